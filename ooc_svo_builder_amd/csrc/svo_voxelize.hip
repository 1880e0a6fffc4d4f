// Partitioner and voxelizer kernels.
//
// Partition (partitioner.cpp:43-77,101-149, BBoxBuffer.h:70-84): per triangle, the box
// of Morton-range partitions whose world box its bbox touches (inclusive test,
// intersection.h:49-53), then per partition an order-preserving flag scan that writes
// the partition's triangle index list (histogram -> scan -> scatter).
//
// Voxelize (voxelizer.cpp:138-307): the Schwarz-Seidel conservative triangle/box test in
// FP32 with the reference's expression order. Work is split in two tiers:
//   * small triangles: a wave takes up to 64 of them, a lane walking its own triangle or all
//     lanes sharing the tile's columns;
//   * large triangles: jobs of some rows of a triangle each, a wave per job.
// Columns run along the axis of the triangle's dominant normal component. Per column the
// projection test in the plane across that axis is evaluated once (it does not depend
// on the position along the column), and only the voxels of the plane slab, widened by
// a margin, are tested; every voxel outside that range fails the reference's plane
// test (the margin is over four times the FP32 error of the test). Triangles with a
// non-finite normal or far-away vertices walk full columns.
// Marked voxels go to a sparse brick grid; compaction of the occupied bricks in Morton
// order yields the sorted unique codes the builder needs (the reference sorts its side
// array, main.cpp:356-359). Payload voxels are resolved to the first triangle in
// partition order that covers them (voxelizer.cpp:263) by a second pass doing
// atomicMin on the triangle index per voxel rank.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <type_traits>

#include "svo_device.h"
#include "svo_internal.h"
#include "svo_scan.h"
#include "svo_walk.h"

namespace svo {

typedef unsigned long long ull;

// The terms of a row of columns (fixed b) that do not depend on a: pb, the hoisted
// plane's h1*pb, plane P's cc*pb, the plane test's term of pb and the slab's term of b.
struct ColRow {
  float pb;
  float hb[3];
  float kp[3];
  float tvb;
  float sb;
};
__device__ __forceinline__ ColRow col_row(const Walk& K, const VoxParams& P, int b) {
  ColRow r;
  r.pb = (float)b * P.unit;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    r.hb[k] = K.f[F_H1 + k] * r.pb;
    r.kp[k] = K.f[F_PC + k] * r.pb;
  }
  r.tvb = K.f[F_NVA] * r.pb;
  r.sb = K.f[F_KB] * (float)b;
  return r;
}

// Rows at least this many columns wide get their columns narrowed to the interval that
// can pass the projection test (row_interval); narrower rows walk every column.
constexpr int kRowSpanMin = 5;

// Columns [a0, a1] of row b: a superset of the columns whose hoisted projection test
// passes (every column outside fails it). An edge's test value at column a,
// fl(fl(fl(h0 * fl(a * u)) + hb) + hd), differs from the real h0 u a + hb + hd by at most
// 5 eps (|h0| |a u| + |hb| + |hd|) (four roundings, eps = 2^-24); with E above that bound,
// a column that passes has h0 u a >= -(hb + hd) - E, a half-line in a. Its end is
// widened by one column for the rounding of its own evaluation (an approximate
// reciprocal, well under a column at these magnitudes). Non-finite constants narrow
// nothing.
__device__ __forceinline__ void row_interval(const Walk& K, const ColRow& R, float u, int& a0,
                                             int& a1) {
  a0 = K.i[I_G0U];
  a1 = K.i[I_G1U];
  if (a1 - a0 + 1 < kRowSpanMin) return;
  const float flo = (float)a0 - 1.0f, fhi = (float)a1 + 1.0f;
  const float amax = fmaxf(fabsf(flo), fabsf(fhi));
  float lo = flo, hi = fhi;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float h0 = K.f[F_H0 + k], hb = R.hb[k], hd = K.f[F_HD + k];
    const float E = 1e-6f * ((fabsf(h0) * amax) * fabsf(u) + fabsf(hb) + fabsf(hd)) + 1e-30f;
    const float rhs = -(hb + hd) - E;
    const float hu = h0 * u;
    if (!(fabsf(rhs) <= 3.0e38f) || !(fabsf(hu) <= 3.0e38f)) continue;
    if (hu > 0.0f)
      lo = fmaxf(lo, rhs * __builtin_amdgcn_rcpf(hu) - 1.0f);
    else if (hu < 0.0f)
      hi = fminf(hi, rhs * __builtin_amdgcn_rcpf(hu) + 1.0f);
    else if (rhs > 0.0f)  // h0 u = 0: no column of the row passes
      hi = flo;
  }
  a0 = max(a0, (int)ceilf(__builtin_amdgcn_fmed3f(lo, flo, fhi)));
  a1 = min(a1, (int)floorf(__builtin_amdgcn_fmed3f(hi, flo, fhi)));
}

// The voxels of column (a, b) that can pass: false when the column's projection test
// fails, else [lo, hi] along w (the bbox, narrowed to the plane slab). Both passes of
// the voxelizer call this with the same inputs, so they see the same ranges.
__device__ __forceinline__ bool column_range(const Walk& K, float pa, const ColRow& R, int a,
                                             int& lo, int& hi) {
  // the three edge tests evaluated together, one branch (their outcome, not their order,
  // decides)
  bool in = true;
#pragma unroll
  for (int k = 0; k < 3; k++)
    in &= !((K.f[F_H0 + k] * pa + R.hb[k]) + K.f[F_HD + k] < 0.0f);
  if (!in) return false;
  lo = K.i[I_G0W];
  hi = K.i[I_G1W];
  if (K.slab()) {
    // the slab ends, clamped to [lo - 1, hi + 1] (finite here: the slab is only used
    // for finite normals and vertices) before the conversion to int
    const float base = K.f[F_KA] * (float)a + R.sb;
    const float l = __builtin_amdgcn_fmed3f(base + K.f[F_ALO], (float)lo - 1.0f, (float)hi + 1.0f);
    const float h = __builtin_amdgcn_fmed3f(base + K.f[F_AHI], (float)lo - 1.0f, (float)hi + 1.0f);
    lo = max(lo, (int)ceilf(l));
    hi = min(hi, (int)floorf(h));
  }
  return lo <= hi;
}

// Pre-pass: flag every brick that a column's candidate voxels fall in (a superset of the
// bricks that will hold marked voxels).
template <typename Act>
__device__ __forceinline__ void touch_column(const Walk& K, const VoxParams& P, int a,
                                             const ColRow& R, int b, Act& act) {
  int lo, hi;
  if (!column_range(K, (float)a * P.unit, R, a, lo, hi)) return;
  const int w = K.w();
  const int ua = (w == 0) ? 1 : 0;
  const int va = (w == 2) ? 1 : 2;
  const uint64_t bbase = (spread3((uint32_t)(a >> 4)) << ua) | (spread3((uint32_t)(b >> 4)) << va);
  for (int cb = lo >> 4; cb <= (hi >> 4); cb++) act.touch(bbase | (spread3((uint32_t)cb) << w));
}

// Morton spreading in the walks from a table in LDS (s_spread[v] = spread3(v) for 8-bit
// v): three lookups and a few shifts instead of the five-step bit spread. Every kernel
// that walks columns fills the table with fill_spread_table before its first walk.
__shared__ uint32_t s_spread[256];
__device__ __forceinline__ void fill_spread_table() {
  for (uint32_t i = threadIdx.x; i < 256u; i += blockDim.x) s_spread[i] = (uint32_t)spread3(i);
}
// spread3(v) for v < 2^21
__device__ __forceinline__ uint64_t spread3_s(uint32_t v) {
  const uint32_t a = s_spread[v & 255u], b = s_spread[(v >> 8) & 255u], c = s_spread[(v >> 16) & 31u];
  return (uint64_t)(a | (b << 24)) | ((uint64_t)((b >> 8) | (c << 16)) << 32);
}

// Every bit of Morton axis k: a coordinate spread onto these bits advances by one with a
// masked add, (m | ~mask) + (1 << k), then & mask.
constexpr uint64_t kAxis0Bits = 0x1249249249249249ull;
__device__ __forceinline__ uint64_t morton_step(uint64_t m, int k) {
  const uint64_t mask = kAxis0Bits << k;
  return ((m | ~mask) + (1ull << k)) & mask;
}

// Test the voxels of column (a, b) and hand every accepted one to act.add(code, tri);
// cbase holds a and b spread onto their Morton axes.
template <typename Act>
__device__ __forceinline__ void walk_column(const Walk& K, const VoxParams& P, int a,
                                            const ColRow& R, uint64_t cbase, Act& act) {
  const float u = P.unit;
  const float pa = (float)a * u;
  int lo, hi;
  if (!column_range(K, pa, R, a, lo, hi)) return;
  const int w = K.w();
  const float tua = K.f[F_NUA] * pa;
  const float Ka = (w == 2) ? (tua + R.tvb) : tua;
  const float Kb = (w == 2) ? 0.0f : R.tvb;
  float KQ[3];
#pragma unroll
  for (int k = 0; k < 3; k++) KQ[k] = K.f[F_QC + k] * pa;
  const float nw = K.f[F_NW], d1 = K.f[F_D1], d2 = K.f[F_D2];
  uint64_t mc = spread3_s((uint32_t)lo) << w;
  for (int c = lo; c <= hi; c++, mc = morton_step(mc, w)) {
    const float pc = (float)c * u;
    const float t = (nw * pc + Ka) + Kb;
    // all seven tests, then one branch
    bool ok = !((t + d1) * (t + d2) > 0.0f);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      ok &= !((K.f[F_PV + k] * pc + R.kp[k]) + K.f[F_PD + k] < 0.0f);
      ok &= !((K.f[F_QV + k] * pc + KQ[k]) + K.f[F_QD + k] < 0.0f);
    }
    if (!ok) continue;
    // cbase and mc occupy disjoint bits: the sum is their union, and an action's
    // loop-invariant offset from cbase folds out of the loop
    act.add(cbase + mc, (uint32_t)K.i[I_TRI]);
  }
}

// Columns [i0, i1] of row b (ma = i0 spread onto axis ua, mb = b onto axis va).
template <typename Act>
__device__ __forceinline__ void walk_row_cols(const Walk& K, const VoxParams& P, int b,
                                              const ColRow& R, int i0, int i1, uint64_t ma,
                                              uint64_t mb, int ua, Act& act) {
  for (int a = i0; a <= i1; a++, ma = morton_step(ma, ua)) {
    if constexpr (Act::kTouch)
      touch_column(K, P, a, R, b, act);
    else
      walk_column(K, P, a, R, ma | mb, act);
  }
}

// Column (a, b) of a walk.
template <typename Act>
__device__ __forceinline__ void walk_one_column(const Walk& K, const VoxParams& P, int a, int b,
                                                Act& act) {
  const int w = K.w();
  const int ua = (w == 0) ? 1 : 0;
  const int va = (w == 2) ? 1 : 2;
  walk_row_cols(K, P, b, col_row(K, P, b), a, a, spread3_s((uint32_t)a) << ua,
                spread3_s((uint32_t)b) << va, ua, act);
}

// All columns of a walk, row by row, the Morton parts of a and b stepped incrementally;
// with 'narrow' rows are narrowed to their interval (rows narrower than kRowSpanMin columns are
// walked whole).
template <typename Act>
__device__ __forceinline__ void walk_all_columns(const Walk& K, const VoxParams& P, Act& act,
                                                 bool narrow) {
  const int w = K.w();
  const int ua = (w == 0) ? 1 : 0;
  const int va = (w == 2) ? 1 : 2;
  uint64_t mb = spread3_s((uint32_t)K.i[I_G0V]) << va;
  const uint64_t ma0 = spread3_s((uint32_t)K.i[I_G0U]) << ua;
  for (int b = K.i[I_G0V]; b <= K.i[I_G1V]; b++, mb = morton_step(mb, va)) {
    const ColRow R = col_row(K, P, b);
    if (narrow) {
      int i0, i1;
      row_interval(K, R, P.unit, i0, i1);
      if (i0 > i1) continue;
      const uint64_t ma = (i0 == K.i[I_G0U]) ? ma0 : (spread3_s((uint32_t)i0) << ua);
      walk_row_cols(K, P, b, R, i0, i1, ma, mb, ua, act);
    } else {
      walk_row_cols(K, P, b, R, K.i[I_G0U], K.i[I_G1U], ma0, mb, ua, act);
    }
  }
}

// Global buffers the actions work on; each action binds its unit's segment.
struct ActArgs {
  uint32_t* table;    // all units' brick tables, concatenated
  uint8_t* cflags;    // dense payload units: a byte per 64-voxel word of every table entry
  uint8_t* pool8;     // touch path: 4096 bytes per slot
  ull* pool;          // 64 bit words per slot (written by the compaction)
  uint32_t* wprefix;  // per word: batch rank of its first voxel
  uint32_t* winner;   // per voxel of the batch: lowest covering triangle
  ull* ctr;
  uint64_t pool_cap;  // touch path slots
};

// What an action keeps per wave in LDS.
struct NoCache {};
// The action of a tile whose lanes walk their own triangles.
template <typename Act>
struct DirectOf {
  using type = Act;
};

// Brick allocation without atomics: the touch pass stores 1 into the table entry of
// every brick a column's candidate voxels fall in; a scan over the table then numbers the
// flagged bricks in Morton order (table entry = slot + 1) and lists them.
struct TouchAction {
  static constexpr bool kTouch = true;
  using Unordered = TouchAction;
  using Cache = NoCache;
  __device__ static bool narrow(const VoxParams&) { return true; }
  uint32_t* table;
  uint64_t brick0;  // first brick of the unit's table segment
  __device__ static TouchAction make(const ActArgs& A, const VoxParams& P, Cache*) {
    return TouchAction{A.table + P.table_base, P.bstart >> kBrickBits};
  }
  __device__ __forceinline__ void touch(uint64_t brick_code) { table[brick_code - brick0] = 1u; }
  __device__ __forceinline__ void add(uint64_t, uint32_t) {}
  __device__ static void drain(const ActArgs&, const VoxParams&, Cache*, bool) {}
};

// Mark voxels with plain byte stores of 1: concurrent marks of one voxel all store the
// same value, so no atomic read-modify-write is needed however many triangles cover it
// (about three per voxel on a terrain).
//  * dense units (MarkDenseT): a byte per voxel of the unit's Morton range (the
//    reference's own layout, voxelizer.cpp:144, kept in HBM); a byte of the brick's table entry
//    is set with a plain store when the thread enters a quarter of it (1 KiB). Only flagged
//    quarters are compacted and cleared afterwards, so the grid is never swept. Dense payload units
//    keep 4 bytes per voxel and resolve the winning triangle in the same walk (atomicMax
//    of ~triangle: voxelizer.cpp:263, the first triangle in partition order wins); they flag
//    64-voxel words as well (256 bytes of cells). Flagged words for all units made the
//    headline's mark 13 us slower for 3 us of its compaction.
//  * touch units (MarkPoolAction): 4096 bytes per pool slot; the slot comes from the table
//    (touch pass + table scan), cached per thread.
// Both store through global (not generic) pointers.
// kWide: some units of the pass carry payload (4-byte cells; the unit's wide flag decides
// per voxel); otherwise every cell is a byte. kSmall: no unit spans more than 2^32 voxels, so a
// voxel's place is 32 bits: the upper half of the Morton stepping goes, and a store takes it as
// its offset from a scalar address (64 mixed meshes 2500 -> 2467 us, payload terrain at 1024 134 ->
// 130).
template <bool kWide, bool kSmall>
struct MarkDenseT {
  static constexpr bool kTouch = false;
  using Rel = std::conditional_t<kSmall, uint32_t, uint64_t>;
  // the same action for queued columns
  using Unordered = MarkDenseT<kWide, kSmall>;
  using Cache = NoCache;  // per wave, in LDS
  // whether a direct walk narrows its rows to their intervals
  __device__ static bool narrow(const VoxParams& P) { return !kWide || !P.wide; }
  gbyte_t* table;  // the unit's table segment, a byte per quarter of a brick
  gbyte_t* words;  // the unit's word flags (payload units)
  gbyte_t* bytes;
  Rel base;  // code of the first voxel of the unit's first brick
  int wide;
  uint32_t cquarter = 0xFFFFFFFFu, cword = 0xFFFFFFFFu;  // the last ones marked
  __device__ static MarkDenseT make(const ActArgs& A, const VoxParams& P, Cache*) {
    MarkDenseT m;
    m.table = (gbyte_t*)(A.table + P.table_base);
    m.words = (gbyte_t*)(A.cflags + P.table_base * kBrickWords);
    m.bytes = (gbyte_t*)P.grid8;
    m.base = (Rel)P.bstart;
    m.wide = kWide ? P.wide : 0;
    return m;
  }
  __device__ __forceinline__ void touch(uint64_t) {}
  __device__ __forceinline__ void add(uint64_t code, uint32_t tri) {
    const Rel rel = (Rel)code - base;
    const uint32_t q = (uint32_t)(rel >> (kBrickBits - 2));
    if (kWide && wide) {
      // the lowest covering triangle as the largest ~tri (0 = unmarked)
      __hip_atomic_fetch_max((gword_t*)bytes + rel, ~tri, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t w = (uint32_t)(rel >> 6);
      if (w != cword) {
        cword = w;
        words[w] = 1;
      }
    } else
      bytes[rel] = 1;
    if (q != cquarter) {
      cquarter = q;
      table[q] = 1;
    }
  }
  __device__ static void drain(const ActArgs&, const VoxParams&, Cache*, bool) {}
};

// Payload marks, gathered in LDS: a wave keeps kLines lines of 32 cells (128 bytes of the grid),
// takes the maximum of ~triangle there, and gives a line to memory whole, a half wave a line. A
// cell whose line's place holds another line goes to memory at once.
//
// The winner atomics bound these marks: at agent scope they are not done in the (per XCD) L2
// but at the memory behind it, ~23 G requests a second whatever they hold (TCC_EA0_ATOMIC =
// TCC_ATOMIC; 12.7 M of them for 17M voxels of a rough sphere at 1024 in 535 us, 4.3 M for a
// fine terrain in 218), so what counts is how many requests there are, and neighbouring
// triangles share both cells and lines.
//
// Lanes walking their own triangles have 64 lines, in the memory that rows and columns are laid
// out in otherwise; a tile laid out so (triangles of more columns, whose lines are few hits each)
// has 16 of its own. With 64 lines besides that memory two blocks fitted a CU instead of three:
// the fine terrain 153 us, 134 so; 320,000 triangles at 512 73 and 61; the rough sphere 453 and 457.
constexpr uint32_t kLineBits = 5;
constexpr uint32_t kLineCells = 1u << kLineBits;
template <uint32_t kLines>
struct MarkLines {
  uint32_t tag[kLines];  // line + 1, 0 = free
  uint32_t val[kLines][kLineCells];
};
template <uint32_t kLines, bool kSmall>
struct MarkGather {
  static constexpr bool kTouch = false;
  using Rel = std::conditional_t<kSmall, uint32_t, uint64_t>;
  static constexpr uint32_t kFull = kLines * 5 / 8;  // lines held at which they go to memory
  using Unordered = MarkDenseT<true, kSmall>;
  using Cache = MarkLines<kLines>;
  __device__ static bool narrow(const VoxParams&) { return false; }
  gbyte_t* table;
  gbyte_t* words;
  gword_t* cells;
  Rel base;
  Cache* L;
  __device__ static MarkGather make(const ActArgs& A, const VoxParams& P, Cache* L) {
    MarkGather m;
    m.table = (gbyte_t*)(A.table + P.table_base);
    m.words = (gbyte_t*)(A.cflags + P.table_base * kBrickWords);
    m.cells = (gword_t*)P.grid8;
    m.base = (Rel)P.bstart;
    m.L = L;
    return m;
  }
  __device__ __forceinline__ void touch(uint64_t) {}
  __device__ __forceinline__ void add(uint64_t code, uint32_t tri) {
    const Rel rel = (Rel)code - base;  // (below 2^37: kDensePayloadBricks)
    const uint32_t line = (uint32_t)(rel >> kLineBits);
    // neighbouring lines in neighbouring places (of a 4 x 4 x 4 block of lines: 6 bits), the
    // blocks mixed
    const uint32_t at = (line ^ ((line >> 6) * 0x9E3779B1u >> 26)) % kLines;
    uint32_t tag = L->tag[at];
    if (tag == 0u) {
      tag = atomicCAS(&L->tag[at], 0u, line + 1u);
      if (tag == 0u) tag = line + 1u;
    }
    if (tag == line + 1u) {
      atomicMax(&L->val[at][(uint32_t)rel % kLineCells], ~tri);
    } else {
      __hip_atomic_fetch_max(cells + rel, ~tri, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      words[line >> 1] = 1;
      table[line >> (kBrickBits - 2 - kLineBits)] = 1;
    }
  }
  // Give the lines to memory (all: else only when there are many). Called by whole waves.
  __device__ static void drain(const ActArgs& A, const VoxParams& P, Cache* L, bool all) {
    const int lane = lane_id();
    wave_lds_sync();
    const uint32_t tag = lane < (int)kLines ? L->tag[lane] : 0u;
    uint64_t used = __ballot(tag != 0u);
    if (!used || (!all && (uint32_t)__popcll(used) < kFull)) return;  // uniform
    const MarkGather m = make(A, P, L);
    while (used) {  // two lines at a time
      const int l0 = __ffsll((long long)used) - 1;
      used &= used - 1ull;
      const int l1 = used ? __ffsll((long long)used) - 1 : -1;
      used &= used - 1ull;
      const int at = lane < kWave / 2 ? l0 : l1;
      const uint32_t line = (uint32_t)__shfl((int)tag, at & (kWave - 1), kWave) - 1u;
      if (at >= 0) {
        const uint32_t cell = (uint32_t)lane % kLineCells;
        const uint32_t v = L->val[at][cell];
        L->val[at][cell] = 0u;
        if (v)
          __hip_atomic_fetch_max(m.cells + (((uint64_t)line << kLineBits) + cell), v,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cell == 0) {
          m.words[line >> 1] = 1;
          m.table[line >> (kBrickBits - 2 - kLineBits)] = 1;
        }
      }
    }
    if (lane < (int)kLines) L->tag[lane] = 0u;
    wave_lds_sync();
  }
};
static_assert(kLineCells == kWave / 2, "drain: two lines a step");
template <bool kSmall>
struct DirectOf<MarkGather<16, kSmall>> {
  using type = MarkGather<64, kSmall>;
};

struct MarkPoolAction {
  static constexpr bool kTouch = false;
  using Unordered = MarkPoolAction;
  using Cache = NoCache;
  __device__ static bool narrow(const VoxParams&) { return true; }
  const gword_t* table;
  gbyte_t* bytes;  // the slot pool
  ull* ctr;
  uint64_t pool_cap;
  uint64_t base;  // code of the first voxel of the unit's first brick
  uint32_t cbrick = 0xFFFFFFFFu, cslot = 0;
  __device__ static MarkPoolAction make(const ActArgs& A, const VoxParams& P, Cache*) {
    MarkPoolAction m;
    m.table = (const gword_t*)(A.table + P.table_base);
    m.bytes = (gbyte_t*)A.pool8;
    m.ctr = A.ctr;
    m.pool_cap = A.pool_cap;
    m.base = P.bstart;
    return m;
  }
  __device__ __forceinline__ void touch(uint64_t) {}
  __device__ __forceinline__ void add(uint64_t code, uint32_t) {
    const uint64_t rel = code - base;
    const uint32_t b = (uint32_t)(rel >> kBrickBits);
    if (b != cbrick) {
      cbrick = b;
      cslot = table[b];
    }
    const uint32_t s = cslot;
    if (s == 0 || s > pool_cap) {
      // s == 0 cannot happen (the touch pass covers every candidate voxel); s > pool_cap
      // means the pool is too small and the pass is redone with a larger one
      atomicAdd(&ctr[s == 0 ? kCtrError : kCtrOverflow], 1ull);
      return;
    }
    bytes[(uint64_t)(s - 1) * kBrickVox + (rel & (kBrickVox - 1))] = 1;
  }
  __device__ static void drain(const ActArgs&, const VoxParams&, Cache*, bool) {}
};

// Second payload pass: lowest triangle index per voxel rank.
struct WinnerAction {
  static constexpr bool kTouch = false;
  using Unordered = WinnerAction;
  using Cache = NoCache;
  __device__ static bool narrow(const VoxParams&) { return false; }
  const uint32_t* table;
  const ull* pool;  // bit form of the bricks, written by the compaction
  const uint32_t* wprefix;
  uint32_t* winner;
  ull* ctr;
  uint64_t base;  // code of the first voxel of the unit's first brick
  __device__ static WinnerAction make(const ActArgs& A, const VoxParams& P, Cache*) {
    return WinnerAction{A.table + P.table_base, A.pool, A.wprefix, A.winner, A.ctr, P.bstart};
  }
  __device__ __forceinline__ void touch(uint64_t) {}
  __device__ __forceinline__ void add(uint64_t code, uint32_t tri) {
    const uint64_t rel = code - base;
    const uint32_t b = (uint32_t)(rel >> kBrickBits);
    const uint32_t s = table[b];
    const uint32_t wi = (uint32_t)(rel >> 6) & (kBrickWords - 1);
    const uint64_t slot = (uint64_t)(s - 1) * kBrickWords + wi;
    const ull bit = 1ull << (rel & 63);
    // both passes evaluate the same predicates, so the voxel is marked; a voxel that is
    // not (which would be a bug) is counted and skipped rather than written
    if (s == 0 || !(pool[slot] & bit)) {
      atomicAdd(&ctr[kCtrError], 1ull);
      return;
    }
    const uint32_t rank = wprefix[slot] + (uint32_t)__popcll(pool[slot] & (bit - 1ull));
    atomicMin(&winner[rank], tri);
  }
  __device__ static void drain(const ActArgs&, const VoxParams&, Cache*, bool) {}
};

// last k with a[k] <= v, for a non-decreasing a[0..n) with a[0] <= v
template <typename T>
__device__ __forceinline__ uint32_t upper_index(const T* __restrict__ a, uint32_t n, T v) {
  uint32_t lo = 0, hi = n - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (a[mid] <= v)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Small tier, persistent: waves take tiles of tt <= 64 consecutive triangles of one unit from
// device work queues (tile_off[u] = first tile of unit u); tt is smaller for passes with few
// triangles, so that their tiles still spread over the chip. Lane l sets up triangle l of
// the tile. A tile whose triangles all have at most direct_cols columns, of about as many
// each, is walked from registers, a lane a triangle. Triangles with more than small_cols columns
// (or non-slab triangles with more than small_cols * 8 tests) go to the column-parallel tier.
// Otherwise a tile is laid out in two steps, each giving every lane of the wave one element
// whatever the triangles' shapes:
//   * rows: 64 rows of the tile's triangles at a time; a lane finds its row's interval of
//     columns, and the terms of its bounds that do not change along it (fast_row);
//   * columns: the columns of these 64 rows, 64 at a time; a lane finds the run of voxels
//     its column holds (fast_column) and marks it without testing them one by one.
// A column whose run is not certain (a bound within its error of an integer: a few in a
// thousand at 2048; most where faces lie on voxel planes) is queued, and the queue walked
// with the reference's own tests once 64 are there. Units the pass does not apply to (skip mask)
// contribute nothing.
//
// Bound by vector instructions (binary meshes) or by the winner atomics (payload). Testing
// every candidate voxel of a row segment per lane left 64% of the lanes of a rough mesh's waves
// idle and took ~43 instructions a candidate: 64 mixed meshes 4.35 -> 2.75 ms, a 1.3M-triangle
// rough sphere at 1024 987 -> 438 us, a 6M-triangle soup at 4096 in 8 partitions 1.71 -> 1.19
// ms, the 2.1M-triangle terrain at 2048 (lanes walking their own triangles) 154 -> 141 us.
// 128 registers and 40 KB of LDS a block keep four blocks on a CU: three cost 10%.
constexpr int kTile = 256;     // threads per block
constexpr int kTileWaves = kTile / kWave;
constexpr int kTileTris = 64;  // triangles per tile: one per lane
constexpr int kRowWords = 8;   // LDS words of a row
constexpr int kTriQuads = (int)sizeof(FastTri) / 16;
constexpr int kRowQuads = (int)(sizeof(FastTri) - sizeof(FastCol)) / 16;  // per-row part of a triangle
constexpr int kQueueCap = 2 * kWave;  // uncertain columns waiting per wave
constexpr uint32_t kColMask = (1u << 26) - 1u;  // columns of a triangle of the small tier, or of a job
constexpr uint32_t kQueues = 8;        // tile queues per persistent launch
constexpr uint32_t kTileRun = 16;      // neighbouring tiles in one queue
constexpr uint32_t kQueueStride = 16;  // words between their counters (own cache lines)
constexpr uint32_t kQueueWords = kQueues * kQueueStride;
constexpr int kSkipBinary = 1;  // geometry-only units (payload winner pass)

__device__ __forceinline__ bool skipped(const VoxParams& P, int skip) {
  return (skip & kSkipBinary) && P.stride == 9;
}

// Per wave: the tile's triangles, the current rows, a 64-entry slot array and the queue of
// uncertain columns (lane of the triangle << 26 | (j - row0) * (number of i) + i).
struct WalkLds {
  uint4 tri[kTileTris][kTriQuads];
  uint4 row[kWave][kRowWords / 4];
  uint32_t q[kQueueCap];
  uint8_t slot[kWave];
};

// The element of lane's position k0 + lane among elements laid out by their start positions
// (lane e holds element e's start, has = it is not empty): the last one that starts at or
// before it. carry: the element the previous window ended in (0 before the first), as
// index + 1.
__device__ __forceinline__ uint32_t locate(uint8_t* slot, uint32_t start, bool has, uint32_t k0,
                                           uint32_t& carry) {
  const int lane = lane_id();
  slot[lane] = (uint8_t)(lane == 0 ? carry : 0u);
  wave_lds_sync();
  if (has && start - k0 < (uint32_t)kWave) slot[start - k0] = (uint8_t)(lane + 1);
  wave_lds_sync();
  const uint32_t v = wave_incl_max(slot[lane]);
  wave_lds_sync();  // (the next call clears the slots)
  carry = (uint32_t)__builtin_amdgcn_readlane((int)v, kWave - 1);
  return v - 1u;
}

// Up to 64 queued columns through the reference's tests: lane l's walk is K.
template <typename Act>
__device__ __forceinline__ void walk_queued(const VoxParams& P, const ActArgs& A, const Walk& K,
                                            uint32_t row0, const uint32_t* q, uint32_t n) {
  const uint32_t e = (uint32_t)lane_id() < n ? q[lane_id()] : 0u;
  const int src = (int)(e >> 26);
  Walk Q;  // the walk of lane src
#pragma unroll
  for (int f = 0; f < kWalkF; f++) Q.f[f] = __shfl(K.f[f], src, kWave);
#pragma unroll
  for (int f = 0; f < kWalkI; f++) Q.i[f] = __shfl(K.i[f], src, kWave);
  if ((uint32_t)lane_id() >= n) return;
  typename Act::Unordered act = Act::Unordered::make(A, P, nullptr);
  const uint32_t col = e & kColMask, na = (uint32_t)(Q.i[I_G1U] - Q.i[I_G0U] + 1);
  const int a = Q.i[I_G0U] + (int)(col % na);
  walk_one_column(Q, P, a, Q.i[I_G0V] + (int)(row0 + col / na), act);
}

// Rows [row0, row0 + nrows) of the lanes' triangles (nall rows each; their walks K, their linear forms in
// L.tri).
template <typename Act>
__device__ __forceinline__ void walk_rows(WalkLds& L, typename Act::Cache* cache,
                                          const VoxParams& P, const ActArgs& A, const Walk& K,
                                          uint32_t nall, uint32_t nrows, uint32_t row0) {
  uint32_t nq = 0;
  const int lane = lane_id();
  const uint32_t rend = wave_incl_scan<uint32_t>(nrows), rstart = rend - nrows;
  const uint32_t R = (uint32_t)__builtin_amdgcn_readlane((int)rend, kWave - 1);
  uint32_t tcarry = 0;
  for (uint32_t r0 = 0; r0 < R; r0 += kWave) {
    const uint32_t t = locate(L.slot, rstart, nrows != 0, r0, tcarry);
    const uint32_t r = r0 + lane;
    const int j = (int)(r - (uint32_t)__shfl((int)rstart, (int)t, kWave) + row0);
    const int nb = __shfl((int)nall, (int)t, kWave);
    uint32_t cnt = 0;
    FastRow W;
    if (r < R) {
      FastTri F;
      const uint4* src = L.tri[t];
      uint4* dst = (uint4*)&F;
#pragma unroll
      for (int k = 0; k < kRowQuads; k++) dst[k] = src[k];
      dst[kRowQuads + 2] = src[kRowQuads + 2];  // (the error)
      fast_row(F, j, nb, W);
      if (W.i1 >= W.i0) cnt = (uint32_t)(W.i1 - W.i0 + 1);
      const int w = (int)(F.rf >> 8) & 3;
      const uint32_t b = (F.rf >> 16) + (uint32_t)j;
      const uint64_t mb = spread3_s(b) << (w == 2 ? 1 : 2);
      // the row's columns are known by their position in the row: its end flags by the count
      L.row[lane][1] = make_uint4(__float_as_uint(W.s_lo), (uint32_t)mb, (uint32_t)(mb >> 32),
                                  (uint32_t)j | (cnt << 16));
      L.row[lane][0] = make_uint4(0u, (uint32_t)W.i0 | (t << 16) | (W.first_unsure ? 1u << 24 : 0u) |
                                          (W.last_unsure ? 1u << 25 : 0u) | (W.all ? 1u << 26 : 0u),
                                  __float_as_uint(W.p_lo), __float_as_uint(W.p_hi));
    }
    const uint32_t cend = wave_incl_scan<uint32_t>(cnt), cstart = cend - cnt;
    const uint32_t C = (uint32_t)__builtin_amdgcn_readlane((int)cend, kWave - 1);
    L.row[lane][0].x = cstart;
    uint32_t ccarry = 0;
    Act act = Act::make(A, P, cache);
    for (uint32_t k0 = 0; k0 < C; k0 += kWave) {
      const uint32_t rr = locate(L.slot, cstart, cnt != 0, k0, ccarry);  // (orders the row stores)
      const uint32_t k = k0 + lane;
      bool push = false;
      uint32_t e = 0;
      if (k < C) {
        const uint4 ra = L.row[rr][0], rb = L.row[rr][1];
        const uint32_t t = (ra.y >> 16) & 0xFFu;
        FastCol F;
        const uint4* src = &L.tri[t][kRowQuads];
        uint4* dst = (uint4*)&F;
#pragma unroll
        for (int q = 0; q < (int)sizeof(FastCol) / 16; q++) dst[q] = src[q];
        const uint32_t at = k - ra.x;
        const int i = (int)((ra.y & 0xFFFFu) + at);
        const int w = (int)(F.qf >> 8) & 3;
        const uint32_t a = (F.qf >> 16) + (uint32_t)i;
        int lo, hi;
        bool sure = fast_column(F, __uint_as_float(ra.z), __uint_as_float(ra.w),
                                __uint_as_float(rb.x), i, lo, hi);
        sure = sure && !((ra.y & (1u << 24)) && at == 0) &&
               !((ra.y & (1u << 25)) && at + 1 == (rb.w >> 16)) && !(ra.y & (1u << 26));
        const bool careful = F.qf & kFastCareful;
        if (lo <= hi || careful) {
          const uint64_t mb = ((uint64_t)rb.z << 32) | rb.y;
          const int c0 = (int)(F.ck & 0xFFFFu);
          if (Act::kTouch ? careful : !sure) {
            push = true;
            const uint32_t na = L.tri[t][kRowQuads - 1].w & 0xFFFFu;
            e = (t << 26) | (((rb.w & 0xFFFFu) - row0) * na + (uint32_t)i);
          } else if constexpr (Act::kTouch) {
            const uint32_t b = (uint32_t)compact3(mb >> (w == 2 ? 1 : 2));
            const uint64_t bb = (spread3(a >> 4) << (w == 0 ? 1 : 0)) |
                                (spread3(b >> 4) << (w == 2 ? 1 : 2));
            for (int cb = (c0 + lo) >> 4; cb <= (c0 + hi) >> 4; cb++)
              act.touch(bb | (spread3((uint32_t)cb) << w));
          } else {
            const uint64_t cbase = mb + (spread3_s(a) << (w == 0 ? 1 : 0));
            uint64_t mc = spread3_s((uint32_t)(c0 + lo)) << w;
            for (int c = lo; c <= hi; c++, mc = morton_step(mc, w)) act.add(cbase + mc, F.tri);
          }
        }
      }
      Act::drain(A, P, cache, false);
      const uint64_t pm = __ballot(push);
      if (pm) {  // uniform
        if (push) L.q[nq + (uint32_t)__popcll(pm & ((1ull << lane) - 1ull))] = e;
        nq += (uint32_t)__popcll(pm);
        wave_lds_sync();
        if (nq >= (uint32_t)kWave) {
          walk_queued<Act>(P, A, K, row0, L.q + (nq - kWave), kWave);
          nq -= kWave;
          wave_lds_sync();
        }
      }
    }
    wave_lds_sync();  // the next rows overwrite these
  }
  if (nq) walk_queued<Act>(P, A, K, row0, L.q, nq);
  wave_lds_sync();
}

// The triangles of the large tier: unit, triangle, rows per job, the linear form and walk of
// the first walk_cap of them (the others are set up again by each of their jobs), and up to job_cap
// jobs after each triangle's first one (triangle's index here, first row).
constexpr uint32_t kJobCols = 1024;  // columns of a job, roughly
constexpr int kLargeQuads = kTriQuads + kWalkWords / 4;
static_assert(kWalkWords % 4 == 0 && sizeof(Walk) == kWalkWords * 4, "walk words");
struct LargeList {
  uint32_t* unit;
  uint32_t* tri;
  uint32_t* rows;
  uint2* jobs;
  uint4* walk;
  uint32_t job_cap, walk_cap;
};
// Rows per job of a triangle with nu x nv columns, and places for its further jobs: n of them
// from 'at' on, to be filled with idx and the rows. With no room for all, the places left are
// filled with none, and the number of its jobs stands above the rows (unlisted: below 2^15, as a
// unit's side): kShareJobs or more are dealt to all waves, fewer are done with its first one.
constexpr int kUnlistedShift = 8;
constexpr uint32_t kShareJobs = 8;
struct JobPlaces {
  uint32_t idx, rows, at, n;
};
__device__ __forceinline__ uint32_t large_jobs(const LargeList& B, ull* ctr, uint32_t idx,
                                               uint32_t nu, uint32_t nv, JobPlaces& J) {
  const uint32_t rows = max(1u, min((uint32_t)kWave, kJobCols / nu));
  const uint32_t more = (nv + rows - 1) / rows - 1;
  if (!more) return rows;
  const ull at = atomicAdd(&ctr[kCtrLargeJobs], (ull)more);
  const bool fits = at + more <= B.job_cap;
  J.idx = fits ? idx : 0xFFFFFFFFu;
  J.rows = rows;
  J.at = (uint32_t)min(at, (ull)B.job_cap);
  J.n = min(more, B.job_cap - J.at);
  return fits ? rows : rows | (more << kUnlistedShift);
}
// Fill the lanes' places (whole waves): a few by their lane, many by the wave, one lane's at a
// time. Hundreds written by a lane one after the other held up its wave, the last of the launch: a
// rotated cube's 12 triangles at 1024 225 us in all, 167 so; at 4096 in 8 partitions 2465 and 1603.
constexpr uint32_t kOwnPlaces = 8;
__device__ __forceinline__ void put_jobs(uint2* jobs, const JobPlaces& J) {
  if (J.n <= kOwnPlaces)
    for (uint32_t q = 0; q < J.n; q++) jobs[J.at + q] = make_uint2(J.idx, (q + 1) * J.rows);
  for (uint64_t m = __ballot(J.n > kOwnPlaces); m; m &= m - 1ull) {
    const int src = __ffsll((long long)m) - 1;
    const uint32_t idx = (uint32_t)__builtin_amdgcn_readlane((int)J.idx, src);
    const uint32_t rows = (uint32_t)__builtin_amdgcn_readlane((int)J.rows, src);
    const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)J.at, src);
    const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)J.n, src);
    for (uint32_t q = lane_id(); q < n; q += kWave) jobs[at + q] = make_uint2(idx, (q + 1) * rows);
  }
}

// blocks of the small tier on a CU (what an action keeps in LDS leaves room for three)
template <typename Act>
constexpr int kTileBlocks = std::is_same<typename Act::Cache, NoCache>::value ? 4 : 3;
template <typename Act>
__global__ __launch_bounds__(kTile, kTileBlocks<Act>) void k_vox_tile(const VoxParams* __restrict__ units,
                                                       uint32_t n_units,
                                                       const uint32_t* __restrict__ tile_off,
                                                       uint64_t payload_runs, ActArgs A,
                                                       ull* queue, LargeList B, uint32_t tt,
                                                       int collect, int skip) {
  __shared__ WalkLds s_walk[kTileWaves];
  __shared__ volatile uint32_t s_empty[kQueues];  // classes found empty
  if (threadIdx.x < kQueues) s_empty[threadIdx.x] = 0;
  fill_spread_table();
  __syncthreads();  // the waves part here
  WalkLds& L = s_walk[threadIdx.x / kWave];
  typename Act::Cache* cache = nullptr;
  if constexpr (!std::is_same<typename Act::Cache, NoCache>::value) {
    __shared__ typename Act::Cache s_cache[kTileWaves];
    cache = &s_cache[threadIdx.x / kWave];
    for (uint32_t k = lane_id(); k < sizeof(*cache) / 4; k += kWave) ((uint32_t*)cache)[k] = 0u;
    wave_lds_sync();
  }
  using Direct = typename DirectOf<Act>::type;
  constexpr bool kOverlay = !std::is_same<typename Direct::Cache, NoCache>::value;
  static_assert(!kOverlay || sizeof(typename Direct::Cache) <= sizeof(WalkLds), "overlay");
  typename Direct::Cache* const overlay = kOverlay ? (typename Direct::Cache*)&L : nullptr;
  bool clean = false;  // the overlay is zero (as a drain leaves it)
  ull* ctr = A.ctr;
  const int lane = lane_id();
  // Runs of geometry-only and of payload tiles, mixed evenly (payload_runs: 2^32 x the payload
  // runs' share, rounded up): the first are bound by vector instructions, the others by their
  // atomics. 64 mixed meshes 2.74 ms job by job, 2.52 so.
  const uint32_t* const off_kind[2] = {tile_off, tile_off + n_units + 1};
  const uint32_t runs = (off_kind[0][n_units] + kTileRun - 1) / kTileRun +
                        (off_kind[1][n_units] + kTileRun - 1) / kTileRun;
  const uint32_t total = runs * kTileRun;
  // Runs of kTileRun tiles are dealt to kQueues classes (one per XCD: blocks are dealt to
  // them in turn), each with its own counter in its own cache line: a run's tiles, neighbours
  // in space, mark lines of one L2, and the classes hold about the same work. One counter's
  // returning atomics serialize (~14 ns each), those that find a class empty included, so a
  // wave looks into one other class only, and a block's waves tell each other which classes
  // are empty. A pass with no more tiles than waves needs no counter.
  const bool one_each = total <= gridDim.x * kTileWaves;
  uint32_t cls = blockIdx.x % kQueues;
  uint32_t next = one_each ? blockIdx.x * kTileWaves + threadIdx.x / kWave : total;
  for (;;) {
    if (!one_each) {
      for (uint32_t tried = 0; tried < 2; tried++) {
        if (!s_empty[cls]) {
          uint32_t k = 0;
          if (lane == 0) k = (uint32_t)atomicAdd(queue + kQueueStride * cls, 1ull);
          k = (uint32_t)__builtin_amdgcn_readfirstlane((int)k);
          next = (k / kTileRun * kQueues + cls) * kTileRun + k % kTileRun;
          if (next < total) break;
          s_empty[cls] = 1u;
        }
        cls = (cls + 1) % kQueues;
      }
    }
    // in a scalar register: the unit search and the unit's parameters run on scalar loads
    const uint32_t at = (uint32_t)__builtin_amdgcn_readfirstlane((int)next);
    if (at >= total) return;
    next = total;
    const uint32_t run = at / kTileRun, pay = (uint32_t)((run * payload_runs) >> 32);
    const bool is_pay = (uint32_t)(((run + 1ull) * payload_runs) >> 32) > pay;
    const uint32_t tile = (is_pay ? pay : run - pay) * kTileRun + at % kTileRun;
    const uint32_t* const off = off_kind[is_pay];
    if (tile >= off[n_units]) continue;  // the kind's last run, not full
    const uint32_t u = upper_index<uint32_t>(off, n_units + 1, tile);
    const VoxParams P = units[u];
    if (skipped(P, skip)) continue;
    const uint32_t i = (tile - off[u]) * tt + lane;
    Walk K;
    uint32_t ncols = 0, nu = 0, nv = 0;  // columns of a triangle of this tier; its sides
    bool large = false;
    if ((uint32_t)lane < tt && i < P.n) {
      const uint32_t t = P.list ? ((const gword_t*)P.list)[i] : i;
      Setup S;
      setup_tri((const gfloat_t*)P.tris + (uint64_t)t * P.stride, P, S);
      make_walk(S, P, t, K);
      const uint64_t nc = K.columns();
      const uint64_t lim = (uint64_t)P.small_cols;
      nu = (uint32_t)(K.i[I_G1U] - K.i[I_G0U] + 1);
      nv = (uint32_t)(K.i[I_G1V] - K.i[I_G0V] + 1);
      // (a bbox end beyond the range of int truncates to INT_MIN, and an end before its start
      // covers nothing)
      if (min(min((int)nu, (int)nv), K.i[I_G1W] - K.i[I_G0W] + 1) > 0) {
        large = (K.slab() ? (nc > lim) : (K.work() > lim * 8)) || nc > (uint64_t)kColMask;
        if (!large) ncols = (uint32_t)nc;
      }
    }
    // A lane walking its own triangle takes ~100 instructions a column, in as many steps as
    // the tile's largest triangle has columns; the rows and columns of the whole tile take
    // ~1200 and ~4 a column (headline, 64 triangles of 9.4 columns: 141 us by lanes, 268 by
    // columns; 16-triangle tiles of the same, 178,802 triangles at 1024: 56 and 55).
    uint32_t all = wave_incl_scan<uint32_t>(min(ncols, 0xFFFFu));
    all = (uint32_t)__builtin_amdgcn_readlane((int)all, kWave - 1);
    uint32_t most = wave_incl_max(ncols);
    most = (uint32_t)__builtin_amdgcn_readlane((int)most, kWave - 1);
    const bool direct = most <= (uint32_t)P.direct_cols && most * 100u <= 1200u + all * 4u;
    uint32_t rows = 0;
    JobPlaces places{0, 0, 0, 0};
    if ((large && collect) || (ncols && !direct)) {
      FastTri F;
      make_fast(K, P, F);
      const uint4* src = (const uint4*)&F;
      if (!large) {
#pragma unroll
        for (int k = 0; k < kTriQuads; k++) L.tri[lane][k] = src[k];
        rows = nv;
      } else {
        const ull idx = atomicAdd(&ctr[kCtrLargeCount], 1ull);
        B.unit[idx] = u;
        B.tri[idx] = (uint32_t)K.i[I_TRI];
        B.rows[idx] = large_jobs(B, ctr, (uint32_t)idx, nu, nv, places);
        if (idx < B.walk_cap) {
          uint4* dst = B.walk + idx * kLargeQuads;
#pragma unroll
          for (int k = 0; k < kTriQuads; k++) dst[k] = src[k];
          const uint4* wk = (const uint4*)&K;
#pragma unroll
          for (int k = 0; k < kWalkWords / 4; k++) dst[kTriQuads + k] = wk[k];
        }
      }
    }
    if (collect) put_jobs(B.jobs, places);
    if (direct) {
      if (kOverlay && !clean) {
        for (uint32_t k = lane; k < sizeof(*overlay) / 4; k += kWave) ((uint32_t*)overlay)[k] = 0u;
        wave_lds_sync();
        clean = true;
      }
      if (ncols) {
        Direct act = Direct::make(A, P, overlay);
        walk_all_columns(K, P, act, Direct::narrow(P));
      }
      Direct::drain(A, P, overlay, true);
      continue;
    }
    clean = false;
    if (__ballot(rows != 0)) {
      wave_lds_sync();
      walk_rows<Act>(L, cache, P, A, K, nv, rows, 0u);
      Act::drain(A, P, cache, true);
    }
  }
}

// Column-parallel tier: a wave per job, a job being some rows of one deferred triangle (at most
// 64, about kJobCols columns), laid out over the wave's lanes as in the small tier; the counts
// live on the device, the grid strides. Triangle idx has its first job at idx, its others at
// n_large + (their place in B.jobs). (A thread per bbox column took 219 us on 20,480 triangles
// of ~2,200 columns, after a launch that scanned the column counts; in rows 160.)
// Once there are more jobs than places, every wave looks through the triangles, 64 at a time, for
// unlisted jobs of its own: job q of triangle idx is wave (idx * jobs + q) mod waves's, which deals
// out triangles of like size evenly. With all rows of such a triangle in one wave, 700 that span
// most of a grid of 4096 took 131 ms (39 with a thread per column), 29 so; 1500 at 2048 38 ms, 17
// and 14.
template <typename Act>
__global__ __launch_bounds__(kTile, 3) void k_vox_large(const VoxParams* __restrict__ units,
                                                        ActArgs A, LargeList B, int skip) {
  __shared__ WalkLds s_walk[kTileWaves];
  const ull* ctr = A.ctr;
  const uint64_t n_large = ctr[kCtrLargeCount], n_jobs = ctr[kCtrLargeJobs];
  const uint64_t total = n_large + min(n_jobs, (uint64_t)B.job_cap);
  const bool unlisted = n_jobs > B.job_cap;
  if ((uint64_t)blockIdx.x * kTileWaves >= total && !unlisted) return;  // uniform per block
  fill_spread_table();
  __syncthreads();
  WalkLds& L = s_walk[threadIdx.x / kWave];
  const int lane = lane_id();
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(
      (int)(blockIdx.x * kTileWaves + threadIdx.x / kWave));
  const uint32_t waves = gridDim.x * kTileWaves;
  uint64_t g = wave, t0 = unlisted ? 0 : n_large;
  uint32_t q = 0, more = 0;  // of the lane's triangle, t0 - 64 + lane: this wave's next job, all
  uint64_t mine = 0;         // lanes whose triangle has a job for this wave
  for (;;) {
    uint32_t idx, row0 = 0;
    if (g < total) {
      idx = (uint32_t)g;
      if (g >= n_large) {
        const uint2 e = B.jobs[g - n_large];
        idx = e.x;
        row0 = e.y;
      }
      g += waves;
      if (idx == 0xFFFFFFFFu) continue;  // a place left empty
    } else {
      while (!mine && t0 < n_large) {
        more = t0 + lane < n_large ? B.rows[t0 + lane] >> kUnlistedShift : 0u;
        const uint32_t first = (uint32_t)((t0 + lane) * more % waves);
        q = wave >= first ? wave - first : wave + waves - first;
        mine = __ballot(more >= kShareJobs && q < more);
        t0 += kWave;
      }
      if (!mine) break;
      const int src = __ffsll((long long)mine) - 1;
      idx = (uint32_t)(t0 - kWave) + (uint32_t)src;
      const uint32_t job = (uint32_t)__builtin_amdgcn_readlane((int)q, src);
      row0 = (job + 1u) * (B.rows[idx] & ((1u << kUnlistedShift) - 1u));
      if (job + waves < (uint32_t)__builtin_amdgcn_readlane((int)more, src)) {
        if (lane == src) q += waves;
      } else {
        mine &= mine - 1ull;
      }
    }
    const VoxParams P = units[B.unit[idx]];
    if (skipped(P, skip)) continue;
    Walk K;  // (the same in every lane)
    if (idx < B.walk_cap) {
      const uint4* src = B.walk + (uint64_t)idx * kLargeQuads;
      if (lane < kTriQuads) L.tri[0][lane] = src[lane];
      uint4* wk = (uint4*)&K;
#pragma unroll
      for (int k = 0; k < kWalkWords / 4; k++) wk[k] = src[kTriQuads + k];
    } else {
      Setup S;
      setup_tri((const gfloat_t*)P.tris + (uint64_t)B.tri[idx] * P.stride, P, S);
      make_walk(S, P, B.tri[idx], K);
      FastTri F;
      make_fast(K, P, F);
      const uint4* src = (const uint4*)&F;
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < kTriQuads; k++) L.tri[0][k] = src[k];
      }
    }
    wave_lds_sync();
    const uint32_t nb = (uint32_t)(K.i[I_G1V] - K.i[I_G0V] + 1);
    const uint32_t rj = B.rows[idx], rows = rj & ((1u << kUnlistedShift) - 1u);
    const uint32_t rest = rj >> kUnlistedShift;  // (of a triangle with few of them: all its rows here)
    const uint32_t end = rest && rest < kShareJobs ? nb : min(row0 + rows, nb);
    for (; row0 < end; row0 += rows)
      walk_rows<Act>(L, nullptr, P, A, K, nb, lane == 0 ? min(rows, end - row0) : 0u, row0);
  }
}

// ---------------------------------------------------------------- compaction
struct OccLoad {
  const uint32_t* table;
  __device__ uint32_t operator()(uint64_t i) const { return table[i] != 0u; }
};
// Touch path: flagged entries become slot + 1 (slots in Morton order).
struct OccStore {
  uint32_t* occ;
  uint32_t* table;
  ull* ctr;
  __device__ void operator()(uint64_t i, uint32_t ex, uint32_t v, bool last) const {
    if (v) {
      occ[ex] = (uint32_t)i;
      table[i] = ex + 1u;
    }
    if (last) ctr[kCtrNumOcc] = (ull)(ex + v);
  }
};
// Dense passes: the list entries carry the brick's flagged quarters above its table index.
constexpr int kOccBits = 28;
constexpr uint32_t kOccMask = (1u << kOccBits) - 1u;
static_assert(kDenseMax >> kBrickBits <= 1ull << kOccBits, "a byte a voxel");
// (payload units' lines of 32 cells go by number + 1)
constexpr uint64_t kDensePayloadBricks = 1ull << (32 + kLineBits - kBrickBits);
struct OccStoreDense {
  uint32_t* occ;
  const uint32_t* table;
  ull* ctr;
  __device__ void operator()(uint64_t i, uint32_t ex, uint32_t v, bool last) const {
    if (v) {
      const uint32_t quarters = __builtin_amdgcn_udot4(table[i], 0x08040201u, 0u, false);
      occ[ex] = (uint32_t)i | (quarters << kOccBits);
    }
    if (last) ctr[kCtrNumOcc] = (ull)(ex + v);
  }
};

// Occupied-brick kernels: one wave per brick (lane = word), striding over the
// ctr[kCtrNumOcc] bricks.
__device__ __forceinline__ uint64_t wave_global() {
  return ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
}
__device__ __forceinline__ uint64_t waves_total() {
  return (uint64_t)gridDim.x * blockDim.x / kWave;
}

// Pack each flagged brick's bytes into 64 bit words (lane l = voxels 64l..64l+63) at the
// brick's rank, count its voxels, and zero the bytes that were set. The bytes live in the
// unit's dense grid (at the brick's index; only its flagged quarters, or words of payload
// cells, are read) or in the slot pool (at its rank). Bound by those reads: an eighth of a
// soup's bricks in 1771 us with whole bricks read.
// ubase[u] = first table entry of unit u (n_units + 1 entries).
// Dense passes flag only bricks that hold voxels, so the rank is the brick's place in the
// brick stream: there 'pool' is the stream's word array, bcode (non-null) receives the
// tagged brick codes and the table entries are cleared here.
// ONE: a single unit (its parameters are uniform, read with scalar loads).

// 16 bytes, each 0 or 1, as 16 bits
__device__ __forceinline__ uint32_t pack16(u32x4 v) {
  const uint32_t lo = __builtin_amdgcn_udot4(v.y, 0x80402010u, __builtin_amdgcn_udot4(v.x, 0x08040201u, 0u, false), false);
  const uint32_t hi = __builtin_amdgcn_udot4(v.w, 0x80402010u, __builtin_amdgcn_udot4(v.z, 0x08040201u, 0u, false), false);
  return lo | (hi << 8);
}
// Brick wv (table entry ti, unit u): its tagged code, and its table entry cleared.
__device__ __forceinline__ void brick_head(uint64_t wv, uint64_t ti, uint32_t u,
                                           const VoxParams* __restrict__ units,
                                           const uint64_t* __restrict__ ubase,
                                           uint64_t* __restrict__ bcode,
                                           uint32_t* __restrict__ table) {
  if (bcode && lane_id() == 0) {
    bcode[wv] = (units[u].bstart + ((ti - ubase[u]) << kBrickBits)) |
                ((uint64_t)units[u].job << kJobShift);
    table[ti] = 0u;
  }
}
// A brick of bytes as occupancy words: load q of lane l is the 16 bytes at q * 1024 + 16 l (each
// load of the wave one contiguous KiB, quarter q of the brick, made if its flag is set); they
// are packed into the lane's word (piece q of lane l holds bits 16 (l % 4) .. + 15 of word
// 16 q + l / 4); pieces that held marks are zeroed.
__device__ __forceinline__ ull pack_bytes(gquad_t* src, uint32_t quarters) {
  ull parts = 0;  // 16 bits per load
  u32x4 v[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    v[q] = u32x4{0u, 0u, 0u, 0u};
    if ((quarters >> q) & 1u) v[q] = src[q * kWave];
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    parts |= (ull)pack16(v[q]) << (16 * q);
    if (v[q].x | v[q].y | v[q].z | v[q].w) src[q * kWave] = u32x4{0u, 0u, 0u, 0u};
  }
  // word L = 16 q + r gathers the parts of load q from lanes 4 r .. 4 r + 3
  const int L = lane_id(), q = L >> 4, r = L & 15;
  ull m = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)parts, 4 * r + k, kWave);
    const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(parts >> 32), 4 * r + k, kWave);
    const ull p = ((ull)hi << 32) | lo;
    m |= ((p >> (16 * q)) & 0xFFFFull) << (16 * k);
  }
  return m;
}
// A payload brick's cells as occupancy words: the lane's own 64 cells (kept: they hold the
// winners), read only when their word's flag is set.
__device__ __forceinline__ ull pack_cells(const gquad_t* cells, uint8_t* flags) {
  const int lane = lane_id();
  const bool set = flags[lane] != 0;
  flags[lane] = 0;
  ull m = 0;
  if (!set) return m;
  const gquad_t* src = cells + lane * 16;
  // four loads at a time: few registers, so that many waves stay resident
#pragma unroll 1
  for (int g = 0; g < 16; g += 4) {
    u32x4 v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = src[g + q];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const uint32_t nib = (v[q].x != 0u ? 1u : 0u) | (v[q].y != 0u ? 2u : 0u) |
                           (v[q].z != 0u ? 4u : 0u) | (v[q].w != 0u ? 8u : 0u);
      m |= (ull)nib << (4 * (g + q));
    }
  }
  return m;
}
// Brick wv's word array, its node shape (dense passes) and its voxel count.
__device__ __forceinline__ void brick_tail(uint64_t wv, ull m, ull* __restrict__ pool,
                                           uint64_t* __restrict__ bcount,
                                           const uint64_t* __restrict__ bcode,
                                           uint32_t* __restrict__ bshape) {
  pool[wv * kBrickWords + lane_id()] = m;
  if (bcode) {  // the brick node's subtree size and child mask, for the build
    const BrickShape B = brick_shape_of(m);
    if (lane_id() == 0) bshape[wv] = brick_shape_word(B);
  }
  const uint32_t c = (uint32_t)__popcll(m);
  const uint32_t tot = wave_incl_scan<uint32_t>(c);
  // voxel count, plus a flag in bit kNonEmptyShift: one scan gives every brick its
  // voxel offset and its rank among the non-empty bricks (the touch pass flags a
  // superset of the bricks that end up holding voxels)
  if (lane_id() == kWave - 1) bcount[wv] = tot + (tot ? (1ull << kNonEmptyShift) : 0ull);
}

template <bool ONE>
__device__ __forceinline__ void brick_count_body(const uint32_t* __restrict__ occ,
                                                 uint64_t n_occ,
                                                 const VoxParams* __restrict__ units,
                                                 const uint64_t* __restrict__ ubase,
                                                 uint32_t n_units, uint8_t* __restrict__ pool8,
                                                 uint8_t* __restrict__ cflags,
                                                 ull* __restrict__ pool,
                                                 uint64_t* __restrict__ bcount,
                                                 uint64_t* __restrict__ bcode,
                                                 uint32_t* __restrict__ bshape,
                                                 uint32_t* __restrict__ table) {
  for (uint64_t wv = wave_global(); wv < n_occ; wv += waves_total()) {
    // the brick is the wave's: its table index in a scalar register, so that the unit
    // search below runs on scalar loads
    const uint32_t oe = (uint32_t)__builtin_amdgcn_readfirstlane((int)occ[wv]);
    const uint64_t ti = bcode ? oe & kOccMask : oe;
    const uint32_t quarters = bcode ? oe >> kOccBits : 15u;
    const uint32_t u = ONE ? 0u : upper_index<uint64_t>(ubase, n_units + 1, ti);
    brick_head(wv, ti, u, units, ubase, bcode, table);
    const uint64_t bi = ti - ubase[u];
    ull m;
    if (units[u].wide)
      m = pack_cells((const gquad_t*)units[u].grid8 + bi * (kBrickVox / 4), cflags + ti * kBrickWords);
    else
      m = pack_bytes((gquad_t*)(units[u].dense ? units[u].grid8 + bi * kBrickVox
                                               : pool8 + wv * kBrickVox) + lane_id(),
                     quarters);
    brick_tail(wv, m, pool, bcount, bcode, bshape);
  }
}

__global__ __launch_bounds__(256) void k_brick_count(const uint32_t* __restrict__ occ,
                                                     const ull* __restrict__ ctr, uint64_t cap,
                                                     const VoxParams* __restrict__ units,
                                                     const uint64_t* __restrict__ ubase,
                                                     uint32_t n_units, uint8_t* __restrict__ pool8,
                                                     uint8_t* __restrict__ cflags,
                                                     ull* __restrict__ pool,
                                                     uint64_t* __restrict__ bcount,
                                                     uint64_t* __restrict__ bcode,
                                                     uint32_t* __restrict__ bshape,
                                                     uint32_t* __restrict__ table) {
  // more flagged bricks than slots (touch path): the pass is redone with a larger pool
  const uint64_t n_occ = min((uint64_t)ctr[kCtrNumOcc], cap);
  if (n_units == 1)
    brick_count_body<true>(occ, n_occ, units, ubase, n_units, pool8, cflags, pool, bcount, bcode,
                           bshape, table);
  else
    brick_count_body<false>(occ, n_occ, units, ubase, n_units, pool8, cflags, pool, bcount, bcode,
                            bshape, table);
}

struct CountStore {
  uint64_t* off;
  ull* total;
  __device__ void operator()(uint64_t i, uint64_t ex, uint64_t v, bool last) const {
    off[i] = ex;
    if (last) *total = (ull)(ex + v);
  }
};
// Brick counts of a dense pass: also each brick's first voxel in the stream (s0 + offset). With
// host (a pass of one unit), the thread that has the total gives the pass's counters to the host,
// which waits for them: the launch that would follow for it took 4 us.
struct BrickOffStore {
  uint64_t* off;
  ull* ctr;
  uint64_t* bvoff;
  uint64_t s0;
  uint64_t* host;  // pinned: kNumCounters words, or nullptr
  volatile uint32_t* flag;
  uint64_t seq;
  __device__ void operator()(uint64_t i, uint64_t ex, uint64_t v, bool last) const {
    off[i] = ex;
    bvoff[i] = s0 + (ex & kVoxMask);
    if (last) done(ex + v);
  }
  __device__ void none() const { done(0); }  // no bricks
  __device__ void done(uint64_t total) const {
    ctr[kCtrNumVox] = total;
    if (!host) return;
    uint64_t h[kNumCounters];
#pragma unroll
    for (int k = 0; k < kNumCounters; k++) h[k] = k == kCtrNumVox ? total : (uint64_t)ctr[k];
#pragma unroll
    for (int k = 0; k < kNumCounters; k++) host[k] = h[k];
    *(volatile uint64_t*)(flag + 2) = wall_clock64();
    __threadfence_system();
    *flag = (uint32_t)seq;
  }
};

// Touched-brick passes: the brick stream entry of every non-empty flagged brick and, with
// kCodes, for payload units the sorted codes of its voxels, tagged with the unit's job in bits
// kJobShift+.
template <bool kCodes>
__global__ __launch_bounds__(256) void k_brick_emit(const uint32_t* __restrict__ occ,
                                                    const ull* __restrict__ ctr,
                                                    const VoxParams* __restrict__ units,
                                                    const uint64_t* __restrict__ ubase,
                                                    uint32_t n_units,
                                                    const ull* __restrict__ pool,
                                                    const uint64_t* __restrict__ boff,
                                                    uint64_t* __restrict__ codes,
                                                    uint32_t* __restrict__ wprefix,
                                                    uint64_t s0, uint64_t* __restrict__ bwords,
                                                    uint64_t* __restrict__ bcode,
                                                    uint64_t* __restrict__ bvoff,
                                                    uint32_t* __restrict__ bshape) {
  const uint64_t n_occ = ctr[kCtrNumOcc];
  for (uint64_t wv = wave_global(); wv < n_occ; wv += waves_total()) {
    const uint64_t ti = (uint32_t)__builtin_amdgcn_readfirstlane((int)occ[wv]);  // wave's brick
    const uint32_t u = upper_index<uint64_t>(ubase, n_units + 1, ti);
    const uint64_t slot = wv * kBrickWords + lane_id();
    ull word = pool[slot];
    const uint64_t bo = boff[wv];
    const uint64_t tag = (uint64_t)units[u].job << kJobShift;
    const uint64_t b0 = units[u].bstart + ((ti - ubase[u]) << kBrickBits);
    // the brick stream (non-empty bricks, appended in stream order)
    if (__ballot(word != 0ull)) {
      const uint64_t sb = bo >> kNonEmptyShift;
      bwords[sb * kBrickWords + lane_id()] = word;
      const BrickShape B = brick_shape_of(word);
      if (lane_id() == 0) {
        bcode[sb] = b0 | tag;
        bvoff[sb] = s0 + (bo & kVoxMask);
        bshape[sb] = brick_shape_word(B);
      }
    }
    if constexpr (!kCodes) continue;
    if (units[u].stride == 9) continue;  // geometry-only unit: codes written on demand
    const uint32_t c = (uint32_t)__popcll(word);
    const uint32_t inc = wave_incl_scan<uint32_t>(c);
    uint64_t pos = (bo & kVoxMask) + (inc - c);
    wprefix[slot] = (uint32_t)pos;
    const uint64_t cb = (b0 + ((uint64_t)lane_id() << 6)) | tag;
    while (word) {
      const int bit = __ffsll(word) - 1;
      codes[pos++] = cb + (uint64_t)bit;
      word &= word - 1;
    }
  }
}

// Codes of the voxels of bricks [0, nb) of the stream, from their occupancy words: one
// wave per brick, lane l = word l, written at the brick's stream offset.
__global__ __launch_bounds__(256) void k_bricks_codes(const uint64_t* __restrict__ bwords,
                                                      const uint64_t* __restrict__ bcode,
                                                      const uint64_t* __restrict__ bvoff,
                                                      uint64_t nb, uint64_t* __restrict__ codes) {
  for (uint64_t b = wave_global(); b < nb; b += waves_total()) {
    ull word = bwords[b * kBrickWords + lane_id()];
    const uint32_t c = (uint32_t)__popcll(word);
    const uint32_t inc = wave_incl_scan<uint32_t>(c);
    uint64_t pos = bvoff[b] + (inc - c);
    const uint64_t cb = bcode[b] + ((uint64_t)lane_id() << 6);
    while (word) {
      const int bit = __ffsll(word) - 1;
      codes[pos++] = cb + (uint64_t)bit;
      word &= word - 1;
    }
  }
}

// restore the all-zero state of the table for the flagged bricks (their bytes were
// cleared by k_brick_count)
__global__ __launch_bounds__(256) void k_brick_clear(const uint32_t* __restrict__ occ,
                                                     const ull* __restrict__ ctr,
                                                     uint32_t* __restrict__ table) {
  const uint64_t n_occ = ctr[kCtrNumOcc];
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_occ; i += stride)
    table[occ[i]] = 0u;
}

// First voxel (batch rank) of each unit: the offset of its first flagged brick.
// (occ_mask: the table index in an occ entry)
__global__ void k_unit_voxels(const uint32_t* __restrict__ occ, uint32_t occ_mask,
                              const ull* __restrict__ ctr,
                              const uint64_t* __restrict__ ubase, uint32_t n_units,
                              const uint64_t* __restrict__ boff, uint64_t* __restrict__ uvoff) {
  const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u > n_units) return;
  const uint64_t n_occ = ctr[kCtrNumOcc];
  const uint64_t V = ctr[kCtrNumVox] & kVoxMask;
  if (u == n_units) {
    uvoff[u] = V;
    return;
  }
  // first occupied brick with table index >= ubase[u]
  uint64_t lo = 0, hi = n_occ;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    if ((uint64_t)(occ[mid] & occ_mask) < ubase[u])
      lo = mid + 1;
    else
      hi = mid;
  }
  uvoff[u] = (lo < n_occ) ? (boff[lo] & kVoxMask) : V;
}

// ---------------------------------------------------------------- payload records
// Exact quotient x / d of a grid coordinate: a power of two d (a unit bbox) needs no division.
__device__ __forceinline__ float coord_over(uint32_t x, float d, float inv_d, bool pow2) {
  return pow2 ? (float)(int)x * inv_d : (float)(int)x / d;
}
// The record of voxel 'code' won by triangle t: BarycentricCoords.h:4-32; colour modes of
// main.cpp:373-382.
__device__ __forceinline__ void make_payload_record(const JobDev& J, uint64_t code, uint32_t t,
                                                    uint4& q0, uint4& q1) {
  float col0, col1, col2, nr0, nr1, nr2;
  const gfloat_t* p = (const gfloat_t*)J.tris + (uint64_t)t * 21;
  const float v0x = p[0], v0y = p[1], v0z = p[2];
  const float v1x = p[3], v1y = p[4], v1z = p[5];
  const float v2x = p[6], v2y = p[7], v2z = p[8];
  nr0 = p[9];
  nr1 = p[10];
  nr2 = p[11];
  uint32_t x, y, z;
  unmorton3(code, x, y, z);
  const int color_mode = J.color_mode;
  const float unit_div = J.unit_div;
  if (color_mode == 0) {
    // n = normalize(cross(e0, e1)) exactly as in the voxelizer
    const float e0x = v1x - v0x, e0y = v1y - v0y, e0z = v1z - v0z;
    const float e1x = v2x - v1x, e1y = v2y - v1y, e1z = v2z - v1z;
    const float cx = e0y * e1z - e1y * e0z;
    const float cy = e0z * e1x - e1z * e0x;
    const float cz = e0x * e1y - e1x * e0y;
    const float inv = 1.0f / sqrtf((cx * cx + cy * cy) + cz * cz);
    const float nx = cx * inv, ny = cy * inv, nz = cz * inv;
    // (a power of two in the middle of the exponent range: its reciprocal is exact)
    const uint32_t ub = __float_as_uint(unit_div);
    const bool pow2 = (ub & 0x807FFFFFu) == 0u && (ub >> 23) > 64u && (ub >> 23) < 190u;
    const float inv_div = __builtin_amdgcn_ldexpf(1.0f, 127 - (int)(ub >> 23));
    const float vx = coord_over(x, unit_div, inv_div, pow2);
    const float vy = coord_over(y, unit_div, inv_div, pow2);
    const float vz = coord_over(z, unit_div, inv_div, pow2);
    const float coeffD = -((v0x * nx + v0y * ny) + v0z * nz);
    const float k = (((vx * nx + vy * ny) + vz * nz) + coeffD) / ((nx * nx + ny * ny) + nz * nz);
    const float qx = vx - k * nx, qy = vy - k * ny, qz = vz - k * nz;
    // glm::inverse(mat3(v0, v1, v2)), m[c][r]
    const float m00 = v0x, m01 = v0y, m02 = v0z;
    const float m10 = v1x, m11 = v1y, m12 = v1z;
    const float m20 = v2x, m21 = v2y, m22 = v2z;
    const float det = (m00 * (m11 * m22 - m21 * m12) - m10 * (m01 * m22 - m21 * m02)) +
                      m20 * (m01 * m12 - m11 * m02);
    const float o = 1.0f / det;
    const float i00 = (m11 * m22 - m21 * m12) * o;
    const float i10 = (-(m10 * m22 - m20 * m12)) * o;
    const float i20 = (m10 * m21 - m20 * m11) * o;
    const float i01 = (-(m01 * m22 - m21 * m02)) * o;
    const float i11 = (m00 * m22 - m20 * m02) * o;
    const float i21 = (-(m00 * m21 - m20 * m01)) * o;
    const float i02 = (m01 * m12 - m11 * m02) * o;
    const float i12 = (-(m00 * m12 - m10 * m02)) * o;
    const float i22 = (m00 * m11 - m10 * m01) * o;
    const float bx = (i00 * qx + i10 * qy) + i20 * qz;
    const float by = (i01 * qx + i11 * qy) + i21 * qz;
    const float bz = (i02 * qx + i12 * qy) + i22 * qz;
    col0 = (bx * p[12] + by * p[15]) + bz * p[18];
    col1 = (bx * p[13] + by * p[16]) + bz * p[19];
    col2 = (bx * p[14] + by * p[17]) + bz * p[20];
  } else if (color_mode == 1) {  // fixed white
    col0 = col1 = col2 = 1.0f;
  } else if (color_mode == 2) {  // mortonToRGB: (z, y, x) / gridsize
    const float g = (float)J.gridsize;
    col0 = (float)z / g;
    col1 = (float)y / g;
    col2 = (float)x / g;
  } else {  // normal -> colour
    const float inv = 1.0f / sqrtf((nr0 * nr0 + nr1 * nr1) + nr2 * nr2);
    const float a = nr0 * inv, b = nr1 * inv, c = nr2 * inv;
    col0 = (a + 1.0f) / 2.0f;
    col1 = (b + 1.0f) / 2.0f;
    col2 = (c + 1.0f) / 2.0f;
  }
  q0.x = (uint32_t)code;
  q0.y = (uint32_t)(code >> 32);
  q0.z = __float_as_uint(canon_nan(col0));
  q0.w = __float_as_uint(canon_nan(col1));
  q1.x = __float_as_uint(canon_nan(col2));
  q1.y = __float_as_uint(canon_nan(nr0));
  q1.z = __float_as_uint(canon_nan(nr1));
  q1.w = __float_as_uint(canon_nan(nr2));
}

// Position of the n-th set bit of w (n below its count)
__device__ __forceinline__ uint32_t nth_set_bit(uint64_t w, uint32_t n) {
  uint32_t lo = (uint32_t)w, at = 0;
  const uint32_t c = (uint32_t)__popc(lo);
  if (n >= c) {
    n -= c;
    lo = (uint32_t)(w >> 32);
    at = 32;
  }
#pragma unroll
  for (int h = 16; h; h >>= 1) {
    const uint32_t k = (uint32_t)__popc(lo & ((1u << h) - 1u));
    const bool up = n >= k;
    n -= up ? k : 0u;
    lo = up ? lo >> h : lo;
    at += up ? h : 0;
  }
  return at;
}

// The records of a dense pass's payload units, straight from their bricks: a wave per brick,
// its voxels 64 at a time in Morton order, so that neighbouring lanes read neighbouring cells
// (~the winning triangle, 0 = unmarked) and write neighbouring records. The cells of non-empty
// words are zeroed afterwards, whole 256-byte words at once. Codes and winners are not written
// (ensure_codes expands the codes for readers that want them). jobs = nullptr: the job is j0.
//
// Bound by memory: 32 bytes written a voxel, the cells' words, and the winners' records
// gathered. A pass that wrote every voxel's code and winner (a lane per word, its voxels one
// after the other) and one that read them back took 242 + 336 us on 17M voxels of a rough
// sphere; this one 403 (1.9M voxels of a fine terrain: 34 + 71 us, 81). With kStaged (more than
// kStagePayload bricks) 64 records go through LDS and out in whole KiB past the caches, not as 16
// bytes of every 32, and cells are zeroed by the 64-byte pieces that hold marks: 392 -> 275 us,
// the terrain 72 -> 61, 64 mixed meshes 876 -> 680 (2500 bricks: 17, staged 18.6).
constexpr uint64_t kStagePayload = 4096;
template <bool kStaged>
__global__ __launch_bounds__(256) void k_payload_bricks(
    const uint32_t* __restrict__ occ, const ull* __restrict__ n_occ_ptr,
    const VoxParams* __restrict__ units, const uint64_t* __restrict__ ubase, uint32_t n_units,
    const ull* __restrict__ words, const uint64_t* __restrict__ boff,
    const JobDev* __restrict__ jobs, JobDev j0, uint64_t s0, float* __restrict__ out, ull* ctr) {
  __shared__ uint8_t s_slot[256];
  __shared__ uint4 s_stage[kStaged ? 256 / kWave : 1][2 * kWave];
  uint8_t* slot = s_slot + (threadIdx.x / kWave) * kWave;
  uint4* stage = s_stage[kStaged ? threadIdx.x / kWave : 0];
  const int lane = lane_id();
  const uint64_t n_occ = *n_occ_ptr;
  for (uint64_t wv = wave_global(); wv < n_occ; wv += waves_total()) {
    const uint32_t ti = (uint32_t)__builtin_amdgcn_readfirstlane((int)occ[wv]) & kOccMask;
    const uint32_t u = upper_index<uint64_t>(ubase, n_units + 1, (uint64_t)ti);
    if (!units[u].wide) continue;
    const ull word = words[wv * kBrickWords + lane];
    gword_t* cells = (gword_t*)units[u].grid8 + (ti - ubase[u]) * kBrickVox;
    const uint64_t code0 = units[u].bstart + ((ti - ubase[u]) << kBrickBits);
    const JobDev J = jobs ? jobs[units[u].job] : j0;
    const uint64_t pos0 = boff[wv] & kVoxMask;  // the brick's first voxel in the pass
    float* rec = out + (J.dbase + 1 + (s0 + pos0 - J.voff)) * 8;
    const uint32_t c = (uint32_t)__popcll(word);
    const uint32_t inc = wave_incl_scan<uint32_t>(c), pre = inc - c;
    const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)inc, kWave - 1);
    // (the next window's cells are on their way while this one's records are made)
    uint32_t carry = 0, v = 0, cell = 0;
    auto fetch = [&](uint32_t k0, uint32_t& vo, uint32_t& co) {
      const uint32_t wi = locate(slot, pre, c != 0, k0, carry) & 63u;
      const uint32_t wlo = (uint32_t)__shfl((int)(uint32_t)word, (int)wi, kWave);
      const uint32_t whi = (uint32_t)__shfl((int)(uint32_t)(word >> 32), (int)wi, kWave);
      const uint32_t wpre = (uint32_t)__shfl((int)pre, (int)wi, kWave);
      const uint32_t k = k0 + lane;
      if (k < n) {
        vo = wi * 64u + nth_set_bit(((uint64_t)whi << 32) | wlo, k - wpre);
        co = cells[vo];
      }
    };
    if (n) fetch(0, v, cell);
    for (uint32_t k0 = 0; k0 < n; k0 += kWave) {
      uint32_t v2 = 0, cell2 = 0;
      if (k0 + kWave < n) fetch(k0 + kWave, v2, cell2);
      const uint32_t k = k0 + lane;
      if (k < n) {
        if (cell == 0u)  // cannot happen: the words were made from the cells
          atomicAdd(&ctr[kCtrError], 1ull);
        else {
          uint4 q0, q1;
          make_payload_record(J, code0 + v, ~cell, q0, q1);
          uint4* to = kStaged ? stage + 2 * lane : (uint4*)(rec + (uint64_t)k * 8);
          to[0] = q0;
          to[1] = q1;
        }
      }
      if constexpr (kStaged) {
        wave_lds_sync();
        const uint32_t quads = 2 * min(n - k0, (uint32_t)kWave);
        u32x4* to = (u32x4*)(rec + (uint64_t)k0 * 8);
#pragma unroll
        for (uint32_t q = 0; q < 2; q++)
          if (lane + kWave * q < quads)
            __builtin_nontemporal_store(((const u32x4*)stage)[lane + kWave * q], to + lane + kWave * q);
        wave_lds_sync();
      }
      v = v2;
      cell = cell2;
    }
    // (every cell has been read: the records were made from them)
    uint64_t ne = __ballot(word != 0ull);
    while (ne) {  // four words at a time, 16 lanes each
      uint32_t mine = 64u;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const uint32_t wi = ne ? (uint32_t)__ffsll((long long)ne) - 1u : 64u;
        if ((lane >> 4) == q) mine = wi;
        ne &= ne - 1ull;
      }
      // (only the 64-byte pieces that hold marks)
      const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)word, (int)(mine & 63u), kWave);
      const uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(word >> 32), (int)(mine & 63u), kWave);
      const uint32_t piece = ((lane & 8) ? hi : lo) >> ((lane & 4) ? 16 : 0);
      if (mine < 64u && (piece & 0xFFFFu))
        ((gquad_t*)(cells + mine * 64u))[lane & 15] = u32x4{0u, 0u, 0u, 0u};
    }
  }
}

// Touched-brick passes: one thread per payload voxel, its code and winner from the arrays that
// k_brick_emit and the winner walk wrote.
// Voxel i of the pass (stream index s0 + i) belongs to the unit whose voxel range holds
// it, and to that unit's job; its record goes to dbase[job] + 1 + (s0 + i - voff[job]).
// Voxels of geometry-only jobs have no record here.
// Threads cover the payload units' voxels only, from payload voxel 'first' on: payload voxel k
// lies in the payload unit j with prange[j] <= k < prange[j + 1] (a block searches for its first voxel, a thread
// steps forward over the rare unit boundaries), unit punit[j], whose voxels start at pass
// voxel pstart[j].
__global__ __launch_bounds__(256) void k_payload_records(
    const JobDev* __restrict__ jobs, const VoxParams* __restrict__ units,
    const uint64_t* __restrict__ prange, const uint64_t* __restrict__ pstart,
    const uint32_t* __restrict__ punit, uint32_t n_pu, const uint64_t* __restrict__ codes,
    uint64_t s0, const uint32_t* __restrict__ winner, uint64_t first, uint64_t n_pv,
    float* __restrict__ out, ull* ctr) {
  __shared__ uint32_t s_j0;
  const uint64_t b0 = first + (uint64_t)blockIdx.x * blockDim.x;
  const uint64_t k = b0 + threadIdx.x;
  if (threadIdx.x == 0) s_j0 = upper_index<uint64_t>(prange, n_pu + 1, b0);
  __syncthreads();
  if (k >= n_pv) return;
  uint32_t j = s_j0;
  while (j + 1 < n_pu && prange[j + 1] <= k) j++;
  const uint32_t u = punit[j];
  const uint64_t i = pstart[j] + (k - prange[j]);  // voxel i of the pass
  const uint64_t tagged = codes[s0 + i];
  const JobDev& J = jobs[units[u].job];
  if (!J.payload) return;
  const uint64_t code = tagged & kCodeMask;
  const uint32_t t = winner[i];
  if (t == 0xFFFFFFFFu)  // cannot happen: both passes evaluate the same predicates
    atomicAdd(&ctr[kCtrError], 1ull);
  else {
    uint4* r = (uint4*)(out + (J.dbase + 1 + (s0 + i - J.voff)) * 8);
    uint4 q0, q1;
    make_payload_record(J, code, t, q0, q1);
    r[0] = q0;
    r[1] = q1;
  }
}

// ---------------------------------------------------------------- partition kernels
// Per triangle, the box [lo, hi] of partition cube coordinates its bbox touches, packed
// as 8-bit fields (x lo, x hi, y lo, y hi, z lo, z hi); ~0 = touches none.
__global__ __launch_bounds__(256) void k_part_hitbox(const float* __restrict__ tris, int stride,
                                                     uint64_t n,
                                                     const float* __restrict__ cube_lo,
                                                     const float* __restrict__ cube_hi, int K,
                                                     uint64_t* __restrict__ hitbox) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  hitbox[t] = part_hitbox_of(tris + t * stride, cube_lo, cube_hi, K);
}

// Up to 64 partitions: a triangle's partitions as a bit mask, and all lists at once. A tile is
// 2048 triangles (kPartItems rows of 64 a wave, in order); cnt[j * ntiles + tile] = its triangles
// in partition j, and their exclusive prefix over that order is where they go, the lists being
// laid out one after the other.
//
// Bound by the records read. A flag scan per partition, with a host wait for each list's length,
// took seven launches a partition: 6M triangles in 8 partitions 0.31 ms of device time and 8 waits,
// 0.14 and one now.
constexpr int kPartItems = 8;
constexpr uint64_t kPartTile = 256 * kPartItems;
constexpr uint64_t kPartMask = 64;  // partitions in a mask
struct PartCubes {
  uint64_t on[3][4];  // partitions whose cube coordinate along an axis is c
};
// Lane j's part of the counts of partition j over a row of 64 masks.
__device__ __forceinline__ uint32_t part_row_count(uint64_t m, uint32_t np) {
  uint32_t c = 0;
  for (uint32_t j = 0; j < np; j++) {
    const uint32_t k = (uint32_t)__popcll(__ballot((m >> j) & 1ull));
    c = (uint32_t)lane_id() == j ? k : c;
  }
  return c;
}
__global__ __launch_bounds__(256) void k_part_masks(const float* __restrict__ tris, int stride,
                                                    uint64_t n, const float* __restrict__ cube_lo,
                                                    const float* __restrict__ cube_hi, int K,
                                                    uint32_t np, PartCubes cubes,
                                                    uint64_t* __restrict__ mask,
                                                    uint32_t* __restrict__ cnt, uint32_t ntiles) {
  __shared__ uint32_t s_cnt[256 / kWave][kWave];
  const int w = threadIdx.x / kWave;
  const uint64_t first = striped_first<kPartItems>(blockIdx.x, 256);
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < kPartItems; k++) {
    const uint64_t i = first + (uint64_t)kWave * k;
    uint64_t m = 0;
    if (i < n) {
      const uint64_t h = part_hitbox_of(tris + i * stride, cube_lo, cube_hi, K);
      if (h != ~0ull) {
        m = ~0ull;
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const int lo = (int)(h >> (16 * a)) & 0xFF, hi = (int)(h >> (16 * a + 8)) & 0xFF;
          uint64_t on = 0;
#pragma unroll
          for (int q = 0; q < 4; q++)
            if (q >= lo && q <= hi) on |= cubes.on[a][q];
          m &= on;
        }
      }
      mask[i] = m;
    }
    c += part_row_count(m, np);
  }
  s_cnt[w][lane_id()] = c;
  __syncthreads();
  if (threadIdx.x < np) {
    uint32_t sum = 0;
    for (int q = 0; q < 256 / kWave; q++) sum += s_cnt[q][threadIdx.x];
    cnt[(uint64_t)threadIdx.x * ntiles + blockIdx.x] = sum;
  }
}
struct PartCountLoad {
  const uint32_t* cnt;
  __device__ uint64_t operator()(uint64_t i) const { return cnt[i]; }
};
struct PartOffStore {
  uint64_t* off;
  uint64_t* start;  // first place of each partition's list; their end
  uint64_t ntiles;
  uint64_t np;
  __device__ void operator()(uint64_t i, uint64_t ex, uint64_t v, bool last) const {
    off[i] = ex;
    if (i % ntiles == 0) start[i / ntiles] = ex;
    if (last) start[np] = ex + v;
  }
};
__global__ __launch_bounds__(256) void k_part_lists(const uint64_t* __restrict__ mask, uint64_t n,
                                                    uint32_t np,
                                                    const uint64_t* __restrict__ off,
                                                    uint32_t ntiles, uint32_t* __restrict__ list) {
  __shared__ uint32_t s_cnt[256 / kWave][kWave];
  const int w = threadIdx.x / kWave, lane = lane_id();
  const uint64_t first = striped_first<kPartItems>(blockIdx.x, 256);
  uint64_t m[kPartItems];
  uint32_t c = 0;
#pragma unroll
  for (int k = 0; k < kPartItems; k++) {
    const uint64_t i = first + (uint64_t)kWave * k;
    m[k] = i < n ? mask[i] : 0ull;
  }
#pragma unroll
  for (int k = 0; k < kPartItems; k++) c += part_row_count(m[k], np);
  s_cnt[w][lane] = c;
  __syncthreads();
  for (uint32_t j = 0; j < np; j++) {
    uint64_t at = off[(uint64_t)j * ntiles + blockIdx.x];
    for (int q = 0; q < w; q++) at += s_cnt[q][j];
#pragma unroll
    for (int k = 0; k < kPartItems; k++) {
      const bool in = (m[k] >> j) & 1ull;
      const uint64_t b = __ballot(in);
      if (in)
        list[at + (uint64_t)__popcll(b & ((1ull << lane) - 1ull))] =
            (uint32_t)(first + (uint64_t)kWave * k);
      at += (uint64_t)__popcll(b);
    }
  }
}

// out[k] = the record of triangle list[k] (list == nullptr: triangle k), stride floats each
__global__ __launch_bounds__(256) void k_gather_records(const float* __restrict__ tris, int stride,
                                                        const uint32_t* __restrict__ list,
                                                        uint64_t n, float* __restrict__ out) {
  const uint64_t total = n * (uint64_t)stride;
  for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
       e += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t k = e / (uint64_t)stride, f = e - k * (uint64_t)stride;
    const uint64_t t = list ? list[k] : k;
    out[e] = tris[t * stride + f];
  }
}

hipError_t gather_records(Context& c, const float* tris, int stride, const uint32_t* list,
                          uint64_t n, float* out) {
  if (!n) return hipSuccess;
  const uint64_t total = n * (uint64_t)stride;
  SVO_LAUNCH(k_gather_records, dim3((unsigned)std::min<uint64_t>((total + 255) / 256, 16384)),
             dim3(256), 0, c.stream, tris, stride, list, n, out);
  return hipGetLastError();
}

struct PartStore {
  uint32_t* list;
  ull* total;
  __device__ void operator()(uint64_t i, uint32_t ex, uint32_t v, bool last) const {
    if (v) list[ex] = (uint32_t)i;
    if (last) *total = (ull)(ex + v);
  }
};

// ---------------------------------------------------------------- fills
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}
__global__ void k_fill_u64(uint64_t* p, uint64_t v, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) p[i] = v;
}
// start of a pass: two small ranges zeroed, the device clock in *stamp
__global__ void k_pass_begin(uint64_t* a, uint64_t na, uint64_t* b, uint64_t nb, uint64_t* stamp) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *stamp = wall_clock64();
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < na + nb; i += stride) {
    if (i < na)
      a[i] = 0;
    else
      b[i - na] = 0;
  }
}
// one job's descriptor by kernel argument (a small copy costs more than a launch)
__global__ void k_put_job(JobDev* dst, JobDev job) { *dst = job; }
static unsigned fill_grid(uint64_t n) {
  uint64_t b = (n + 255) / 256;
  return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(b, 8192));
}
hipError_t fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s) {
  if (!n) return hipSuccess;
  SVO_LAUNCH(k_fill_u32, dim3(fill_grid(n)), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}
hipError_t fill_u64(uint64_t* p, uint64_t v, uint64_t n, hipStream_t s) {
  if (!n) return hipSuccess;
  SVO_LAUNCH(k_fill_u64, dim3(fill_grid(n)), dim3(256), 0, s, p, v, n);
  return hipGetLastError();
}

// ---------------------------------------------------------------- host drivers
#define SVO_TRY(x)                        \
  do {                                    \
    hipError_t _e = (x);                  \
    if (_e != hipSuccess) return _e;      \
  } while (0)

hipError_t upload_async(Context& c, void* dst, const void* src, size_t bytes) {
  if (!bytes) return hipSuccess;
  const size_t need = (bytes + 255) & ~(size_t)255;
  if (c.stage_used + need > c.stage_cap) {
    // every copy from the staging buffer has completed after this
    SVO_TRY(stream_sync(c.stream));
    c.stage_used = 0;
    if (need > c.stage_cap) {
      if (c.stage) (void)hipHostFree(c.stage);
      c.stage = nullptr;
      c.stage_cap = 0;
      // (pinned pages cost 0.15 us each to get: 4 MB of them 600 us of a new context's first pass)
      const size_t cap = std::max<size_t>(4 * need, 128u << 10);
      SVO_TRY(hipHostMalloc(&c.stage, cap, hipHostMallocDefault));
      c.stage_cap = cap;
    }
  }
  void* h = (char*)c.stage + c.stage_used;
  memcpy(h, src, bytes);
  c.stage_used += need;
  return hipMemcpyAsync(dst, h, bytes, hipMemcpyHostToDevice, c.stream);
}

// Small read-backs: one kernel copies every request into the pinned host buffer (mapped
// into the device's address space), instead of one DMA copy per request.
constexpr int kGatherMax = 4;
struct GatherArgs {
  const uint64_t* src[kGatherMax];
  uint64_t* dst[kGatherMax];
  uint32_t words[kGatherMax];
  int n;
};
// Then it leaves the device clock after the flag and raises *flag = seq (after a system-scope
// fence), which the host polls: a shorter wait than a stream synchronization.
__global__ __launch_bounds__(256) void k_gather_host(GatherArgs g, volatile uint32_t* flag,
                                                     uint32_t seq) {
  for (int k = 0; k < g.n; k++)
    for (uint32_t i = threadIdx.x; i < g.words[k]; i += blockDim.x) g.dst[k][i] = g.src[k][i];
  if (threadIdx.x == 0) *(volatile uint64_t*)(flag + 2) = wall_clock64();
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) *flag = seq;
}

// The pinned landing area, at least 'total' bytes.
static hipError_t ensure_hread(Context& c, size_t total) {
  if (total <= c.hread_cap) return hipSuccess;
  SVO_TRY(hipStreamSynchronize(c.stream));
  if (c.hread) (void)hipHostFree(c.hread);
  c.hread = nullptr;
  c.hread_cap = 0;
  const size_t cap = std::max<size_t>(2 * total, 72u << 10);  // (every small read-back fits)
  SVO_TRY(hipHostMalloc(&c.hread, cap, hipHostMallocDefault));
  // memory freed by another context may hold its last flag: a value this one will wait for
  memset(c.hread, 0, 256);
  c.hread_cap = cap;
  return hipSuccess;
}
// Wait until a kernel has raised the landing area's flag to seq: polled for a short while (the
// usual case: the stream is almost done), then a blocking synchronization (long kernels ahead,
// or a failed launch).
static hipError_t wait_flag(Context& c, uint32_t seq) {
  volatile uint32_t* flag = (volatile uint32_t*)c.hread;
  bool seen = false;
  const auto t0 = std::chrono::steady_clock::now();
  for (uint32_t k = 0;; k++) {
    if (*flag == seq) {
      seen = true;
      break;
    }
    if ((k & 255) == 255 &&
        std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(2000))
      break;
  }
  if (seen)
    std::atomic_thread_fence(std::memory_order_acquire);
  else
    SVO_TRY(hipStreamSynchronize(c.stream));
  return hipSuccess;
}

hipError_t read_back(Context& c, const ReadReq* reqs, int n) {
  t_syncs++;  // one host wait, whichever way it is done
  size_t total = 0;
  bool small = n <= kGatherMax;
  for (int k = 0; k < n; k++) {
    total += (reqs[k].bytes + 255) & ~(size_t)255;
    small = small && reqs[k].bytes % 8 == 0 && (uintptr_t)reqs[k].src % 8 == 0;
  }
  small = small && total <= (64u << 10);
  total += 256;  // the completion flag
  SVO_TRY(ensure_hread(c, total));
  const size_t base = 256;
  size_t off = base;
  if (small) {
    GatherArgs g{};
    g.n = n;
    for (int k = 0; k < n; k++) {
      g.src[k] = (const uint64_t*)reqs[k].src;
      g.dst[k] = (uint64_t*)((char*)c.hread + off);
      g.words[k] = (uint32_t)(reqs[k].bytes / 8);
      off += (reqs[k].bytes + 255) & ~(size_t)255;
    }
    volatile uint32_t* flag = (volatile uint32_t*)c.hread;
    const uint32_t seq = ++c.hread_seq;
    SVO_LAUNCH(k_gather_host, dim3(1), dim3(256), 0, c.stream, g, flag, seq);
    SVO_TRY(hipGetLastError());
    SVO_TRY(wait_flag(c, seq));
    c.stamp_read = ((volatile uint64_t*)c.hread)[1];
  } else {
    for (int k = 0; k < n; k++) {
      if (reqs[k].bytes)
        SVO_TRY(hipMemcpyAsync((char*)c.hread + off, reqs[k].src, reqs[k].bytes,
                               hipMemcpyDeviceToHost, c.stream));
      off += (reqs[k].bytes + 255) & ~(size_t)255;
    }
    SVO_TRY(hipStreamSynchronize(c.stream));
  }
  off = base;
  for (int k = 0; k < n; k++) {
    memcpy(reqs[k].dst, (char*)c.hread + off, reqs[k].bytes);
    off += (reqs[k].bytes + 255) & ~(size_t)255;
  }
  return hipSuccess;
}

// n elements of 16 bytes (8-byte aligned: wide accesses need no more) and, with tail, one of 8
// after them: a block copies kItems x 4 KB in one piece, a wave's load or store 1 KB of it. A copy
// of few blocks also raises the read-back flag: the block that finishes last, by a counter it
// leaves at zero for the next copy (flag = nullptr: no flag).
//
// Bound by memory: 6.2 TB/s read and written at 0.5 GB, 6.3 at 2.4 GB, 7.0 at 0.25 GB, a thread an
// element, streamed past the caches on the way out only. Four elements a thread a grid apart (32
// MB: the same channels) and streamed both ways reached 5.2, 5.1 and 5.0; four in one piece 6.2,
// 5.7 and 6.2.
typedef u32x4 u32x4_u __attribute__((aligned(8)));
template <int kItems>
__global__ __launch_bounds__(256) void k_copy(u32x4_u* __restrict__ dst,
                                              const u32x4_u* __restrict__ src, uint64_t n,
                                              int tail, volatile uint32_t* flag, uint32_t seq,
                                              ull* done) {
  if (tail && blockIdx.x == 0 && threadIdx.x == 0)
    *(uint64_t*)(dst + n) = *(const uint64_t*)(src + n);
  for (uint64_t b = (uint64_t)blockIdx.x * 256 * kItems; b < n;
       b += (uint64_t)gridDim.x * 256 * kItems) {
    u32x4 v[kItems];
#pragma unroll
    for (int k = 0; k < kItems; k++) {
      const uint64_t i = b + 256 * k + threadIdx.x;
      if (i < n) v[k] = src[i];
    }
#pragma unroll
    for (int k = 0; k < kItems; k++) {
      const uint64_t i = b + 256 * k + threadIdx.x;
      if (i < n) __builtin_nontemporal_store(v[k], dst + i);
    }
  }
  if (!flag) return;
  __builtin_amdgcn_s_waitcnt(0);  // the wave's stores have reached the L2
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence_system();  // (writes the L2 back)
    if (gridDim.x == 1) {
      *flag = seq;
    } else if (atomicAdd(done, 1ull) == gridDim.x - 1) {
      *done = 0;
      *flag = seq;
    }
  }
}
// blocks up to which the copy raises the flag itself: 2 MB in four elements a thread
constexpr unsigned kCopyFlagBlocks = 128;
// (HIP takes less than 2^32 threads in a launch; the blocks stride)
constexpr uint64_t kCopyMaxBlocks = (1u << 24) - 1;
hipError_t copy_records(Context& c, void* dst, const void* src, size_t bytes) {
  const uint64_t n = bytes / 16;
  const int tail = bytes % 16 != 0;
  if (n > kCopyFlagBlocks * 1024ull) {
    SVO_LAUNCH(k_copy<1>, dim3((unsigned)std::min<uint64_t>((n + 255) / 256, kCopyMaxBlocks)),
               dim3(256), 0, c.stream, (u32x4_u*)dst, (const u32x4_u*)src, n, tail,
               (volatile uint32_t*)nullptr, 0u, (ull*)nullptr);
    SVO_TRY(hipGetLastError());
    return read_back(c, nullptr, 0);
  }
  SVO_TRY(ensure_hread(c, 256));
  const uint32_t seq = ++c.hread_seq;
  auto copy = [&](auto kernel, uint64_t per_block) {
    SVO_LAUNCH(kernel, dim3((unsigned)std::max<uint64_t>(1, (n + per_block - 1) / per_block)),
               dim3(256), 0, c.stream, (u32x4_u*)dst, (const u32x4_u*)src, n, tail,
               (volatile uint32_t*)c.hread, seq, c.counters.as<ull>() + kCtrCopyDone);
  };
  n <= kCopyFlagBlocks * 256ull ? copy(k_copy<1>, 256) : copy(k_copy<4>, 1024);
  SVO_TRY(hipGetLastError());
  t_syncs++;
  return wait_flag(c, seq);
}

static hipError_t ensure_scan_scratch(Context& c, uint64_t n, size_t elem) {
  return ensure(c.scan_scratch, scan_scratch_elems(n) * elem + 256);
}

hipError_t partition_job(Context& c, uint32_t jid, float unitlength, uint64_t gridsize,
                         uint64_t n_parts) {
  Job& J = c.jobs[jid];
  J.n_parts = n_parts;
  J.part_off.assign(n_parts, 0);
  J.part_cnt.assign(n_parts, 0);
  if (n_parts <= 1) {
    J.part_cnt[0] = J.n_tris;
    return hipSuccess;
  }
  // partitions are the 8^k aligned Morton cubes; K cubes per axis
  int k = 0;
  while ((1ull << (3 * k)) < n_parts) k++;
  const int K = 1 << k;
  if (K > 256) {
    set_error("more than 256 partitions per axis are not supported");
    return hipErrorInvalidValue;
  }
  const uint64_t side = gridsize / (uint64_t)K;
  // world box of cube c along any axis: [c*side*u, (c+1)*side*u] (partitioner.cpp:56-61)
  std::vector<float> lohi(2 * 256, 0.0f);
  for (int i = 0; i < K; i++) {
    lohi[i] = (float)(uint32_t)(i * side) * unitlength;
    lohi[256 + i] = (float)(uint32_t)((i + 1) * side) * unitlength;
  }
  const uint64_t n = J.n_tris;
  const int stride = J.payload ? 21 : 9;
  const bool masks = n_parts <= kPartMask && n > 0;
  const uint64_t ntiles = (n + kPartTile - 1) / kPartTile, ncnt = masks ? n_parts * ntiles : 0;
  // hit boxes (or masks) | cube bounds | tile counts, their places, the lists' first places
  const uint64_t b_box = (n * 8 + 255) & ~255ull;
  SVO_TRY(ensure(c.hitbox, b_box + 2 * 256 * sizeof(float) + ncnt * 12 + 8 * (kPartMask + 2) + 256));
  float* d_lo = (float*)((char*)c.hitbox.p + b_box);
  float* d_hi = d_lo + 256;
  SVO_TRY(upload_async(c, d_lo, lohi.data(), 2 * 256 * sizeof(float)));
  if (masks) {
    uint64_t* d_off = (uint64_t*)(d_hi + 256);
    uint64_t* d_start = d_off + ncnt;
    uint32_t* d_cnt = (uint32_t*)(d_start + kPartMask + 2);
    PartCubes cubes{};
    for (uint64_t j = 0; j < n_parts; j++) {
      uint32_t x[3];
      unmorton3(j, x[0], x[1], x[2]);
      for (int a = 0; a < 3; a++) cubes.on[a][x[a]] |= 1ull << j;
    }
    ktimer_begin(c, "part_hitbox");
    SVO_LAUNCH(k_part_masks, dim3((unsigned)ntiles), dim3(256), 0, c.stream, J.tris, stride, n,
               d_lo, d_hi, K, (uint32_t)n_parts, cubes, c.hitbox.as<uint64_t>(), d_cnt,
               (uint32_t)ntiles);
    ktimer_end(c);
    SVO_TRY(hipGetLastError());
    SVO_TRY(ensure_scan_scratch(c, ncnt, 8));
    SVO_TRY((scan_exclusive<uint64_t>(PartCountLoad{d_cnt},
                                      PartOffStore{d_off, d_start, ntiles, n_parts}, ncnt,
                                      c.scan_scratch.as<uint64_t>(), c.stream)));
    uint64_t start[kPartMask + 1];
    const ReadReq rq{start, d_start, (n_parts + 1) * 8};
    SVO_TRY(read_back(c, &rq, 1));
    if ((c.part_used + start[n_parts]) * 4 > c.part_lists.cap)
      SVO_TRY(ensure_keep(c.part_lists, (c.part_used + start[n_parts]) * 4 + 256, c.part_used * 4,
                          c.stream));
    SVO_LAUNCH(k_part_lists, dim3((unsigned)ntiles), dim3(256), 0, c.stream,
               c.hitbox.as<uint64_t>(), n, (uint32_t)n_parts, d_off, (uint32_t)ntiles,
               c.part_lists.as<uint32_t>() + c.part_used);
    SVO_TRY(hipGetLastError());
    for (uint64_t j = 0; j < n_parts; j++) {
      J.part_off[j] = c.part_used + start[j];
      J.part_cnt[j] = start[j + 1] - start[j];
    }
    c.part_used += start[n_parts];
    return hipSuccess;
  }
  if (n) {
    ktimer_begin(c, "part_hitbox");
    SVO_LAUNCH(k_part_hitbox, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c.stream,
                       J.tris, stride, n, d_lo, d_hi, K, c.hitbox.as<uint64_t>());
    ktimer_end(c);
    SVO_TRY(hipGetLastError());
  }
  // one order-preserving flag scan per partition; lists concatenated in partition order
  SVO_TRY(ensure_scan_scratch(c, n, 4));
  ull* d_tot = c.counters.as<ull>() + kCtrPartTotal;
  for (uint64_t j = 0; j < n_parts; j++) {
    // list capacity: grow if the previous partitions filled it
    if ((c.part_used + n) * 4 > c.part_lists.cap)
      SVO_TRY(ensure_keep(c.part_lists, (c.part_used + n) * 4 * 2 + 256, c.part_used * 4,
                          c.stream));
    SVO_TRY(fill_u64((uint64_t*)d_tot, 0, 1, c.stream));
    uint32_t cx, cy, cz;
    unmorton3(j, cx, cy, cz);
    if (n) {
      PartLoad ld{c.hitbox.as<uint64_t>(), cx, cy, cz};
      PartStore st{c.part_lists.as<uint32_t>() + c.part_used, d_tot};
      SVO_TRY((scan_exclusive<uint32_t>(ld, st, n, c.scan_scratch.as<uint32_t>(), c.stream)));
    }
    ull tot = 0;
    const ReadReq rq{&tot, d_tot, 8};
    SVO_TRY(read_back(c, &rq, 1));
    J.part_off[j] = c.part_used;
    J.part_cnt[j] = tot;
    c.part_used += tot;
  }
  return hipSuccess;
}

// The unit's brick-table segment covers its Morton range in bricks.
static uint64_t unit_bricks(const VoxUnit& u) {
  return (u.mend - (u.mstart & ~(uint64_t)(kBrickVox - 1)) + kBrickVox - 1) >> kBrickBits;
}

static void fill_params(const VoxUnit& h, const Context& c, VoxParams& P) {
  P.tris = h.tris;
  P.list = h.list;
  P.n = (uint32_t)h.n;
  P.stride = h.stride;
  P.mstart = h.mstart;
  P.bstart = h.mstart & ~(uint64_t)(kBrickVox - 1);
  uint32_t x, y, z;
  unmorton3(h.mstart, x, y, z);
  P.pmin[0] = (int)x;
  P.pmin[1] = (int)y;
  P.pmin[2] = (int)z;
  unmorton3(h.mend - 1, x, y, z);
  P.pmax[0] = (int)x;
  P.pmax[1] = (int)y;
  P.pmax[2] = (int)z;
  P.unit = h.unit;
  P.unit_div = 1.0f / h.unit;  // voxelizer.cpp:164, IEEE on the host as on the reference
  P.coord_limit = 4.0f * (float)h.gridsize * h.unit;
  // Along a column the voxels c that pass the reference's plane test lie, in exact
  // arithmetic, in [l, h] (the two zeros of (t + d1) and (t + d2)). Its FP32 evaluation
  // moves them by at most: t = n.p with |p| <= G u: 3 roundings of terms <= |n|_1 G u,
  // ~3.1e-7 G u; d1, d2 with |v0| <= coord_limit = 4 G u: ~1.7e-6 G u; so ~2e-6 G u, i.e.
  // 3.5e-6 G voxels along the column axis (|n_w| >= 1/sqrt(3)); p = fl(x u) adds ~3e-7 G.
  // This range is computed from float coefficients (KA, KB, alpha rounded to float, base
  // summed in float): below 1.8e-6 G voxels. The margin, 0.03 + 2.5e-5 G voxels, is over
  // four times the sum; the candidates are the integers in [l - margin, h + margin].
  P.slab_margin = 0.03 + 2.5e-5 * (double)h.gridsize;
  P.inv_unit = 1.0 / (double)h.unit;
  P.small_cols = c.tune.small_cols;
  P.direct_cols = c.tune.direct_cols;
  P.job = h.job;
  P.dense = 0;
  P.wide = 0;
  P.table_base = 0;
  P.grid8 = nullptr;
}

// What a pass marks is cleared by its later kernels. One that returns before they are all on the
// stream leaves marks behind: the next pass is to zero everything again.
struct MarksLeft {
  Context& c;
  bool cleared = false;
  ~MarksLeft() {
    if (!cleared) c.table_entries = c.cflags_zeroed = c.grid_zeroed = c.pool_cap = 0;
  }
};

hipError_t voxelize_units(Context& c, const std::vector<VoxUnit>& hu, bool batch,
                          uint64_t* nfilled) {
  *nfilled = 0;
  std::vector<VoxUnit> units;
  for (const VoxUnit& u : hu)
    if (u.n) units.push_back(u);  // main.cpp:330 skips empty partitions
  const uint32_t nu = (uint32_t)units.size();
  if (nu == 0) return hipSuccess;
  // unit table: VoxParams[nu] | ubase[nu+1] | 2 x tile_off[nu+1] | uvoff[nu+1]
  std::vector<VoxParams> P(nu);
  std::vector<uint64_t> ubase(nu + 1);
  // tiles before each unit: of the geometry-only units, of the payload ones
  std::vector<uint32_t> toff(2 * (nu + 1), 0);
  uint32_t* const toff_kind[2] = {&toff[0], &toff[nu + 1]};
  uint64_t ntab = 0, ntiles = 0, ntri = 0;
  // triangles per tile: kTileTris once the pass has about four tiles of them per wave of the
  // persistent grid, else fewer; up to 16 a wave, one tile for each wave
  uint32_t tt = (uint32_t)kTileTris;
  int small_cols = c.tune.small_cols;
  {
    uint64_t all = 0;
    for (uint32_t u = 0; u < nu; u++) all += units[u].n;
    const uint64_t blocks = (uint64_t)std::max(1, c.tune.tile_blocks);
    const uint64_t waves = kTileWaves * blocks;
    if (all <= 16 * waves) {
      tt = (uint32_t)std::max<uint64_t>(1, (all + waves - 1) / waves);
      // (a wave has few triangles: it keeps those of four times as many columns, which saves
      // their trip through the large tier's list; 20,480 triangles at 2048: 137 + 161 us in
      // the two tiers, 138 in this one)
      small_cols = (int)std::max<int64_t>(small_cols, std::min<int64_t>(4ll * small_cols, 1 << 16));
    } else
      tt = (uint32_t)std::min<uint64_t>(kTileTris, (all / (4 * waves) + 7) / 8 * 8);
    // A pass of one mesh with 12 or more tiles of 64 triangles per wave of the persistent grid
    // keeps triangles of up to 16 x small_cols columns in the small tier: its waves are busy, and
    // the large tier would list them and read them again. Soups in 8 partitions, so and with 1024
    // columns: 6M triangles at 4096 4.8 and 6.6 ms, 50M at 8192 40.5 and 46.4, 50M at 4096 (few such
    // triangles) 13.4 and 13.5. Batches keep their autotuned threshold.
    if (!batch && all >= 16 * blocks * 192)
      small_cols = std::max(small_cols, (int)std::min<int64_t>(16ll * small_cols, 1 << 16));
  }
  for (uint32_t u = 0; u < nu; u++) {
    // a unit smaller than a brick shares its brick with its neighbours: the brick stream
    // would hold that brick more than once
    const uint64_t G = units[u].gridsize;
    if (units[u].mend - units[u].mstart < std::min<uint64_t>(kBrickVox, G * G * G))
      c.bricks_ok = false;
    if (units[u].n > 0xFFFFFFF0ull) {
      set_error("partition holds more than 2^32 triangles");
      return hipErrorInvalidValue;
    }
    fill_params(units[u], c, P[u]);
    P[u].small_cols = small_cols;
    P[u].table_base = ntab;
    ubase[u] = ntab;
    ntab += unit_bricks(units[u]);
    const uint64_t tiles = (units[u].n + tt - 1) / tt;
    for (int k = 0; k < 2; k++)
      toff_kind[k][u + 1] = toff_kind[k][u] + ((units[u].stride == 21) == (k == 1) ? (uint32_t)tiles : 0u);
    ntiles += tiles;
    ntri += units[u].n;
  }
  ubase[nu] = ntab;
  if (ntab > 0xFFFFFFF0ull || ntiles > 0xFFFFFFF0ull || ntri > 0xFFFFFFF0ull) {
    set_error("voxelize pass too large for 32-bit brick, tile or triangle indices");
    return hipErrorInvalidValue;
  }
  // dense path: a cell per voxel of every unit (a byte, 4 bytes for payload units) when
  // that fits the HBM budget (no allocation pass needed); otherwise bricks get pool slots
  // from a touch pass
  std::vector<uint64_t> goff(nu + 1, 0);
  for (uint32_t u = 0; u < nu; u++)
    goff[u + 1] = goff[u] + ((ubase[u + 1] - ubase[u]) << kBrickBits) *
                                (units[u].stride == 21 ? 4 : 1);
  const uint64_t dense_bytes = goff[nu];
  bool dense = dense_bytes <= c.dense_limit;
  for (uint32_t u = 0; u < nu; u++)
    dense = dense && (units[u].stride == 9 || ubase[u + 1] - ubase[u] < kDensePayloadBricks);
  bool geometry_only = true;  // no unit carries payload records
  bool small_units = true;    // no unit spans more than 2^32 voxels
  for (uint32_t u = 0; u < nu; u++) {
    geometry_only = geometry_only && units[u].stride == 9;
    small_units = small_units && (ubase[u + 1] - ubase[u]) <= (1ull << (32 - kBrickBits));
  }
  // the table, the word flags, the dense grid and the byte pool are all-zero whenever no pass
  // is running, as far as the context's counts of them go
  const bool new_table = c.table_entries < ntab;
  const bool new_flags = dense && !geometry_only && c.cflags_zeroed < ntab * kBrickWords;
  // (allocated before the first fill: an allocation while the GPU works waits for it. What is
  // replaced counts as zero only once its fill is on the stream: a later allocation may fail)
  if (new_table) {
    c.table_entries = 0;
    SVO_TRY(ensure(c.table, ntab * 4));
  }
  if (new_flags) {
    c.cflags_zeroed = 0;
    SVO_TRY(ensure(c.cflags, ntab * kBrickWords));
  }
  uint64_t grid_fill = 0;
  if (dense) {
    if (c.grid_zeroed < dense_bytes) {
      // grown to at least twice its size (at most the dense limit), so that passes of
      // slowly growing spans (a server's batches) reallocate it a few times only
      uint64_t target = dense_bytes;
      c.grid_zeroed = 0;
      if (c.grid8.cap < dense_bytes) {
        target = std::max<uint64_t>(dense_bytes,
                                    std::min<uint64_t>(c.dense_limit, 2 * (uint64_t)c.grid8.cap));
        release(c.grid8);
        SVO_TRY(ensure(c.grid8, target));
      }
      grid_fill = target;
    }
    for (uint32_t u = 0; u < nu; u++) {
      P[u].dense = 1;
      P[u].wide = units[u].stride == 21 ? 1 : 0;
      P[u].grid8 = c.grid8.as<uint8_t>() + goff[u];
    }
  } else if (c.pool_cap == 0) {
    const uint64_t cap = std::max<uint64_t>(1024, ntri / 64);
    SVO_TRY(ensure(c.pool, cap * kBrickWords * 8));
    SVO_TRY(ensure(c.pool8, cap * kBrickVox));
    SVO_TRY(fill_u64(c.pool8.as<uint64_t>(), 0, cap * kBrickVox / 8, c.stream));
    c.pool_cap = cap;
  }
  const size_t szP = ((nu * sizeof(VoxParams)) + 255) & ~(size_t)255;
  const size_t szB = (((nu + 1) * 8) + 255) & ~(size_t)255;
  const size_t szT = ((toff.size() * 4) + 255) & ~(size_t)255;
  {
    const void* prev = c.unitdev.p;
    const size_t prev_cap = c.unitdev.cap;
    SVO_TRY(ensure(c.unitdev, szP + 2 * szB + szT));
    if (c.unitdev.p != prev || c.unitdev.cap != prev_cap) c.unit_img.clear();
  }
  VoxParams* d_units = (VoxParams*)c.unitdev.p;
  uint64_t* d_ubase = (uint64_t*)((char*)c.unitdev.p + szP);
  uint32_t* d_toff = (uint32_t*)((char*)c.unitdev.p + szP + szB);
  uint64_t* d_uvoff = (uint64_t*)((char*)c.unitdev.p + szP + szB + szT);
  {  // one upload for the unit table (same layout as on the device)
    std::vector<uint8_t> img(szP + szB + szT, 0);
    memcpy(img.data(), P.data(), nu * sizeof(VoxParams));
    memcpy(img.data() + szP, ubase.data(), (nu + 1) * 8);
    memcpy(img.data() + szP + szB, toff.data(), toff.size() * 4);
    // a pass over the same units as the last one (the same mesh again) finds them there
    if (img != c.unit_img) {
      SVO_TRY(upload_async(c, d_units, img.data(), img.size()));
      c.unit_img.swap(img);
    }
  }

  // dense passes write their bricks straight into the brick stream (every flagged brick
  // holds voxels): room for all of the pass's bricks after the nb0 already there
  const uint64_t s0 = c.n_vox;
  const uint64_t nb0 = c.n_bricks;
  if (dense) {
    SVO_TRY(ensure_keep(c.bwords, (nb0 + ntab) * kBrickWords * 8, nb0 * kBrickWords * 8,
                        c.stream));
    SVO_TRY(ensure_keep(c.bcode, (nb0 + ntab) * 8, nb0 * 8, c.stream));
    SVO_TRY(ensure_keep(c.bvoff, (nb0 + ntab) * 8, nb0 * 8, c.stream));
    SVO_TRY(ensure_keep(c.bshape, (nb0 + ntab) * 4, nb0 * 4, c.stream));
  }
  ull* pool_words = dense ? c.bwords.as<ull>() + nb0 * kBrickWords : c.pool.as<ull>();
  // (one allocation: a large one the runtime has to map takes 250 us)
  const uint32_t walk_cap = (uint32_t)std::min<uint64_t>(ntri, c.tune.large_walks);
  const size_t b_tri = ((size_t)ntri * 4 + 255) & ~(size_t)255;
  const size_t b_jobs = ((size_t)c.tune.large_jobs * sizeof(uint2) + 255) & ~(size_t)255;
  SVO_TRY(ensure(c.large, 3 * b_tri + b_jobs + (size_t)walk_cap * kLargeQuads * sizeof(uint4)));
  SVO_TRY(ensure(c.occ_list, ntab * 4));
  SVO_TRY(ensure_scan_scratch(c, ntab, 8));
  if (new_table) {
    SVO_TRY(fill_u32(c.table.as<uint32_t>(), 0, ntab, c.stream));
    c.table_entries = ntab;
  }
  if (grid_fill) {
    SVO_TRY(fill_u64(c.grid8.as<uint64_t>(), 0, grid_fill / 8, c.stream));
    c.grid_zeroed = grid_fill;
  }
  if (new_flags) {
    SVO_TRY(fill_u64(c.cflags.as<uint64_t>(), 0, ntab * kBrickWords / 8, c.stream));
    c.cflags_zeroed = ntab * kBrickWords;
  }
  ull* ctr = c.counters.as<ull>();
  ull hc[kNumCounters];
  const unsigned large_grid = (unsigned)c.tune.large_blocks;
  auto brick_grid = [&](uint64_t bricks) {
    return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((bricks * kWave + 255) / 256, 8192));
  };
  auto args = [&]() {
    ActArgs A;
    A.table = c.table.as<uint32_t>();
    A.cflags = c.cflags.as<uint8_t>();
    A.pool8 = c.pool8.as<uint8_t>();
    A.pool = pool_words;
    A.wprefix = c.wprefix.as<uint32_t>();
    A.winner = c.winner.as<uint32_t>();
    A.ctr = ctr;
    A.pool_cap = c.pool_cap;
    return A;
  };
  char* const lb = (char*)c.large.p;
  const LargeList large{(uint32_t*)lb,
                        (uint32_t*)(lb + b_tri),
                        (uint32_t*)(lb + 2 * b_tri),
                        (uint2*)(lb + 3 * b_tri),
                        (uint4*)(lb + 3 * b_tri + b_jobs),
                        c.tune.large_jobs,
                        walk_cap};
  const uint64_t runs_kind[2] = {(toff_kind[0][nu] + (uint64_t)kTileRun - 1) / kTileRun,
                                 (toff_kind[1][nu] + (uint64_t)kTileRun - 1) / kTileRun};
  const uint64_t runs = runs_kind[0] + runs_kind[1];
  const uint64_t payload_runs = ((runs_kind[1] << 32) + runs - 1) / runs;
  auto tile_pass = [&](auto tag, const char* name, ull* queue, int collect, int skip) {
    using Act = decltype(tag);
    const unsigned tile_grid = (unsigned)std::min<uint64_t>(
        runs * kTileRun / kTileWaves,
        std::max<uint64_t>(
            1, (uint64_t)std::max(1, c.tune.tile_blocks) * kTileBlocks<Act> / kTileBlocks<TouchAction>));
    ktimer_begin(c, name);
    SVO_LAUNCH((k_vox_tile<Act>), dim3(tile_grid), dim3(kTile), 0, c.stream, d_units, nu,
                       d_toff, payload_runs, args(), queue, large, tt, collect, skip);
    ktimer_end(c);
    return hipGetLastError();
  };
  auto large_pass = [&](auto tag, const char* name, int skip) {
    using Act = decltype(tag);
    ktimer_begin(c, name);
    SVO_LAUNCH((k_vox_large<Act>), dim3(large_grid), dim3(256), 0, c.stream, d_units,
                       args(), large, skip);
    ktimer_end(c);
    return hipGetLastError();
  };
  // single-pass scans, each with its own zeroed status words: flagged bricks, brick counts (the last only while its packed prefixes stay below 2^62:
  // at most bricks * (2^kNonEmptyShift + 4096))
  const uint64_t w_occ = scan_single_words(ntab);
  ull* st_occ = nullptr;
  ull* st_bc = nullptr;
  ull* queues = nullptr;  // 3 x kQueueWords: the tile queues of the mark/touch, second and winner passes
  auto occ_scan = [&]() {
    if (dense)
      return scan_single<uint32_t>(
          OccLoad{c.table.as<uint32_t>()},
          OccStoreDense{c.occ_list.as<uint32_t>(), c.table.as<uint32_t>(), ctr}, ntab, st_occ,
          ctr + kCtrError, c.stream);
    return scan_single<uint32_t>(
        OccLoad{c.table.as<uint32_t>()},
        OccStore{c.occ_list.as<uint32_t>(), c.table.as<uint32_t>(), ctr}, ntab, st_occ,
        ctr + kCtrError, c.stream);
  };

  // ---- phase A: mark, compact counts; one synchronization at its end
  MarksLeft marks{c};
  std::vector<uint64_t> uvoff(nu + 1);
  for (int attempt = 0;; attempt++) {
    const uint64_t bc_bound = dense ? ntab : std::min<uint64_t>(ntab, c.pool_cap);
    const bool bc_single = bc_bound <= (3ull << 20);
    const uint64_t w_bc = bc_single ? scan_single_words(bc_bound) : 0;
    SVO_TRY(ensure(c.bcount, bc_bound * 8 + 8));
    // status words of the scans, then the tile queues of the three tile passes
    SVO_TRY(ensure(c.scan_status, (w_occ + w_bc + 3 * kQueueWords) * 8));
    st_occ = c.scan_status.as<ull>();
    st_bc = st_occ + w_occ;
    queues = st_bc + w_bc;
    // one unit: the scan of the brick counts reads back (not in a graph, whose arguments stay)
    uint64_t* host_ctr = nullptr;
    volatile uint32_t* host_flag = nullptr;
    uint64_t seq = 0;
    if (nu == 1 && dense && bc_single && !c.graphs) {
      SVO_TRY(ensure_hread(c, 256 + kNumCounters * sizeof(ull)));
      host_ctr = (uint64_t*)((char*)c.hread + 256);
      host_flag = (volatile uint32_t*)c.hread;
      seq = ++c.hread_seq;
    }
    // the pass's kernels up to its read-back: one graph segment
    SVO_TRY(run_segment(c, [&]() -> hipError_t {
      {  // pass counters, scan status words and tile queues
        const uint64_t ns = w_occ + w_bc + 3 * kQueueWords;
        const uint64_t nc = c.clear_counters ? (uint64_t)kCtrStamp : (uint64_t)kCtrPassClear;
        SVO_LAUNCH(k_pass_begin, dim3(fill_grid(nc + ns)), dim3(256), 0, c.stream,
                   (uint64_t*)ctr, nc, c.scan_status.as<uint64_t>(), ns,
                   (uint64_t*)(ctr + kCtrStamp));
        SVO_TRY(hipGetLastError());
      }
      // first pass: dense units mark directly, touch units flag their bricks; both collect
      // the large triangles
      // (units of both kinds: the payload marks' lines in LDS would leave room for half the waves
      // of the others; apart, in two launches, 64 mixed meshes took 1.15 + 1.89 ms against 2.74)
      auto mark_dense = [&](auto small) -> hipError_t {
        constexpr bool kSmall = decltype(small)::value;
        if (geometry_only)
          SVO_TRY(tile_pass(MarkDenseT<false, kSmall>{}, "vox_small_mark", queues, 1, 0));
        else if (!toff_kind[0][nu])
          SVO_TRY(tile_pass(MarkGather<16, kSmall>{}, "vox_small_mark", queues, 1, 0));
        else
          SVO_TRY(tile_pass(MarkDenseT<true, kSmall>{}, "vox_small_mark", queues, 1, 0));
        if (geometry_only) return large_pass(MarkDenseT<false, kSmall>{}, "vox_large_mark", 0);
        return large_pass(MarkDenseT<true, kSmall>{}, "vox_large_mark", 0);
      };
      if (dense) {
        SVO_TRY(small_units ? mark_dense(std::true_type{}) : mark_dense(std::false_type{}));
        // list the flagged bricks in Morton order, with their flagged quarters
        SVO_TRY(occ_scan());
      } else {
        SVO_TRY(tile_pass(TouchAction{}, "vox_small_touch", queues, 1, 0));
        SVO_TRY(large_pass(TouchAction{}, "vox_large_touch", 0));
        SVO_TRY(occ_scan());
        // mark pass: byte stores into the slots
        SVO_TRY(tile_pass(MarkPoolAction{}, "vox_small_mark", queues + kQueueWords, 0, 0));
        SVO_TRY(large_pass(MarkPoolAction{}, "vox_large_mark", 0));
      }
      // per-brick voxel counts (bytes packed to bits, bytes cleared) and their offsets
      ktimer_begin(c, "brick_count");
      SVO_LAUNCH(k_brick_count, dim3(brick_grid(bc_bound)), dim3(256), 0, c.stream,
                         c.occ_list.as<uint32_t>(), ctr, bc_bound, d_units, d_ubase, nu,
                         c.pool8.as<uint8_t>(), c.cflags.as<uint8_t>(), pool_words,
                         c.bcount.as<uint64_t>(), dense ? c.bcode.as<uint64_t>() + nb0 : (uint64_t*)nullptr,
                         dense ? c.bshape.as<uint32_t>() + nb0 : (uint32_t*)nullptr,
                         dense ? c.table.as<uint32_t>() : (uint32_t*)nullptr);
      ktimer_end(c);
      SVO_TRY(hipGetLastError());
      if (bc_single && dense)
        SVO_TRY((scan_single<uint64_t>(
            ArrayLoad<uint64_t>{c.bcount.as<uint64_t>()},
            BrickOffStore{c.bcount.as<uint64_t>(), ctr, c.bvoff.as<uint64_t>() + nb0, s0,
                          host_ctr, host_flag, seq},
            bc_bound, st_bc, ctr + kCtrError, c.stream, ctr + kCtrNumOcc)));
      else if (bc_single)
        SVO_TRY((scan_single<uint64_t>(
            ArrayLoad<uint64_t>{c.bcount.as<uint64_t>()},
            CountStore{c.bcount.as<uint64_t>(), ctr + kCtrNumVox}, bc_bound,
            st_bc, ctr + kCtrError, c.stream, ctr + kCtrNumOcc)));
      else if (dense)
        SVO_TRY((scan_exclusive<uint64_t>(
            ArrayLoad<uint64_t>{c.bcount.as<uint64_t>()},
            BrickOffStore{c.bcount.as<uint64_t>(), ctr, c.bvoff.as<uint64_t>() + nb0, s0, nullptr,
                          nullptr, 0},
            bc_bound, c.scan_scratch.as<uint64_t>(), c.stream, ctr + kCtrNumOcc)));
      else
        SVO_TRY((scan_exclusive<uint64_t>(
            ArrayLoad<uint64_t>{c.bcount.as<uint64_t>()},
            CountStore{c.bcount.as<uint64_t>(), ctr + kCtrNumVox}, bc_bound,
            c.scan_scratch.as<uint64_t>(), c.stream, ctr + kCtrNumOcc)));
      if (nu > 1) {
        SVO_LAUNCH(k_unit_voxels, dim3((nu + 256) / 256), dim3(256), 0, c.stream,
                   c.occ_list.as<uint32_t>(), dense ? kOccMask : 0xFFFFFFFFu, ctr, d_ubase, nu,
                   c.bcount.as<uint64_t>(), d_uvoff);
        SVO_TRY(hipGetLastError());
      }
      return hipSuccess;
    }));
    if (nu == 1) {
      // one unit: its voxels are the whole pass, [0, voxel count)
      if (host_ctr) {
        t_syncs++;
        SVO_TRY(wait_flag(c, (uint32_t)seq));
        c.stamp_read = ((volatile uint64_t*)c.hread)[1];
        memcpy(hc, host_ctr, sizeof(hc));
      } else {
        const ReadReq rq = {hc, c.counters.p, kNumCounters * sizeof(ull)};
        SVO_TRY(read_back(c, &rq, 1));
      }
      uvoff[0] = 0;
      uvoff[1] = hc[kCtrNumVox] & kVoxMask;
    } else {
      const ReadReq rq[2] = {{uvoff.data(), d_uvoff, (nu + 1) * 8},
                             {hc, c.counters.p, kNumCounters * sizeof(ull)}};
      SVO_TRY(read_back(c, rq, 2));
    }
    c.clear_counters = false;
    if (attempt == 0) c.stamp_pass = hc[kCtrStamp];
    ktimer_flush(c);
    if (dense || (!hc[kCtrOverflow] && hc[kCtrNumOcc] <= c.pool_cap)) break;
    // pool too small for the flagged bricks: clear everything, grow, redo
    const uint64_t want = std::max<uint64_t>(c.pool_cap * 2, hc[kCtrNumOcc] + 1024);
    if (attempt > 8 || want > (1ull << 26)) {
      set_error("brick pool could not be sized");
      return hipErrorOutOfMemory;
    }
    SVO_TRY(fill_u32(c.table.as<uint32_t>(), 0, ntab, c.stream));
    release(c.pool);
    release(c.pool8);
    SVO_TRY(ensure(c.pool, want * kBrickWords * 8));
    SVO_TRY(ensure(c.pool8, want * kBrickVox));
    SVO_TRY(fill_u64(c.pool8.as<uint64_t>(), 0, want * kBrickVox / 8, c.stream));
    c.pool_cap = want;
    pool_words = c.pool.as<ull>();
  }
  const uint64_t n_occ = hc[kCtrNumOcc];
  const uint64_t nvox = hc[kCtrNumVox] & kVoxMask;
  const uint64_t n_nonempty = hc[kCtrNumVox] >> kNonEmptyShift;
  const uint64_t n_large = hc[kCtrLargeCount];
  if (c.n_vox + nvox >= (1ull << 40)) {
    set_error("voxel stream too long");
    return hipErrorInvalidValue;
  }

  // ---- job layout: voxel and data-record ranges
  const bool any_payload = !geometry_only;
  if (batch) {
    // the passes of a batch take its jobs' partitions in job order: a job's range starts
    // at its first voxel and grows with every pass that holds its partitions (jobs start
    // with voff = ~0, nvox = 0; the caller places jobs without voxels afterwards)
    for (uint32_t u = 0; u < nu; u++) {
      Job& J = c.jobs[units[u].job];
      const uint64_t k = uvoff[u + 1] - uvoff[u];
      if (J.voff == ~0ull && k) J.voff = s0 + uvoff[u];
      J.nvox += k;
    }
  } else {
    Job& J = c.jobs[0];
    J.voff = 0;
    J.nvox = s0 + nvox;
  }
  // data ranges: a job's records start after the complete ranges of the jobs before it
  // (jobs after the last one of this pass have no records yet, their bases move later)
  uint64_t n_records = 0;
  for (size_t j = 0; j < c.jobs.size(); j++) {
    Job& J = c.jobs[j];
    J.dbase = n_records;
    J.n_data = J.payload ? 1 + J.nvox : 2;
    n_records += J.n_data;
  }
  std::vector<JobDev> jd(c.jobs.size());
  for (size_t j = 0; j < c.jobs.size(); j++) {
    const Job& J = c.jobs[j];
    JobDev& d = jd[j];
    memset(&d, 0, sizeof(d));
    d.tris = J.tris;
    d.unit_div = 1.0f / J.unit_vox;
    d.color_mode = J.color_mode;
    d.payload = J.payload;
    d.gridsize = J.gridsize;
    int D = 0;
    while ((1ull << D) < J.gridsize) D++;
    d.depth = D;
    d.voff = J.voff == ~0ull ? 0 : J.voff;
    d.nvox = J.nvox;
    d.dbase = J.dbase;
  }
  c.jobdev_img.clear();  // (before what it tells of may be replaced)
  SVO_TRY(ensure(c.jobdev, jd.size() * sizeof(JobDev)));
  if (batch) {
    SVO_TRY(upload_async(c, c.jobdev.p, jd.data(), jd.size() * sizeof(JobDev)));
    c.jobdev_img = jd;
  } else if (any_payload && !dense) {  // (else the build is its first reader, and writes it)
    SVO_LAUNCH(k_put_job, dim3(1), dim3(1), 0, c.stream, c.jobdev.as<JobDev>(), jd[0]);
    SVO_TRY(hipGetLastError());
  }

  JobDev job0;  // a single job's descriptor, for the kernels' arguments
  memset(&job0, 0, sizeof(job0));
  if (!batch) job0 = jd[0];

  // ---- phase B: emit sorted codes, payload, clear; no synchronization
  if (n_occ) {
    // dense passes resolve payload winners while marking (emitted with the codes); the
    // touched-brick path finds them with a second walk
    const bool winner_walk = any_payload && !dense;
    if (any_payload && nvox > 0xFFFFFFF0ull) {
      set_error("voxelize pass holds more than 2^32 voxels");
      return hipErrorInvalidValue;
    }
    if (winner_walk) SVO_TRY(ensure(c.wprefix, n_occ * kBrickWords * 4));
    if (winner_walk) SVO_TRY(ensure(c.winner, nvox * 4));
    // dense and geometry-only passes write no codes: the build reads the brick stream, and
    // ensure_codes writes the codes for readers that want them
    const bool codes_now = winner_walk;
    if (codes_now) SVO_TRY(ensure_keep(c.codes, (s0 + nvox) * 8, s0 * 8, c.stream));
    if (!dense) {
      SVO_TRY(ensure_keep(c.bwords, (nb0 + n_occ) * kBrickWords * 8, nb0 * kBrickWords * 8,
                          c.stream));
      SVO_TRY(ensure_keep(c.bcode, (nb0 + n_occ) * 8, nb0 * 8, c.stream));
      SVO_TRY(ensure_keep(c.bvoff, (nb0 + n_occ) * 8, nb0 * 8, c.stream));
      SVO_TRY(ensure_keep(c.bshape, (nb0 + n_occ) * 4, nb0 * 4, c.stream));
    }
    // the payload units' voxel ranges, for the records kernel: prange (n_pu + 1) |
    // pstart (n_pu) | punit (n_pu, as u64)
    uint64_t n_pv = 0;
    uint32_t n_pu = 0;
    const uint64_t* d_prange = nullptr;
    const uint64_t* d_pstart = nullptr;
    const uint32_t* d_punit = nullptr;
    if (any_payload) {
      // records: each job's first record is its null record
      const uint64_t keep = batch ? c.records.cap : (1 + s0) * 32;
      SVO_TRY(ensure_keep(c.records, n_records * 32, keep, c.stream));
    }
    if (winner_walk) {
      std::vector<uint64_t> pr(1, 0), ps, pu;
      for (uint32_t u = 0; u < nu; u++) {
        const uint64_t cnt = uvoff[u + 1] - uvoff[u];
        if (units[u].stride != 21 || cnt == 0) continue;
        pr.push_back(pr.back() + cnt);
        ps.push_back(uvoff[u]);
        pu.push_back(u);
      }
      n_pu = (uint32_t)ps.size();
      n_pv = pr.back();
      if (n_pv) {
        std::vector<uint64_t> img(pr);
        img.insert(img.end(), ps.begin(), ps.end());
        std::vector<uint32_t> pu32(pu.begin(), pu.end());
        const size_t b64 = img.size() * 8;
        SVO_TRY(ensure(c.payload_map, b64 + pu32.size() * 4));
        SVO_TRY(upload_async(c, c.payload_map.p, img.data(), b64));
        SVO_TRY(upload_async(c, (char*)c.payload_map.p + b64, pu32.data(), pu32.size() * 4));
        d_prange = c.payload_map.as<uint64_t>();
        d_pstart = d_prange + n_pu + 1;
        d_punit = (const uint32_t*)((const char*)c.payload_map.p + b64);
      }
    }
    // the pass's remaining kernels: one graph segment
    SVO_TRY(run_segment(c, [&]() -> hipError_t {
      // a dense pass has its brick stream entries already (k_brick_count)
      if (!dense) {
        ktimer_begin(c, "brick_emit");
        SVO_LAUNCH(codes_now ? k_brick_emit<true> : k_brick_emit<false>,
                   dim3(brick_grid(n_occ)), dim3(256), 0, c.stream,
                   c.occ_list.as<uint32_t>(), ctr, d_units, d_ubase, nu, pool_words,
                   c.bcount.as<uint64_t>(), c.codes.as<uint64_t>() + s0,
                   winner_walk ? c.wprefix.as<uint32_t>() : (uint32_t*)nullptr, s0,
                   c.bwords.as<uint64_t>() + nb0 * kBrickWords, c.bcode.as<uint64_t>() + nb0,
                   c.bvoff.as<uint64_t>() + nb0, c.bshape.as<uint32_t>() + nb0);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      } else if (any_payload) {
        ktimer_begin(c, "payload_records");
        SVO_LAUNCH(n_occ > kStagePayload ? k_payload_bricks<true> : k_payload_bricks<false>,
                   dim3(brick_grid(n_occ)), dim3(256), 0, c.stream,
                   c.occ_list.as<uint32_t>(), (const ull*)(ctr + kCtrNumOcc),
                   (const VoxParams*)d_units, d_ubase, nu, (const ull*)pool_words,
                   c.bcount.as<uint64_t>(),
                   batch ? (const JobDev*)c.jobdev.p : (const JobDev*)nullptr, job0, s0,
                   c.records.as<float>(), ctr);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }
      if (winner_walk) {
        {
          SVO_TRY(fill_u32(c.winner.as<uint32_t>(), 0xFFFFFFFFu, nvox, c.stream));
          SVO_TRY(tile_pass(WinnerAction{}, "vox_small_winner", queues + 2 * kQueueWords, 0,
                            kSkipBinary));
          if (n_large) SVO_TRY(large_pass(WinnerAction{}, "vox_large_winner", kSkipBinary));
        }
        if (n_pv) {
          ktimer_begin(c, "payload_records");
          const uint64_t part = 1ull << 31;  // (a launch takes less than 2^32 threads)
          for (uint64_t first = 0; first < n_pv; first += part)
            SVO_LAUNCH(k_payload_records,
                       dim3((unsigned)((std::min(n_pv - first, part) + 255) / 256)), dim3(256), 0,
                       c.stream, c.jobdev.as<JobDev>(), (const VoxParams*)d_units, d_prange,
                       d_pstart, d_punit, n_pu, c.codes.as<uint64_t>(), s0,
                       c.winner.as<uint32_t>(), first, n_pv, c.records.as<float>(), ctr);
          ktimer_end(c);
          SVO_TRY(hipGetLastError());
        }
      }
      if (!dense) {  // (dense passes cleared their table entries in k_brick_count)
        ktimer_begin(c, "brick_clear");
        SVO_LAUNCH(k_brick_clear,
                   dim3((unsigned)std::min<uint64_t>((n_occ + 255) / 256, 4096)),
                   dim3(256), 0, c.stream, c.occ_list.as<uint32_t>(), ctr,
                   c.table.as<uint32_t>());
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }
      return hipSuccess;
    }));
    c.n_bricks = nb0 + n_nonempty;
    bool any_binary = false;
    for (uint32_t u = 0; u < nu; u++) any_binary |= units[u].stride == 9;
    if (!codes_now || any_binary) c.codes_lazy = true;
  }
  marks.cleared = true;
  c.n_vox = s0 + nvox;
  *nfilled = nvox;
  return hipSuccess;
}

hipError_t ensure_codes(Context& c) {
  if (!c.codes_lazy) return hipSuccess;
  SVO_TRY(ensure_keep(c.codes, std::max<uint64_t>(c.n_vox, 1) * 8, c.n_vox * 8, c.stream));
  // every brick again (rewriting codes already there with the same values)
  if (c.n_bricks) {
    const unsigned grid =
        (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((c.n_bricks * kWave + 255) / 256, 8192));
    SVO_LAUNCH(k_bricks_codes, dim3(grid), dim3(256), 0, c.stream,
                       c.bwords.as<uint64_t>(), c.bcode.as<uint64_t>(), c.bvoff.as<uint64_t>(),
                       c.n_bricks, c.codes.as<uint64_t>());
    SVO_TRY(hipGetLastError());
  }
  c.codes_lazy = false;
  return hipSuccess;
}

}  // namespace svo
