// Bottom-up SVO build from the sorted unique Morton codes, replacing the streaming
// OctreeBuilder (OctreeBuilder.cpp:34-168, OctreeBuilder.h:50-91) with level passes.
//
// Node order. The streaming builder writes, each time a node completes, its non-null
// children consecutively in child order (groupNodes, OctreeBuilder.cpp:58-79), and the
// root last (:42). Nodes complete in post-order, so the children written for the whole
// subtree of a node P occupy one contiguous range of size(P) - 1 records (size = nodes in
// the subtree, P included), laid out as: the ranges of P's children subtrees in child
// order, then P's own children. Hence, with start(P) the first record of P's range:
//   start(root)        = 0
//   start(child r)     = start(P) + sum_{r' < r} (size(child r') - 1)
//   children_base(P)   = start(P) + size(P) - 1 - popcount(mask(P))
//   position(child r)  = children_base(P) + r,   root at n_nodes - 1 = size(root) - 1.
// Bottom-up passes build each level (parent = code >> 3, child mask, subtree size) with
// one scan per level; top-down passes give every node its start and position and write
// its 24-byte record (Node.h:16-18, octree_io.h:62-66), one thread per node, level by
// level from the root.
#include <algorithm>
#include <cstring>
#include <vector>

#include "svo_device.h"
#include "svo_internal.h"
#include "svo_scan.h"

namespace svo {

typedef unsigned long long ull;

// child offsets of a node with child mask m: rank of each present child, -1 otherwise
__device__ __forceinline__ uint64_t offsets_of(uint32_t m) {
  uint64_t o = 0;
  uint32_t r = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const uint64_t byte = (m >> k & 1u) ? (uint64_t)(r++) : 0xFFull;
    o |= byte << (8 * k);
  }
  return o;
}

// A node's data index and children_base as written: moved by the job's placement in a
// larger node stream (zero but for a streamed partition), data indices only past the
// leading records (the null record, and the white record of geometry-only leaves).
__device__ __forceinline__ uint64_t placed_data(const JobDev& J, uint64_t data) {
  return data >= (J.payload ? 1ull : 2ull) ? data + J.data_add : data;
}

__device__ __forceinline__ void put_node(const JobDev& J, uint64_t* nodes, uint64_t pos,
                                         uint64_t data, uint64_t cb, uint64_t offs) {
  uint64_t* r = nodes + 3 * pos;
  r[0] = placed_data(J, data);
  r[1] = offs != ~0ull ? cb + J.cb_add : cb;
  r[2] = offs;
}

// Jobs. The voxel stream may hold several jobs (meshes), job-major, each tagged in the
// code bits selected by tag_mask (0 for a single job). Levels are indexed by height above
// the leaves, h = 0 (leaves) .. H: a node of job j at height h has depth D_j - h, so the
// root of job j is its only node at height D_j, and one pass per height serves all jobs.
// parent(c) keeps the tag and drops the lowest Morton digit.
struct Tags {
  uint64_t tag_mask;  // bits of the job index (shifted by kJobShift)
  __device__ __forceinline__ uint32_t job(uint64_t c) const {
    return (uint32_t)((c & tag_mask) >> kJobShift);
  }
  __device__ __forceinline__ uint64_t parent(uint64_t c) const {
    return (c & tag_mask) | ((c & ~tag_mask) >> 3);
  }
};

// Level arrays live in arenas (code, size, mask, first child, start, parent index),
// height h >= 1 at element offset off[h]; the per-height counts n[h] and offsets are kept
// on the device so that the passes run back to back without host round trips. Height 0
// (the leaves) is the voxel code stream itself, with implicit size 1.
struct LevelMeta {
  unsigned long long* n;    // n[h], h = 0..H
  unsigned long long* off;  // off[h], h = 1..H+1
  unsigned long long* flag; // [0] arena overflow, [1] node range error, [2] total nodes
};

struct Arena {
  uint64_t* code;
  uint64_t* size;
  uint8_t* mask;
  uint32_t* first;
  uint64_t* start;
  uint32_t* pidx;  // index of the node's parent within the parent level
  uint64_t cap;
  // -levels only (nullptr otherwise): internal nodes in the subtree (the node included),
  // the node's averaged colour and normal, and the first data-record rank of its subtree
  uint64_t* isize;
  float* cache;  // 6 floats per node
  uint64_t* pstart;
  // sum of (size - 1) over the node's preceding siblings: its start is its parent's start
  // plus this (written by the bottom-up pass that creates the parent)
  uint64_t* sib;
};

// -levels data record of an internal node (OctreeBuilder.cpp:82-99): the caches of its
// children summed in child order (a null child adds zeros, which change no sum that started
// from +0), divided by the number of non-null children, the normal then normalized
// (glm::normalize = v * (1 / sqrt(dot))). Children i .. i + cnt - 1 of the child level; leaf
// caches are the voxels' own records (payload) or zero (geometry-only builds: leaves carry no
// data).
//
// Bound by latency: every child's loads are issued before the first sum. One child after the
// other, the levels of 487,600 payload voxels took 128 us, 116 now.
__device__ __forceinline__ void average_children(const Arena& A, uint64_t coff, bool leaf,
                                                 const float* __restrict__ leaf_rec,
                                                 int payload, uint64_t i, uint32_t cnt,
                                                 uint64_t& isz, float* out) {
  float2 v[8][3];
  uint64_t inner[8];
  const bool any = !leaf || payload;
  // (8-byte aligned: 32-byte records from their third float on, 24-byte caches)
  const float2* row = (const float2*)(leaf ? leaf_rec + i * 8 + 2 : A.cache + (coff + i) * 6);
  const uint32_t step = leaf ? 4 : 3;
#pragma unroll
  for (uint32_t r = 0; r < 8; r++) {
    const bool live = r < cnt;
#pragma unroll
    for (int q = 0; q < 3; q++) v[r][q] = live && any ? row[r * step + q] : make_float2(0.0f, 0.0f);
    inner[r] = live && !leaf ? A.isize[coff + i + r] : 0ull;
  }
  float s[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  isz = 1;
#pragma unroll
  for (int r = 0; r < 8; r++) {
    isz += inner[r];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      s[2 * q] = s[2 * q] + v[r][q].x;
      s[2 * q + 1] = s[2 * q + 1] + v[r][q].y;
    }
  }
  const float notnull = (float)cnt;
  out[0] = s[0] / notnull;
  out[1] = s[1] / notnull;
  out[2] = s[2] / notnull;
  const float t0 = s[3] / notnull, t1 = s[4] / notnull, t2 = s[5] / notnull;
  const float inv = 1.0f / sqrtf((t0 * t0 + t1 * t1) + t2 * t2);
  out[3] = t0 * inv;
  out[4] = t1 * inv;
  out[5] = t2 * inv;
}

// Parent height h+1 from child height h: head = first child of a parent group; a job's
// root (height D_j) has no parent.
struct HeadLoad {
  Arena A;
  LevelMeta M;
  Tags T;
  const JobDev* jobs;
  const uint64_t* leaves;
  int h;
  int pad = 0;  // no padding bytes: launch logs compare arguments byte by byte
  __device__ uint32_t operator()(uint64_t i) const {
    // an overflowed child level is not read (its tail lies beyond the arena)
    if (h > 0 && M.off[h] + M.n[h] > A.cap) return 0u;
    const uint64_t* code = (h == 0) ? leaves : A.code + M.off[h];
    const uint64_t c = code[i];
    const uint64_t cp = i ? code[i - 1] : 0ull;
    // one job (no tags): its depth does not wait for the code
    const int depth = T.tag_mask ? jobs[T.job(c)].depth : jobs[0].depth;
    if (depth <= h) return 0u;
    return (i == 0 || T.parent(c) != T.parent(cp)) ? 1u : 0u;
  }
};
struct ParentStore {
  Arena A;
  LevelMeta M;
  Tags T;
  const JobDev* jobs;
  const uint64_t* leaves;
  uint32_t* leaf_parent;  // height 0 only: parent index of every leaf
  unsigned long long* root_size;  // per job: nodes in its tree
  unsigned long long* root_isize; // per job: internal nodes in its tree (-levels)
  const float* leaf_rec;          // -levels, payload: voxel i's record at leaf_rec + 8 i
  int h;
  int pad = 0;  // no padding bytes: launch logs compare arguments byte by byte
  __device__ void operator()(uint64_t i, uint32_t ex, uint32_t head, bool) const {
    const bool leaf = (h == 0);
    if (leaf)
      leaf_parent[i] = ex + head - 1;
    else if (M.off[h] + i < A.cap)
      A.pidx[M.off[h] + i] = ex + head - 1;
    if (!leaf && M.off[h] + M.n[h] > A.cap) {
      M.flag[0] = 1;
      return;
    }
    const uint64_t* code = leaf ? leaves : A.code + M.off[h];
    const uint64_t* csize = leaf ? nullptr : A.size + M.off[h];
    const uint64_t nch = M.n[h];
    const uint64_t base = M.off[h + 1];
    if (head) {
      if (base + ex >= A.cap) {
        M.flag[0] = 1;
      } else {
        // the (at most 8) children follow the head: all their loads issued at once
        uint64_t cj[8], sj[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
          cj[k] = (i + k < nch) ? code[i + k] : ~0ull;  // ~0: no node has this parent
          sj[k] = (csize && i + k < nch) ? csize[i + k] : 1ull;
        }
        const uint64_t pc = T.parent(cj[0]);
        uint32_t m = 0;
        uint64_t sz = 1;
        bool more = true;
#pragma unroll
        for (int k = 0; k < 8; k++) {
          more = more && T.parent(cj[k]) == pc;
          if (more) {
            m |= 1u << (cj[k] & 7);
            if (csize) A.sib[M.off[h] + i + k] = sz - 1 - (uint64_t)k;
            sz += sj[k];
          }
        }
        A.code[base + ex] = pc;
        A.size[base + ex] = sz;
        A.mask[base + ex] = (uint8_t)m;
        A.first[base + ex] = (uint32_t)i;
        const uint32_t jb = T.job(pc);
        uint64_t isz = 1;
        if (A.isize) {
          float avg[6];
          average_children(A, leaf ? 0 : M.off[h], leaf, leaf_rec, jobs[jb].payload, i,
                           (uint32_t)__popc(m), isz, avg);
          A.isize[base + ex] = isz;
#pragma unroll
          for (int q = 0; q < 6; q++) A.cache[(base + ex) * 6 + q] = avg[q];
        }
        if (jobs[jb].depth == h + 1) {
          root_size[jb] = sz;
          root_isize[jb] = isz;
        }
      }
    }
    if (i == nch - 1) {
      const uint64_t np = (uint64_t)ex + head;
      M.n[h + 1] = np;
      M.off[h + 2] = base + np;
    }
  }
};

// Level bookkeeping before a build from the codes: all zero, n[0] = V; the device clock in
// flag[3]; a single job's descriptor (job, unless null) from the arguments.
constexpr int kStampWord = 2 * 64 + 3;
__global__ __launch_bounds__(256) void k_build_init(unsigned long long* meta, uint64_t words,
                                                    uint64_t V, JobDev* job, JobDev j0) {
  const unsigned long long now = wall_clock64();
  for (uint64_t i = threadIdx.x; i < words; i += blockDim.x) {
    unsigned long long v = 0;
    if (i == 0) v = V;
    if (i == kStampWord) v = now;
    meta[i] = v;
  }
  if (job && threadIdx.x == 0) *job = j0;
}

// Per job, after the bottom-up passes: node count (a single null root for an empty
// grid, finalizeTree pads it; the single leaf of a 1^3 grid), node base (exclusive scan
// over the jobs), data count (-levels adds one record per internal node), the records
// the builder writes itself (OctreeBuilder.cpp:25-29: the null record, plus the white
// record of geometry-only builds), and the hazard flag. One block.
// BLOCK threads of one block; wsum holds BLOCK / 64 words.
template <int BLOCK>
__device__ __forceinline__ void job_bases(JobDev* jobs, uint32_t n_jobs,
                                          const unsigned long long* root_size,
                                          const unsigned long long* root_isize,
                                          const unsigned long long* brick_hazard,
                                          const uint64_t* codes, Tags T, LevelMeta M,
                                          uint64_t node_cap, uint64_t* nodes,
                                          const float* in_rec, float* records, uint64_t* wsum,
                                          uint64_t& carry) {
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (uint32_t j0 = 0; j0 < n_jobs; j0 += BLOCK) {
    const uint32_t j = j0 + threadIdx.x;
    uint64_t nn = 0;
    if (j < n_jobs) {
      const JobDev& J = jobs[j];
      nn = (J.nvox == 0 || J.depth == 0) ? 1ull : root_size[j];
    }
    uint64_t tot;
    const uint64_t inc = block_incl_scan<uint64_t, BLOCK>(nn, wsum, tot);
    const uint64_t nb = carry + inc - nn;
    if (j < n_jobs) {
      JobDev& J = jobs[j];
      J.n_nodes = nn;
      J.nbase = nb;
      const bool trivial = (J.nvox == 0 || J.depth == 0);
      J.n_data = (J.payload ? 1 + J.nvox : 2) + ((J.levels && !trivial) ? root_isize[j] : 0);
      const uint64_t G3 = J.gridsize * J.gridsize * J.gridsize;
      uint64_t hz = 0;
      if (J.nvox == 0) {
        hz = (J.gridsize == 1) ? 1 : 0;
      } else if (brick_hazard) {  // found in the brick stream (codes not written)
        hz = brick_hazard[j];
      } else {
        const uint64_t last = codes[J.voff + J.nvox - 1] & ~T.tag_mask;
        // OctreeBuilder.cpp:36-42 leaves the root undefined when the last voxel is the
        // second-to-last code; the completed tree is built and the hazard reported
        hz = (G3 >= 2 && last == G3 - 2) ? 1 : 0;
      }
      J.hazard = hz;
      if (trivial) {
        if (nb < node_cap) {
          put_node(J, nodes, nb, J.nvox ? 1ull : 0ull, 0ull, ~0ull);
        } else {
          M.flag[1] = 1;
        }
      }
      float* d = records + J.dbase * 8;
      if (J.levels && J.payload && J.depth == 0 && J.nvox && in_rec != records) {
        // 1^3 grid: the single voxel's record keeps its place after the null record
        for (int k = 0; k < 8; k++) d[8 + k] = in_rec[(J.dbase + 1) * 8 + k];
      }
      for (int k = 0; k < 8; k++) d[k] = 0.0f;
      if (!J.payload) {
        // data[1] = {0, colour (1,1,1), normal (0,0,0)}
        for (int k = 0; k < 8; k++) d[8 + k] = 0.0f;
        d[8 + 2] = d[8 + 3] = d[8 + 4] = 1.0f;
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) carry += tot;
    __syncthreads();
  }
  if (threadIdx.x == 0) M.flag[2] = carry;
}

// The bottom-up levels h_lo .. H-1 whose element counts are small (bounded on the host),
// in one block, level after level (a level's scan in chunks of the block with a running
// carry, a barrier before the next level reads it), then the per-job bases.
constexpr int kTailBlock = 1024;
constexpr uint64_t kTailLevelMax = 8192;  // largest level bound the tail block takes
// The level scans' stores walk a parent's children (dependent loads, and with -levels their
// averages): one element a thread up to this many keeps enough blocks in flight. With eight,
// the levels of 487,600 voxels ran on 60 blocks: 375 us for four of them. Without -levels a store
// does less, and the blocks' look-back costs more than their number gives from 2M elements on: added
// voxels' builds, one and eight a thread, 1.4M 337 and 362 us, 2.0M 304 and 397, 2.5M 1171 and 1094,
// 4M 1709 and 1402, 8M 1047 and 866.
constexpr uint64_t kLevelScanSmall = 1ull << 23;
constexpr uint64_t kPlainScanSmall = 1ull << 21;
constexpr uint64_t kTopLevelMax = 4096;  // largest level bound k_emit_levels_top takes
__global__ __launch_bounds__(kTailBlock) void k_levels_tail(
    Arena A, LevelMeta M, Tags T, JobDev* jobs, uint32_t n_jobs, const uint64_t* leaves,
    uint32_t* leaf_parent, unsigned long long* root_size, unsigned long long* root_isize,
    const float* leaf_rec, int h_lo, int H, const unsigned long long* brick_hazard,
    uint64_t node_cap, uint64_t* __restrict__ nodes, const float* __restrict__ in_rec,
    float* __restrict__ records) {
  __shared__ uint32_t wsum32[kTailBlock / kWave];
  __shared__ uint64_t wsum[kTailBlock / kWave];
  __shared__ uint64_t carry;
  for (int h = h_lo; h < H; h++) {
    HeadLoad ld{A, M, T, jobs, leaves, h};
    ParentStore st{A, M, T, jobs, leaves, leaf_parent, root_size, root_isize, leaf_rec, h};
    __syncthreads();  // the previous level's nodes and counts are written
    const uint64_t n = M.n[h];
    uint32_t run = 0;
    for (uint64_t b = 0; b < n; b += kTailBlock) {
      const uint64_t i = b + threadIdx.x;
      const uint32_t v = i < n ? ld(i) : 0u;
      uint32_t tot;
      const uint32_t inc = block_incl_scan<uint32_t, kTailBlock>(v, wsum32, tot);
      if (i < n) st(i, run + inc - v, v, i == n - 1);
      run += tot;
    }
  }
  __syncthreads();
  job_bases<kTailBlock>(jobs, n_jobs, root_size, root_isize, brick_hazard, leaves, T, M,
                        node_cap, nodes, in_rec, records, wsum, carry);
}

// -levels: the data records of a subtree are written in post-order (a node completes
// after its children, OctreeBuilder.cpp:58-99, 149-168), so node P's record is at
// base + pstart(P) + S(P) - 1, with S = nodes that write a record (every node for
// payload builds, internal nodes only for geometry-only ones) and
// pstart(child r) = pstart(P) + sum_{r' < r} S(child r').
__device__ __forceinline__ uint64_t levels_weight(const Arena& A, uint64_t k, int payload) {
  return payload ? A.size[k] : A.isize[k];
}

__device__ __forceinline__ void put_data(float* rec, uint64_t idx, const float* avg) {
  float* r = rec + idx * 8;
  *(uint64_t*)r = 0ull;  // internal nodes' records carry morton 0
#pragma unroll
  for (int q = 0; q < 6; q++) r[2 + q] = canon_nan(avg[q]);
}

// One thread per node at height h >= 1: a job's root starts at 0 and sits last; any
// other node's start is its parent's start plus the (size - 1) of its preceding
// siblings, and its position is the parent's children_base plus its rank. It writes its
// own record (children_base relative to its job's node array) and start; with -levels
// also its data record. Consecutive nodes land in consecutive records, so the stores
// coalesce.
__device__ __forceinline__ void emit_level_node(const Arena& A, const LevelMeta& M, const Tags& T,
                                                const JobDev* __restrict__ jobs, int h,
                                                uint64_t i, uint64_t node_cap,
                                                uint64_t* __restrict__ nodes,
                                                float* __restrict__ out_rec) {
  const uint64_t co = M.off[h];
  const uint64_t code = A.code[co + i];
  const JobDev& J = jobs[T.job(code)];
  const bool lv = A.isize && J.levels;
  const uint64_t sz = A.size[co + i];
  const uint32_t cm = A.mask[co + i];
  uint64_t st, pos, pst = 0;
  if (J.depth == h) {
    st = 0;
    pos = sz - 1;
  } else {
    const uint64_t po = M.off[h + 1] + A.pidx[co + i];
    const uint32_t f = A.first[po];
    const uint32_t pcnt = (uint32_t)__popc((uint32_t)A.mask[po]);
    const uint64_t ps = A.start[po];
    const uint64_t cb = ps + A.size[po] - 1 - pcnt;
    const uint64_t sib = A.sib[co + i];
    st = ps + sib;
    if (lv) {
      pst = A.pstart[po];
      if (J.payload)
        pst += sib + (i - f);  // the siblings' sizes
      else
        for (uint64_t j = f; j < i; j++) pst += A.isize[co + j];
    }
    pos = cb + (i - f);
  }
  const uint64_t gpos = J.nbase + pos;
  if (pos >= J.n_nodes || gpos >= node_cap) {
    M.flag[1] = 1;
    return;
  }
  A.start[co + i] = st;
  uint64_t data = 0;
  if (lv) {
    A.pstart[co + i] = pst;
    const uint64_t idx = (J.payload ? 1 : 2) + pst + levels_weight(A, co + i, J.payload) - 1;
    if (idx >= J.n_data) {
      M.flag[1] = 1;
      return;
    }
    data = idx;
    put_data(out_rec, J.dbase + idx, A.cache + (co + i) * 6);
  }
  put_node(J, nodes, gpos, data, st + sz - 1 - (uint32_t)__popc(cm), offsets_of(cm));
}
__global__ __launch_bounds__(256) void k_emit_level(Arena A, LevelMeta M, Tags T,
                                                    const JobDev* __restrict__ jobs, int h,
                                                    uint64_t node_cap,
                                                    uint64_t* __restrict__ nodes,
                                                    float* __restrict__ out_rec) {
  if (M.flag[0]) return;  // arena overflow: the build is redone with a larger arena
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < M.n[h]) emit_level_node(A, M, T, jobs, h, i, node_cap, nodes, out_rec);
}
// Heights H .. h_lo, all small, in one block (a height reads what the one above it wrote):
// a launch each took 5 us whatever it did.
__global__ __launch_bounds__(kTailBlock) void k_emit_levels_top(Arena A, LevelMeta M, Tags T,
                                                                const JobDev* __restrict__ jobs,
                                                                int h_lo, int H, uint64_t node_cap,
                                                                uint64_t* __restrict__ nodes,
                                                                float* __restrict__ out_rec) {
  if (M.flag[0]) return;
  for (int h = H; h >= h_lo; h--) {
    const uint64_t n = M.n[h];
    for (uint64_t i = threadIdx.x; i < n; i += kTailBlock)
      emit_level_node(A, M, T, jobs, h, i, node_cap, nodes, out_rec);
    __syncthreads();
  }
}

// Every node of heights hs..H in one launch (geometry records, no -levels data): one
// thread per node, flattened over the contiguous levels of the arena. A node's start is
// the sum of the sibling offsets along its path to the root (start(P) plus its own sib),
// which needs only the bottom-up results, so all levels are written at once.
__global__ __launch_bounds__(256) void k_emit_upper(Arena A, LevelMeta M, Tags T,
                                                    const JobDev* __restrict__ jobs, int hs,
                                                    int H, uint64_t node_cap,
                                                    uint64_t* __restrict__ nodes) {
  if (M.flag[0]) return;
  const uint64_t g = M.off[hs] + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int h = hs;
  while (h <= H && g >= M.off[h] + M.n[h]) h++;
  if (h > H) return;
  const uint64_t i = g - M.off[h];
  const uint64_t code = A.code[g];
  const JobDev& J = jobs[T.job(code)];
  const uint64_t sz = A.size[g];
  const uint32_t cm = A.mask[g];
  uint64_t st, pos;
  if (J.depth == h) {  // the job's root: start 0, last record
    st = 0;
    pos = sz - 1;
  } else {
    const uint64_t po = M.off[h + 1] + A.pidx[g];
    uint64_t sp = 0;  // start of the parent
    uint64_t cur = po;
    for (int l = h + 1; l < J.depth; l++) {
      sp += A.sib[cur];
      cur = M.off[l + 1] + A.pidx[cur];
    }
    st = sp + A.sib[g];
    pos = sp + A.size[po] - 1 - (uint32_t)__popc((uint32_t)A.mask[po]) + (i - A.first[po]);
  }
  const uint64_t gpos = J.nbase + pos;
  if (pos >= J.n_nodes || gpos >= node_cap) {
    M.flag[1] = 1;
    return;
  }
  A.start[g] = st;
  put_node(J, nodes, gpos, 0ull, st + sz - 1 - (uint32_t)__popc(cm), offsets_of(cm));
}

// One thread per leaf: position = children_base(parent) + rank among its siblings.
// OctreeBuilder.cpp:137-139 (binary: data 1) / :157-159 (payload: its data index; with
// -levels its record moves to its post-order place).
__global__ __launch_bounds__(256) void k_emit_leaves(Arena A, LevelMeta M, Tags T,
                                                     const JobDev* __restrict__ jobs,
                                                     uint64_t node_cap,
                                                     const uint64_t* __restrict__ codes,
                                                     const uint32_t* __restrict__ leaf_parent,
                                                     uint64_t* __restrict__ nodes,
                                                     const float* __restrict__ in_rec,
                                                     float* __restrict__ out_rec) {
  if (M.flag[0]) return;
  const uint64_t nl = M.n[0];
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nl) return;
  const JobDev& J = jobs[T.job(codes[i])];
  if (J.depth == 0) return;  // 1^3 grid: its leaf is the root, written with the job bases
  const uint64_t po = M.off[1] + leaf_parent[i];
  const uint32_t cnt = (uint32_t)__popc((uint32_t)A.mask[po]);
  const uint64_t cb = A.start[po] + A.size[po] - 1 - cnt;
  const uint64_t rank = i - A.first[po];
  const uint64_t pos = cb + rank;
  const uint64_t gpos = J.nbase + pos;
  if (pos >= J.n_nodes || gpos >= node_cap) {
    M.flag[1] = 1;
    return;
  }
  uint64_t data = J.payload ? (1ull + (i - J.voff)) : 1ull;
  if (A.isize && J.levels && J.payload) {
    const uint64_t idx = 1 + A.pstart[po] + rank;
    if (idx >= J.n_data) {
      M.flag[1] = 1;
      return;
    }
    const float4* src = (const float4*)(in_rec + (J.dbase + data) * 8);
    float4* dst = (float4*)(out_rec + (J.dbase + idx) * 8);
    dst[0] = src[0];
    dst[1] = src[1];
    data = idx;
  }
  put_node(J, nodes, gpos, data, 0ull, ~0ull);
}

// ---------------------------------------------------------------- brick fast path
// Every occupied 16^3 brick of the voxel stream is an aligned subtree of height 4 whose
// occupancy is its 64 words (word w = voxels 64w..64w+63 in Morton order). Within it:
//   height 1: a byte of a word (8 voxels), child mask = the byte;
//   height 2: a word, child mask = its non-zero bytes;
//   height 3: 8 consecutive words, child mask = its non-zero words;
//   height 4: the brick, child mask = its non-zero word groups.
// The voxelizer's brick kernels compute each brick node's subtree size and child mask
// (brick_shape_of, one wave per brick, lane = word) into the brick stream; here one wave
// per brick writes every record below the brick node at its post-order position, and
// the heights above come from the brick codes at once (upper levels, above).

// Every record below each brick node, a wave per brick. The brick's records form the contiguous
// range [S, S + s4 - 1) laid out as the word groups' subtree ranges, then the group nodes; a
// group's range is its words' ranges, then its word nodes; a word's range is its voxels, then
// its byte nodes. So the voxels' records come in voxel order, whatever lies between them: the
// wave lists its inner nodes (first child, child mask) in record order in LDS, with a bitmap of
// their places, and lane r then writes records r, r + 64, ...: an inner node's from the list
// (its place there is the count of bitmap bits before it), a voxel's from the count of clear
// bits before it. Consecutive lanes store consecutive records.
//
// Bound by the writes, 24 bytes a node. Finding each record's node by searches in the ranges'
// offsets took 740 vector instructions a brick, two thirds of the kernel's time. With kStaged
// (more than kStageBricks bricks) a window's records go through LDS and out by whole 128-byte
// lines, past the caches; a line shared with another brick goes through them. Three 8-byte stores
// a record, 16 bytes a lane staged but not by lines, by lines: 30M nodes 198, 165, 143 us (5.0
// TB/s), 64 mixed meshes 1107, 955, 894, a 6M-triangle soup in 8 partitions 1660, 1501, 1242 (past
// the caches without regard to lines the mixed meshes took 1190). A few bricks wait for the LDS
// longer than for the stores: 900 of them 11.3 us, staged 13.2.
constexpr int kEmitWaves = 4;  // waves per block of k_emit_bricks
typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kLineWords = 16;  // 64-bit words of a memory line
constexpr int kInnerMax = 8 + 64 + 512;                        // inner nodes below a brick node
constexpr int kInnerBits = (kBrickVox + kInnerMax + 63) / 64 * 2;  // bitmap, 32-bit words

// the child offsets of a mask (offsets_of) in two halves by multiplications: four mask bits
// spread over the low bits of four bytes, their exclusive prefix sums, 0xFF where clear
__device__ __forceinline__ uint64_t offsets_fast(uint32_t m) {
  const uint32_t lo = ((m & 15u) * 0x00204081u) & 0x01010101u;
  const uint32_t hi = ((m >> 4) * 0x00204081u) & 0x01010101u;
  const uint32_t below = (uint32_t)__popc(m & 15u) * 0x01010101u;
  const uint32_t l = (lo * 0x01010100u) | ((lo ^ 0x01010101u) * 0xFFu);
  const uint32_t h = (hi * 0x01010100u + below) | ((hi ^ 0x01010101u) * 0xFFu);
  return ((uint64_t)h << 32) | l;
}

// kPlaced: the job's records go to a larger node stream (a streamed partition), their
// children_base and data indices moved by its placement.
constexpr uint64_t kStageBricks = 4096;
template <bool kPlaced, bool kStaged>
__global__ __launch_bounds__(kWave * kEmitWaves) void k_emit_bricks(
    Arena A, LevelMeta M, Tags T, const JobDev* __restrict__ jobs,
    const uint64_t* __restrict__ bwords, const uint64_t* __restrict__ bcode,
    const uint64_t* __restrict__ bvoff, uint64_t nb, uint64_t node_cap,
    uint64_t* __restrict__ nodes) {
  __shared__ uint32_t s_inner[kEmitWaves][kInnerMax];  // first child (relative to S) | mask << 16
  __shared__ uint32_t s_bits[kEmitWaves][kInnerBits + 2];
  __shared__ uint64_t s_offs[256];  // offsets of every child mask
  __shared__ __attribute__((aligned(16))) uint64_t s_rec[kStaged ? kEmitWaves : 1][kLineWords + 3 * kWave];
  const int ws = threadIdx.x / kWave;
  const int lane = lane_id();
  const int g = lane >> 3, q = lane & 7;
  const uint64_t w = (uint64_t)blockIdx.x * kEmitWaves + ws;
  const bool live = w < nb && !M.flag[0];
  // the brick's own words and offsets, in flight while the offset table is built
  uint64_t word = 0, bc = 0, bvo = 0, S = 0;
  if (live) {
    word = bwords[w * kBrickWords + lane];
    bc = bcode[w];
    bvo = bvoff[w];
    S = A.start[M.off[4] + w];
  }
  s_offs[threadIdx.x] = offsets_fast(threadIdx.x);  // the block has 256 threads
  uint32_t* inner = s_inner[ws];
  uint32_t* bits = s_bits[ws];
#pragma unroll
  for (int k = 0; k < (kInnerBits + 2 + kWave - 1) / kWave; k++)
    if (lane + kWave * k < kInnerBits + 2) bits[lane + kWave * k] = 0u;
  __syncthreads();
  if (!live) return;
  // the word: its voxels, its non-empty bytes (byte nodes)
  uint32_t m2 = 0;
#pragma unroll
  for (int j = 0; j < 8; j++)
    if ((word >> (8 * j)) & 0xFFull) m2 |= 1u << j;
  const uint32_t nv = (uint32_t)__popcll(word), nbz = (uint32_t)__popc(m2);
  const uint64_t nz = __ballot(word != 0ull);
  const uint32_t mask3 = (uint32_t)(nz >> (8 * g)) & 0xFFu;  // the group's non-empty words
  const uint32_t nw = (uint32_t)__popc(mask3);
  uint32_t mask4 = 0;
#pragma unroll
  for (int k = 0; k < 8; k++)
    if ((nz >> (8 * k)) & 0xFFull) mask4 |= 1u << k;
  // within the group: records of the words before this one (voxels and byte nodes), and byte
  // nodes of the words before it (upper half)
  const uint32_t mine = (nv + nbz) | (nbz << 16);
  int x = (int)mine;
  {
    const int o1 = __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1
    x += (q >= 1) ? o1 : 0;
    const int o2 = __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);  // row_shr:2
    x += (q >= 2) ? o2 : 0;
    const int o4 = __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);  // row_shr:4
    x += (q >= 4) ? o4 : 0;
  }
  const uint32_t before = (uint32_t)x - mine;
  const uint32_t all = group8_sum(mine);  // of the whole group
  // over the groups: records of a group's range (its words' and the word nodes), inner nodes
  const uint32_t grp = ((all & 0xFFFFu) + nw) | (((all >> 16) + nw) << 16);
  const uint32_t ginc = wave_incl_scan<uint32_t>(q == 0 ? grp : 0u);
  const uint32_t gpre = ginc - grp;  // (only group heads add; every lane knows its group's term)
  const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)ginc, kWave - 1);
  const uint32_t RG = tot & 0xFFFFu;                      // records inside the groups' ranges
  const uint32_t R = RG + (uint32_t)__popc(mask4);        // records below the brick node
  const uint32_t go = gpre & 0xFFFFu, gi = gpre >> 16;    // the group's range, its inner nodes
  const uint32_t wo = go + (before & 0xFFFFu);            // the word's range
  auto set_bits = [&](uint32_t at, uint32_t n) {          // n <= 8 bits
    const uint64_t v = (uint64_t)((1u << n) - 1u) << (at & 31u);
    atomicOr(&bits[at >> 5], (uint32_t)v);
    if (v >> 32) atomicOr(&bits[(at >> 5) + 1], (uint32_t)(v >> 32));
  };
  if (word) {
    uint32_t i = gi + (before >> 16), vo = wo;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint32_t byte = (uint32_t)(word >> (8 * j)) & 0xFFu;
      if (byte) inner[i++] = vo | (byte << 16);  // its voxels start at vo
      vo += (uint32_t)__popc(byte);
    }
    set_bits(wo + nv, nbz);
    const uint32_t rank = (uint32_t)__popc(mask3 & ((1u << q) - 1u));
    inner[gi + (all >> 16) + rank] = (wo + nv) | (m2 << 16);  // the word node
  }
  if (q == 0 && mask3) {
    set_bits(go + (all & 0xFFFFu), nw);
    const uint32_t rank = (uint32_t)__popc(mask4 & ((1u << g) - 1u));
    inner[(tot >> 16) + rank] = (go + (all & 0xFFFFu)) | (mask3 << 16);  // the group node
  }
  if (lane == 0) set_bits(RG, R - RG);
  wave_lds_sync();
  const JobDev& J = jobs[T.job(bc)];
  if (S + R > J.n_nodes || J.nbase + S + R > node_cap) {
    if (lane == 0) M.flag[1] = 1;
    return;
  }
  uint64_t* out = nodes + 3 * (J.nbase + S);
  uint64_t* rec = s_rec[kStaged ? ws : 0];
  const int payload = J.payload;
  // the job's placement, read once (the record stores below could alias the job table)
  const uint64_t cb0 = S + (kPlaced ? J.cb_add : 0);
  // the first voxel's data index; geometry-only voxels share record 1
  uint64_t leaf0 = payload ? 1ull + (bvo - J.voff) : 1ull;
  if (kPlaced && leaf0 >= (payload ? 1ull : 2ull)) leaf0 += J.data_add;
  uint32_t prior = 0;  // inner nodes before the window
  // staged words lie in rec as in their 128-byte lines: 'fill' words wait there for their line's
  // others, the first 'skip' of them not the brick's; line = the first one's place
  const uint32_t lead = (uint32_t)((uintptr_t)out >> 3) % kLineWords;
  uint32_t fill = lead, skip = lead;
  uint64_t* line = out - lead;
  for (uint32_t r0 = 0; r0 < R; r0 += kWave) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits[r0 >> 5]);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)bits[(r0 >> 5) + 1]);
    const uint32_t below = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
    const bool is_inner = ((lane < 32 ? lo : hi) >> (lane & 31)) & 1u;
    const uint32_t r = r0 + lane;
    if (r < R) {
      uint64_t d0, d1, d2;
      if (is_inner) {
        const uint32_t e = inner[prior + below];
        d0 = 0;
        d1 = cb0 + (e & 0xFFFFu);
        d2 = s_offs[e >> 16];
      } else {
        d0 = leaf0 + (payload ? r - prior - below : 0u);
        d1 = 0;
        d2 = ~0ull;
      }
      uint64_t* to = kStaged ? rec + fill + 3 * lane : out + 3 * (uint64_t)r;
      to[0] = d0;
      to[1] = d1;
      to[2] = d2;
    }
    if constexpr (kStaged) {
      wave_lds_sync();
      const uint32_t total = fill + 3 * min(R - r0, (uint32_t)kWave);
      const uint32_t whole = total / kLineWords * kLineWords;
      const uint32_t words = r0 + kWave >= R ? total : whole;  // to store now
#pragma unroll
      for (uint32_t k = 0; k < 2; k++) {
        const uint32_t at = 2 * (lane + kWave * k);
        if (at < words) {
          const u64x2 v = *(const u64x2*)(rec + at);
          const bool first = at >= skip, second = at + 1 < words && at + 1 >= skip;
          if (at >= whole || at / kLineWords < (skip + kLineWords - 1) / kLineWords) {
            // a line shared with another brick: through the cache
            if (first && second)
              *(u64x2*)(line + at) = v;
            else if (first)
              line[at] = v.x;
            else if (second)
              line[at + 1] = v.y;
          } else {
            __builtin_nontemporal_store(v, (u64x2*)(line + at));
          }
        }
      }
      uint64_t rest = 0;
      if (lane < (int)kLineWords) rest = rec[whole + lane];
      wave_lds_sync();
      if (lane < (int)kLineWords) rec[lane] = rest;
      line += whole;
      fill = total - whole;
      skip = 0;
      wave_lds_sync();
    }
    prior += (uint32_t)__popc(lo) + (uint32_t)__popc(hi);
  }
}

// ---------------------------------------------------------------- upper levels at once
// Fast path: every height >= 5 straight from the sorted brick nodes (height 4) in four
// launches, instead of one scan per height. Brick i heads its ancestor at height l (is the
// first brick below it) iff l <= T(i): T(i) = the job's depth D for the first brick of a
// job, else 4 + (highest bit where its code differs from brick i-1's) / 3, capped at D.
// So the index of brick i's ancestor at height l is incl_l(i) - 1, incl_l(i) = the number
// of bricks j <= i with T(j) >= l. With S4(i) = the brick subtree sizes before brick i and
//   A_l(i) = S4(i) + sum_{m=5..l} (bricks before i with T >= m)
// (the nodes below height l+1 that precede brick i in the stream), a node P of height l
// whose bricks are [i0, i1) has size(P) = A_l(i1) - A_l(i0), and the sizes of P's
// preceding siblings sum to A_l(head of P) - A_l(head of its parent's first child).
// k_up_count counts per tile of 256 bricks, k_up_scan scans the counts per height (one
// block), k_up_apply writes every node's code, first child, parent index and A_l at its
// head brick (and A_l at every job's end), k_up_finish turns them into sizes, child masks
// and sibling offsets. No atomics.
constexpr int kUpTile = 256;
constexpr int kUpLevels = 17;  // heights 5 .. 21
constexpr int kUpRows = 8;

// job_bases for one job with bricks: its fields (one thread), and the null record and the white
// one of geometry-only builds (16 threads).
__device__ __forceinline__ void put_single_base(JobDev* job, const JobDev& j0, const LevelMeta& M,
                                                uint64_t n_nodes, uint64_t hazard) {
  job->n_nodes = n_nodes;
  job->nbase = 0;
  job->hazard = hazard;
  job->n_data = j0.payload ? 1 + j0.nvox : 2;
  M.flag[2] = n_nodes;
}
__device__ __forceinline__ void put_leading_records(float* records, const JobDev& j0) {
  if (threadIdx.x < (j0.payload ? 8u : 16u))
    records[j0.dbase * 8 + threadIdx.x] = threadIdx.x >= 10 && threadIdx.x < 13 ? 1.0f : 0.0f;
}

// T(i) from brick i's node code c and the previous brick's p (has_prev = i > 0)
__device__ __forceinline__ int brick_top(uint64_t c, uint64_t p, bool has_prev, Tags T, int D) {
  if (D <= 4) return 4;
  if (!has_prev || (c & T.tag_mask) != (p & T.tag_mask)) return D;
  const uint64_t x = (c ^ p) & ~T.tag_mask;
  if (!x) return 4;
  return min(D, 4 + (63 - __clzll((long long)x)) / 3);
}
// the height-4 node code of a brick (its first voxel's code without the 12 in-brick bits)
__device__ __forceinline__ uint64_t brick_node_code(uint64_t c0, Tags T) {
  return (c0 & T.tag_mask) | ((c0 & ~T.tag_mask) >> 12);
}
__device__ __forceinline__ int job_depth(const JobDev* jobs, Tags T, uint64_t code) {
  return T.tag_mask ? jobs[T.job(code)].depth : jobs[0].depth;
}

// Per brick: its height-4 node (code, subtree size and child mask from the voxelizer's
// brick shape) and the hazard case (the job's last voxel is code G^3 - 2: bits 62 and 63
// of the last word of the grid's last brick; a job's last brick answers for it); per tile: counts
// of T >= l for l = 5 .. H, and the sum of the brick subtree sizes. The first block also leaves
// the device clock in *stamp and, with put, the single job's descriptor j0 in *jobs.
__global__ __launch_bounds__(kUpTile) void k_up_count(Arena A, Tags T, JobDev* jobs, int put,
                                                      JobDev j0, unsigned long long* stamp,
                                                      const uint64_t* __restrict__ bwords,
                                                      const uint64_t* __restrict__ bcode,
                                                      const uint32_t* __restrict__ bshape,
                                                      uint64_t NB, int H,
                                                      uint32_t* __restrict__ tile_cnt,
                                                      uint64_t* __restrict__ tile_s4,
                                                      unsigned long long* hazard) {
  __shared__ uint32_t wcnt[kUpTile / kWave][kUpLevels];
  __shared__ uint64_t ws4[kUpTile / kWave];
  const uint64_t i = (uint64_t)blockIdx.x * kUpTile + threadIdx.x;
  int t = 4;
  uint64_t s4 = 0;
  if (i == 0) {
    *stamp = wall_clock64();
    if (put) *jobs = j0;
  }
  if (i < NB) {
    const uint64_t c0 = bcode[i];
    const uint64_t code = brick_node_code(c0, T);
    const uint64_t prev = i ? brick_node_code(bcode[i - 1], T) : 0ull;
    const uint32_t sh = bshape[i];
    s4 = sh & 0xFFFFu;
    A.code[i] = code;
    A.size[i] = s4;
    A.mask[i] = (uint8_t)(sh >> 16);
    A.first[i] = 0;
    const uint32_t jb = T.job(c0);
    // (one job: not from the memory that it is being put into)
    const uint64_t G = T.tag_mask ? jobs[jb].gridsize : j0.gridsize;
    const int D = T.tag_mask ? jobs[jb].depth : j0.depth;
    if (i + 1 == NB || (T.tag_mask && T.job(bcode[i + 1]) != jb))
      hazard[jb] = (c0 & ~T.tag_mask) == G * G * G - kBrickVox &&
                   (bwords[i * kBrickWords + kWave - 1] >> 62) == 1ull;
    t = brick_top(code, prev, i > 0, T, D);
  }
  const int w = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k < kUpLevels; k++) {
    const uint64_t b = __ballot(t >= 5 + k);
    if (lane_id() == 0) wcnt[w][k] = (uint32_t)__popcll(b);
  }
  const uint64_t sw = wave_last<uint64_t>(wave_incl_scan<uint64_t>(s4));
  if (lane_id() == 0) ws4[w] = sw;
  __syncthreads();
  if (threadIdx.x < kUpLevels && 5 + (int)threadIdx.x <= H) {
    uint32_t sum = 0;
    for (int q = 0; q < kUpTile / kWave; q++) sum += wcnt[q][threadIdx.x];
    tile_cnt[(uint64_t)blockIdx.x * kUpLevels + threadIdx.x] = sum;
  }
  if (threadIdx.x == 0) {
    uint64_t sum = 0;
    for (int q = 0; q < kUpTile / kWave; q++) sum += ws4[q];
    tile_s4[blockIdx.x] = sum;
  }
}

// one block, a wave per height (and one for the sizes): the exclusive prefix of the tile
// counts (in place, kUpRows x 64 tiles at a time: 270,000 bricks' 1056 tiles took 12.8 us one row of
// 64 after the other, 6.1 so); then the node counts and arena offsets of all
// heights and A_l at the end of the stream; an arena too small is flagged. One job (jobs not
// null; it has bricks, so it is not trivial): job_bases' results as well.
__global__ __launch_bounds__(1024) void k_up_scan(Arena A, LevelMeta M, uint64_t NB, int H,
                                                  JobDev* jobs, JobDev j0,
                                                  const unsigned long long* hazard,
                                                  float* records, uint32_t ntiles,
                                                  uint32_t* __restrict__ tile_cnt,
                                                  uint64_t* __restrict__ tile_s4,
                                                  uint64_t* __restrict__ a_end) {
  __shared__ uint64_t s_tot[kUpLevels + 1];
  const int w = threadIdx.x / kWave;
  for (int task = w; task <= kUpLevels; task += 1024 / kWave) {
    const int k = task ? task - 1 : kUpLevels;  // (the sizes first: a wave of their own below H = 20)
    if (k < kUpLevels && 5 + k > H) continue;   // uniform per wave
    uint64_t carry = 0;
    for (uint32_t t0 = 0; t0 < ntiles; t0 += kWave * kUpRows) {
      uint64_t v[kUpRows];  // all loads issued before the first scan
#pragma unroll
      for (int q = 0; q < kUpRows; q++) {
        const uint32_t t = t0 + kWave * q + lane_id();
        v[q] = t >= ntiles ? 0ull
               : k == kUpLevels ? tile_s4[t]  // the brick subtree sizes
                                : (uint64_t)tile_cnt[(uint64_t)t * kUpLevels + k];
      }
#pragma unroll
      for (int q = 0; q < kUpRows; q++) {
        const uint32_t t = t0 + kWave * q + lane_id();
        const uint64_t inc = wave_incl_scan<uint64_t>(v[q]);
        const uint64_t ex = carry + inc - v[q];
        if (t < ntiles) {
          if (k == kUpLevels)
            tile_s4[t] = ex;
          else
            tile_cnt[(uint64_t)t * kUpLevels + k] = (uint32_t)ex;
        }
        carry += wave_last<uint64_t>(inc);
      }
    }
    if (lane_id() == 0) s_tot[k] = carry;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t off = NB;  // off[5]
    uint64_t a = s_tot[kUpLevels];  // S4 at the end
    M.n[4] = M.off[5] = NB;
    M.off[4] = 0;
    for (int l = 5; l <= H; l++) {
      const uint64_t n = s_tot[l - 5];
      M.n[l] = n;
      M.off[l] = off;
      off += n;
      M.off[l + 1] = off;
      a += n;
      a_end[l - 5] = a;
    }
    M.flag[0] = off > A.cap;
    M.flag[1] = 0;
    if (jobs) put_single_base(jobs, j0, M, a, *hazard);
  }
  if (jobs) put_leading_records(records, j0);
}

// Per brick: the parent index of its brick node, the fields of every node it heads, A_l at
// each of those nodes (kept in the node's start slot until the records are written), and
// at a job's first brick A_l as the previous job's end (the last brick: its job's end is
// the end of the stream).
__global__ __launch_bounds__(kUpTile) void k_up_apply(Arena A, LevelMeta M, Tags T,
                                                      const JobDev* jobs, uint64_t NB, int H,
                                                      const uint32_t* __restrict__ tile_pre,
                                                      const uint64_t* __restrict__ tile_s4,
                                                      const uint64_t* __restrict__ a_end,
                                                      uint64_t* __restrict__ job_end) {
  __shared__ uint32_t wpre[kUpTile / kWave][kUpLevels];
  __shared__ uint64_t ws4[kUpTile / kWave];
  if (M.flag[0]) return;  // arena too small: the build is redone with a larger one
  const uint64_t i = (uint64_t)blockIdx.x * kUpTile + threadIdx.x;
  const bool live = i < NB;
  uint64_t c = 0, s4 = 0, cp = 0;
  int D = 4, t = 4;
  if (live) {
    c = A.code[i];
    s4 = A.size[i];
    if (i) cp = A.code[i - 1];
    D = job_depth(jobs, T, c);
    t = brick_top(c, cp, i > 0, T, D);
  }
  const int w = threadIdx.x / kWave;
  const uint64_t le = (2ull << lane_id()) - 1ull;  // lanes <= this one
  uint64_t bal[kUpLevels];
#pragma unroll
  for (int k = 0; k < kUpLevels; k++) {
    bal[k] = __ballot(t >= 5 + k);
    if (lane_id() == 0) wpre[w][k] = (uint32_t)__popcll(bal[k]);
  }
  const uint64_t s4i = wave_incl_scan<uint64_t>(s4);
  if (lane_id() == kWave - 1) ws4[w] = s4i;
  __syncthreads();
  if (threadIdx.x < kUpLevels) {  // exclusive prefix over the waves, per height
    uint32_t run = 0;
    for (int q = 0; q < kUpTile / kWave; q++) {
      const uint32_t x = wpre[q][threadIdx.x];
      wpre[q][threadIdx.x] = run;
      run += x;
    }
  }
  __syncthreads();
  uint64_t S4 = tile_s4[blockIdx.x] + s4i - s4;
  for (int q = 0; q < w; q++) S4 += ws4[q];
  if (!live) return;
  const uint64_t tag = c & T.tag_mask, rest = c & ~T.tag_mask;
  const bool job_first = i == 0 || (cp & T.tag_mask) != tag;
  const uint32_t jb = T.job(c);
  A.start[i] = S4;  // A_4 at the brick
  if (D >= 5)
    A.pidx[i] = tile_pre[(uint64_t)blockIdx.x * kUpLevels] + wpre[w][0] +
                (uint32_t)__popcll(bal[0] & le) - 1u;
  uint64_t a = S4;
  uint32_t prev_incl = 0;
#pragma unroll
  for (int k = 0; k < kUpLevels; k++) {
    const int l = 5 + k;
    if (l > H) break;
    const uint32_t incl = tile_pre[(uint64_t)blockIdx.x * kUpLevels + k] + wpre[w][k] +
                          (uint32_t)__popcll(bal[k] & le);
    const bool head = t >= l;
    a += incl - (head ? 1u : 0u);  // A_l(i)
    if (head && l <= D) {
      const uint64_t g = M.off[l] + incl - 1u;
      A.code[g] = tag | (rest >> (3 * (l - 4)));
      A.first[g] = l == 5 ? (uint32_t)i : prev_incl - 1u;
      if (k + 1 < kUpLevels && l < D) {
        const uint32_t nxt = tile_pre[(uint64_t)blockIdx.x * kUpLevels + k + 1] +
                             wpre[w][k + 1] + (uint32_t)__popcll(bal[k + 1] & le);
        A.pidx[g] = nxt - 1u;
      }
      A.start[g] = a;
    }
    if (job_first && i) job_end[(uint64_t)T.job(cp) * kUpLevels + k] = a;
    if (i == NB - 1) job_end[(uint64_t)jb * kUpLevels + k] = a_end[k];
    prev_incl = incl;
  }
}

// Every node of heights 4 .. H: size and child mask (heights >= 5), sibling offset (below
// its job's root); each job: its tree size.
__global__ __launch_bounds__(256) void k_up_finish(Arena A, LevelMeta M, Tags T,
                                                   const JobDev* jobs, int H,
                                                   const uint64_t* __restrict__ job_end,
                                                   unsigned long long* root_size) {
  if (M.flag[0]) return;
  const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int l = 4;
  while (l <= H && g >= M.off[l] + M.n[l]) l++;
  if (l > H) return;
  const uint64_t co = M.off[l], i = g - co;
  const uint64_t code = A.code[g];
  const uint32_t jb = T.job(code);
  const int D = job_depth(jobs, T, code);
  const uint64_t a0 = A.start[g];
  if (l >= 5) {
    const bool last = i + 1 == M.n[l] || T.job(A.code[g + 1]) != jb;
    const uint64_t a1 = last ? job_end[(uint64_t)jb * kUpLevels + (l - 5)] : A.start[g + 1];
    const uint64_t size = a1 - a0;
    A.size[g] = size;
    // children: the nodes of height l-1 from the first child on whose parent is this node
    const uint64_t cco = M.off[l - 1], nch = M.n[l - 1];
    const uint64_t f = A.first[g];
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (f + k < nch) {
        const uint64_t cc = A.code[cco + f + k];
        if (T.parent(cc) == code) m |= 1u << (cc & 7);
      }
    }
    A.mask[g] = (uint8_t)m;
    if (l == D) root_size[jb] = size;
  }
  if (l == 4 && D == 4) root_size[jb] = A.size[g];  // a 16^3 job: the brick is the root
  if (l < D) {
    const uint64_t p = M.off[l + 1] + A.pidx[g];
    const uint64_t f = A.first[p];
    A.sib[g] = a0 - A.start[co + f] - (i - f);
  }
}

// All of the above for few bricks, in one block and one launch, the nodes in LDS: the build's
// bookkeeping (k_build_init), the upper levels, the per-job bases (k_levels_tail) and the upper
// nodes' records (k_emit_upper). A thread is a brick, then a node.
//
// Bound by its chain of accesses, as are the seven launches it replaces (2 to 5 us each whatever
// they do; with the nodes in global memory one launch of it took 14 us for 40 bricks, 21 for 900,
// no less than they did).
constexpr uint32_t kSmallNodes = 2816;  // nodes of heights 4 .. H, at most
struct SmallNode {
  uint64_t code;
  uint32_t a;          // A_l of its first brick, then its start
  uint32_t size, sib;
  uint16_t first, pidx;
};
__global__ __launch_bounds__(kTailBlock) void k_up_small(
    uint64_t* __restrict__ start, LevelMeta M, Tags T, JobDev* jobs, uint32_t n_jobs,
    const uint64_t* __restrict__ bwords, const uint64_t* __restrict__ bcode,
    const uint32_t* __restrict__ bshape, uint32_t NB, int H, uint64_t meta_words, int put,
    JobDev j0, unsigned long long* root_size, unsigned long long* root_isize,
    unsigned long long* hazard, uint64_t* job_end, uint64_t node_cap, uint64_t* nodes,
    float* records) {
  constexpr int kWaves = kTailBlock / kWave;
  __shared__ SmallNode s_node[kSmallNodes];
  __shared__ uint8_t s_mask[kSmallNodes];
  __shared__ uint32_t s_cnt[kUpLevels], s_off[kUpLevels + 2], wpre[kWaves][kUpLevels];
  __shared__ uint32_t s_end[kUpLevels];  // one job: A_l at its end
  __shared__ uint32_t ws4[kWaves], s_hazard;
  __shared__ uint64_t s_scan[kWaves], s_carry;
  const int w = threadIdx.x / kWave, lane = lane_id();
  const uint64_t le = (2ull << lane) - 1ull;  // lanes <= this one
  const bool tagged = T.tag_mask != 0ull;
  const unsigned long long now = wall_clock64();
  for (uint64_t i = threadIdx.x; i < meta_words; i += kTailBlock)
    M.n[i] = i == (uint64_t)kStampWord ? now : 0ull;
  if (put && threadIdx.x == 0) *jobs = j0;
  if (threadIdx.x == 0) s_hazard = 0;
  const uint32_t i = threadIdx.x;
  const bool live = i < NB;
  uint64_t c0 = 0, c = 0, cp = 0;
  uint32_t sh = 0, jb = 0;
  int D = 4, t = 4;
  if (live) {
    c0 = bcode[i];
    sh = bshape[i];
    c = brick_node_code(c0, T);
    if (i) cp = brick_node_code(bcode[i - 1], T);
    jb = T.job(c0);
    D = tagged ? jobs[jb].depth : j0.depth;
    t = brick_top(c, cp, i > 0, T, D);
  }
  const uint32_t s4 = sh & 0xFFFFu;
  for (int k = 0; 5 + k <= H; k++) {
    const uint64_t m = __ballot(t >= 5 + k);
    if (lane == 0) wpre[w][k] = (uint32_t)__popcll(m);
  }
  const uint32_t s4i = wave_incl_scan<uint32_t>(s4);
  if (lane == kWave - 1) ws4[w] = s4i;
  __syncthreads();
  if (threadIdx.x < kWave) {  // exclusive prefixes over the waves, per height; the heights' offsets
    uint32_t n = 0;
    if (5 + lane <= H)
      for (int q = 0; q < kWaves; q++) {
        const uint32_t x = wpre[q][lane];
        wpre[q][lane] = n;
        n += x;
      }
    const uint32_t inc = wave_incl_scan<uint32_t>(n);
    if (5 + lane <= H) {
      s_cnt[lane] = n;
      s_off[lane + 2] = NB + inc;
    }
    if (lane == 0) {
      s_off[0] = 0;
      s_off[1] = NB;
    }
  }
  uint32_t S4 = s4i - s4, all4 = 0;
  for (int q = 0; q < kWaves; q++) {
    if (q < w) S4 += ws4[q];
    all4 += ws4[q];
  }
  __syncthreads();
  // s_off[l - 4]: first node of height l
  const uint32_t total = s_off[H - 3];
  if (live) {
    SmallNode& B = s_node[i];
    B.code = c;
    B.a = S4;
    B.size = s4;
    B.first = 0;
    s_mask[i] = (uint8_t)(sh >> 16);
    const uint64_t G = tagged ? jobs[jb].gridsize : j0.gridsize;
    if ((c0 & ~T.tag_mask) == G * G * G - kBrickVox &&
        (bwords[(uint64_t)i * kBrickWords + kWave - 1] >> 62) == 1ull) {
      if (tagged) hazard[jb] = 1;
      s_hazard = 1;
    }
  }
  {
    const uint64_t tag = c & T.tag_mask, rest = c & ~T.tag_mask;
    const bool job_first = live && i && (cp & T.tag_mask) != tag;
    uint32_t a = S4, a_end = all4;
    uint32_t below = i;  // its ancestor's index a height down
    for (int k = 0; 5 + k <= H; k++) {
      const int l = 5 + k;
      const uint64_t m = __ballot(t >= l);  // (all lanes)
      const uint32_t incl = wpre[w][k] + (uint32_t)__popcll(m & le);
      const bool head = t >= l;
      a += incl - (head ? 1u : 0u);  // A_l(i)
      a_end += s_cnt[k];             // A_l at the end
      if (live) {
        // the node it heads a height down learns its parent
        if (t >= l - 1 && l <= D) s_node[s_off[k] + below].pidx = (uint16_t)(incl - 1u);
        if (head && l <= D) {
          SmallNode& P = s_node[s_off[k + 1] + incl - 1u];
          P.code = tag | (rest >> (3 * (l - 4)));
          P.first = (uint16_t)below;
          P.a = a;
        }
        if (job_first) job_end[(uint64_t)T.job(cp) * kUpLevels + k] = a;
        if (i == NB - 1) {
          if (tagged) job_end[(uint64_t)jb * kUpLevels + k] = a_end;
          s_end[k] = a_end;
        }
      }
      below = incl - 1u;
    }
  }
  __syncthreads();
  auto height = [&](uint32_t g) {
    int l = 4;
    while (g >= s_off[l - 3]) l++;
    return l;
  };
  for (uint32_t g = threadIdx.x; g < total; g += kTailBlock) {  // sizes, masks, sibling offsets
    const int l = height(g);
    const uint32_t co = s_off[l - 4], n = s_off[l - 3] - co, j = g - co;
    SmallNode& P = s_node[g];
    const uint64_t code = P.code;
    const uint32_t job = T.job(code);
    const int Dj = tagged ? jobs[job].depth : j0.depth;
    if (l >= 5) {
      const bool last = j + 1 == n || T.job(s_node[g + 1].code) != job;
      const uint32_t a1 = !last ? s_node[g + 1].a
                          : tagged ? (uint32_t)job_end[(uint64_t)job * kUpLevels + (l - 5)]
                                   : s_end[l - 5];
      P.size = a1 - P.a;
      const uint32_t cco = s_off[l - 5], nch = co - cco, f = P.first;
      uint32_t m = 0;
#pragma unroll
      for (uint32_t k = 0; k < 8; k++) {
        const uint64_t cc = s_node[cco + min(f + k, nch - 1u)].code;
        if (f + k < nch && T.parent(cc) == code) m |= 1u << (cc & 7);
      }
      s_mask[g] = (uint8_t)m;
    }
    if (l == Dj && tagged) root_size[job] = P.size;
    if (l < Dj) {
      const uint32_t f = s_node[s_off[l - 3] + P.pidx].first;
      P.sib = P.a - s_node[co + f].a - (j - f);
    }
  }
  __syncthreads();
  uint32_t n_nodes = 0;
  if (tagged) {
    job_bases<kTailBlock>(jobs, n_jobs, root_size, root_isize, hazard, nullptr, T, M, node_cap,
                          nodes, records, records, s_scan, s_carry);
    __syncthreads();
  } else {
    n_nodes = s_node[total - 1].size;
    if (threadIdx.x == 0) put_single_base(jobs, j0, M, n_nodes, s_hazard);
    put_leading_records(records, j0);
  }
  for (uint32_t g = threadIdx.x; g < total; g += kTailBlock) {  // records
    int l = height(g);
    const uint32_t j = g - s_off[l - 4];
    const SmallNode& P = s_node[g];
    const uint32_t cm = s_mask[g];
    uint64_t nbase = 0, nn = n_nodes, cb_add = j0.cb_add;
    int Dj = j0.depth;
    if (tagged) {
      const JobDev& J = jobs[T.job(P.code)];
      nbase = J.nbase;
      nn = J.n_nodes;
      cb_add = J.cb_add;
      Dj = J.depth;
    }
    uint32_t st = 0, pos = P.size - 1;
    if (l < Dj) {
      const SmallNode& Q = s_node[s_off[l - 3] + P.pidx];
      const uint32_t qm = s_mask[s_off[l - 3] + P.pidx];
      uint32_t sp = 0, cur = P.pidx;  // start of the parent
      for (l++; l < Dj; l++) {
        const SmallNode& X = s_node[s_off[l - 4] + cur];
        sp += X.sib;
        cur = X.pidx;
      }
      st = sp + P.sib;
      pos = sp + Q.size - 1 - (uint32_t)__popc(qm) + (j - Q.first);
    }
    if (pos >= nn || nbase + pos >= node_cap) {
      M.flag[1] = 1;
      continue;
    }
    if (g < NB) start[g] = st;
    uint64_t* r = nodes + 3 * (nbase + pos);
    r[0] = 0;
    r[1] = st + P.size - 1 - (uint32_t)__popc(cm) + cb_add;
    r[2] = offsets_of(cm);
  }
}

#define SVO_TRY(x)                   \
  do {                               \
    hipError_t _e = (x);             \
    if (_e != hipSuccess) return _e; \
  } while (0)

hipError_t build_jobs(Context& c, uint32_t n_jobs, bool tagged, int levels,
                      const BuildOut* out) {
  if ((levels || out) && (tagged || n_jobs != 1)) {
    set_error(levels ? "-levels is supported for single builds only"
                     : "internal: a placed build is a single build");
    return hipErrorNotSupported;
  }
  const uint64_t V = c.n_vox;
  if (V >= (1ull << 32)) {
    set_error("more than 2^32 voxels in one build");
    return hipErrorInvalidValue;
  }
  if (n_jobs == 0 || n_jobs > kMaxJobs || (!tagged && n_jobs != 1)) {
    set_error("invalid job count");
    return hipErrorInvalidValue;
  }
  // host view of the jobs: depth, voxel range, data range
  std::vector<JobDev> jd(n_jobs);
  uint64_t n_records = 0;
  int H = 0;
  std::vector<uint64_t> bound;
  for (uint32_t j = 0; j < n_jobs; j++) {
    Job& J = c.jobs[j];
    JobDev& d = jd[j];
    memset(&d, 0, sizeof(d));
    int D = 0;
    while ((1ull << D) < J.gridsize) D++;
    if (tagged && D > 16) {
      set_error("a batched job's gridsize is at most 65536");
      return hipErrorInvalidValue;
    }
    d.tris = J.tris;
    d.unit_div = J.unit_vox != 0.0f ? 1.0f / J.unit_vox : 0.0f;
    d.color_mode = J.color_mode;
    d.payload = J.payload;
    d.depth = D;
    d.levels = levels ? 1 : 0;
    d.gridsize = J.gridsize;
    d.voff = J.voff;
    d.nvox = J.nvox;
    J.dbase = n_records;
    J.n_data = J.payload ? 1 + J.nvox : 2;
    d.dbase = J.dbase;
    if (out) {
      d.cb_add = out->cb_add;
      d.data_add = out->data_add;
    }
    n_records += J.n_data;
    if (J.nvox) H = std::max(H, D);
  }
  // brick fast path: the four lowest levels come from the voxelizer's brick stream (not
  // for -levels, for voxels added from outside, or for meshes below 16^3)
  bool fast = c.bricks_ok && !levels && c.n_bricks > 0;
  for (uint32_t j = 0; j < n_jobs; j++)
    if (jd[j].nvox && jd[j].depth < 4) fast = false;
  if (!fast) SVO_TRY(ensure_codes(c));  // the level scans start from the codes
  const uint64_t NB = fast ? c.n_bricks : 0;
  const int h0 = fast ? 4 : 0;  // lowest height the level scans start from
  // per-height upper bounds (host) size the launch grids
  bound.assign(H + 2, 0);
  bound[0] = V;
  for (int h = 1; h <= H; h++) {
    uint64_t b = 0;
    for (uint32_t j = 0; j < n_jobs; j++) {
      if (!jd[j].nvox || jd[j].depth < h) continue;
      const int e = jd[j].depth - h;
      b += (3 * e >= 63) ? jd[j].nvox : std::min<uint64_t>(jd[j].nvox, 1ull << (3 * e));
    }
    bound[h] = std::min(bound[h - 1], b);
    if (fast && h == 4) bound[h] = NB;
  }
  // a batch's last upload usually holds these already (the kernels of a tagged build read them
  // there, a batch of one job as well); the plain flow's job goes by kernel argument
  // (not into a graph, whose launches are compared by their argument bytes)
  const bool job_arg = !tagged && !c.graphs;
  SVO_TRY(ensure(c.jobdev, n_jobs * sizeof(JobDev)));
  if (c.clear_counters) {  // no pass came first
    SVO_TRY(fill_u64(c.counters.as<uint64_t>(), 0, kNumCounters, c.stream));
    c.clear_counters = false;
  }
  if (job_arg) {
  } else if (c.jobdev_img.size() != jd.size() ||
      memcmp(c.jobdev_img.data(), jd.data(), n_jobs * sizeof(JobDev)) != 0) {
    SVO_TRY(upload_async(c, c.jobdev.p, jd.data(), n_jobs * sizeof(JobDev)));
  }
  c.jobdev_img.clear();  // the job bases are written into it
  // data records: payload records were written by the voxelizer at dbase + 1 ..
  SVO_TRY(ensure_keep(c.records, n_records * 32, n_records * 32, c.stream));
  JobDev* d_jobs = c.jobdev.as<JobDev>();
  const Tags T{tagged ? ~kCodeMask : 0ull};
  JobDev job0;  // a single job's descriptor, for the kernels' arguments
  memset(&job0, 0, sizeof(job0));
  if (!tagged) job0 = jd[0];

  // arena: the internal nodes the level scans produce (heights >= h0)
  uint64_t cap = fast ? NB + NB / 2 + 4096 : std::max<uint64_t>(V / 2 + 1024, 4096);
  // internal nodes below the brick nodes (fast path): bytes, words, word groups
  const uint64_t in_brick =
      fast ? std::min<uint64_t>(V, 512 * NB) + std::min<uint64_t>(V, 64 * NB) + 8 * NB : 0;
  for (int attempt = 0;; attempt++) {
    SVO_TRY(ensure(c.lvl_code, cap * 8));
    SVO_TRY(ensure(c.lvl_size, cap * 8));
    SVO_TRY(ensure(c.lvl_mask, cap + 8));  // (+: masks are or-ed as 32-bit words)
    SVO_TRY(ensure(c.lvl_first, cap * 4));
    SVO_TRY(ensure(c.lvl_start, cap * 8));
    SVO_TRY(ensure(c.lvl_pidx, cap * 4));
    SVO_TRY(ensure(c.lvl_sib, cap * 8));
    // meta | per job: root size, root internal size, hazard | single-pass scan status
    const uint64_t meta_words = 2 * 64 + 8 + 3 * (uint64_t)n_jobs;
    // heights from h_tail up go to the single-block tail kernel; on the fast path all
    // heights above the bricks come from the brick codes at once (no level scans)
    const bool up_once = fast;
    int h_tail = H;
    for (int h = h0; h < H && !up_once; h++)
      if (bound[h] <= kTailLevelMax) {
        h_tail = h;
        break;
      }
    uint64_t nup = 0;  // nodes from the bricks up, at most
    for (int h = 4; h <= H && up_once; h++) nup += bound[h];
    // all of it in one launch
    const bool up_small = up_once && NB <= kTailBlock && nup <= kSmallNodes;
    const int h_scan_end = up_once ? h0 : h_tail;  // level scans for h0 .. h_scan_end-1
    uint64_t st_words = 0;
    const uint64_t scan_small = levels ? kLevelScanSmall : kPlainScanSmall;
    for (int h = h0; h < h_scan_end; h++) st_words += scan_single_words(bound[h], scan_small);
    SVO_TRY(ensure(c.lvl_aux, (meta_words + st_words) * 8));
    if (levels) {
      SVO_TRY(ensure(c.lvl_isize, cap * 8));
      SVO_TRY(ensure(c.lvl_cache, cap * 24));
      SVO_TRY(ensure(c.lvl_pstart, cap * 8));
      // null (+ white) record, one per voxel (payload), one per internal node (<= cap)
      SVO_TRY(ensure(c.records2, (n_records + cap) * 32));
    }
    float* out_rec = levels ? c.records2.as<float>() : c.records.as<float>();
    if (!fast) SVO_TRY(ensure(c.lvl_leafp, std::max<uint64_t>(V, 1) * 4));
    const uint64_t node_cap = cap + V + in_brick + n_jobs;
    uint64_t* nodes;
    if (out) {
      SVO_TRY(ensure_keep(*out->nodes, (out->at + node_cap) * 24, out->at * 24, c.stream));
      nodes = out->nodes->as<uint64_t>() + 3 * out->at;
    } else {
      SVO_TRY(ensure(c.nodes, node_cap * 24));
      nodes = c.nodes.as<uint64_t>();
    }
    Arena A{c.lvl_code.as<uint64_t>(), c.lvl_size.as<uint64_t>(), c.lvl_mask.as<uint8_t>(),
            c.lvl_first.as<uint32_t>(), c.lvl_start.as<uint64_t>(), c.lvl_pidx.as<uint32_t>(),
            cap, levels ? c.lvl_isize.as<uint64_t>() : nullptr,
            levels ? c.lvl_cache.as<float>() : nullptr,
            levels ? c.lvl_pstart.as<uint64_t>() : nullptr, c.lvl_sib.as<uint64_t>()};
    unsigned long long* meta = c.lvl_aux.as<unsigned long long>();
    LevelMeta M{meta, meta + 64, meta + 128};
    unsigned long long* root_size = meta + 136;
    unsigned long long* root_isize = root_size + n_jobs;
    unsigned long long* brick_hazard = root_isize + n_jobs;
    // the upper levels' tile scratch (fast path)
    const uint32_t ntiles = (uint32_t)((NB + kUpTile - 1) / kUpTile);
    const uint64_t b_cnt = ((uint64_t)ntiles * kUpLevels * 4 + 255) & ~255ull;
    const uint64_t b_s4 = ((uint64_t)ntiles * 8 + 255) & ~255ull;
    const uint64_t b_end = ((uint64_t)kUpLevels * 8 + 255) & ~255ull;
    if (up_once)
      SVO_TRY(ensure(c.up_tiles, b_cnt + b_s4 + b_end + (uint64_t)n_jobs * kUpLevels * 8));
    // the build's kernels up to its read-back: one graph segment
    SVO_TRY(run_segment(c, [&]() -> hipError_t {
      // n[0] = V, off[1] = 0, flags = 0, root sizes = 0, hazard flags = 0, scan status = 0
      // (the brick path writes what it reads itself)
      if (!up_once)
        SVO_LAUNCH(k_build_init, dim3(1), dim3(256), 0, c.stream, meta, meta_words + st_words, V,
                   job_arg ? d_jobs : (JobDev*)nullptr, job0);
      SVO_TRY(hipGetLastError());

      if (up_small) {
        ktimer_begin(c, "upper_levels");
        SVO_LAUNCH(k_up_small, dim3(1), dim3(kTailBlock), 0, c.stream, A.start, M, T, d_jobs,
                   n_jobs, c.bwords.as<uint64_t>(), c.bcode.as<uint64_t>(),
                   c.bshape.as<uint32_t>(), (uint32_t)NB, H, meta_words, (int)job_arg, job0,
                   root_size, root_isize, brick_hazard,
                   (uint64_t*)((char*)c.up_tiles.p + b_cnt + b_s4 + b_end), node_cap, nodes,
                   c.records.as<float>());
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      } else if (up_once) {
        char* ub = (char*)c.up_tiles.p;
        uint32_t* tile_cnt = (uint32_t*)ub;
        uint64_t* tile_s4 = (uint64_t*)(ub + b_cnt);
        uint64_t* a_end = (uint64_t*)(ub + b_cnt + b_s4);
        uint64_t* job_end = (uint64_t*)(ub + b_cnt + b_s4 + b_end);
        ktimer_begin(c, "upper_levels");
        SVO_LAUNCH(k_up_count, dim3(ntiles), dim3(kUpTile), 0, c.stream, A, T,
                           d_jobs, (int)job_arg, job0, M.flag + 3, c.bwords.as<uint64_t>(),
                           c.bcode.as<uint64_t>(), c.bshape.as<uint32_t>(), NB, H, tile_cnt,
                           tile_s4, brick_hazard);
        SVO_LAUNCH(k_up_scan, dim3(1), dim3(1024), 0, c.stream, A, M, NB, H,
                           tagged ? (JobDev*)nullptr : d_jobs, job0,
                           (const unsigned long long*)brick_hazard, c.records.as<float>(), ntiles,
                           tile_cnt, tile_s4, a_end);
        SVO_LAUNCH(k_up_apply, dim3(ntiles), dim3(kUpTile), 0, c.stream, A, M, T,
                           (const JobDev*)d_jobs, NB, H, (const uint32_t*)tile_cnt,
                           (const uint64_t*)tile_s4, (const uint64_t*)a_end, job_end);
        SVO_LAUNCH(k_up_finish, dim3((unsigned)((nup + 255) / 256)), dim3(256), 0,
                           c.stream, A, M, T, (const JobDev*)d_jobs, H,
                           (const uint64_t*)job_end, root_size);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }

      // ---- bottom-up: heights 1 .. H
      unsigned long long* status = meta + meta_words;
      for (int h = h0; h < h_scan_end; h++) {
        HeadLoad ld{A, M, T, d_jobs, c.codes.as<uint64_t>(), h};
        ParentStore st{A, M, T, d_jobs, c.codes.as<uint64_t>(), c.lvl_leafp.as<uint32_t>(),
                       root_size, root_isize, c.records.as<float>() + 8, h};
        SVO_TRY((scan_single<uint32_t>(ld, st, bound[h], status,
                                       c.counters.as<unsigned long long>() + kCtrError, c.stream,
                                       M.n + h, scan_small)));
        status += scan_single_words(bound[h], scan_small);
      }
      if (!up_once || (tagged && !up_small))
        SVO_LAUNCH(k_levels_tail, dim3(1), dim3(kTailBlock), 0, c.stream, A, M, T, d_jobs,
                         n_jobs, c.codes.as<uint64_t>(), c.lvl_leafp.as<uint32_t>(), root_size,
                         root_isize, c.records.as<float>() + 8, h_tail, H,
                         fast ? brick_hazard : nullptr, node_cap,
                         nodes, c.records.as<float>(), out_rec);
      SVO_TRY(hipGetLastError());
      // ---- top-down: heights H .. 1 (one launch without -levels), then the leaves
      const int hs = std::max(h0, 1);
      if (!levels && !up_small && H >= hs) {
        uint64_t nup = 0;
        for (int h = hs; h <= H; h++) nup += bound[h];
        ktimer_begin(c, "emit_children");
        SVO_LAUNCH(k_emit_upper, dim3((unsigned)std::max<uint64_t>((nup + 255) / 256, 1)),
                           dim3(256), 0, c.stream, A, M, T, (const JobDev*)d_jobs, hs, H, node_cap,
                           nodes);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }
      int h_top = H + 1;  // heights from here up in one launch
      while (levels && h_top > hs && bound[h_top - 1] <= kTopLevelMax) h_top--;
      if (h_top <= H) {
        ktimer_begin(c, "emit_children");
        SVO_LAUNCH(k_emit_levels_top, dim3(1), dim3(kTailBlock), 0, c.stream, A, M, T,
                   (const JobDev*)d_jobs, h_top, H, node_cap, nodes, out_rec);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }
      for (int h = h_top - 1; levels && h >= hs; h--) {
        ktimer_begin(c, "emit_children");
        SVO_LAUNCH(k_emit_level, dim3((unsigned)std::max<uint64_t>((bound[h] + 255) / 256, 1)),
                           dim3(256), 0, c.stream, A, M, T, (const JobDev*)d_jobs, h, node_cap,
                           nodes, out_rec);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }
      if (fast) {
        ktimer_begin(c, "emit_bricks");
        const dim3 eg((unsigned)((NB + kEmitWaves - 1) / kEmitWaves)), eb(kWave * kEmitWaves);
        auto emit = [&](auto kernel) {
          SVO_LAUNCH(kernel, eg, eb, 0, c.stream, A, M, T, (const JobDev*)d_jobs,
                     c.bwords.as<uint64_t>(), c.bcode.as<uint64_t>(), c.bvoff.as<uint64_t>(), NB,
                     node_cap, nodes);
        };
        if (NB > kStageBricks)
          out ? emit(k_emit_bricks<true, true>) : emit(k_emit_bricks<false, true>);
        else
          out ? emit(k_emit_bricks<true, false>) : emit(k_emit_bricks<false, false>);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      } else if (V) {
        ktimer_begin(c, "emit_leaves");
        SVO_LAUNCH(k_emit_leaves, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, c.stream,
                           A, M, T, (const JobDev*)d_jobs, node_cap, c.codes.as<uint64_t>(),
                           c.lvl_leafp.as<uint32_t>(), nodes,
                           c.records.as<float>(), out_rec);
        ktimer_end(c);
        SVO_TRY(hipGetLastError());
      }
      return hipSuccess;
    }));
    unsigned long long flags[4] = {0, 0, 0, 0};
    if (c.build_done_ev) SVO_TRY(hipEventRecord(c.build_done_ev, c.stream));
    {
      const ReadReq rq[3] = {{flags, M.flag, 32},
                             {jd.data(), d_jobs, n_jobs * sizeof(JobDev)},
                             {&c.err_count, c.counters.as<unsigned long long>() + kCtrError, 8}};
      SVO_TRY(read_back(c, rq, 3));
    }
    c.stamp_build = flags[3];
    ktimer_flush(c);
    if (flags[1] && !flags[0]) {
      set_error("internal: node record out of range");
      return hipErrorUnknown;
    }
    if (!flags[0]) {
      c.n_nodes = flags[2];
      break;
    }
    if (attempt > 8) {
      set_error("internal: level arena could not be sized");
      return hipErrorUnknown;
    }
    cap *= 4;
  }
  n_records = 0;
  for (uint32_t j = 0; j < n_jobs; j++) {
    Job& J = c.jobs[j];
    J.n_nodes = jd[j].n_nodes;
    J.nbase = jd[j].nbase;
    J.hazard = (int)jd[j].hazard;
    J.n_data = jd[j].n_data;
    n_records += J.n_data;
  }
  c.n_data = n_records;
  c.data_in_records2 = levels != 0;  // the post-order records are the output
  return hipSuccess;
}

}  // namespace svo
