// Triangle set-up of the voxelizer (voxelizer.cpp:189-254), its column walk, and the linear
// form of its tests that classifies whole runs of voxels at once. Everything here runs on
// the host as well, where the classification is checked against the tests themselves.
//
// Every FP32 operation that decides a voxel is in the reference's order (see svo_device.h);
// the classification only ever answers "passes", "fails" or "not certain", the last being
// left to those tests.
#pragma once

#include <cmath>

#include "svo_device.h"

namespace svo {

#define SVO_HD __host__ __device__ __forceinline__

// One voxelize unit: one Morton-range partition of one job (a mesh). A batch voxelizes
// many units in the same launches.
struct VoxParams {
  const float* tris;
  const uint32_t* list;  // partition's triangle indices, nullptr = identity
  uint32_t n;
  int stride;  // floats per record: 9 binary, 21 payload
  uint64_t mstart;
  uint64_t bstart;  // mstart rounded down to a brick: origin of the brick table segment
  int pmin[3], pmax[3];
  float unit, unit_div;
  float coord_limit;  // |vertex| beyond this walks full columns
  double slab_margin; // voxels added on each side of the exact plane slab
  double inv_unit;    // 1 / unit in double
  int small_cols;
  int direct_cols;     // triangles with at most this many columns: walked by their thread
  uint32_t job;        // tag of the unit's codes (bits kJobShift and up)
  int dense;           // 1: voxels in grid8; 0: in pool slots flagged by the touch pass
  int wide;            // dense payload unit: 4-byte cells holding ~(first triangle)
  uint64_t table_base; // first entry of the unit's segment of the brick table
  uint8_t* grid8;      // dense byte grid of the unit (nullptr on the touch path)
};

struct Setup {
  float n[3];
  float d1, d2;
  float ne[9][2];  // edge normals: xy e0..e2, yz e0..e2, zx e0..e2
  float de[9];
  int g0[3], g1[3];
  int w;          // column axis
  bool slab;      // restrict columns to the plane slab
  double nv0, nc, nm;
};

// voxelizer.cpp:189-254 (bbox, clamp, normal, critical point, edge functions) of the nine
// floats at p
template <typename FloatPtr>
SVO_HD void setup_tri(FloatPtr p, const VoxParams& P, Setup& S) {
  const float v0x = p[0], v0y = p[1], v0z = p[2];
  const float v1x = p[3], v1y = p[4], v1z = p[5];
  const float v2x = p[6], v2y = p[7], v2z = p[8];
  const float u = P.unit;
  {
    const float mn0 = min_std(v0x, min_std(v1x, v2x)), mx0 = max_std(v0x, max_std(v1x, v2x));
    const float mn1 = min_std(v0y, min_std(v1y, v2y)), mx1 = max_std(v0y, max_std(v1y, v2y));
    const float mn2 = min_std(v0z, min_std(v1z, v2z)), mx2 = max_std(v0z, max_std(v1z, v2z));
    S.g0[0] = clamp_i(trunc_i32_x86(mn0 * P.unit_div), P.pmin[0], P.pmax[0]);
    S.g0[1] = clamp_i(trunc_i32_x86(mn1 * P.unit_div), P.pmin[1], P.pmax[1]);
    S.g0[2] = clamp_i(trunc_i32_x86(mn2 * P.unit_div), P.pmin[2], P.pmax[2]);
    S.g1[0] = clamp_i(trunc_i32_x86(mx0 * P.unit_div), P.pmin[0], P.pmax[0]);
    S.g1[1] = clamp_i(trunc_i32_x86(mx1 * P.unit_div), P.pmin[1], P.pmax[1]);
    S.g1[2] = clamp_i(trunc_i32_x86(mx2 * P.unit_div), P.pmin[2], P.pmax[2]);
  }
  const float e0x = v1x - v0x, e0y = v1y - v0y, e0z = v1z - v0z;
  const float e1x = v2x - v1x, e1y = v2y - v1y, e1z = v2z - v1z;
  const float e2x = v0x - v2x, e2y = v0y - v2y, e2z = v0z - v2z;
  const float cx = e0y * e1z - e1y * e0z;
  const float cy = e0z * e1x - e1z * e0x;
  const float cz = e0x * e1y - e1x * e0y;
  const float ss = (cx * cx + cy * cy) + cz * cz;
  const float inv = 1.0f / sqrtf(ss);
  const float nx = cx * inv, ny = cy * inv, nz = cz * inv;
  S.n[0] = nx;
  S.n[1] = ny;
  S.n[2] = nz;
  const float ccx = (nx > 0) ? u : 0.0f;
  const float ccy = (ny > 0) ? u : 0.0f;
  const float ccz = (nz > 0) ? u : 0.0f;
  S.d1 = (nx * (ccx - v0x) + ny * (ccy - v0y)) + nz * (ccz - v0z);
  S.d2 = (nx * ((u - ccx) - v0x) + ny * ((u - ccy) - v0y)) + nz * ((u - ccz) - v0z);

  const float E[3][3] = {{e0x, e0y, e0z}, {e1x, e1y, e1z}, {e2x, e2y, e2z}};
  const float V[3][3] = {{v0x, v0y, v0z}, {v1x, v1y, v1z}, {v2x, v2y, v2z}};
#pragma unroll
  for (int k = 0; k < 3; k++) {
    // XY plane (voxelizer.cpp:220-230)
    float a = -1.0f * E[k][1], b = E[k][0];
    if (nz < 0.0f) {
      a = -1.0f * a;
      b = -1.0f * b;
    }
    S.ne[k][0] = a;
    S.ne[k][1] = b;
    S.de[k] = ((-1.0f * (a * V[k][0] + b * V[k][1])) + max_std(0.0f, u * a)) + max_std(0.0f, u * b);
    // YZ plane (:232-242)
    a = -1.0f * E[k][2];
    b = E[k][1];
    if (nx < 0.0f) {
      a = -1.0f * a;
      b = -1.0f * b;
    }
    S.ne[3 + k][0] = a;
    S.ne[3 + k][1] = b;
    S.de[3 + k] = ((-1.0f * (a * V[k][1] + b * V[k][2])) + max_std(0.0f, u * a)) + max_std(0.0f, u * b);
    // ZX plane (:244-254)
    a = -1.0f * E[k][0];
    b = E[k][2];
    if (ny < 0.0f) {
      a = -1.0f * a;
      b = -1.0f * b;
    }
    S.ne[6 + k][0] = a;
    S.ne[6 + k][1] = b;
    S.de[6 + k] = ((-1.0f * (a * V[k][2] + b * V[k][0])) + max_std(0.0f, u * a)) + max_std(0.0f, u * b);
  }

  // column axis and slab restriction
  const float ax = fabsf(nx), ay = fabsf(ny), az = fabsf(nz);
  S.w = (az >= ax && az >= ay) ? 2 : (ax >= ay ? 0 : 1);
  const float L = P.coord_limit;
  const bool finite = (ax <= 2.0f) && (ay <= 2.0f) && (az <= 2.0f);  // false for NaN/inf
  const bool near = fabsf(v0x) <= L && fabsf(v0y) <= L && fabsf(v0z) <= L && fabsf(v1x) <= L &&
                    fabsf(v1y) <= L && fabsf(v1z) <= L && fabsf(v2x) <= L && fabsf(v2y) <= L &&
                    fabsf(v2z) <= L;
  S.slab = finite && near && fmaxf(ax, fmaxf(ay, az)) >= 0.5f;
  S.nv0 = ((double)nx * v0x + (double)ny * v0y) + (double)nz * v0z;
  S.nc = ((double)nx * ccx + (double)ny * ccy) + (double)nz * ccz;
  S.nm = ((double)nx * (u - ccx) + (double)ny * (u - ccy)) + (double)nz * (u - ccz);
}

// ---------------------------------------------------------------- column walk
// A triangle's voxels are tested column by column along its column axis w (the axis of
// the dominant normal component); a column is fixed by its coordinates (a, b) on the two
// other axes ua < va. The per-triangle constants are re-slotted once so that one
// branch-free code path serves all three axes:
//   * plane test t = (n0*px + n1*py) + n2*pz becomes t = (nw*pc + Ka) + Kb with
//     Ka, Kb per column (Kb = +0 when w = z; a zero's sign never changes the decision);
//   * the projection test in the plane across w (3 edges) depends on (pa, pb) only and
//     is evaluated once per column: (h0*pa + h1*pb) + hd;
//   * each edge of the two other planes is (cv*pc + cc*pconst) + de per voxel, where
//     pconst is pb for one of them (plane P) and pa for the other (plane Q).
// Every product and sum is the reference's own (voxelizer.cpp:257-287); only operands of
// single additions are swapped, which is exact in IEEE arithmetic. The products of pb
// (h1*pb, cc*pb of plane P, the plane-test term of b, the slab term of b) are the same
// along a row of columns and are computed once per row.
enum WalkF {
  F_NW = 0, F_D1, F_D2, F_NUA, F_NVA,
  F_H0 = 5, F_H1 = 8, F_HD = 11,
  F_PV = 14, F_PC = 17, F_PD = 20,
  F_QV = 23, F_QC = 26, F_QD = 29,
  F_KA = 32, F_KB, F_ALO, F_AHI,
  kWalkF = 36
};
enum WalkI { I_G0U = 0, I_G1U, I_G0V, I_G1V, I_G0W, I_G1W, I_WS, I_TRI, kWalkI = 8 };
constexpr int kWalkWords = kWalkF + kWalkI;

struct Walk {
  float f[kWalkF];
  int i[kWalkI];
  SVO_HD int w() const { return i[I_WS] & 3; }
  SVO_HD bool slab() const { return (i[I_WS] >> 2) & 1; }
  SVO_HD uint64_t columns() const {
    return (uint64_t)(i[I_G1U] - i[I_G0U] + 1) * (uint64_t)(i[I_G1V] - i[I_G0V] + 1);
  }
  SVO_HD uint64_t work() const {
    return slab() ? columns() : columns() * (uint64_t)(i[I_G1W] - i[I_G0W] + 1);
  }
};

// The plane roles for column axis w, as value selects: the hoisted plane's edges (H0, H1
// in operand order (pa, pb), HD), plane P (its other coordinate is pb) and plane Q (pa)
// with their column-coordinate factor (PV, QV), the other factor (PC, QC) and the offset
// (PD, QD). Edges: xy = ne[0..2], yz = ne[3..5], zx = ne[6..8].
//   w = 2: hoisted xy(pa, pb); P = yz(pb, pc); Q = zx(pc, pa)
//   w = 0: hoisted yz(pa, pb); P = zx(pb, pc); Q = xy(pc, pa)
//   w = 1: hoisted zx(pb, pa); P = yz(pc, pb); Q = xy(pa, pc)
// (A branch per axis is merged by the compiler into an index on the edge arrays, which
// puts them in scratch memory.)
SVO_HD void fill_planes(const Setup& S, Walk& K, int w) {
  const bool w2 = (w == 2), w0 = (w == 0);
  auto pick = [&](float a2, float a0, float a1) { return w2 ? a2 : (w0 ? a0 : a1); };
#pragma unroll
  for (int k = 0; k < 3; k++) {
    K.f[F_H0 + k] = pick(S.ne[k][0], S.ne[3 + k][0], S.ne[6 + k][1]);
    K.f[F_H1 + k] = pick(S.ne[k][1], S.ne[3 + k][1], S.ne[6 + k][0]);
    K.f[F_HD + k] = pick(S.de[k], S.de[3 + k], S.de[6 + k]);
    K.f[F_PV + k] = pick(S.ne[3 + k][1], S.ne[6 + k][1], S.ne[3 + k][0]);
    K.f[F_PC + k] = pick(S.ne[3 + k][0], S.ne[6 + k][0], S.ne[3 + k][1]);
    K.f[F_PD + k] = pick(S.de[3 + k], S.de[6 + k], S.de[3 + k]);
    K.f[F_QV + k] = pick(S.ne[6 + k][0], S.ne[k][0], S.ne[k][1]);
    K.f[F_QC + k] = pick(S.ne[6 + k][1], S.ne[k][1], S.ne[k][0]);
    K.f[F_QD + k] = pick(S.de[6 + k], S.de[k], S.de[k]);
  }
}

// Re-slot a triangle's setup (voxelizer.cpp:189-254, see setup_tri) for the column walk.
SVO_HD void make_walk(const Setup& S, const VoxParams& P, uint32_t tri,
                                          Walk& K) {
  const int w = S.w;
  const int ua = (w == 0) ? 1 : 0;
  const int va = (w == 2) ? 1 : 2;
  fill_planes(S, K, w);
  const float n0 = S.n[0], n1 = S.n[1], n2 = S.n[2];
  const float nw = (w == 0) ? n0 : (w == 1 ? n1 : n2);
  const float nua = (ua == 0) ? n0 : n1;
  const float nva = (va == 1) ? n1 : n2;
  K.f[F_NW] = nw;
  K.f[F_D1] = S.d1;
  K.f[F_D2] = S.d2;
  K.f[F_NUA] = nua;
  K.f[F_NVA] = nva;
  // plane slab in index space along w: c in [ka*a + kb*b + alpha_lo, ... + alpha_hi]
  if (S.slab) {
    const double inw = 1.0 / (double)nw, iu = P.inv_unit;
    const double a1 = -(S.nc - S.nv0) * inw * iu, a2 = -(S.nm - S.nv0) * inw * iu;
    K.f[F_KA] = (float)(-(double)nua * inw);
    K.f[F_KB] = (float)(-(double)nva * inw);
    K.f[F_ALO] = (float)(fmin(a1, a2) - P.slab_margin);
    K.f[F_AHI] = (float)(fmax(a1, a2) + P.slab_margin);
  } else {
    K.f[F_KA] = K.f[F_KB] = K.f[F_ALO] = K.f[F_AHI] = 0.0f;
  }
  // bbox along (ua, va, w) by value selects (a branch per axis would let the compiler
  // index the bbox arrays with w, which puts them in scratch memory)
  const int x0 = S.g0[0], y0 = S.g0[1], z0 = S.g0[2];
  const int x1 = S.g1[0], y1 = S.g1[1], z1 = S.g1[2];
  K.i[I_G0U] = (w == 0) ? y0 : x0;
  K.i[I_G1U] = (w == 0) ? y1 : x1;
  K.i[I_G0V] = (w == 2) ? y0 : z0;
  K.i[I_G1V] = (w == 2) ? y1 : z1;
  K.i[I_G0W] = (w == 0) ? x0 : (w == 1 ? y0 : z0);
  K.i[I_G1W] = (w == 0) ? x1 : (w == 1 ? y1 : z1);
  K.i[I_WS] = w | (S.slab ? 4 : 0);
  K.i[I_TRI] = (int)tri;
}


// ---------------------------------------------------------------- linear form of the tests
// The tests of a voxel (a, b, c) (column coordinates a, b along ua < va, c along the column)
// are signs of functions that are linear in its coordinates: three edge functions in each
// coordinate plane, and the two faces of the plane slab. For a triangle (local coordinates
// i = a - a0, j = b - b0, k = c - c0 from its clamped bbox corner) each becomes a bound
//   on i given j  (the plane across the column axis: H),
//   on k given j  (plane P, whose other coordinate is b),
//   on k given i  (plane Q), and on k given i and j (the slab),
// a lower bound where the function grows with the bounded coordinate, an upper one where it
// falls. The three edge functions of a plane sum to a constant, so there is at least one of
// each kind (slots 1 and 2; slot 3 is of either kind).
//
// Error. An edge test is the sign of fl(fl(h0 * pa) + fl(h1 * pb)) + hd with pa = fl(a u):
// the last addition keeps the sign of its exact sum, so the value it tests differs from the
// real h0 u a + h1 u b + hd by at most 2 eps (|h0| pa + |h1| pb) for the four products and
// eps (|h0| pa + |h1| pb) for the first sum, eps = 2^-24. The plane test's t has three
// products and two sums: at most 4 eps of its terms' magnitudes. The bounds themselves are
// evaluated from a corner value computed in double, with coefficients off by at most 5 eps
// and one rounding: 8 eps of their terms covers that. A bound x with error d then decides
// every integer outside (x - d, x + d); a triangle keeps the largest d of its bounds.
//
// Edges along the bounded axis (their function does not change with it by more than its
// error) bound the other coordinate instead: i in [il, iu], j in [jl, ju], the bbox but for a
// column or a row.
//
// Where a coefficient is zero the test has one coordinate, its values are monotonic in it (every
// rounding is), and the one integer within the error of the bound is decided by the test itself,
// once for the triangle: the bound is then half an integer off. Faces in a voxel plane would
// otherwise leave all their columns uncertain (20,000 boxes of 4 to 40 voxels at 1024: a run 1526 us,
// 1133 so, 1432 with every candidate tested; 500 boxes of 100 to 300: 2781, 1992 and 2363).
//
// A triangle whose bounds are not usable (no slab, non-finite values, an error of a quarter voxel)
// is 'careful': all columns of its rows' intervals go through the tests, all its columns where those
// of plane H are not usable either (2,000 triangles without area of ~5,600 columns at 512: 829 us
// with all columns, 231 so).
constexpr float kEps24 = 5.9604645e-8f;
constexpr float kFar = 1.0e9f;
constexpr float kMaxErr = 0.25f;
enum FastFlag : uint32_t {
  kFastQ3Lower = 1u, kFastH3Lower = 2u, kFastP3Lower = 4u, kFastCareful = 8u,
  kFastIl = 16u, kFastIu = 32u, kFastJl = 64u, kFastJu = 128u,  // that bound's integer is not certain
  kFastNoRows = 1u << 10  // (bits 8 and 9: w)
};
// 28 words: 12 read per column (the last four of them per row too), 16 per row.
struct FastCol {
  float q1A, q1B, q2A, q2B;
  float q3A, q3B, KA, thick;
  float d;       // the largest error of the bounds
  uint32_t qf;   // FastFlag | w << 8 | a0 << 16
  uint32_t ck;   // c0 | (number of k) << 16
  uint32_t tri;
};
struct FastTri {
  float h1A, h1B, h2A, h2B;
  float h3A, h3B, SL, KB;
  float p1A, p1B, p2A, p2B;
  float p3A, p3B;
  uint32_t rf;   // FastFlag | w << 8 | b0 << 16
  uint32_t trim; // number of i | il << 16 | (last i - iu) << 20 | jl << 24 | (last j - ju) << 28
  FastCol c;
};
static_assert(sizeof(FastCol) == 48 && sizeof(FastTri) == 112, "words");
constexpr int kMaxTrim = 15;  // (a triangle trimmed by more is careful)

SVO_HD float fast_rcp(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.0f / x;
#endif
}
SVO_HD float fast_med3(float x, float lo, float hi) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_fmed3f(x, lo, hi);
#else
  return fminf(fmaxf(x, lo), hi);
#endif
}

// The test of an edge whose other coefficient is zero, at integer x of its coordinate
struct AxisTest {
  float coef, D, u;
  int base;
  SVO_HD bool passes(int x) const { return !(coef * ((float)(base + x) * u) + D < 0.0f); }
};
// The integer a bound starts (lower) or ends at, given the outer and the inner one within its
// error: the same, or decided by the test.
SVO_HD int exact_end(const AxisTest& T, int outer, int inner) {
  return outer == inner || T.passes(outer) ? outer : inner;
}

// Integer bounds [lo, hi] on one coordinate, and whether their end integers are certain.
struct IntBounds {
  int lo, hi;
  bool lo_unsure, hi_unsure;
};
// x * coefficient >= 0 beyond x = at (coefficient's sign: lower or upper), error d; exact: T is
// its test
SVO_HD bool add_bound(IntBounds& B, float at, float d, bool lower, bool exact, const AxisTest& T) {
  if (!(d < kMaxErr)) return false;
  const float x = fast_med3(at, -2.0f, 65536.0f);
  if (lower) {
    int o = (int)ceilf(x - d), in = (int)ceilf(x + d);
    if (exact) o = in = exact_end(T, o, in);
    if (o > B.lo || (o == B.lo && in > o)) {
      B.lo_unsure = (in > o) || (o == B.lo && B.lo_unsure);
      B.lo = o;
    } else if (in > B.lo) {
      B.lo_unsure = true;
    }
  } else {
    int o = (int)floorf(x + d), in = (int)floorf(x - d);
    if (exact) o = in = exact_end(T, o, in);
    if (o < B.hi || (o == B.hi && in < o)) {
      B.hi_unsure = (in < o) || (o == B.hi && B.hi_unsure);
      B.hi = o;
    } else if (in < B.hi) {
      B.hi_unsure = true;
    }
  }
  return true;
}
// A bound that does not change along the other coordinate, moved half an integer off the one that
// its test decides (out of the bbox: left where it is).
SVO_HD float exact_bound(const AxisTest& T, float at, float d, bool lower, float n) {
  if (!(at > -1.0f && at < n && d < kMaxErr)) return at;
  if (lower) return (float)exact_end(T, (int)ceilf(at - d), (int)ceilf(at + d)) - 0.5f;
  return (float)exact_end(T, (int)floorf(at + d), (int)floorf(at - d)) + 0.5f;
}

struct Slots {
  float A1, B1, A2, B2, A3, B3;
  bool third_lower;
};
// The three edge functions N0[e] + s[e] x + m[e] p >= 0 (x bounded, nx values; p the other
// coordinate, np values; E[e] the error of the test's value) as bounds on x linear in p;
// functions that hardly change with x bound p. fx, fp, D: the functions' coefficients and
// constants, bx and bp: where x and p start. False: not usable.
SVO_HD bool make_slots(const float s[3], const float m[3], const float N0[3], const float E[3],
                       const float* fx, const float* fp, const float* D, float u, int bx, int bp,
                       float nx, float np, Slots& S, IntBounds& pb, float& d_max) {
  bool ok = true;
  float A[3], B[3], key[3];
#pragma unroll
  for (int e = 0; e < 3; e++) {
    const float sv = s[e];
    ok = ok && (E[e] < 1.0e30f);
    const bool flat = !(fabsf(sv) * nx > E[e]);
    if (!flat) {
      const float r = fast_rcp(sv);
      A[e] = -N0[e] * r;
      B[e] = -m[e] * r;
      key[e] = sv;
      const float d = 1.0001f * E[e] * fabsf(r) + 8.0f * kEps24 * (fabsf(A[e]) + fabsf(B[e]) * np);
      ok = ok && (d < kMaxErr);
      d_max = fmaxf(d_max, d);
      if (fp[e] == 0.0f) A[e] = exact_bound(AxisTest{fx[e], D[e], u, bx}, A[e], d, sv > 0.0f, nx);
    } else {
      A[e] = B[e] = key[e] = 0.0f;
      if (sv == 0.0f && m[e] == 0.0f) {
        ok = ok && (N0[e] >= 0.0f);  // the test's value is its constant, exactly
      } else {
        const float E2 = 2.0f * E[e];
        if (fabsf(m[e]) * np <= E2) {
          ok = ok && (N0[e] >= 2.0f * E2);
        } else {
          const float r = fast_rcp(m[e]);
          const float at = -N0[e] * r;
          ok = add_bound(pb, at, 1.0001f * E2 * fabsf(r) + 8.0f * kEps24 * fabsf(at), m[e] > 0.0f,
                         fx[e] == 0.0f, AxisTest{fp[e], D[e], u, bp}) && ok;
        }
      }
    }
  }
  // slot 1: the steepest rising function, slot 2: the steepest falling one
  const bool m01 = key[0] >= key[1];
  const float kh = m01 ? key[0] : key[1], kl = m01 ? key[1] : key[0];
  const float Ah = m01 ? A[0] : A[1], Bh = m01 ? B[0] : B[1];
  const float Al = m01 ? A[1] : A[0], Bl = m01 ? B[1] : B[0];
  const bool top = key[2] > kh, bot = key[2] < kl;
  const float k1 = top ? key[2] : kh, k2 = bot ? key[2] : kl;
  const float k3 = top ? kh : (bot ? kl : key[2]);
  S.A1 = top ? A[2] : Ah;
  S.B1 = top ? B[2] : Bh;
  S.A2 = bot ? A[2] : Al;
  S.B2 = bot ? B[2] : Bl;
  S.A3 = top ? Ah : (bot ? Al : A[2]);
  S.B3 = top ? Bh : (bot ? Bl : B[2]);
  S.third_lower = k3 >= 0.0f;
  if (!(k1 > 0.0f)) {
    S.A1 = -kFar;
    S.B1 = 0.0f;
  }
  if (!(k2 < 0.0f)) {
    S.A2 = kFar;
    S.B2 = 0.0f;
  }
  if (k3 == 0.0f) {
    S.A3 = -kFar;
    S.B3 = 0.0f;
  }
  return ok;
}

// The linear form of a triangle's walk.
SVO_HD void make_fast(const Walk& K, const VoxParams& P, FastTri& F) {
  const int w = K.w();
  const int a0 = K.i[I_G0U], b0 = K.i[I_G0V], c0 = K.i[I_G0W];
  const int na = K.i[I_G1U] - a0 + 1, nb = K.i[I_G1V] - b0 + 1, nc = K.i[I_G1W] - c0 + 1;
  const float u = P.unit;
  const double ud = (double)u;
  const double pa0 = ud * a0, pb0 = ud * b0, pc0 = ud * c0;
  const float ua = fabsf(u);
  const float pam = ua * (float)(a0 + na - 1), pbm = ua * (float)(b0 + nb - 1),
              pcm = ua * (float)(c0 + nc - 1);
  const float fna = (float)na, fnb = (float)nb, fnc = (float)nc;
  IntBounds ib{0, na - 1, false, false}, jb{0, nb - 1, false, false};
  bool ok = K.slab(), rows_ok;
  float d = 0.0f, d_rows;
  IntBounds jb_rows;
  Slots H, Pp, Q;
  const float k3 = 3.01f * kEps24;
  {
    float s[3], m[3], N[3], E[3];
#pragma unroll
    for (int e = 0; e < 3; e++) {  // bound on i given j
      const float x = K.f[F_H0 + e], y = K.f[F_H1 + e];
      s[e] = x * u;
      m[e] = y * u;
      N[e] = (float)((double)x * pa0 + ((double)y * pb0 + (double)K.f[F_HD + e]));
      E[e] = k3 * (fabsf(x) * pam + fabsf(y) * pbm) + 1e-37f;
    }
    rows_ok = make_slots(s, m, N, E, K.f + F_H0, K.f + F_H1, K.f + F_HD, u, a0, b0, fna, fnb, H, jb, d);
    d_rows = d;
    jb_rows = jb;
    ok = rows_ok && ok;
#pragma unroll
    for (int e = 0; e < 3; e++) {  // bound on k given j
      const float x = K.f[F_PV + e], y = K.f[F_PC + e];
      s[e] = x * u;
      m[e] = y * u;
      N[e] = (float)((double)x * pc0 + ((double)y * pb0 + (double)K.f[F_PD + e]));
      E[e] = k3 * (fabsf(x) * pcm + fabsf(y) * pbm) + 1e-37f;
    }
    ok = make_slots(s, m, N, E, K.f + F_PV, K.f + F_PC, K.f + F_PD, u, c0, b0, fnc, fnb, Pp, jb, d) && ok;
#pragma unroll
    for (int e = 0; e < 3; e++) {  // bound on k given i
      const float x = K.f[F_QV + e], y = K.f[F_QC + e];
      s[e] = x * u;
      m[e] = y * u;
      N[e] = (float)((double)x * pc0 + ((double)y * pa0 + (double)K.f[F_QD + e]));
      E[e] = k3 * (fabsf(x) * pcm + fabsf(y) * pam) + 1e-37f;
    }
    ok = make_slots(s, m, N, E, K.f + F_QV, K.f + F_QC, K.f + F_QD, u, c0, a0, fnc, fna, Q, ib, d) && ok;
  }
  // the slab: k between the zeros of t + d1 and t + d2
  const float nw = K.f[F_NW], nua = K.f[F_NUA], nva = K.f[F_NVA];
  const double t0 = (double)nw * pc0 + ((double)nua * pa0 + (double)nva * pb0);
  const float r = fast_rcp(nw * u), rn = fast_rcp(nw);
  const float z1 = -(float)(t0 + (double)K.f[F_D1]) * r, z2 = -(float)(t0 + (double)K.f[F_D2]) * r;
  F.c.KA = -nua * rn;
  F.KB = -nva * rn;
  F.SL = fminf(z1, z2);
  float SH = fmaxf(z1, z2);
  {
    // 1e-18: a product of two distances below it could underflow to zero in the test
    const float E = 4.01f * kEps24 * (fabsf(nw) * pcm + fabsf(nua) * pam + fabsf(nva) * pbm) + 1e-18f;
    const float ds = 1.0001f * E * fabsf(r) +
                     8.0f * kEps24 * (fabsf(F.SL) + fabsf(SH) + fabsf(F.c.KA) * fna + fabsf(F.KB) * fnb);
    ok = ok && (ds < kMaxErr);
    d = fmaxf(d, ds);
    if (nua == 0.0f && nva == 0.0f && ds < kMaxErr) {  // a face in a voxel plane: t has one term
      auto passes = [&](int k) {
        const float t = nw * ((float)(c0 + k) * u);
        return !((t + K.f[F_D1]) * (t + K.f[F_D2]) > 0.0f);
      };
      if (F.SL > -1.0f && F.SL < fnc) {
        const int o = (int)ceilf(F.SL - ds), in = (int)ceilf(F.SL + ds);
        F.SL = (float)(o == in || passes(o) ? o : in) - 0.5f;
      }
      if (SH > -1.0f && SH < fnc) {
        const int o = (int)floorf(SH + ds), in = (int)floorf(SH - ds);
        SH = (float)(o == in || passes(o) ? o : in) + 0.5f;
      }
    }
    F.c.thick = SH - F.SL;
  }
  int il = max(ib.lo, 0), iu = na - 1 - min(ib.hi, na - 1), jl = max(jb.lo, 0),
      ju = nb - 1 - min(jb.hi, nb - 1);
  ok = ok && (d < kMaxErr) && max(max(il, iu), max(jl, ju)) <= kMaxTrim;
  if (!ok) {  // what plane H says alone
    il = iu = 0;
    jl = min(max(jb_rows.lo, 0), kMaxTrim);
    ju = min(nb - 1 - min(jb_rows.hi, nb - 1), kMaxTrim);
  }
  uint32_t fl = (Q.third_lower ? kFastQ3Lower : 0u) | (H.third_lower ? kFastH3Lower : 0u) |
                (Pp.third_lower ? kFastP3Lower : 0u) | (ok ? 0u : kFastCareful) |
                (rows_ok ? 0u : kFastNoRows);
  // (a bound outside the bbox is certain for every voxel of it)
  fl |= (ib.lo_unsure && ib.lo >= 0 ? kFastIl : 0u) | (ib.hi_unsure && ib.hi < na ? kFastIu : 0u) |
        (jb.lo_unsure && jb.lo >= 0 ? kFastJl : 0u) | (jb.hi_unsure && jb.hi < nb ? kFastJu : 0u);
  fl |= (uint32_t)w << 8;
  F.c.q1A = Q.A1; F.c.q1B = Q.B1; F.c.q2A = Q.A2; F.c.q2B = Q.B2; F.c.q3A = Q.A3; F.c.q3B = Q.B3;
  F.h1A = H.A1; F.h1B = H.B1; F.h2A = H.A2; F.h2B = H.B2; F.h3A = H.A3; F.h3B = H.B3;
  F.p1A = Pp.A1; F.p1B = Pp.B1; F.p2A = Pp.A2; F.p2B = Pp.B2; F.p3A = Pp.A3; F.p3B = Pp.B3;
  F.c.d = ok ? d : d_rows;
  F.c.qf = fl | ((uint32_t)a0 << 16);
  F.rf = fl | ((uint32_t)b0 << 16);
  F.c.ck = (uint32_t)c0 | ((uint32_t)nc << 16);
  F.c.tri = (uint32_t)K.i[I_TRI];
  F.trim = (uint32_t)na | ((uint32_t)il << 16) | ((uint32_t)iu << 20) | ((uint32_t)jl << 24) |
           ((uint32_t)ju << 28);
}

// Row j of a triangle's nb rows: its columns [i0, i1] that are not certain to fail (none: i0 > i1);
// the columns strictly inside are certain to pass the projection test, an end column unless
// it is flagged. all: every column of the row is uncertain. p_lo, p_hi: plane P's bounds on
// k along the row; s_lo: the slab's lower bound at i = 0.
struct FastRow {
  int i0, i1;
  bool first_unsure, last_unsure, all;
  float p_lo, p_hi, s_lo;
};
SVO_HD void fast_row(const FastTri& F, int j, int nb, FastRow& R) {
  const int na = (int)(F.trim & 0xFFFFu);
  const float fj = (float)j, fna = (float)na;
  const float h3 = fmaf(F.h3B, fj, F.h3A), p3 = fmaf(F.p3B, fj, F.p3A);
  const bool hl = F.rf & kFastH3Lower, pl = F.rf & kFastP3Lower;
  float L = fmaf(F.h1B, fj, F.h1A), U = fmaf(F.h2B, fj, F.h2A);
  L = fmaxf(L, hl ? h3 : -kFar);
  U = fminf(U, hl ? kFar : h3);
  // into [-1, na] before the conversions; an integer of the bbox keeps its answer
  L = fast_med3(L, -1.0f, fna + 1.0f);
  U = fast_med3(U, -2.0f, fna);
  const int lo_o = (int)ceilf(L - F.c.d), lo_i = (int)ceilf(L + F.c.d);
  const int hi_o = (int)floorf(U + F.c.d), hi_i = (int)floorf(U - F.c.d);
  const int il = (int)(F.trim >> 16) & 15, iu = na - 1 - ((int)(F.trim >> 20) & 15);
  const int jl = (int)(F.trim >> 24) & 15, ju = nb - 1 - (int)(F.trim >> 28);
  R.i0 = max(lo_o, il);
  R.i1 = min(hi_o, iu);
  R.first_unsure = lo_i > R.i0 || (R.i0 == il && (F.rf & kFastIl));
  R.last_unsure = hi_i < R.i1 || (R.i1 == iu && (F.rf & kFastIu));
  R.all = (j == jl && (F.rf & kFastJl)) || (j == ju && (F.rf & kFastJu));
  if (j < jl || j > ju) R.i1 = R.i0 - 1;
  if (F.rf & kFastCareful) {
    R.all = true;
    if (F.rf & kFastNoRows) {
      R.i0 = 0;
      R.i1 = na - 1;
    }
  }
  R.p_lo = fmaxf(fmaf(F.p1B, fj, F.p1A), pl ? p3 : -kFar);
  R.p_hi = fminf(fmaf(F.p2B, fj, F.p2A), pl ? kFar : p3);
  R.s_lo = fmaf(F.KB, fj, F.SL);
}

// Column i of a row: the voxels k in [lo, hi] that are not certain to fail (none: lo > hi),
// and whether every one of them is certain to pass the plane tests of P and Q and the slab.
SVO_HD bool fast_column(const FastCol& F, float p_lo, float p_hi, float s_lo, int i, int& lo,
                        int& hi) {
  const float fi = (float)i;
  const float q3 = fmaf(F.q3B, fi, F.q3A);
  const float s = fmaf(F.KA, fi, s_lo);
  const bool ql = F.qf & kFastQ3Lower;
  float L = fmaxf(fmaxf(p_lo, s), fmaf(F.q1B, fi, F.q1A));
  float U = fminf(fminf(p_hi, s + F.thick), fmaf(F.q2B, fi, F.q2A));
  L = fmaxf(L, ql ? q3 : -kFar);
  U = fminf(U, ql ? kFar : q3);
  const int nc = (int)(F.ck >> 16);
  L = fast_med3(L, -1.0f, (float)nc + 1.0f);
  U = fast_med3(U, -2.0f, (float)nc);
  lo = (int)ceilf(L - F.d);
  hi = (int)floorf(U + F.d);
  const int lo_i = (int)ceilf(L + F.d), hi_i = (int)floorf(U - F.d);
  lo = max(lo, 0);
  hi = min(hi, nc - 1);
  return max(lo_i, 0) == lo && min(hi_i, nc - 1) == hi;
}

}  // namespace svo
