// Host check of the voxelizer's linear classification (svo_walk.h) against the tests it
// stands for: every voxel of a triangle's clamped bbox through the reference's FP32 tests
// (voxelizer.cpp:257-287) and through fast_row / fast_column.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../ooc_svo_builder_amd/csrc/svo_walk.h"

using namespace svo;

static bool passes(const Setup& S, float u, int x, int y, int z) {
  const float px = (float)x * u, py = (float)y * u, pz = (float)z * u;
  const float t = (S.n[0] * px + S.n[1] * py) + S.n[2] * pz;
  if ((t + S.d1) * (t + S.d2) > 0.0f) return false;
  for (int k = 0; k < 3; k++) {
    if ((S.ne[k][0] * px + S.ne[k][1] * py) + S.de[k] < 0.0f) return false;
    if ((S.ne[3 + k][0] * py + S.ne[3 + k][1] * pz) + S.de[3 + k] < 0.0f) return false;
    if ((S.ne[6 + k][0] * pz + S.ne[6 + k][1] * px) + S.de[6 + k] < 0.0f) return false;
  }
  return true;
}

// out: voxels tested, wrong "certain" answers, columns in a row's interval, uncertain columns,
// careful triangles, accepted voxels
extern "C" void walk_check(const float* tris, uint64_t n, float unit, uint64_t gridsize,
                           const int* pmin, const int* pmax, uint64_t* out) {
  VoxParams P{};
  P.unit = unit;
  P.unit_div = 1.0f / unit;
  P.coord_limit = 4.0f * (float)gridsize * unit;
  P.slab_margin = 0.03 + 2.5e-5 * (double)gridsize;
  P.inv_unit = 1.0 / (double)unit;
  for (int k = 0; k < 3; k++) {
    P.pmin[k] = pmin[k];
    P.pmax[k] = pmax[k];
  }
  for (uint64_t q = 0; q < n; q++) {
    Setup S;
    setup_tri(tris + 9 * q, P, S);
    Walk K;
    make_walk(S, P, (uint32_t)q, K);
    FastTri F;
    make_fast(K, P, F);
    const int w = K.w(), ua = w == 0 ? 1 : 0, va = w == 2 ? 1 : 2;
    const int nb = K.i[I_G1V] - K.i[I_G0V] + 1, na = K.i[I_G1U] - K.i[I_G0U] + 1, nc = (int)(F.c.ck >> 16);
    if (na < 1 || nb < 1 || nc < 1) continue;  // nothing to test (an inverted bbox)
    if (F.rf & kFastCareful) out[4]++;
    for (int j = 0; j < nb; j++) {
      FastRow R;
      fast_row(F, j, nb, R);
      if (R.i0 <= R.i1 && (R.i0 < 0 || R.i1 >= na)) out[1]++;
      for (int i = 0; i < na; i++) {
        const bool in_row = i >= R.i0 && i <= R.i1;
        int lo = 0, hi = -1;
        bool sure = true;
        if (in_row) {
          sure = fast_column(F.c, R.p_lo, R.p_hi, R.s_lo, i, lo, hi);
          sure = sure && !(R.first_unsure && i == R.i0) && !(R.last_unsure && i == R.i1) && !R.all;
          const bool careful = F.rf & kFastCareful;
          out[2]++;
          if (careful || (lo <= hi && !sure)) out[3]++;
          if (careful) {
            lo = 0;
            hi = nc - 1;
          }
        }
        for (int k = 0; k < nc; k++) {
          int v[3];
          v[ua] = K.i[I_G0U] + i;
          v[va] = K.i[I_G0V] + j;
          v[w] = K.i[I_G0W] + k;
          const bool want = passes(S, unit, v[0], v[1], v[2]);
          const bool cand = in_row && k >= lo && k <= hi;
          out[0]++;
          out[5] += want;
          if (want && !cand) out[1]++;
          if (!want && cand && sure && !(F.rf & kFastCareful)) out[1]++;
        }
      }
    }
  }
}
