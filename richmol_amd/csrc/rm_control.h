// richmol_amd: what the kernels with a control wave share (rm_block.hip,
// rm_team.hip): the workgroup's sums and the adaptive rule's metric.
#pragma once

#include "rm_slice.h"

namespace {

constexpr int NT = 1024, NW = NT / 64, NWORK = NW - 1;   // the last wave is the control wave
constexpr int GL = 32;   // Gram matrix order held in LDS (adaptive)

// Sum of NQ values over the workgroup, the same on every thread; one barrier.
// red: [2][NW][4], the halves used in turn.
template <int NQ>
__device__ __forceinline__ void blk_sum(double (&v)[NQ], double (*red)[NW][4], int& half) {
#pragma unroll
  for (int q = 0; q < NQ; ++q) v[q] = wave_allsum(v[q]);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < NQ; ++q) red[half][wv][q] = v[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double t = red[half][lane & 15][q];
    t += dpp_mov<0x128>(t);   // sums over the 16 lanes of a row
    t += dpp_mov<0x124>(t);
    t += dpp_mov<0x122>(t);
    t += dpp_mov<0x121>(t);
    v[q] = t;
  }
  half ^= 1;
}

// LDS of a workgroup besides the vectors.
template <bool FIXED>
struct BlkShared {
  double2 alpha[KMAX];
  double beta[KMAX + 1];
  double2 cf[KMAX];
  double2 gram[FIXED ? 1 : GL * GL];
  double2 cv[FIXED ? 1 : 2 * GL];
  double red[2][NW][4];
  double conv;
};

// The adaptive rule's metric after Krylov vector k (adaptive_metric) for
// k < 16, by one wave: lane 16 q + i takes row i and the columns 4 q .. 4 q + 3
// of the quadratic form; c and c_prev also go to cv (c, then c_prev) as the
// general form keeps them.
__device__ __forceinline__ double metric16(int k, bool breakdown, double2* G, int ld, const double2* alpha,
                                           const double* beta, double2 f, bool herm, double2* cv, double2* tmp) {
  const int lane = threadIdx.x & 63, i = lane & 15, q = lane >> 4;
  if (!breakdown && i < k && q == 0) {
    double2 hv;
    const double2 g1 = G[i * ld + k - 1];
    if (i == k - 1) {
      hv = cconj(alpha[k - 1]);
    } else {
      hv = cscale(beta[i + 1], G[(i + 1) * ld + k - 1]);
      hv = fmac(cconj(alpha[i]), g1, hv);
      if (i > 0) hv = cadd(hv, cscale(beta[i], G[(i - 1) * ld + k - 1]));
    }
    double2 t = csub(hv, cmul(alpha[k - 1], g1));
    if (k >= 2) t = csub(t, cscale(beta[k - 1], G[i * ld + k - 2]));
    const double be = beta[k];
    t = make_double2(t.x / be, t.y / be);
    G[i * ld + k] = t;
    G[k * ld + i] = cconj(t);
  }
  if (lane == 0) G[k * ld + k] = make_double2(1.0, 0.0);
  const double2 c = herm ? expm_row16_herm<false>(k + 1, alpha, beta, f.y, tmp) : expm_row16(k + 1, alpha, beta, f);
  double2 d = make_double2(0.0, 0.0);
  if (i <= k) d = csub(c, i < k ? cv[ld + i] : make_double2(0.0, 0.0));
  if (q == 0) cv[i] = d;
  wave_sync();
  double2 r = make_double2(0.0, 0.0);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int j = 4 * q + u;
    if (i <= k && j <= k) r = fmac(G[i * ld + j], cv[j], r);
  }
  const double part = d.x * r.x + d.y * r.y;
  wave_sync();
  if (q == 0) {
    cv[i] = c;
    cv[ld + i] = c;
  }
  return wave_allsum(part);
}

}  // namespace
