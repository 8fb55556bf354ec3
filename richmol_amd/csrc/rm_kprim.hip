// richmol_amd: the Kronecker-block operator in the primitive symmetric-top
// basis, and the batched Lanczos propagator on it.
//
// A K block of a rigid rotor is K_w = C1^H P_w C2 with C the states'
// coefficients over primitive k and P_w the tensor's matrix between primitive
// functions, which only couples k1 - k2 = s, |s| <= w <= 2
// (labtens.py:482-496).  C is unitary and acts on k alone, so the whole Krylov
// recurrence of a step can run on X' = X C^T: the wavepackets are transformed
// once before it (k_pr_tr, matrix cores) and what the step adds to them once
// after it, and inside it the operator is a stencil,
//   Y'[J1](m1, k1) = sum_{J2, w} sum_sigma MF_sigma(m1) sum_s P_s(k1) X'[J2](m1 - sigma, k1 - s),
// at most 5 x (5 + 5) complex multiply-adds per element and tensor rank instead
// of a row of dense products over all k (9 x 161 per element at J = 80 for a
// dipole and a polarizability).  The same operator, the same Lanczos
// recurrence (tdse.py:417-486): results agree to rounding, as C is unitary.
// The state's own part of a step, c_0 phi, is taken from psi and does not go
// through C and back: C is unitary to 1e-15 only, which left an error of 1e-15
// after one step and of 3-4e-13 after 1 000 (the dense form's norm drifts by
// 0.3-0.9e-13 in these).  Now only what a step adds carries it: 1.6e-16 after one
// step at J = 80 (dense form 2.0e-16), after 1 000 steps at J <= 20 a norm
// drift of 0.2-1.0e-13 in a field of 1e9 V/m, 1.3-2.1e-13 in one of 5e9; at
// J = 80 in one of 1e8 7.6e-14 (dense form 7.9e-14).
//
// Vectors are (wavepacket, internal order) arrays of complex values, as the
// caller's rows: J blocks of (m, k), k fastest.  The basis is kept as the
// unnormalised W_k with V_k = W_k / beta_k, so an iteration moves W (read), Y
// (written), then Y, W_k, W_{k-1} (read) and W_{k+1} (written): 6 passes of
// 16 n bytes per wavepacket.
//
// Measured (MI355X, J <= 80 all m: 708 561 states, 64 wavepackets, Krylov
// dimension 12, dipole + full polarizability in an XY field): 20.4 ms per step
// FP64, 17.6 ms with FP32 products, where the dense form (m-mixed input stored,
// rocBLAS products) takes 157.5 and 112.2 ms; J <= 31, 16 wavepackets, adaptive,
// <cos^2> read: 0.36 ms per step against 4.8.  Of the 20.4 ms the stencils take
// 10.8 (0.90 each), the vector updates 6.0 (0.55 each: 2.9 GB at 5.2 TB/s), the
// final combination 1.7 (8.9 GB at 5.2 TB/s), the transforms 1.7.  FP32 error
// against 64-bit dense products 2.6e-9 (dense form 3.2e-9).

#include <algorithm>
#include <cmath>
#include <vector>

#include "rm_kprim.h"

namespace {

constexpr int SR = 8;            // output rows (m1) of one wave of the stencil
constexpr int SW = 4;            // waves per workgroup
constexpr int MPAD = SR;         // MF rows are padded to a multiple of this
constexpr int EB = 2048;         // elements per workgroup of the vector kernels
constexpr int TR = 32, TC = 64, TK = 16;   // rows, columns, depth of a transform tile

// s and sigma sets the stencil is compiled for; a block runs the smallest
// one that holds its own
enum { S_0 = 0, S_1 = 1, S_02 = 2, S_2 = 3 };                    // {0}, {-1..1}, {-2,0,2}, {-2..2}
enum { G_0 = 0, G_PM1 = 1, G_1 = 2, G_02 = 3, G_2 = 4, G_NONE = 5 };   // {0}, {-1,1}, {-1..1}, {-2,0,2}, {-2..2}, {}

struct PTask {          // one source block of an output J
  int32_t J2, dpad;     // J2; row length of its MF table
  int32_t spat, blk;
  int64_t voff2;        // J2 block in a wavepacket's row
  int64_t p_off;        // [5][2 J1 + 1]
  int64_t mf_off;       // [5][dpad]
};

struct PJ {             // one output J
  int32_t J, task0, ntask, nb;   // nb: wavepackets side by side in a wave
  int64_t voff;
};

struct PMf {            // MF assembly of one block
  int32_t dm1, nsig, ncart, slot0, dpad;
  int32_t sig[5];
  int32_t pe;           // P is kept times 2^-pe, so that its largest element is in [1, 2)
  int64_t d_off, mf_off;
};

}  // namespace

struct KPrim {
  std::vector<int32_t> Js;
  std::vector<int64_t> voff;
  int64_t n = 0;
  bool cplx = false;               // some C has an imaginary part
  int32_t nblk = 0;
  std::vector<PMf> h_mfd;
  const double2* mdiag = nullptr;  // the plan's
  std::vector<PJ> h_pj;
  PJ* d_pj = nullptr;
  PTask* d_task = nullptr;
  PMf* d_mfd = nullptr;
  int32_t* d_gpat = nullptr;       // per block: the sigma set of the step's MF
  double2* d_p = nullptr;
  float2* d_p32 = nullptr;
  double2* d_mf = nullptr;
  float2* d_mf32 = nullptr;
  double* d_T = nullptr;           // per J the forward (C^T) and backward (conj C) matrices, re then im planes
  int64_t* d_toff = nullptr;
  // per number of wavepackets (the last one used): stencil items, transform tiles
  int32_t ncols = 0;
  int4* d_items = nullptr;
  int64_t items_cap = 0, nitems = 0;
  int32_t nslots = 0;              // stencil partial sums per wavepacket
  int4* d_tiles = nullptr;
  int64_t tiles_cap = 0, ntiles = 0;
  char* ws = nullptr;
  size_t ws_bytes = 0;
  int32_t* h_run = nullptr;        // pinned: wavepackets going on, per iteration
  int32_t kpred = 0;               // dimension of the last adaptive step
};

namespace {

__host__ __device__ inline int64_t jd(int32_t J) { return 2 * (int64_t)J + 1; }
size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

template <typename T> struct C2;
template <> struct C2<double> { using V = double2; };
template <> struct C2<float> { using V = float2; };

__device__ __forceinline__ double sh1(double v, bool up) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return up ? __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, 0x130, 0xf, 0xf, true),
                               __builtin_amdgcn_update_dpp(0, lo, 0x130, 0xf, 0xf, true))
            : __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, 0x138, 0xf, 0xf, true),
                               __builtin_amdgcn_update_dpp(0, lo, 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float sh1(float v, bool up) {
  const int i = __float_as_int(v);
  return __int_as_float(up ? __builtin_amdgcn_update_dpp(0, i, 0x130, 0xf, 0xf, true)
                           : __builtin_amdgcn_update_dpp(0, i, 0x138, 0xf, 0xf, true));
}
// lane l <- lane l + 1 (up) or l - 1; 0 past the wave's ends
template <typename V>
__device__ __forceinline__ V shc(V v, bool up) {
  v.x = sh1(v.x, up);
  v.y = sh1(v.y, up);
  return v;
}
// acc + a b as four fused multiply-adds
__device__ __forceinline__ double2 mac(double2 a, double2 b, double2 c) {
  return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
__device__ __forceinline__ float2 mac(float2 a, float2 b, float2 c) {
  return make_float2(fmaf(a.x, b.x, fmaf(-a.y, b.y, c.x)), fmaf(a.x, b.y, fmaf(a.y, b.x, c.y)));
}
__device__ __forceinline__ void conv2(double2 v, double2& o) { o = v; }
__device__ __forceinline__ void conv2(double2 v, float2& o) { o = make_float2((float)v.x, (float)v.y); }

// MF_sigma(m1) of every block for the step's field products, times 2^(pe + e),
// in the padded [sigma + 2][m1] tables (entries of sigmas a block lacks stay zero), and the
// smallest compiled sigma set that holds the non-zero ones: a field along Z
// leaves sigma = 0, one in the XY plane +-1 (dipole) or 0, +-2 (polarizability).
__global__ __launch_bounds__(256) void k_pr_mf(const PMf* __restrict__ d, const double2* __restrict__ mdiag,
                                               const double2* __restrict__ fp, int e, double2* __restrict__ mf,
                                               float2* __restrict__ mf32, int32_t* __restrict__ gpat) {
  const PMf b = d[blockIdx.x];
  int mask = 0;
  for (int t = 0; t < b.nsig; ++t)
    for (int m = threadIdx.x; m < b.dm1; m += blockDim.x) {
      double2 acc = make_double2(0.0, 0.0);
      for (int c = 0; c < b.ncart; ++c)
        acc = cfma(fp[b.slot0 + c], mdiag[b.d_off + ((int64_t)t * b.ncart + c) * b.dm1 + m], acc);
      acc = make_double2(scalbn(acc.x, b.pe + e), scalbn(acc.y, b.pe + e));
      const int64_t o = b.mf_off + (int64_t)(b.sig[t] + 2) * b.dpad + m;
      mf[o] = acc;
      mf32[o] = make_float2((float)acc.x, (float)acc.y);
      if (!(acc.x == 0.0 && acc.y == 0.0)) mask |= 1 << (b.sig[t] + 2);
    }
  __shared__ int s_mask;
  if (threadIdx.x == 0) s_mask = 0;
  __syncthreads();
  if (mask) atomicOr(&s_mask, mask);
  __syncthreads();
  if (threadIdx.x == 0) {
    const int k = s_mask;
    gpat[blockIdx.x] = k == 0 ? G_NONE : k == 4 ? G_0 : !(k & ~10) ? G_PM1 : !(k & ~14) ? G_1 : !(k & ~21) ? G_02 : G_2;
  }
}

// One source block's contribution to the SR output rows of a wave: per output
// row the m mixing z = sum_sigma MF_sigma(m1) x(m1 - sigma), then the k mixing
// acc += sum_s P_s z(k1 - s) -- the neighbours in k are the neighbouring lanes.
// (The k mixing first, on the SR + 4 source rows, costs 37 % more operations
// for a full rank-2 tensor: 0.97 against 0.89 ms per matvec.  Loading the
// rows once for all blocks of one J2 took 1.00 ms: more registers, fewer waves.)
// xp: this lane's element of source row m2 = 0; row r of the window is
// m2 = m0 + r - (largest sigma).
template <typename T, int SP, int GP>
__device__ __forceinline__ void sten_task(const double2* __restrict__ xp, int m2_0, int dm2, int ld2,
                                          const typename C2<T>::V* __restrict__ P, int d1,
                                          const typename C2<T>::V* __restrict__ mf, int dpad,
                                          typename C2<T>::V (&acc)[SR]) {
  using V = typename C2<T>::V;
  constexpr int GM = GP == G_0 ? 0 : (GP == G_PM1 || GP == G_1) ? 1 : 2;   // largest sigma
  constexpr int NR = SR + 2 * GM;
  V x[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    // rows outside J2 have MF = 0: any row of the wavepacket stands in
    const int m2 = min(max(m2_0 + r - GM, 0), dm2 - 1);
    conv2(xp[(int64_t)m2 * ld2], x[r]);
  }
  V p[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int s = i - 2;
    if (s == 0 || (SP == S_1 && (s == 1 || s == -1)) || (SP == S_02 && (s == 2 || s == -2)) || SP == S_2)
      p[i] = P[(int64_t)i * d1];
  }
#pragma unroll
  for (int o = 0; o < SR; ++o) {
    V z{0, 0};
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const int sg = i - 2;
      const bool use = GP == G_0 ? sg == 0 : GP == G_PM1 ? (sg == 1 || sg == -1) : GP == G_1 ? (sg >= -1 && sg <= 1)
                       : GP == G_02 ? (sg == 0 || sg == 2 || sg == -2) : true;
      if (use) z = mac(mf[(int64_t)i * dpad + o], x[o + GM - sg < 0 || o + GM - sg >= NR ? 0 : o + GM - sg], z);
    }
    acc[o] = mac(p[2], z, acc[o]);
    if constexpr (SP != S_0) {
      const V dn = shc(z, false), up = shc(z, true);   // k1 - 1, k1 + 1
      if constexpr (SP == S_1 || SP == S_2) {
        acc[o] = mac(p[3], dn, acc[o]);
        acc[o] = mac(p[1], up, acc[o]);
      }
      if constexpr (SP == S_02 || SP == S_2) {
        acc[o] = mac(p[4], shc(dn, false), acc[o]);
        acc[o] = mac(p[0], shc(up, true), acc[o]);
      }
    }
  }
}

template <typename T, int SP>
__device__ __forceinline__ void sten_g(int gp, const double2* xp, int m2_0, int dm2, int ld2,
                                       const typename C2<T>::V* P, int d1, const typename C2<T>::V* mf, int dpad,
                                       typename C2<T>::V (&acc)[SR]) {
  switch (gp) {
    case G_0: sten_task<T, SP, G_0>(xp, m2_0, dm2, ld2, P, d1, mf, dpad, acc); break;
    case G_PM1: sten_task<T, SP, G_PM1>(xp, m2_0, dm2, ld2, P, d1, mf, dpad, acc); break;
    case G_1: sten_task<T, SP, G_1>(xp, m2_0, dm2, ld2, P, d1, mf, dpad, acc); break;
    case G_02: sten_task<T, SP, G_02>(xp, m2_0, dm2, ld2, P, d1, mf, dpad, acc); break;
    case G_2: sten_task<T, SP, G_2>(xp, m2_0, dm2, ld2, P, d1, mf, dpad, acc); break;
    default: break;
  }
}

// Y = H(F) (ib W) and the partials of vdot(Y, ib W).  One wave per item:
// SR rows m1 of one output J and 60 consecutive k1 of one wavepacket, or all
// k1 of nb wavepackets side by side when a row with its margins fits a wave
// (2 J + 5 <= 64).  Two margin lanes on either side of a row or chunk supply
// the neighbours in k.  The rows' MF values are the same on every lane (scalar
// loads); P_s(k1) is loaded once per source block and used for all rows.
// Items are ordered by wavepacket, then J, and split into 8 contiguous parts,
// one per XCD (workgroups go round robin over the XCDs): the source blocks
// J1 - 2 .. J1 + 2 of a wavepacket (2 MB at J = 80) are then re-read from that
// XCD's L2.
// part[b][slot]: (re, im) partials, slot = item within a wavepacket; NULL: none.
template <typename T, typename YT>
__global__ __launch_bounds__(64 * SW) void k_pr_sten(const int4* __restrict__ items, int nitems, int seg,
                                                     const PJ* __restrict__ pj, const PTask* __restrict__ tasks,
                                                     const int32_t* __restrict__ gpat,
                                                     const typename C2<T>::V* __restrict__ P,
                                                     const typename C2<T>::V* __restrict__ mf,
                                                     const double2* __restrict__ W, int64_t n, int32_t ncols,
                                                     const double* __restrict__ ib, typename C2<YT>::V* __restrict__ Y,
                                                     double2* __restrict__ part, int32_t nslots) {
  using V = typename C2<T>::V;
  __shared__ double2 s_red[SW][64];
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int q = (blockIdx.x >> 3) * SW + wv;
  const int itm = (blockIdx.x & 7) * seg + q;
  if (q >= seg || itm >= nitems) return;
  const int4 it = items[itm];
  const PJ j = pj[it.x];
  const int m0 = it.y & 0xffff, kc = it.y >> 16, b0 = it.z;
  const int J = j.J, d = 2 * J + 1;
  int i1, b;
  bool live;
  if (j.nb > 1 || d + 4 <= 64) {
    const int bi = lane / (d + 4);
    i1 = lane - bi * (d + 4) - 2;
    b = b0 + bi;
    live = bi < j.nb && b < ncols && i1 >= 0 && i1 < d;
  } else {
    i1 = kc * 60 - 2 + lane;
    b = b0;
    live = lane >= 2 && lane < 62 && i1 < d;
  }
  const int bb = min(b, ncols - 1);
  const double2* xb = W + (int64_t)bb * n;
  const int ic = min(max(i1, 0), d - 1);
  V acc[SR];
#pragma unroll
  for (int r = 0; r < SR; ++r) acc[r] = V{0, 0};
  for (int t = 0; t < j.ntask; ++t) {
    const PTask tk = tasks[j.task0 + t];
    const int gp = gpat[tk.blk];
    if (gp == G_NONE) continue;
    const int d2 = 2 * tk.J2 + 1;
    const int i2 = min(max(i1 - J + tk.J2, 0), d2 - 1);
    const double2* xp = xb + tk.voff2 + i2;
    const V* Pt = P + tk.p_off + ic;
    const V* mt = mf + tk.mf_off + m0;
    const int m2_0 = m0 - J + tk.J2;
    switch (tk.spat) {
      case S_0: sten_g<T, S_0>(gp, xp, m2_0, d2, d2, Pt, d, mt, tk.dpad, acc); break;
      case S_1: sten_g<T, S_1>(gp, xp, m2_0, d2, d2, Pt, d, mt, tk.dpad, acc); break;
      case S_02: sten_g<T, S_02>(gp, xp, m2_0, d2, d2, Pt, d, mt, tk.dpad, acc); break;
      default: sten_g<T, S_2>(gp, xp, m2_0, d2, d2, Pt, d, mt, tk.dpad, acc); break;
    }
  }
  const double s = ib ? ib[bb] : 1.0;
  double a0 = 0.0, a1 = 0.0;
  const int64_t e0 = j.voff + ic;
#pragma unroll
  for (int r = 0; r < SR; ++r) {
    const int m1 = m0 + r;
    if (live && m1 < d) {
      const int64_t e = e0 + (int64_t)m1 * d;
      const double yr = s * (double)acc[r].x, yi = s * (double)acc[r].y;
      if (Y) {
        typename C2<YT>::V yo;
        conv2(make_double2(yr, yi), yo);
        Y[(int64_t)b * n + e] = yo;
      }
      if (part) {
        const double2 w = xb[e];
        const double vr = s * w.x, vi = s * w.y;
        a0 += yr * vr + yi * vi;
        a1 += yr * vi - yi * vr;
      }
    }
  }
  if (!part) return;
  if (j.nb == 1) {
    a0 = wave_allsum(a0);
    a1 = wave_allsum(a1);
    if (lane == 0) part[(int64_t)b0 * nslots + it.w] = make_double2(a0, a1);
  } else {
    s_red[wv][lane] = make_double2(a0, a1);
    wave_sync();
    if (lane < j.nb && b0 + lane < ncols) {
      double2 t = make_double2(0.0, 0.0);
      for (int i = 0; i < d + 4; ++i) t = cadd(t, s_red[wv][lane * (d + 4) + i]);
      part[(int64_t)(b0 + lane) * nslots + it.w] = t;
    }
  }
}

// out[r][c] = sum_q in[r][q] T[q][c] per J on the matrix cores, rows r =
// (wavepacket, m); FWD: in = phase x rows of psi, T = C^T; backward: T =
// conj(C), and with c0 (the step's first coefficient per wavepacket, ldc0
// apart) out = phase x (c0 phase out + result), psi's own part of the step.  TR x TC output tiles, the re and im parts of a
// row as two rows of the real product (a real C) -- a quarter of the flops
// of the complex product in real form -- or with a complex C two products
// more.  One wave per 16 columns; the next TK-deep slice is loaded while the
// current one is multiplied.  (FP64 16x16x4: lane l supplies A[l % 16][l / 16]
// and B[l / 16][l % 16], item v of lane l is D[l / 16 + 4 v][l % 16].)
template <bool CT, bool FWD>
__global__ __launch_bounds__(256) void k_pr_tr(const int4* __restrict__ tiles, const PJ* __restrict__ pj,
                                               const int64_t* __restrict__ toff, const double* __restrict__ T,
                                               const double2* __restrict__ in, int64_t ldi, double2* __restrict__ out,
                                               int64_t ldo, const double2* __restrict__ ph, int32_t ncols,
                                               const double2* __restrict__ c0_, int32_t ldc0) {
  typedef double V4 __attribute__((ext_vector_type(4)));
  constexpr int NP = CT ? 2 : 1;
  __shared__ double sA[2][2][TK][TR + 1];
  __shared__ double sB[2][NP][TK][TC];
  const int4 tl = tiles[blockIdx.x];
  const PJ j = pj[tl.x];
  const int d = 2 * j.J + 1;
  const int64_t M = (int64_t)ncols * d;
  const int64_t r0 = (int64_t)tl.y * TR;
  const int c0 = tl.z * TC;
  const double* Tj = T + toff[tl.x] + (FWD ? 0 : (int64_t)NP * d * d);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  // loads of one slice: two complex inputs and four T values (per plane) per thread
  const int qa = t & 15;
  int64_t ra[2];
  bool rv[2];
  int64_t pa[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int64_t r = r0 + (t >> 4) + 16 * u;
    rv[u] = r < M;
    const int64_t b = rv[u] ? r / d : 0, m = rv[u] ? r - b * d : 0;
    ra[u] = b * ldi + j.voff + m * d;
    pa[u] = j.voff + m * d;
  }
  double2 ga[2];
  double gb[NP][4];
  auto fetch = [&](int q0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      double2 v = make_double2(0.0, 0.0);
      if (rv[u] && q0 + qa < d) {
        v = in[ra[u] + q0 + qa];
        if (FWD && ph) v = cmul(v, ph[pa[u] + q0 + qa]);
      }
      ga[u] = v;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = t + 256 * u, q = q0 + e / TC, c = c0 + e % TC;
#pragma unroll
      for (int p = 0; p < NP; ++p) gb[p][u] = (q < d && c < d) ? Tj[(int64_t)p * d * d + (int64_t)q * d + c] : 0.0;
    }
  };
  auto stash = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      sA[buf][0][qa][(t >> 4) + 16 * u] = ga[u].x;
      sA[buf][1][qa][(t >> 4) + 16 * u] = ga[u].y;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = t + 256 * u;
#pragma unroll
      for (int p = 0; p < NP; ++p) sB[buf][p][e / TC][e % TC] = gb[p][u];
    }
  };
  V4 acc[2][2];   // [re / im][row block]
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 2; ++r) acc[a][r] = V4{0, 0, 0, 0};
  const int nch = (d + TK - 1) / TK;
  fetch(0);
  stash(0);
  __syncthreads();
  for (int ch = 0; ch < nch; ++ch) {
    const int cur = ch & 1;
    if (ch + 1 < nch) fetch((ch + 1) * TK);
#pragma unroll
    for (int ks = 0; ks < TK / 4; ++ks) {
      const int kq = ks * 4 + (lane >> 4);
      const double br = sB[cur][0][kq][w * 16 + (lane & 15)];
      const double bi = CT ? sB[cur][NP - 1][kq][w * 16 + (lane & 15)] : 0.0;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const double ar = sA[cur][0][kq][r * 16 + (lane & 15)], ai = sA[cur][1][kq][r * 16 + (lane & 15)];
        acc[0][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, acc[0][r], 0, 0, 0);
        acc[1][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, acc[1][r], 0, 0, 0);
        if constexpr (CT) {
          acc[0][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, acc[0][r], 0, 0, 0);
          acc[1][r] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, acc[1][r], 0, 0, 0);
        }
      }
    }
    if (ch + 1 < nch) stash(cur ^ 1);
    __syncthreads();
  }
  const int c = c0 + w * 16 + (lane & 15);
  if (c >= d) return;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t row = r0 + r * 16 + (lane >> 4) + 4 * v;
      if (row >= M) continue;
      const int64_t b = row / d, m = row - b * d;
      double2 o = make_double2(acc[0][r][v], acc[1][r][v]);
      double2* q = out + b * ldo + j.voff + m * d + c;
      if (!FWD) {
        const double2 p = ph ? ph[j.voff + m * d + c] : make_double2(1.0, 0.0);
        if (c0_) o = mac(c0_[b * ldc0], ph ? cmul(*q, p) : *q, o);
        if (ph) o = cmul(o, p);
      }
      *q = o;
    }
}

// Start of a step's recurrence: per wavepacket ib_0 = 1, beta_0 = 0, and the
// adaptive rule's counters.
__global__ void k_pr_begin(int32_t ncols, int32_t kcap, double* __restrict__ ibs, double* __restrict__ beta,
                           int32_t* __restrict__ kdone, int32_t* __restrict__ running) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (running && b < kcap) running[b] = 0;
  if (b >= ncols) return;
  ibs[b] = 1.0;
  beta[(int64_t)b * (kcap + 1)] = 0.0;
  if (kdone) kdone[b] = 0;
}

// Partials of |W|^2, one per workgroup; UPD: first W = Y - alpha V_k - beta V_{k-1}
// (V = ib W), in place of Y when Y is FP64.
template <bool UPD, typename YT>
__global__ __launch_bounds__(256) void k_pr_upd(int64_t n, const typename C2<YT>::V* Y, const double2* __restrict__ Wk,
                                                const double2* __restrict__ Wp, const double2* __restrict__ alpha,
                                                const double* __restrict__ beta, const double* __restrict__ ibs,
                                                int32_t ncols, int32_t it, int32_t kcap, double2* W,
                                                double* __restrict__ part) {
  const int b = blockIdx.y;
  const int64_t base = (int64_t)b * n;
  double2 al = make_double2(0.0, 0.0);
  double be = 0.0;
  if (UPD) {
    const double ib = ibs[(int64_t)it * ncols + b];
    al = cscale(ib, alpha[(int64_t)b * kcap + it]);
    if (it > 0) be = beta[(int64_t)b * (kcap + 1) + it] * ibs[(int64_t)(it - 1) * ncols + b];
  }
  double acc = 0.0;
  const int64_t i0 = (int64_t)blockIdx.x * EB + threadIdx.x;
#pragma unroll
  for (int u = 0; u < EB / 256; ++u) {
    const int64_t i = i0 + 256 * u;
    if (i < n) {
      double2 w;
      if (UPD) {
        const typename C2<YT>::V y = Y[base + i];
        const double2 v = Wk[base + i];
        w = csub(make_double2((double)y.x, (double)y.y), cmul(al, v));
        if (it > 0) w = csub(w, cscale(be, Wp[base + i]));
        W[base + i] = w;
      } else {
        w = Wk[base + i];
      }
      acc += w.x * w.x + w.y * w.y;
    }
  }
  __shared__ double red[4];
  acc = wave_allsum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) part[(int64_t)b * gridDim.x + blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// beta_{it+1} and 1/beta per wavepacket from the partials (one wave each).
// An exact breakdown gives ib = 0, a zero vector in place of the reference's
// restart vector (its coefficient in exp(fT) e0 is exactly zero).
// it < 0: G_00 = |V_0|^2 of the adaptive rule and c_prev = [1] instead.
__global__ __launch_bounds__(64) void k_pr_beta(const double* __restrict__ part, int32_t np, int32_t ncols, int32_t it,
                                                int32_t kcap, double* __restrict__ beta, double* __restrict__ ibs,
                                                double2* __restrict__ G, double2* __restrict__ cb) {
  const int b = blockIdx.x, lane = threadIdx.x;
  double s = 0.0;
  for (int i = lane; i < np; i += 64) s += part[(int64_t)b * np + i];
  s = wave_allsum(s);
  if (lane != 0) return;
  if (it < 0) {
    G[(int64_t)b * kcap * kcap] = make_double2(s, 0.0);
    cb[(int64_t)b * 2 * kcap + kcap] = make_double2(1.0, 0.0);
  } else {
    const double be = sqrt(s);
    beta[(int64_t)b * (kcap + 1) + it + 1] = be;
    ibs[(int64_t)(it + 1) * ncols + b] = be != 0.0 ? 1.0 / be : 0.0;
  }
}

// alpha_it per wavepacket from the stencil's partials (one wave each) and,
// under the adaptive rule from it = 1 on, the stopping rule for dimension
// it + 1 (tdse.py:466-476): Gram column it, c = exp(f T) e0 and conv = |u_it -
// u_{it-1}|^2; a stopped wavepacket keeps its coefficients (times ib) while
// the others go on.
__global__ __launch_bounds__(64) void k_pr_alpha(const double2* __restrict__ part, int32_t np, int32_t ncols,
                                                 int32_t it, int32_t kcap, double2* __restrict__ alpha,
                                                 const double* __restrict__ beta, const double* __restrict__ ibs,
                                                 int rule, double2 f, double tol, int32_t maxorder,
                                                 double2* __restrict__ G, double2* __restrict__ cb,
                                                 int32_t* __restrict__ kdone, double2* __restrict__ coef,
                                                 int32_t* __restrict__ status, int32_t* __restrict__ running) {
  __shared__ double2 s_a[KMAX];
  __shared__ double s_b[KMAX + 1];
  const int b = blockIdx.x, lane = threadIdx.x;
  double2 s = make_double2(0.0, 0.0);
  for (int i = lane; i < np; i += 64) s = cadd(s, part[(int64_t)b * np + i]);
  s.x = wave_allsum(s.x);
  s.y = wave_allsum(s.y);
  if (lane == 0) alpha[(int64_t)b * kcap + it] = s;
  if (!rule || it < 1 || kdone[b] != 0) return;
  for (int i = lane; i <= it; i += 64) {
    s_a[i] = i == it ? s : alpha[(int64_t)b * kcap + i];
    s_b[i] = beta[(int64_t)b * (kcap + 1) + i];
  }
  wave_sync();
  double2* Gb = G + (int64_t)b * kcap * kcap;
  double2* c = cb + (int64_t)b * 2 * kcap;
  const bool brk = !(s_b[it] != 0.0);
  if (brk)
    for (int i = lane; i < it; i += 64) {
      Gb[i * kcap + it] = make_double2(0.0, 0.0);
      Gb[it * kcap + i] = make_double2(0.0, 0.0);
    }
  wave_sync();
  const double conv = adaptive_metric<false>(it, brk, Gb, kcap, s_a, s_b, f, c, c + kcap);
  wave_sync();
  if (!(it + 1 < maxorder && conv > tol)) {
    for (int i = lane; i <= it; i += 64)
      coef[(int64_t)b * kcap + i] = cscale(ibs[(int64_t)i * ncols + b], c[kcap + i]);
    if (lane == 0) {
      kdone[b] = it + 1;
      if (it + 1 >= maxorder && status) status[b] |= RM_NOT_CONVERGED;
    }
  } else if (lane == 0) {
    atomicAdd(running + it, 1);
  }
}

// exp(f T) e0 times ib per wavepacket (one wave each), fixed dimension m
__global__ __launch_bounds__(64) void k_pr_expm(const double2* __restrict__ alpha, const double* __restrict__ beta,
                                                const double* __restrict__ ibs, int32_t ncols, int32_t m, int32_t kcap,
                                                double2 f, double2* __restrict__ coef) {
  __shared__ double2 s_a[KMAX];
  __shared__ double s_b[KMAX + 1];
  __shared__ double2 s_c[KMAX];
  const int b = blockIdx.x, l = threadIdx.x;
  for (int i = l; i < m; i += 64) {
    s_a[i] = alpha[(int64_t)b * kcap + i];
    s_b[i] = beta[(int64_t)b * (kcap + 1) + i];
  }
  wave_sync();
  if (m == 1) {
    if (l == 0) s_c[0] = make_double2(1.0, 0.0);
  } else {
    expm_e0_any(m, s_a, s_b, f, s_c);
  }
  wave_sync();
  for (int i = l; i < m; i += 64) coef[(int64_t)b * kcap + i] = cscale(ibs[(int64_t)i * ncols + b], s_c[i]);
}

// W_0 <- sum_{j > 0} coef_j W_j (kd: the wavepacket's own dimension, or NULL: m)
__global__ __launch_bounds__(256) void k_pr_comb(int64_t n, double2* W0, int64_t vstride,
                                                 const double2* __restrict__ coef, int32_t m, int32_t kcap,
                                                 const int32_t* __restrict__ kd, int32_t* __restrict__ kused) {
  const int b = blockIdx.y;
  if (kd) m = kd[b];
  if (kused && blockIdx.x == 0 && threadIdx.x == 0) kused[b] = m;
  const int64_t base = (int64_t)b * n;
  const double2* cf = coef + (int64_t)b * kcap;
  const int64_t i0 = (int64_t)blockIdx.x * EB + threadIdx.x;
#pragma unroll 4
  for (int u = 0; u < EB / 256; ++u) {
    const int64_t i = i0 + 256 * u;
    if (i >= n) break;
    double2 s = make_double2(0.0, 0.0);
    for (int q = 1; q < m; ++q) s = mac(cf[q], W0[q * vstride + base + i], s);
    W0[base + i] = s;
  }
}

// A step without field: psi = P P psi (tdse.py:368-380 with the expv skipped)
__global__ void k_pr_phase2(int64_t n, double2* __restrict__ psi, int64_t ld, const double2* __restrict__ ph,
                            int32_t* __restrict__ kused) {
  const int b = blockIdx.y;
  if (kused && blockIdx.x == 0 && threadIdx.x == 0) kused[b] = 0;
  if (!ph) return;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double2* q = psi + (int64_t)b * ld + i;
    *q = cmul(cmul(*q, ph[i]), ph[i]);
  }
}

__global__ void k_pr_ifill(int32_t* __restrict__ x, int32_t n, int32_t v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}

// ex[b] = <S_b|Y_b>: the partials hold vdot(Y, S), its conjugate
__global__ __launch_bounds__(64) void k_pr_ofin(const double2* __restrict__ part, int32_t np,
                                                double2* __restrict__ ex) {
  const int b = blockIdx.x, lane = threadIdx.x;
  double2 s = make_double2(0.0, 0.0);
  for (int i = lane; i < np; i += 64) s = cadd(s, part[(int64_t)b * np + i]);
  s.x = wave_allsum(s.x);
  s.y = wave_allsum(s.y);
  if (lane == 0) ex[b] = make_double2(s.x, -s.y);
}

// Stencil items and transform tiles for ncols wavepackets (kept for the next
// call with as many).
int prim_lists(KPrim* p, int32_t ncols) {
  if (p->ncols == ncols) return RM_OK;
  std::vector<int4> items, tiles;
  const int nJ = (int)p->Js.size();
  int32_t slot = 0;
  for (int a = 0; a < nJ; ++a) {
    const PJ& j = p->h_pj[a];
    const int d = (int)jd(j.J);
    const int nc = d + 4 <= 64 ? 1 : (d + 59) / 60;
    for (int m0 = 0; m0 < d; m0 += SR)
      for (int c = 0; c < nc; ++c, ++slot)
        for (int b = 0; b < ncols; b += j.nb) items.push_back(make_int4(a, m0 | (c << 16), b, slot));
    const int64_t nrt = ((int64_t)ncols * d + TR - 1) / TR, nct = (d + TC - 1) / TC;
    for (int64_t rt = 0; rt < nrt; ++rt)
      for (int64_t ct = 0; ct < nct; ++ct) tiles.push_back(make_int4(a, (int)rt, (int)ct, 0));
  }
  // by wavepacket, then (within one) in J order
  std::stable_sort(items.begin(), items.end(), [](const int4& x, const int4& y) { return x.z < y.z; });
  // the longest products first
  std::stable_sort(tiles.begin(), tiles.end(), [](const int4& x, const int4& y) { return x.x > y.x; });
  if (items.size() > (size_t)INT32_MAX / 2 || tiles.size() > (size_t)INT32_MAX)
    return fail(RM_ERR_ARG, "too many work items for %d wavepackets", ncols);
  p->ncols = 0;
  int rc;
  if ((rc = grow(&p->d_items, &p->items_cap, (int64_t)items.size()))) return rc;
  if ((rc = grow(&p->d_tiles, &p->tiles_cap, (int64_t)tiles.size()))) return rc;
  // earlier launches may still read the lists
  HIPCHK(hipDeviceSynchronize());
  HIPCHK(hipMemcpy(p->d_items, items.data(), sizeof(int4) * items.size(), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(p->d_tiles, tiles.data(), sizeof(int4) * tiles.size(), hipMemcpyHostToDevice));
  p->nitems = (int64_t)items.size();
  p->ntiles = (int64_t)tiles.size();
  p->nslots = slot;
  p->ncols = ncols;
  return RM_OK;
}

struct PWork {
  double2 *W, *alpha, *coef, *G, *cb, *part;
  double *beta, *ibs, *epart;
  float2* Yf;
  int32_t *kdone, *running;
  int64_t vs;
};

// m Krylov vectors (FP64: the product of W_k goes where W_{k+1} will be; a
// matvec alone needs two)
int prim_work(KPrim* p, int32_t ncols, int32_t m, bool f32, bool adaptive, PWork* w) {
  const int64_t vs = p->n * ncols;
  const int64_t ne = (p->n + EB - 1) / EB;
  const size_t b_vec = al256(sizeof(double2) * (size_t)vs * (size_t)(f32 ? m : std::max(m, 2)));
  const size_t b_yf = f32 ? al256(sizeof(float2) * (size_t)vs) : 0;
  const size_t b_part = al256(sizeof(double2) * (size_t)ncols * p->nslots);
  const size_t b_ep = al256(sizeof(double) * (size_t)ncols * ne);
  const size_t b_al = al256(sizeof(double2) * (size_t)ncols * m);
  const size_t b_be = al256(sizeof(double) * (size_t)ncols * (m + 1));
  const size_t b_g = adaptive ? al256(sizeof(double2) * (size_t)ncols * m * m) : 0;
  const size_t b_cb = adaptive ? al256(sizeof(double2) * (size_t)ncols * 2 * m) : 0;
  const size_t b_kd = al256(sizeof(int32_t) * (size_t)ncols) + al256(sizeof(int32_t) * (size_t)(m + 1));
  const size_t need = b_vec + b_yf + b_part + b_ep + 2 * b_al + 2 * b_be + b_g + b_cb + b_kd;
  if (p->ws_bytes < need) {
    if (p->ws) {
      HIPCHK(hipDeviceSynchronize());
      HIPCHK(hipFree(p->ws));
      p->ws = nullptr;
      p->ws_bytes = 0;
    }
    HIPCHK(hipMalloc((void**)&p->ws, need));
    p->ws_bytes = need;
  }
  char* c = p->ws;
  auto take = [&](size_t b) { char* r = c; c += b; return r; };
  w->W = (double2*)take(b_vec);
  w->Yf = (float2*)take(b_yf);
  w->part = (double2*)take(b_part);
  w->epart = (double*)take(b_ep);
  w->alpha = (double2*)take(b_al);
  w->coef = (double2*)take(b_al);
  w->beta = (double*)take(b_be);
  w->ibs = (double*)take(b_be);
  w->G = (double2*)take(b_g);
  w->cb = (double2*)take(b_cb);
  w->kdone = (int32_t*)take(al256(sizeof(int32_t) * (size_t)ncols));
  w->running = (int32_t*)take(al256(sizeof(int32_t) * (size_t)(m + 1)));
  w->vs = vs;
  return RM_OK;
}

// The step's operator is taken times 2^e so that its elements are of order 1,
// and the exponent factor f times 2^-e: exact, and in FP32 no product of the
// unnormalised vectors leaves the range whatever the units of H and the field
// (in joules 1e9 V/m x 1e-21 J x 1e-30 C m is not a normal number).
int step_exponent(const KPrim* p, const double* fprod) {
  double top = 0.0;
  for (const PMf& b : p->h_mfd)
    for (int c = 0; c < b.ncart; ++c)
      for (int q = 0; q < 2; ++q) top = std::max(top, scalbn(std::fabs(fprod[2 * (b.slot0 + c) + q]), b.pe));
  return top > 0.0 && std::isfinite(top) ? -std::ilogb(top) : 0;
}

int launch_mf(KPrim* p, const double2* fp, int e, hipStream_t s) {
  if (p->nblk)
    hipLaunchKernelGGL(k_pr_mf, dim3((unsigned)p->nblk), dim3(256), 0, s, p->d_mfd, p->mdiag, fp, e, p->d_mf,
                       p->d_mf32, p->d_gpat);
  HIPCHK(hipGetLastError());
  return RM_OK;
}

// T: precision of the stencil, YT: of its output
template <typename T, typename YT>
int launch_sten(KPrim* p, const double2* W, int32_t ncols, const double* ib, void* Y, double2* part, hipStream_t s) {
  const int seg = (int)((p->nitems + 7) / 8);
  const unsigned grid = 8u * (unsigned)((seg + SW - 1) / SW);
  const typename C2<T>::V *P, *mf;
  if constexpr (sizeof(T) == 4) {
    P = p->d_p32;
    mf = p->d_mf32;
  } else {
    P = p->d_p;
    mf = p->d_mf;
  }
  hipLaunchKernelGGL((k_pr_sten<T, YT>), dim3(grid), dim3(64 * SW), 0, s, p->d_items, (int)p->nitems, seg, p->d_pj,
                     p->d_task, p->d_gpat, P, mf, W, p->n, ncols, ib, (typename C2<YT>::V*)Y, part, p->nslots);
  HIPCHK(hipGetLastError());
  return RM_OK;
}

int launch_tr(KPrim* p, bool fwd, const double2* in, int64_t ldi, double2* out, int64_t ldo, const double2* ph,
              int32_t ncols, hipStream_t s, const double2* c0 = nullptr, int32_t ldc0 = 0) {
  const dim3 g((unsigned)p->ntiles), b(256);
#define RM_TR(CT, FWD)                                                                                          \
  hipLaunchKernelGGL((k_pr_tr<CT, FWD>), g, b, 0, s, p->d_tiles, p->d_pj, p->d_toff, p->d_T, in, ldi, out, ldo, \
                     ph, ncols, c0, ldc0)
  if (p->cplx) {
    if (fwd) RM_TR(true, true);
    else RM_TR(true, false);
  } else {
    if (fwd) RM_TR(false, true);
    else RM_TR(false, false);
  }
#undef RM_TR
  HIPCHK(hipGetLastError());
  return RM_OK;
}

}  // namespace

void kprim_free(KPrim* p) {
  if (!p) return;
  void* bufs[] = {p->d_pj, p->d_task, p->d_mfd, p->d_gpat, p->d_p, p->d_p32, p->d_mf, p->d_mf32, p->d_T, p->d_toff,
                  p->d_items, p->d_tiles, p->ws};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  if (p->h_run) (void)hipHostFree(p->h_run);
  delete p;
}

int kprim_create(KPrim** out, const std::vector<int32_t>& Js, const std::vector<int64_t>& voff, int64_t n,
                 const std::vector<KPrimBlock>& blk, const double2* mdiag, const double* C, const double* P) {
  *out = nullptr;
  KPrim* p = new (std::nothrow) KPrim();
  if (!p) return fail(RM_ERR_ALLOC, "primitive-basis operator: host allocation");
  p->Js = Js;
  p->voff = voff;
  p->n = n;
  p->nblk = (int32_t)blk.size();
  p->mdiag = mdiag;
  const int nJ = (int)Js.size();
  // transforms: T forward [s][k] = C[k][s], backward [k][s] = conj(C[k][s]); re plane, then im
  int64_t cpos = 0;
  for (int a = 0; a < nJ; ++a) cpos += jd(Js[a]) * jd(Js[a]);
  for (int64_t i = 0; i < cpos && !p->cplx; ++i) p->cplx = C[2 * i + 1] != 0.0;
  const int np = p->cplx ? 2 : 1;
  std::vector<double> T((size_t)(2 * np * cpos));
  std::vector<int64_t> toff;
  cpos = 0;
  for (int a = 0; a < nJ; ++a) {
    const int64_t d = jd(Js[a]);
    toff.push_back(2 * np * cpos);
    double* fw = T.data() + 2 * np * cpos;
    double* bw = fw + np * d * d;
    for (int64_t k = 0; k < d; ++k)
      for (int64_t s = 0; s < d; ++s) {
        const double cr = C[2 * (cpos + k * d + s)], ci = C[2 * (cpos + k * d + s) + 1];
        fw[s * d + k] = cr;
        bw[k * d + s] = cr;
        if (p->cplx) {
          fw[d * d + s * d + k] = ci;
          bw[d * d + k * d + s] = -ci;
        }
      }
    cpos += d * d;
  }
  // tasks per output J, its blocks ordered by J2
  std::vector<PTask> tasks;
  std::vector<PMf> mfd(blk.size());
  std::vector<int64_t> poff(blk.size());
  int64_t ppos = 0, mpos = 0;
  for (size_t q = 0; q < blk.size(); ++q) {
    const int64_t d1 = jd(blk[q].J1);
    poff[q] = ppos;
    ppos += 5 * d1;
    PMf& m = mfd[q];
    m.dm1 = (int32_t)d1;
    m.dpad = (int32_t)((d1 + MPAD - 1) / MPAD * MPAD);
    m.nsig = blk[q].nsig;
    m.ncart = blk[q].ncart;
    m.slot0 = blk[q].slot0;
    for (int t = 0; t < 5; ++t) m.sig[t] = t < m.nsig ? blk[q].sig[t] : 0;
    m.pe = 0;
    m.d_off = blk[q].d_off;
    m.mf_off = mpos;
    mpos += 5 * (int64_t)m.dpad;
  }
  for (int a = 0; a < nJ; ++a) {
    PJ j;
    j.J = Js[a];
    const int d = (int)jd(Js[a]);
    j.nb = d + 4 <= 64 ? 64 / (d + 4) : 1;
    j.voff = voff[a];
    j.task0 = (int32_t)tasks.size();
    std::vector<int> qs;
    for (size_t q = 0; q < blk.size(); ++q)
      if (blk[q].J1 == Js[a]) qs.push_back((int)q);
    std::stable_sort(qs.begin(), qs.end(), [&](int x, int y) { return blk[x].J2 < blk[y].J2; });
    for (int q : qs) {
      PTask t;
      t.J2 = blk[q].J2;
      t.dpad = mfd[q].dpad;
      t.blk = q;
      t.voff2 = voff[std::lower_bound(Js.begin(), Js.end(), t.J2) - Js.begin()];
      t.p_off = poff[q];
      t.mf_off = mfd[q].mf_off;
      int mask = 0;
      double top = 0.0;
      for (int s = 0; s < 5; ++s)
        for (int64_t k = 0; k < d; ++k) {
          const double* v = P + 2 * (poff[q] + s * (int64_t)d + k);
          if (v[0] != 0.0 || v[1] != 0.0) mask |= 1 << s;
          top = std::max(top, std::max(std::fabs(v[0]), std::fabs(v[1])));
        }
      mfd[q].pe = top > 0.0 && std::isfinite(top) ? std::ilogb(top) : 0;
      t.spat = !(mask & ~4) ? S_0 : !(mask & ~14) ? S_1 : !(mask & ~21) ? S_02 : S_2;
      tasks.push_back(t);
    }
    j.ntask = (int32_t)tasks.size() - j.task0;
    p->h_pj.push_back(j);
  }
  std::vector<double> ps(P, P + 2 * ppos);
  for (size_t q = 0; q < blk.size(); ++q)
    for (int64_t i = 2 * poff[q]; i < 2 * (poff[q] + 5 * (int64_t)mfd[q].dm1); ++i) ps[i] = scalbn(ps[i], -mfd[q].pe);
  const std::vector<float> p32(ps.begin(), ps.end());
  p->h_mfd = mfd;
  const std::vector<double2> zero((size_t)std::max<int64_t>(mpos, 1), make_double2(0.0, 0.0));
  int rc;
  if ((rc = upload(&p->d_T, T.data(), (int64_t)T.size())) || (rc = upload(&p->d_toff, toff.data(), nJ)) ||
      (rc = upload(&p->d_pj, p->h_pj.data(), nJ)) || (rc = upload(&p->d_task, tasks.data(), (int64_t)tasks.size())) ||
      (rc = upload(&p->d_mfd, mfd.data(), (int64_t)mfd.size())) ||
      (rc = upload(&p->d_p, (const double2*)ps.data(), ppos)) || (rc = upload(&p->d_p32, (const float2*)p32.data(), ppos)) ||
      (rc = upload(&p->d_mf, zero.data(), (int64_t)zero.size())) ||
      (rc = upload(&p->d_mf32, (const float2*)zero.data(), (int64_t)zero.size())) ||
      (rc = upload(&p->d_gpat, (const int32_t*)nullptr, (int64_t)blk.size()))) {
    kprim_free(p);
    return rc;
  }
  if (hipHostMalloc((void**)&p->h_run, sizeof(int32_t) * (KMAX + 1)) != hipSuccess) {
    p->h_run = nullptr;
    kprim_free(p);
    return fail(RM_ERR_HIP, "primitive-basis operator: pinned allocation failed");
  }
  *out = p;
  return RM_OK;
}

int kprim_matvec(KPrim* p, const double2* x, double2* y, int64_t ld, int32_t ncols, const double2* fprod, bool f32,
                 hipStream_t s) {
  int rc;
  PWork w;
  if ((rc = prim_lists(p, ncols)) || (rc = prim_work(p, ncols, 1, false, false, &w))) return rc;
  if ((rc = launch_mf(p, fprod, 0, s)) || (rc = launch_tr(p, true, x, ld, w.W, p->n, nullptr, ncols, s))) return rc;
  double2* Y = w.W + w.vs;
  rc = f32 ? launch_sten<float, double>(p, w.W, ncols, nullptr, Y, nullptr, s)
           : launch_sten<double, double>(p, w.W, ncols, nullptr, Y, nullptr, s);
  if (rc) return rc;
  return launch_tr(p, false, Y, p->n, y, ld, nullptr, ncols, s);
}

int kprim_propagate(KPrim* p, double2* psi, int64_t ld, int32_t ncols, int64_t nsteps, int32_t nslot,
                    const double* fprod, const double2* d_fp, double2 f, const double2* phase, int32_t krylov_fixed,
                    int32_t maxorder, double tol, int32_t* kused, int32_t* status, bool f32, KPrim* obs,
                    const double2* d_ofp, double2* ex, hipStream_t s) {
  const bool adaptive = krylov_fixed == 0;
  const int32_t m = adaptive ? maxorder : krylov_fixed;
  int rc;
  PWork w;
  if ((rc = prim_lists(p, ncols)) || (rc = prim_work(p, ncols, m, f32, adaptive, &w))) return rc;
  if (obs && ((rc = prim_lists(obs, ncols)) || (rc = launch_mf(obs, d_ofp, 0, s)))) return rc;
  const unsigned ne = (unsigned)((p->n + EB - 1) / EB);
  const dim3 eg(ne, (unsigned)ncols), eb(256), cg((unsigned)ncols), cb(64);
  const bool rule = adaptive && m > 1;   // maxorder 1: V_0 itself, as a fixed dimension
  const dim3 bg(grid_for(std::max(ncols, m), 256));
  for (int64_t st = 0; st < nsteps; ++st) {
    int32_t* ku = kused ? kused + st * ncols : nullptr;
    bool field = false;
    for (int32_t c = 0; c < nslot && !field; ++c)
      field = fprod[2 * (st * nslot + c)] != 0.0 || fprod[2 * (st * nslot + c) + 1] != 0.0;
    if (!field) {
      hipLaunchKernelGGL(k_pr_phase2, dim3(std::min<unsigned>(ne, 256), (unsigned)ncols), eb, 0, s, p->n, psi, ld,
                         phase, ku);
      HIPCHK(hipGetLastError());
    } else {
      const int e = step_exponent(p, fprod + 2 * st * nslot);
      const double2 fe = make_double2(scalbn(f.x, -e), scalbn(f.y, -e));
      if ((rc = launch_mf(p, d_fp + st * nslot, e, s))) return rc;
      if ((rc = launch_tr(p, true, psi, ld, w.W, p->n, phase, ncols, s))) return rc;
      hipLaunchKernelGGL(k_pr_begin, bg, eb, 0, s, ncols, m, w.ibs, w.beta, rule ? w.kdone : nullptr,
                         rule ? w.running : nullptr);
      if (rule) {
        hipLaunchKernelGGL((k_pr_upd<false, double>), eg, eb, 0, s, p->n, (const double2*)nullptr, w.W,
                           (const double2*)nullptr, w.alpha, w.beta, w.ibs, ncols, 0, m, (double2*)nullptr, w.epart);
        hipLaunchKernelGGL(k_pr_beta, cg, cb, 0, s, w.epart, (int)ne, ncols, -1, m, w.beta, w.ibs, w.G, w.cb);
      }
      int32_t kdim = m;
      for (int32_t it = 0; it < m; ++it) {
        double2* Wk = w.W + it * w.vs;
        const double2* Wp = it > 0 ? Wk - w.vs : Wk;
        const double* ib = w.ibs + (int64_t)it * ncols;
        const bool last = it + 1 == m;   // its product is only needed for alpha
        rc = f32 ? launch_sten<float, float>(p, Wk, ncols, ib, last ? nullptr : w.Yf, w.part, s)
                 : launch_sten<double, double>(p, Wk, ncols, ib, last ? nullptr : Wk + w.vs, w.part, s);
        if (rc) return rc;
        hipLaunchKernelGGL(k_pr_alpha, cg, cb, 0, s, w.part, p->nslots, ncols, it, m, w.alpha, w.beta, w.ibs,
                           rule ? 1 : 0, fe, tol, maxorder, w.G, w.cb, w.kdone, w.coef, status, w.running);
        if (rule && it >= 1 && (it + 1 >= p->kpred || last)) {
          // the counts of wavepackets going on after each iteration so far: the
          // host waits for them from the previous step's dimension on
          // (iterations a shorter step did not need change nothing: a stopped
          // wavepacket keeps its coefficients)
          HIPCHK(hipMemcpyAsync(p->h_run, w.running, sizeof(int32_t) * (size_t)(it + 1), hipMemcpyDeviceToHost, s));
          HIPCHK(hipStreamSynchronize(s));
          if (p->h_run[it] == 0) {
            kdim = it + 1;
            p->kpred = kdim;
            for (int32_t q = 1; q <= it; ++q)
              if (p->h_run[q] == 0) {
                p->kpred = q + 1;
                break;
              }
            break;
          }
        }
        if (last) break;
        if (f32)
          hipLaunchKernelGGL((k_pr_upd<true, float>), eg, eb, 0, s, p->n, w.Yf, Wk, Wp, w.alpha, w.beta, w.ibs, ncols,
                             it, m, Wk + w.vs, w.epart);
        else
          hipLaunchKernelGGL((k_pr_upd<true, double>), eg, eb, 0, s, p->n, Wk + w.vs, Wk, Wp, w.alpha, w.beta, w.ibs,
                             ncols, it, m, Wk + w.vs, w.epart);
        hipLaunchKernelGGL(k_pr_beta, cg, cb, 0, s, w.epart, (int)ne, ncols, it, m, w.beta, w.ibs, w.G, w.cb);
      }
      if (!rule) {
        hipLaunchKernelGGL(k_pr_expm, cg, cb, 0, s, w.alpha, w.beta, w.ibs, ncols, m, m, fe, w.coef);
        if (adaptive && status)   // maxorder 1 is reached at once
          hipLaunchKernelGGL(k_pr_ifill, dim3(grid_for(ncols, 256)), dim3(256), 0, s, status, ncols,
                             RM_NOT_CONVERGED);
      }
      hipLaunchKernelGGL(k_pr_comb, eg, eb, 0, s, p->n, w.W, w.vs, w.coef, kdim, m,
                         rule ? (const int32_t*)w.kdone : nullptr, ku);
      HIPCHK(hipGetLastError());
      if ((rc = launch_tr(p, false, w.W, p->n, psi, ld, phase, ncols, s, w.coef, m))) return rc;
    }
    if (obs) {
      // <S|O|S> in the observable's primitive basis: the wavepackets once more
      // forward, its stencil with its partial sums (FP64, output not kept)
      if ((rc = launch_tr(obs, true, psi, ld, w.W, p->n, nullptr, ncols, s))) return rc;
      if ((rc = launch_sten<double, double>(obs, w.W, ncols, nullptr, nullptr, w.part, s))) return rc;
      hipLaunchKernelGGL(k_pr_ofin, cg, cb, 0, s, w.part, obs->nslots, ex + st * ncols);
      HIPCHK(hipGetLastError());
    }
  }
  return RM_OK;
}
