// richmol_amd: device code shared by the kernels on the sliced operator
// (rm_block.hip, rm_wave.hip): pairs of entries and the small exponential.
#pragma once

#include "rm_common.h"

namespace {

// a lane's pair of entries: values v0, v1 (real or complex) in the matvec's
// precision
template <bool F32, bool REAL> struct PairT;
template <> struct PairT<false, true> { using T = double2; };
template <> struct PairT<true, true> { using T = float2; };
template <> struct PairT<false, false> { struct T { double2 a, b; }; };
template <> struct PairT<true, false> { using T = float4; };

__device__ __forceinline__ double2 fmac(double2 a, double2 b, double2 c) {
  return make_double2(fma(a.x, b.x, fma(-a.y, b.y, c.x)), fma(a.x, b.y, fma(a.y, b.x, c.y)));
}
// acc += pair . (x0, x1)
__device__ __forceinline__ void pair_mac(double2 p, double2 x0, double2 x1, double2& acc) {
  acc.x = fma(p.y, x1.x, fma(p.x, x0.x, acc.x));
  acc.y = fma(p.y, x1.y, fma(p.x, x0.y, acc.y));
}
// (FP32 entries: the vector and the sum stay FP64.  Their own loads are what
// FP32 saves; the gathers and sums in FP32 were no faster, and added one by one
// they lost up to 1.8 times more than the sums of 16 lanes per row did.  What
// is rounded is the step's F B; with one slot k_blk holds B_0 rounded for the
// run, whose error is the same at every step: 1.1e-7 after 200 steps)
__device__ __forceinline__ void pair_mac(float2 p, double2 x0, double2 x1, double2& acc) {
  pair_mac(make_double2(p.x, p.y), x0, x1, acc);
}
__device__ __forceinline__ void pair_mac(const PairT<false, false>::T& p, double2 x0, double2 x1, double2& acc) {
  acc = fmac(p.b, x1, fmac(p.a, x0, acc));
}
__device__ __forceinline__ void pair_mac(float4 p, double2 x0, double2 x1, double2& acc) {
  acc = fmac(make_double2(p.z, p.w), x1, fmac(make_double2(p.x, p.y), x0, acc));
}
// a pair's value as the compiler must take it from here on
__device__ __forceinline__ void keep(double2& v) { asm volatile("" : "+v"(v.x)); }
__device__ __forceinline__ void keep(float2& v) { asm volatile("" : "+v"(v.x)); }
__device__ __forceinline__ void keep(float4& v) { asm volatile("" : "+v"(v.x)); }
__device__ __forceinline__ void keep(PairT<false, false>::T& v) { asm volatile("" : "+v"(v.a.x)); }
// the FP64 pair of slot s, and its sum over the slots in FP64, rounded once
template <bool REAL>
__device__ __forceinline__ typename PairT<false, REAL>::T pair_load(const SubOp& op, int64_t s, int64_t q) {
  return ((const typename PairT<false, REAL>::T*)op.sval)[s * op.npairs + q];
}
__device__ __forceinline__ void pair_add(double2& t, double2 f, double2 v) {
  t.x = fma(f.x, v.x, t.x);
  t.y = fma(f.x, v.y, t.y);
}
__device__ __forceinline__ void pair_add(PairT<false, false>::T& t, double2 f, const PairT<false, false>::T& v) {
  t.a = fmac(f, v.a, t.a);
  t.b = fmac(f, v.b, t.b);
}
__device__ __forceinline__ void pair_round(double2 v, double2& o) { o = v; }
__device__ __forceinline__ void pair_round(double2 v, float2& o) { o = make_float2((float)v.x, (float)v.y); }
__device__ __forceinline__ void pair_round(const PairT<false, false>::T& v, PairT<false, false>::T& o) { o = v; }
__device__ __forceinline__ void pair_round(const PairT<false, false>::T& v, float4& o) {
  o = make_float4((float)v.a.x, (float)v.a.y, (float)v.b.x, (float)v.b.y);
}

// exp(f T) e0 of the s x s tridiagonal T, s <= 16, returned per lane: every
// 16-lane row holds the whole problem, lane i % 16 = row i (as expm_e0_16).
// PAIR: the halves of the wave hold two problems.
template <bool PAIR = false>
__device__ __forceinline__ double2 expm_row16(int s, const double2* alpha, const double* beta, double2 f) {
  const int i = threadIdx.x & 15;
  double2 a = make_double2(0.0, 0.0), bl = a, bu = a;
  double col1 = 0.0;
  if (i < s) {
    a = cmul(f, alpha[i]);
    if (i >= 1) bl = cscale(beta[i], f);
    if (i + 1 < s) bu = cscale(beta[i + 1], f);
    col1 = fabs(a.x) + fabs(a.y) + fabs(bl.x) + fabs(bl.y) + fabs(bu.x) + fabs(bu.y);
  }
  const double norm1 = row_max16(col1);
  int nsub = 1;
  if (norm1 > 0.5) nsub = (int)ceil(2.0 * norm1);
  if (!(nsub >= 1) || nsub > (1 << 20)) nsub = 1;
  const double h = 1.0 / (double)nsub;
  int nt, nmax;
  if constexpr (PAIR) {
    int c0, c1;
    taylor_terms_halves(h * norm1, &c0, &c1);
    nt = (threadIdx.x & 63) < 32 ? c0 : c1;
    nmax = max(c0, c1);
  } else {
    nt = nmax = taylor_terms_hi((uint32_t)__builtin_amdgcn_readfirstlane((int)abs_hi(h * norm1)));
  }
  double2 y = make_double2(i == 0 ? 1.0 : 0.0, 0.0);
  for (int sub = 0; sub < nsub; ++sub) {
    double2 term = y, acc = y;
    cplx_terms<1>(nmax, nt, h, a, bl, bu, term, acc);
    y = acc;
  }
  return y;
}

// exp(f T) e0, s <= 16, per lane (expm_row16), for a real T and f = i phi: the
// real recursion of expm_e0_16_herm_row.  Each half's own 1-norm decides.
template <bool PAIR>
__device__ __forceinline__ double2 expm_row16_herm(int s, const double2* alpha, const double* beta, double phi,
                                                   double2* tmp) {
  const int i = threadIdx.x & 15;
  double a = 0.0, bl = 0.0, bu = 0.0, col1 = 0.0;
  if (i < s) {
    a = phi * alpha[i].x;
    if (i >= 1) bl = phi * beta[i];
    if (i + 1 < s) bu = phi * beta[i + 1];
    col1 = fabs(a) + fabs(bl) + fabs(bu);
  }
  expm_e0_16_herm_row<PAIR>(s, a, bl, bu, row_max16(col1), tmp);
  wave_sync();
  const double2 c = tmp[i];
  return i < s ? c : make_double2(0.0, 0.0);
}

}  // namespace
