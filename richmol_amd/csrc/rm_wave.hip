// richmol_amd: propagation of wavepackets on domains of at most 64 rows, one
// wave per wavepacket, or two of the same operator side by side on at most 32
// rows (lanes 32 h + i hold row i of wavepacket h), every step of the run in
// one launch.  The adaptive rule, and the fixed dimensions and operators that
// k_sub_pair (rm_subspace.hip) does not take.
//
// A lane owns a row: its entries (sliced operator, rm_plan::sslice) stay in
// registers for the whole step, or with one field slot for the whole run, so a
// matvec is LDS gathers and multiply-adds.  The first Krylov vectors, the Gram
// matrix of the adaptive rule up to order 16 and everything small sit in LDS;
// longer recurrences continue in the wave's global region.  A real symmetric
// operator under real field products has real alpha: its imaginary sum is not
// formed, and with a real-time exponent the Krylov exponential runs the real
// recursion.  Per half of a pair every operation is lane- or row-local, so a
// wavepacket's result does not depend on its partner; a half that has stopped
// (adaptive rule) keeps its coefficients while its partner goes on.
//
// Bound by the latency of the recurrence; LDS per wave sets how many run beside
// each other (8 per CU).  Measured: 4096 wavepackets, J <= 60, adaptive, 40 steps,
// 477 us against 1 830 with a wave per wavepacket on entries read at every
// matvec (776 before the real exponential and the smaller Gram block).

#include <algorithm>

#include "rm_slice.h"
#include "rm_wave.h"

namespace {

constexpr int GO = 16, GLD = 17;   // Gram matrix order in LDS and its row length
constexpr int LB_FIX = 20, LB_AD = 8;   // Krylov vectors in LDS, fixed and adaptive

// alpha and beta held in LDS: all of a fixed dimension, 16 under the adaptive
// rule (8 waves of a CU then fit its LDS; longer recurrences move to global memory)
__host__ __device__ constexpr int lds_orders(int kcap, bool fixed) { return fixed || kcap < GO + 1 ? kcap : GO + 1; }

__host__ __device__ constexpr int lds_vectors(int kcap, bool fixed) {
  return kcap < (fixed ? LB_FIX : LB_AD) ? kcap : (fixed ? LB_FIX : LB_AD);
}

// Orders beyond 16, as calls: they are rare and would set the registers of the
// whole kernel.
__device__ __attribute__((noinline)) double long_metric(int k, bool brk, double2* G, int kc, const double2* alpha,
                                                        const double* beta, double2 f, double2* c) {
  return adaptive_metric<false>(k, brk, G, kc, alpha, beta, f, c, c + kc);
}
__device__ __attribute__((noinline)) void long_expm(int k, const double2* alpha, const double* beta, double2 f,
                                                    double2* c) {
  expm_e0(k, alpha, beta, f, c);
}

template <bool FIXED, bool F32, bool REAL, bool PAIR, int NP>
__global__ __launch_bounds__(64, NP == 2 ? 2 : 1) void k_wav(SubArgs a) {
  using PT = typename PairT<F32, REAL>::T;
  constexpr int H = PAIR ? 2 : 1;         // wavepackets per wave
  constexpr int LP = 64 / H;              // lanes of each
  extern __shared__ char s_dyn[];
  const int kc = a.kcap;
  const int lb = lds_vectors(kc, FIXED);
  // LDS: matvec input, basis [lb][64] (between steps the observable's state),
  // alpha and beta per half (kl of them), coefficients
  const int kl = lds_orders(kc, FIXED);
  double2* s_x = (double2*)s_dyn;
  double2* s_V = (double2*)(s_dyn + 64 * sizeof(double2));
  double2* s_o = s_V;
  double2* s_al = s_V + (size_t)lb * 64;                   // [H][kl]
  double* s_be = (double*)(s_al + (size_t)H * kl);         // [H][kl + 1]
  __shared__ double2 s_c[H][GO];                           // coefficients of the combination (orders <= 16)
  __shared__ double2 s_d[FIXED ? 1 : H][FIXED ? 1 : GO];
  __shared__ double2 s_g[FIXED ? 1 : H][FIXED ? 1 : GO * GLD];
  const int l = threadIdx.x;
  const int h = PAIR ? l >> 5 : 0, i = PAIR ? l & 31 : l;
  const int i16 = l & 15;
  const double2 zero = make_double2(0.0, 0.0);
  double2* Vg = a.basis + (int64_t)blockIdx.x * kc * 64;
  double2* Gg = a.gram + (int64_t)blockIdx.x * kc * kc * H;
  const int cs = 4 * kc + 1;              // c, c_prev, alpha, beta (as reals) of a half in global memory
  double2* Cg = a.cscr + (int64_t)blockIdx.x * cs * H;
  double2* al_ = s_al + (size_t)h * kl;
  double* be_ = s_be + (size_t)h * (kl + 1);
  auto hsum = [&](double v) __attribute__((always_inline)) -> double {
    if constexpr (PAIR)
      return half_allsum32(v);
    else
      return wave_allsum(v);
  };
  auto vec = [&](int j) __attribute__((always_inline)) -> double2* {
    return j < lb ? s_V + j * 64 + l : Vg + (int64_t)j * 64 + l;
  };
  const int nunit = (a.nitems + H - 1) / H;
  for (int un = blockIdx.x; un < nunit; un += gridDim.x) {
    const int itm = H * un + h;
    int4 item = itm < a.nitems ? a.items[itm] : make_int4(-1, 0, 0, 0);
    // an empty half repeats its partner's wavepacket and stores nothing
    const bool own = item.x >= 0;
    if (PAIR && !own) item = a.items[itm ^ 1];
    const int b = item.x, lo = item.y, len = item.z;
    const SubOp op = a.ops ? a.ops[__builtin_amdgcn_readfirstlane(item.w)] : a.op0;
    if (op.stale && *op.stale == op.call_id) {
      // reused domains that failed their check: the wavepackets are left as they are
      if (i == 0 && own && op.status) op.status[b - op.kcol0] |= RM_STALE_DOMAIN;
      continue;
    }
    const bool ok = i < len;
    const int nslot = op.nslot;
    const int gq = lo + (ok ? i : 0);
    const int orig = op.perm[gq];
    double2 st = load_or_zero(ok, op.psi + (int64_t)b * op.ld + orig);
    double2 ph = make_double2(1.0, 0.0);
    if (op.phase) ph = op.phase[orig];
    // my row's entries: the domain lies in one slice
    const int sl_i = op.srow[lo];
    const int4 sl = op.sslice[sl_i];
    const int64_t e0 = op.soff[sl_i] + (gq - sl.x);
    // (a slice may be wider than its shorter rows, whose subspace sets NP)
    const int z = min(sl.z, NP);
    const int np = __builtin_amdgcn_readfirstlane(PAIR ? max(z, __shfl_xor(z, 32)) : z);
    // the columns' byte offsets count from the slice's base row; mine from my half of s_x
    const uint32_t cb = (uint32_t)(sl.w - lo + LP * h) * 0x100010u;
    PT A[NP];
    uint32_t cc[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const bool in = p < z && ok;
      cc[p] = (uint32_t)(LP * h) * 0x100010u;
      typename PairT<false, REAL>::T v{};
      if (in) {
        cc[p] = op.scol[e0 + 64 * p] + cb;
        if (nslot == 1) v = pair_load<REAL>(op, 0, e0 + 64 * p);
      }
      pair_round(v, A[p]);
    }
    int built = -1;
    // the observable's first entries of my row (source lane, value); the others from memory
    constexpr int OWR = 4;
    int osrc[OWR];
    double2 oval[OWR];
    if (a.obs) {
#pragma unroll
      for (int j = 0; j < OWR; ++j) {
        const bool e = ok && j < op.ow;
        const int c = e ? op.ocol[(int64_t)j * op.n + gq] - lo : -1;
        const bool in = c >= 0 && c < len;
        oval[j] = load_or_zero(in, op.oval + (int64_t)j * op.n + gq);
        osrc[j] = LP * h + (in ? c : 0);
      }
    }
    auto observe = [&](int step) __attribute__((always_inline)) {
      if (!(a.obs && op.ow > 0)) return;
      wave_sync();   // the basis' readers are done
      s_o[l] = st;
      wave_sync();
      double2 y = zero;
#pragma unroll
      for (int j = 0; j < OWR; ++j) y = fmac(oval[j], s_o[osrc[j]], y);
      for (int j = OWR; j < op.ow; ++j) {
        const int c = ok ? op.ocol[(int64_t)j * op.n + gq] - lo : -1;
        if (c >= 0 && c < len) y = fmac(op.oval[(int64_t)j * op.n + gq], s_o[LP * h + c], y);
      }
      const double e0_ = hsum(st.x * y.x + st.y * y.y), e1_ = hsum(st.x * y.y - st.y * y.x);
      if (i == 0 && own && op.expect)
        op.expect[(int64_t)step * op.expect_ld + b - op.kcol0] = make_double2(e0_, e1_);
      wave_sync();   // s_o is rewritten only after these reads
    };
    // acc += a pair's two products (columns as byte offsets of an FP64 vector)
    auto gather = [&](uint32_t c, const PT& v, double2& acc) __attribute__((always_inline)) {
      const double2 x0 = *(const double2*)(s_dyn + (c & 0xffffu)), x1 = *(const double2*)(s_dyn + (c >> 16));
      pair_mac(v, x0, x1, acc);
    };

    for (int step = 0; step < op.nsteps; ++step) {
      double2 vk = op.phase ? cmul(st, ph) : st;
      if (!step_on(op, step)) {
        // no field: the expv is skipped (tdse.py:377), phases only
        st = op.phase ? cmul(vk, ph) : vk;
        if (i == 0 && own && op.kused) op.kused[(int64_t)step * op.kused_ld + b - op.kcol0] = 0;
        observe(step);
        continue;
      }
      const double2* fp = op.table + (int64_t)step * nslot;
      // the step's operator from the real field products, unless it is the one
      // already built; with one slot B_0 itself is used and its sums are scaled
      // (not in FP32: the rounding of B_0 would add up over the steps, that of
      // F B_0 differs from step to step)
      bool imag = false;
      if (nslot > 1 || F32) {
        bool same = built >= 0;
        const double2* fb = op.table + (int64_t)max(built, 0) * nslot;
        for (int s = 0; s < nslot; ++s) {
          const double2 f = fp[s];
          imag = imag || (REAL && f.y != 0.0);
          same = same && f.x == fb[s].x && f.y == fb[s].y;
        }
        if (!same && !imag) {
          built = step;
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            typename PairT<false, REAL>::T t{};
            if (p < z && ok)
              for (int s = 0; s < nslot; ++s) pair_add(t, fp[s], pair_load<REAL>(op, s, e0 + 64 * p));
            pair_round(t, A[p]);
          }
        }
      }
      const double2 f0 = nslot == 1 && !F32 ? fp[0] : make_double2(1.0, 0.0);
      const bool realal = REAL && (op.sflags & 1) && !imag && f0.y == 0.0;
      const bool realexp = realal && op.f.x == 0.0;
      auto matvec = [&]() __attribute__((always_inline)) -> double2 {
        double2 y;
        if (REAL && imag) {
          // complex field products of a real operator: slot by slot
          y = zero;
          for (int s = 0; s < nslot; ++s) {
            double2 t = zero;
            for (int p = 0; ok && p < z; ++p) {
              PT v;
              pair_round(pair_load<REAL>(op, s, e0 + 64 * p), v);
              gather(op.scol[e0 + 64 * p] + cb, v, t);
            }
            y = fmac(fp[s], t, y);
          }
        } else {
          double2 acc = zero, acc1 = zero;
#pragma unroll
          for (int p = 0; p < NP; p += 2)
            if (p < np) {
              gather(cc[p], A[p], acc);
              gather(cc[p + 1], A[p + 1], acc1);
            }
          const double2 t = cadd(acc, acc1);
          y = realal ? cscale(f0.x, t) : cmul(f0, t);
        }
        return ok ? y : zero;
      };
      // per half: dimension of a stopped wavepacket, still running, c_prev of my row
      int kk = 1;
      bool live = true;
      double2 cprev = i16 == 0 ? make_double2(1.0, 0.0) : zero, Wr = zero, vp = zero, vl = vk;
      double beta = 0.0;
      bool brk = false, big = false;   // big: order beyond 16, Gram matrix in global memory
      for (int it = 0;; ++it) {
        *vec(it) = vk;
        s_x[l] = vk;
        wave_sync();
        if (!FIXED && brk && live && it > 0) {
          // Gram column of the restart vector, explicit dots
          for (int j = 0; j < it; ++j) {
            const double2 x = *vec(j);
            const double d0 = hsum(x.x * vk.x + x.y * vk.y), d1 = hsum(x.x * vk.y - x.y * vk.x);
            if (i == 0) {
              if (it < GO) {
                s_g[h][j * GLD + it] = make_double2(d0, d1);
                s_g[h][it * GLD + j] = make_double2(d0, -d1);
              } else {
                double2* G = Gg + (int64_t)h * kc * kc;
                G[j * kc + it] = make_double2(d0, d1);
                G[it * kc + j] = make_double2(d0, -d1);
              }
            }
          }
        }
        // w = H V_it; alpha = vdot(w, V_it); W = w - alpha V_it - beta V_{it-1}
        Wr = matvec();
        double2 al = make_double2(hsum(Wr.x * vk.x + Wr.y * vk.y), 0.0);
        if (!realal) al.y = hsum(Wr.x * vk.y - Wr.y * vk.x);
        Wr = csub(Wr, cscale(beta, vp));
        Wr = realal ? csub(Wr, cscale(al.x, vk)) : csub(Wr, cmul(al, vk));
        if (i == 0) {
          if (FIXED || it < GO)
            al_[it] = al;
          else
            Cg[(int64_t)h * cs + 2 * kc + it] = al;
        }
        if (live) vl = vk;
        const int k = it + 1;
        if (FIXED) {
          kk = k;
          if (k >= a.fixed_m) break;
        } else {
          if (it == 0) {
            const double g = hsum(vk.x * vk.x + vk.y * vk.y);
            if (i == 0) s_g[h][0] = make_double2(g, 0.0);
            live = k < a.maxorder;
          } else {
            wave_sync();
            double conv;
            if (it < GO) {
              // Gram column it from the three-term relation (adaptive_metric)
              double2* G = s_g[h];
              if (!brk && i < it) {
                const double2 g1 = G[i * GLD + it - 1];
                double2 hv;
                if (i == it - 1) {
                  hv = cconj(al_[it - 1]);
                } else {
                  hv = cscale(be_[i + 1], G[(i + 1) * GLD + it - 1]);
                  hv = fmac(cconj(al_[i]), g1, hv);
                  if (i > 0) hv = cadd(hv, cscale(be_[i], G[(i - 1) * GLD + it - 1]));
                }
                double2 t = csub(hv, cmul(al_[it - 1], g1));
                if (it >= 2) t = csub(t, cscale(be_[it - 1], G[i * GLD + it - 2]));
                t = make_double2(t.x / beta, t.y / beta);
                G[i * GLD + it] = t;
                G[it * GLD + i] = cconj(t);
              }
              if (i == 0) G[it * GLD + it] = make_double2(1.0, 0.0);
              const double2 c = realexp ? expm_row16_herm<PAIR>(k, al_, be_, op.f.y, s_d[h])
                                        : expm_row16<PAIR>(k, al_, be_, op.f);
              const double2 d = i16 < k ? csub(c, cprev) : zero;
              wave_sync();
              if (i < 16) s_d[h][i] = d;
              wave_sync();
              // conv = d^H G d: row i16, my 16-lane row's share of the columns
              constexpr int NC = 16 / (LP / 16);
              const int j0 = (i >> 4) * NC;
              double2 r = zero;
              if (i16 < k)
#pragma unroll
                for (int u = 0; u < NC; ++u)
                  if (j0 + u < k) r = fmac(G[i16 * GLD + j0 + u], s_d[h][j0 + u], r);
              conv = hsum(d.x * r.x + d.y * r.y);
              if (live) {
                cprev = c;
                kk = k;
              }
            } else {
              if (it == GO) {
                // the next Gram column has index 16: matrix and coefficients move to global memory
#pragma unroll
                for (int q = 0; q < H; ++q) {
                  double2* G = Gg + (int64_t)q * kc * kc;
                  for (int e = l; e < GO * GO; e += 64) G[(e / GO) * kc + e % GO] = s_g[q][(e / GO) * GLD + e % GO];
                }
                if (live && i < 16) Cg[(int64_t)h * cs + kc + i] = cprev;
                if (i < 16) {
                  Cg[(int64_t)h * cs + 2 * kc + i] = al_[i];
                  ((double*)(Cg + (int64_t)h * cs + 3 * kc))[i] = be_[i];
                }
                if (i == 0) ((double*)(Cg + (int64_t)h * cs + 3 * kc))[it] = be_[it];
                __threadfence_block();
                wave_sync();
              }
              conv = 0.0;
#pragma unroll
              for (int q = 0; q < H; ++q) {
                // one half after the other, all 64 lanes on its matrices
                const bool lq = __any(live && h == q);
                if (!lq) continue;
                const double bq = __shfl(beta, LP * q);
                double2* c = Cg + (int64_t)q * cs;
                const double cq = long_metric(it, !(bq != 0.0), Gg + (int64_t)q * kc * kc, kc, c + 2 * kc,
                                              (const double*)(c + 3 * kc), op.f, c);
                if (h == q) conv = cq;
              }
              if (live) {
                kk = k;
                big = true;
              }
            }
            live = live && k < a.maxorder && conv > a.tol;
          }
          if (!__any(live)) break;
        }
        // beta_k = |W| (tdse.py:453)
        const double ww = hsum(Wr.x * Wr.x + Wr.y * Wr.y);
        double ib = 0.0;
        beta = 0.0;
        if (ww != 0.0) sqrt_rcp_nb(ww, &beta, &ib);
        brk = !(ww != 0.0);
        if (i == 0) {
          if (FIXED || k <= GO)
            be_[k] = beta;
          else
            ((double*)(Cg + (int64_t)h * cs + 3 * kc))[k] = beta;
        }
        vp = vk;
        if (!brk) {
          vk = cscale(ib, Wr);
        } else if (live) {
          // exact breakdown: Gram-Schmidt of ones against the basis (tdse.py:459-465);
          // nothing left: the basis spans the domain, zero stands for the
          // reference's restart vector (its coefficient is exactly zero)
          Wr = ok ? make_double2(1.0, 0.0) : zero;
          for (int j = 0; j < k; ++j) {
            const double2 x = *vec(j);
            const double2 proj = make_double2(hsum(x.x * Wr.x + x.y * Wr.y), hsum(x.x * Wr.y - x.y * Wr.x));
            Wr = csub(Wr, cmul(proj, x));
          }
          const double nv = sqrt(hsum(Wr.x * Wr.x + Wr.y * Wr.y));
          vk = nv > 0.0 ? make_double2(Wr.x / nv, Wr.y / nv) : zero;
        } else {
          vk = zero;
        }
      }
      // u = sum_j c_j V_j with c = exp(f T) e0; psi = P u
      wave_sync();
      if (FIXED) {
        if (kk > 16) {
#pragma unroll
          for (int q = 0; q < H; ++q)
            long_expm(kk, s_al + (size_t)q * kl, s_be + (size_t)q * (kl + 1), op.f, Cg + (int64_t)q * cs);
          big = true;
          __threadfence_block();
        } else if (kk > 1) {
          cprev = realexp ? expm_row16_herm<PAIR>(kk, al_, be_, op.f.y, s_c[h]) : expm_row16<PAIR>(kk, al_, be_, op.f);
        }
      }
      wave_sync();
      if (i < 16) s_c[h][i] = cprev;
      wave_sync();
      const double2* cf = big ? Cg + (int64_t)h * cs + (FIXED ? 0 : kc) : s_c[h];
      double2 u0 = zero, u1 = zero;
      const int kmax = PAIR ? max(kk, __shfl_xor(kk, 32)) : kk;
      for (int j = 0; j < kmax - 1; ++j) {
        const double2 x = *vec(j);
        if (j < kk - 1) {
          if (j & 1)
            u1 = fmac(cf[j], x, u1);
          else
            u0 = fmac(cf[j], x, u0);
        }
      }
      const double2 uu = fmac(cf[kk - 1], vl, cadd(u0, u1));
      st = ok ? (op.phase ? cmul(uu, ph) : uu) : zero;
      if (i == 0 && own) {
        if (op.kused) op.kused[(int64_t)step * op.kused_ld + b - op.kcol0] = kk;
        if (!FIXED && kk >= a.maxorder && op.status) op.status[b - op.kcol0] = RM_NOT_CONVERGED;
      }
      observe(step);
      wave_sync();
    }
    if (ok && own) op.psi[(int64_t)b * op.ld + orig] = st;
  }
}

template <bool FIXED, bool F32, bool REAL, bool PAIR, int NP>
hipError_t launch_k(const SubArgs& a0, int n_cu, hipStream_t s, int* waves_out, bool dry) {
  auto kern = k_wav<FIXED, F32, REAL, PAIR, NP>;
  constexpr int H = PAIR ? 2 : 1;
  const size_t lds = 64 * sizeof(double2) +
                     sizeof(double2) * (size_t)(lds_vectors(a0.kcap, FIXED) * 64 + H * lds_orders(a0.kcap, FIXED)) +
                     sizeof(double) * (size_t)(H * (lds_orders(a0.kcap, FIXED) + 1));
  int occ = 0;
  hipError_t e = occupancy((const void*)kern, 64, lds, &occ);
  if (e != hipSuccess) return e;
  int waves = (int)std::min<int64_t>(((int64_t)a0.nitems + H - 1) / H, (int64_t)std::max(occ, 1) * n_cu);
  if (a0.max_waves > 0) waves = std::min(waves, a0.max_waves);
  *waves_out = std::max(waves, 1);
  if (dry) return hipSuccess;
  hipLaunchKernelGGL(kern, dim3((unsigned)*waves_out), dim3(64), lds, s, a0);
  return hipGetLastError();
}

template <bool FIXED, bool F32>
hipError_t launch_t(int kind, const SubArgs& a, int n_cu, hipStream_t s, int* waves, bool dry) {
  switch (kind) {
    case WAV_S2: return launch_k<FIXED, F32, true, false, 2>(a, n_cu, s, waves, dry);
    case WAV_S32: return launch_k<FIXED, F32, true, false, 32>(a, n_cu, s, waves, dry);
    case WAV_P2: return launch_k<FIXED, F32, true, true, 2>(a, n_cu, s, waves, dry);
    case WAV_P16: return launch_k<FIXED, F32, true, true, 16>(a, n_cu, s, waves, dry);
    case WAV_SC: return launch_k<FIXED, F32, false, false, 32>(a, n_cu, s, waves, dry);
    default: return launch_k<FIXED, F32, false, true, 16>(a, n_cu, s, waves, dry);
  }
}

}  // namespace

hipError_t launch_wav(int kind, const SubArgs& a, bool f32, int n_cu, hipStream_t s, int* waves, bool dry) {
  const bool fixed = a.fixed_m > 0;
  if (fixed)
    return f32 ? launch_t<true, true>(kind, a, n_cu, s, waves, dry) : launch_t<true, false>(kind, a, n_cu, s, waves, dry);
  return f32 ? launch_t<false, true>(kind, a, n_cu, s, waves, dry) : launch_t<false, false>(kind, a, n_cu, s, waves, dry);
}
