// richmol_amd: propagation of wavepackets on domains of up to BLK_MAX_ROWS rows,
// one workgroup of 16 waves each, every step of the run in one launch.
//
// Layout.  The operator comes in slices of up to 64 rows (of one subspace, or
// of several whole small ones), entries column by column in pairs
// (SubOp::sslice, scol, sval): lane l of a wave holds
// row l of a slice, its loads are contiguous over the lanes and 16 bytes wide,
// and there is no reduction over lanes in a row's sum.  A domain with fewer
// slices than waves splits each slice's columns over several waves (parts):
// part 0 owns the rows (Krylov vectors in its registers), the others hand
// their partial sums over in LDS.  When a lane's entries fit BLK_PAIRS pairs
// (REG) they stay in registers for the whole step -- with one field slot for
// the whole run -- and a matvec reads nothing but the vector in LDS; otherwise
// they are read (L2) at every matvec, from the step's assembled operator or,
// with one field slot, straight from B_0.
//
// An iteration has two barriers: the matvec's with the alpha sum -- each
// wave adds conj(its partial sums) . V, linear in them, so the parts meet
// in the same barrier -- and the update's with the beta sum, which also
// publishes W, the next matvec's input (scaled by 1/beta where it is used).
// Sums are wave DPP sums, then the waves' values added by every wave in
// the same order.  The adaptive rule's metric runs on the last wave while
// the others update W, before the second barrier.  That wave, which
// also takes the Krylov exponentials, has no rows (blk_control): its code
// then does not set the register pressure of the other waves' loop.
//
// Bound by barriers and reductions where the entries are in registers, by one
// CU's L2 reads (0.9 MB a matvec at 44 000 pairs) where they are not.
// Measured, us a step under the adaptive rule against the kernel before it
// (rm_coop.hip's block form, 16 lanes per row): 96 off-axis wavepackets, J <= 21,
// 19 against 69; 64 on an asymmetric top, J <= 12 (741 rows, 49 218 entries, 3
// slots), 39 against 470.  Steps' operators formed once for all wavepackets
// (k_blk_operators) instead of by each: 39 against 95 there, 195 against 486 on
// 3 101 rows.

#include <algorithm>
#include <climits>

#include "rm_block.h"
#include "rm_control.h"

namespace {

struct BlkArgs {
  const SubOp* ops;        // the jobs, or NULL: the one job is op0
  SubOp op0;
  const int4* items;       // (column, lo, len, op)
  int32_t nitems;
  char* ws;                // one region per workgroup: basis [kcap][lmax], operator pairs
  int64_t wg_bytes, offA, offG;
  const void* pre;         // the steps' operators (k_blk_operators), entry 0 of the plan's slices; or NULL
  int64_t pre_ld;          // pairs from one step's to the next one's
  int32_t kcap, fixed_m, maxorder, lmax;
  double tol;
};

constexpr int PRE_STEPS = 8;   // steps of one thread

// The operators A(F) = sum_s F_s B_s of steps 0 .. nsteps-1 on the pairs [q0,
// q0 + count) of the sliced form, for every wavepacket of the launch: a step
// whose products are those of the step before is left out, as its readers
// leave it out.  Bound by its stores; a thread loads a pair's slots once for
// PRE_STEPS steps.
template <bool F32, bool REAL>
__global__ __launch_bounds__(256) void k_blk_operators(SubOp op, int64_t q0, int64_t count,
                                                       typename PairT<F32, REAL>::T* __restrict__ out) {
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int t0 = blockIdx.y * PRE_STEPS, nt = min(PRE_STEPS, op.nsteps - t0);
  if (q >= count) return;
  const double2* fp = op.table + (int64_t)t0 * op.nslot;
  bool need[PRE_STEPS];
  typename PairT<false, REAL>::T acc[PRE_STEPS];
#pragma unroll
  for (int t = 0; t < PRE_STEPS; ++t) {
    acc[t] = {};
    need[t] = t < nt && t0 + t == 0;
    if (t < nt && t0 + t > 0)
      for (int s = 0; s < op.nslot; ++s) {
        const double2 f = fp[(int64_t)t * op.nslot + s], g = fp[(int64_t)(t - 1) * op.nslot + s];
        need[t] = need[t] || !(f.x == g.x && f.y == g.y);
      }
  }
  for (int s = 0; s < op.nslot; ++s) {
    const auto v = pair_load<REAL>(op, s, q0 + q);
#pragma unroll
    for (int t = 0; t < PRE_STEPS; ++t)
      if (need[t]) pair_add(acc[t], fp[(int64_t)t * op.nslot + s], v);
  }
#pragma unroll
  for (int t = 0; t < PRE_STEPS; ++t)
    if (need[t]) {
      typename PairT<F32, REAL>::T o;
      pair_round(acc[t], o);
      out[(int64_t)(t0 + t) * count + q] = o;
    }
}

// The control wave's part of one item: it adds nothing to the sums, and runs
// the Krylov exponentials, the stopping rule and the bookkeeping, passing the
// same barriers as the others.
template <bool FIXED>
__device__ __forceinline__ void blk_control(const BlkArgs& a, const SubOp& op, int b, BlkShared<FIXED>& sh,
                                            double2* G2, int& half) {
  const int lane = threadIdx.x & 63;
  const int kc = a.kcap;
  auto observe = [&](int step) __attribute__((always_inline)) {
    if (op.ow <= 0) return;
    __syncthreads();
    __syncthreads();
    double d[2] = {0.0, 0.0};
    blk_sum<2>(d, sh.red, half);
    if (lane == 0 && op.expect) op.expect[(int64_t)step * op.expect_ld + b - op.kcol0] = make_double2(d[0], d[1]);
  };
  for (int step = 0; step < op.nsteps; ++step) {
    if (!step_on(op, step)) {
      if (lane == 0 && op.kused) op.kused[(int64_t)step * op.kused_ld + b - op.kcol0] = 0;
      observe(step);
      continue;
    }
    // a real symmetric operator under real field products: alpha is real, and
    // with a real-time exponent the exponentials take the real recursion
    bool herm = (op.sflags & 1) && op.f.x == 0.0;
    for (int s = 0; s < op.nslot; ++s) herm = herm && op.table[(int64_t)step * op.nslot + s].y == 0.0;
    __syncthreads();
    double2* Gm = sh.gram;
    double2* cv = sh.cv;
    int g_ld = GL, k = 1;
    bool brk = false;
    for (int it = 0;; ++it) {
      double red[3] = {0.0, 0.0, 0.0};
      if (it == 0 && !FIXED) {
        blk_sum<3>(red, sh.red, half);
      } else {
        double r2[2] = {0.0, 0.0};
        blk_sum<2>(r2, sh.red, half);
        red[0] = r2[0];
        red[1] = r2[1];
      }
      k = it + 1;
      if (lane == 0) sh.alpha[it] = make_double2(red[0], herm ? 0.0 : red[1]);
      if (FIXED && k >= a.fixed_m) break;
      if (!FIXED) {
        if (it == 0) {
          if (lane == 0) {
            Gm[0] = make_double2(red[2], 0.0);
            cv[g_ld] = make_double2(1.0, 0.0);   // c_prev = [1]
            sh.conv = 1.0;
          }
        } else {
          wave_sync();
          const double c = it < 16 ? metric16(it, brk, Gm, g_ld, sh.alpha, sh.beta, op.f, herm, cv, sh.cf)
                                   : adaptive_metric<false>(it, brk, Gm, g_ld, sh.alpha, sh.beta, op.f, cv, cv + g_ld);
          if (lane == 0) sh.conv = c;
        }
      }
      double bs[1] = {0.0};
      blk_sum<1>(bs, sh.red, half);
      if (!FIXED) {
        if (!(k < a.maxorder && sh.conv > a.tol)) break;
        if (k == GL) {
          // the next Gram column has index GL: matrix and coefficients move to global memory
          double2* c2 = G2 + (int64_t)kc * kc;
          for (int q = lane; q < GL * GL; q += 64) G2[(q / GL) * kc + q % GL] = sh.gram[q];
          for (int q = lane; q < GL; q += 64) {
            c2[q] = sh.cv[q];
            c2[kc + q] = sh.cv[GL + q];
          }
          __threadfence_block();
          Gm = G2;
          cv = c2;
          g_ld = kc;
        }
      }
      const double beta = sqrt(bs[0]);
      if (lane == 0) sh.beta[k] = beta;
      brk = !(beta != 0.0);
      if (!brk) continue;
      for (int j = 0; j < k; ++j) {
        double d[2] = {0.0, 0.0};
        blk_sum<2>(d, sh.red, half);
      }
      double nv[1] = {0.0};
      blk_sum<1>(nv, sh.red, half);
      if (!FIXED) {
        // Gram column of the restart vector, explicit dots
        for (int j = 0; j < k; ++j) {
          double d[2] = {0.0, 0.0};
          blk_sum<2>(d, sh.red, half);
          if (lane == 0) {
            Gm[j * g_ld + k] = make_double2(d[0], d[1]);
            Gm[k * g_ld + j] = make_double2(d[0], -d[1]);
          }
        }
      }
      __syncthreads();
    }
    if (FIXED || k == 1) {
      wave_sync();
      if (k == 1) {
        if (lane == 0) sh.cf[0] = make_double2(1.0, 0.0);
      } else if (k <= 16) {
        const double2 c = herm ? expm_row16_herm<false>(k, sh.alpha, sh.beta, op.f.y, sh.cf)
                               : expm_row16(k, sh.alpha, sh.beta, op.f);
        wave_sync();
        if (lane < k) sh.cf[lane] = c;
      } else {
        expm_e0(k, sh.alpha, sh.beta, op.f, sh.cf);
      }
      __syncthreads();
    }
    if (lane == 0) {
      if (op.kused) op.kused[(int64_t)step * op.kused_ld + b - op.kcol0] = k;
      if (!FIXED && k >= a.maxorder && op.status) op.status[b - op.kcol0] |= RM_NOT_CONVERGED;
    }
    observe(step);
  }
}

// The other waves' part: rows, vectors and matvecs.  RS: slices per wave;
// REG (RS = 1): the lane's entries in registers.
template <bool FIXED, bool F32, bool REAL, int RS, bool REG>
__device__ __forceinline__ void blk_work(const BlkArgs& a, const SubOp& op, int b, int lo, int len, int wv,
                                         char* s_dyn, double2* s_w, double2* s_part, BlkShared<FIXED>& sh,
                                         double2* __restrict__ V, char* base, int& half) {
  using PT = typename PairT<F32, REAL>::T;
  constexpr int NP = REG ? BLK_PAIRS(F32, REAL) : 1;
  const int lane = threadIdx.x & 63;
  const double2 zero = make_double2(0.0, 0.0);
  PT* Ast = (PT*)(base + a.offA);
  const int ns0 = op.srow[lo], nsl = op.srow[lo + len - 1] - ns0 + 1;   // the domain's slices
  const int G = RS == 1 ? NWORK / nsl : 1;       // parts per slice
  const int part = RS == 1 ? wv / nsl : 0;
  const bool act = part < G, own = act && part == 0;
  const int nslot = op.nslot;
  const int lmax = a.lmax;
  // this wave's slices: local row of this lane, in range or not, its entries
  int row[RS], np[RS], orig[RS];
  uint32_t cb[RS];
  bool ok[RS];
  int64_t e0[RS];
  double2 S[RS], W[RS], Vk[RS], Vp[RS];
#pragma unroll
  for (int r = 0; r < RS; ++r) {
    const int si = RS == 1 ? wv % nsl : wv + NWORK * r;
    const bool has = act && si < nsl;
    const int4 sl = op.sslice[ns0 + (has ? si : 0)];   // (first row, rows, pairs per row, row that columns count from)
    row[r] = sl.x - lo + lane;
    ok[r] = has && lane < sl.y && row[r] >= 0 && row[r] < len;
    if (!ok[r]) row[r] = 0;
    cb[r] = (uint32_t)(sl.w - lo) * 0x100010u;   // added to both columns of a pair
    const int p0 = (int)((int64_t)sl.z * part / G), p1 = (int)((int64_t)sl.z * (part + 1) / G);
    np[r] = has ? p1 - p0 : 0;                   // this part's range of pairs
    e0[r] = op.soff[ns0 + (has ? si : 0)] + (int64_t)p0 * 64 + lane;
    W[r] = Vk[r] = Vp[r] = zero;
    orig[r] = op.perm[lo + row[r]];
    S[r] = load_or_zero(own && ok[r], op.psi + (int64_t)b * op.ld + orig[r]);
  }
  PT A[NP];
  uint32_t cc[NP];
  if constexpr (REG) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const bool in = p < np[0] && ok[0];
      cc[p] = 0;
      typename PairT<false, REAL>::T v{};
      if (in) {
        cc[p] = op.scol[e0[0] + 64 * p] + cb[0];
        if (nslot == 1) v = pair_load<REAL>(op, 0, e0[0] + 64 * p);
      }
      pair_round(v, A[p]);
    }
  }
  int built = -1;
  // acc += a pair's two products; c: the two columns' offsets in
  // bytes of the vector
  auto gather = [&](uint32_t c, const PT& v, double2& acc) __attribute__((always_inline)) {
    const double2 x0 = *(const double2*)(s_dyn + (c & 0xffffu)), x1 = *(const double2*)(s_dyn + (c >> 16));
    pair_mac(v, x0, x1, acc);
  };
  // the row's sum with pairs read from q
  auto row_sum = [&](int r, const PT* __restrict__ q) __attribute__((always_inline)) -> double2 {
    double2 acc = zero, acc2 = zero;
    const uint32_t* __restrict__ qc = op.scol;
    constexpr int U = 4;   // pairs loaded together (8: more spilled registers, 7 % slower)
    int p = 0;
    const int n = np[r];
    if (!ok[r]) return acc;
    for (; p + U <= n; p += U) {
      PT v[U];
      uint32_t c[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        v[u] = q[e0[r] + 64 * (p + u)];
        c[u] = qc[e0[r] + 64 * (p + u)];
      }
#pragma unroll
      for (int u = 0; u < U; u += 2) {
        gather(c[u] + cb[r], v[u], acc);
        gather(c[u + 1] + cb[r], v[u + 1], acc2);
      }
    }
    for (; p < n; ++p) gather(qc[e0[r] + 64 * p] + cb[r], q[e0[r] + 64 * p], acc);
    return cadd(acc, acc2);
  };
  auto publish = [&](int r) __attribute__((always_inline)) {
    if (own && ok[r]) {
      s_w[row[r]] = W[r];
    }
  };
  // <psi|O|psi> after step `step` (the state in S)
  auto observe = [&](int step) __attribute__((always_inline)) {
    if (op.ow <= 0) return;
    __syncthreads();   // the matvec input's readers are done
#pragma unroll
    for (int r = 0; r < RS; ++r)
      if (own && ok[r]) s_w[row[r]] = S[r];
    __syncthreads();
    double d[2] = {0.0, 0.0};
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      if (!(own && ok[r])) continue;
      double2 y = zero;
      for (int j = 0; j < op.ow; ++j) {
        const int64_t q = (int64_t)j * op.n + lo + row[r];
        const int c = op.ocol[q] - lo;
        if (c >= 0 && c < len) y = fmac(op.oval[q], s_w[c], y);
      }
      d[0] += S[r].x * y.x + S[r].y * y.y;
      d[1] += S[r].x * y.y - S[r].y * y.x;
    }
    blk_sum<2>(d, sh.red, half);   // its barrier: s_w is rewritten only after these reads
  };

  for (int step = 0; step < op.nsteps; ++step) {
    if (!step_on(op, step)) {
      // no field: the expv is skipped (tdse.py:377), phases only
      if (op.phase)
#pragma unroll
        for (int r = 0; r < RS; ++r) S[r] = cmul(cmul(S[r], op.phase[orig[r]]), op.phase[orig[r]]);
      observe(step);
      continue;
    }
    const double2* fp = op.table + (int64_t)step * nslot;
    // the step's operator from the real field products, unless it is the one
    // already built; with one slot B_0 itself is used and its sums are scaled
    bool imag = false, same = built >= 0;
    if (nslot > 1) {
      const double2* fb = op.table + (int64_t)max(built, 0) * nslot;
      for (int s = 0; s < nslot; ++s) {
        const double2 f = fp[s];
        imag = imag || (REAL && f.y != 0.0);
        same = same && f.x == fb[s].x && f.y == fb[s].y;
      }
      if (!same && !imag) {
        built = step;
        if constexpr (REG) {
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            typename PairT<false, REAL>::T t{};
            if (p < np[0] && ok[0])
              for (int s = 0; s < nslot; ++s) pair_add(t, fp[s], pair_load<REAL>(op, s, e0[0] + 64 * p));
            pair_round(t, A[p]);
          }
        } else if (!a.pre) {
#pragma unroll
          for (int r = 0; r < RS; ++r) {
            const int64_t ea = e0[r] - op.soff[ns0];
#pragma unroll 4
            for (int p = 0; p < np[r]; ++p) {
              typename PairT<false, REAL>::T t{};
              for (int s = 0; s < nslot; ++s) pair_add(t, fp[s], pair_load<REAL>(op, s, e0[r] + 64 * p));
              pair_round(t, Ast[ea + 64 * p]);
            }
          }
        }
      }
    }
    const double2 f0 = nslot == 1 ? fp[0] : make_double2(1.0, 0.0);
    const bool realal = (op.sflags & 1) && op.f.x == 0.0 && !imag && f0.y == 0.0;
    // V_0 = phi = P psi (unnormalised, tdse.py:443-446), the first matvec input
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      W[r] = op.phase ? cmul(S[r], op.phase[orig[r]]) : S[r];
      Vp[r] = zero;
      publish(r);
    }
    __syncthreads();
    int k = 1;
    double beta = 0.0, ib = 1.0;
    for (int it = 0;; ++it) {
      // this lane's part of w = A (W / beta), and its part of alpha = vdot(w, V_it)
      double red[3] = {0.0, 0.0, 0.0};
      double2 yp[RS];
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        double2 y;
        if (REAL && imag) {
          // complex field products of a real operator: slot by slot
          y = zero;
          for (int s = 0; s < nslot; ++s) {
            double2 tot = zero;
            for (int p = 0; ok[r] && p < np[r]; ++p) {
              PT v;
              pair_round(pair_load<REAL>(op, s, e0[r] + 64 * p), v);
              gather(op.scol[e0[r] + 64 * p] + cb[r], v, tot);
            }
            y = fmac(fp[s], tot, y);
          }
        } else {
          double2 acc;
          if constexpr (REG) {
            // (the empty asm: without it the compiler spills 470 registers in
            // the FP64 kernel of a fixed dimension, 50 us an iteration)
#pragma unroll
            for (int p = 0; p < NP; ++p) keep(A[p]);
            double2 acc1 = zero;
            acc = zero;
#pragma unroll
            for (int p = 0; p < NP; p += 2) {
              // (the empty asm keeps the columns packed: unpacked ahead of the
              // loop they would take two more registers per pair)
              asm volatile("" : "+v"(cc[p]));
              asm volatile("" : "+v"(cc[p + 1]));
              if (p < np[0]) {
                gather(cc[p], A[p], acc);
                gather(cc[p + 1], A[p + 1], acc1);
              }
            }
            acc = cadd(acc, acc1);
          } else if (nslot == 1) {
            acc = row_sum(r, F32 ? (const PT*)op.sval32 : (const PT*)op.sval);
          } else {
            acc = row_sum(r, a.pre ? (const PT*)a.pre + (int64_t)built * a.pre_ld : Ast - op.soff[ns0]);
          }
          y = cmul(f0, acc);
        }
        y = cscale(ib, y);
        yp[r] = ok[r] ? y : zero;
        double2 v = zero;
        if (own) {
          v = cscale(ib, W[r]);
          Vk[r] = v;
          if (ok[r]) V[(int64_t)it * lmax + row[r]] = v;
          red[2] += v.x * v.x + v.y * v.y;
        } else if (act) {
          v = cscale(ib, s_w[row[r]]);
          if (!ok[r]) v = zero;
          s_part[((part - 1) * nsl + wv % nsl) * 64 + lane] = yp[r];
        }
        red[0] += yp[r].x * v.x + yp[r].y * v.y;
        red[1] += yp[r].x * v.y - yp[r].y * v.x;
      }
      if (it == 0 && !FIXED) {
        blk_sum<3>(red, sh.red, half);
      } else {
        double r2[2] = {red[0], red[1]};
        blk_sum<2>(r2, sh.red, half);
        red[0] = r2[0];
        red[1] = r2[1];
      }
      const double2 al = make_double2(red[0], realal ? 0.0 : red[1]);
      k = it + 1;
      if (FIXED && k >= a.fixed_m) break;
      // W = w - alpha V_it - beta V_{it-1}, and |W|^2
      double bs[1] = {0.0};
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        if (!own) continue;
        double2 y = yp[r];
        if (RS == 1)
          for (int g = 1; g < G; ++g) y = cadd(y, s_part[((g - 1) * nsl + wv) * 64 + lane]);
        y = csub(csub(y, cscale(beta, Vp[r])), cmul(al, Vk[r]));
        W[r] = y;
        publish(r);
        bs[0] += y.x * y.x + y.y * y.y;
      }
      // beta_k = |W| (tdse.py:453); publishes W, the next matvec input
      blk_sum<1>(bs, sh.red, half);
      if (!FIXED && !(k < a.maxorder && sh.conv > a.tol)) break;
      beta = sqrt(bs[0]);
#pragma unroll
      for (int r = 0; r < RS; ++r) Vp[r] = Vk[r];
      if (beta != 0.0) {
        ib = __builtin_amdgcn_rcp(beta);   // and two Newton steps (within an ulp of the quotient)
        ib = fma(fma(-beta, ib, 1.0), ib, ib);
        ib = fma(fma(-beta, ib, 1.0), ib, ib);
        continue;
      }
      // exact breakdown: Gram-Schmidt of ones against the basis (tdse.py:459-465);
      // the restart vector becomes the next matvec input with ib = 1
      ib = 1.0;
#pragma unroll
      for (int r = 0; r < RS; ++r) W[r] = own && ok[r] ? make_double2(1.0, 0.0) : zero;
      for (int j = 0; j < k; ++j) {
        double d[2] = {0.0, 0.0};
#pragma unroll
        for (int r = 0; r < RS; ++r) {
          const double2 vj = load_or_zero(own && ok[r], V + (int64_t)j * lmax + row[r]);
          d[0] += vj.x * W[r].x + vj.y * W[r].y;
          d[1] += vj.x * W[r].y - vj.y * W[r].x;
        }
        blk_sum<2>(d, sh.red, half);
#pragma unroll
        for (int r = 0; r < RS; ++r)
          W[r] = csub(W[r], cmul(make_double2(d[0], d[1]), load_or_zero(own && ok[r], V + (int64_t)j * lmax + row[r])));
      }
      double nv[1] = {0.0};
#pragma unroll
      for (int r = 0; r < RS; ++r) nv[0] += W[r].x * W[r].x + W[r].y * W[r].y;
      blk_sum<1>(nv, sh.red, half);
      const double nrm = sqrt(nv[0]);
      // nrm == 0: the basis spans the domain; the reference's restart vector
      // lies outside it and enters with coefficient exactly zero
#pragma unroll
      for (int r = 0; r < RS; ++r) {
        W[r] = nrm > 0.0 ? make_double2(W[r].x / nrm, W[r].y / nrm) : zero;
        publish(r);
      }
      if (!FIXED)   // Gram column of the restart vector, explicit dots
        for (int j = 0; j < k; ++j) {
          double d[2] = {0.0, 0.0};
#pragma unroll
          for (int r = 0; r < RS; ++r) {
            const double2 vj = load_or_zero(own && ok[r], V + (int64_t)j * lmax + row[r]);
            d[0] += vj.x * W[r].x + vj.y * W[r].y;
            d[1] += vj.x * W[r].y - vj.y * W[r].x;
          }
          blk_sum<2>(d, sh.red, half);
        }
      __syncthreads();
    }
    // u = sum_j c_j V_j with c = exp(f T) e0; psi = P u
    const double2* cf = sh.cf;
    if (FIXED || k == 1)
      __syncthreads();
    else if (k <= GL)
      cf = sh.cv;
    else
      cf = (const double2*)(base + a.offG) + (int64_t)a.kcap * a.kcap;
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      if (!own) continue;
      double2 u = zero;
      if (ok[r]) {
        const double2* Vr = V + row[r];
#pragma unroll 4
        for (int j = 0; j < k - 1; ++j) u = fmac(cf[j], Vr[(int64_t)j * lmax], u);
        u = fmac(cf[k - 1], Vk[r], u);
      }
      S[r] = op.phase ? cmul(u, op.phase[orig[r]]) : u;
    }
    observe(step);
    // the coefficients are rewritten only after the next step's first barrier
  }
#pragma unroll
  for (int r = 0; r < RS; ++r)
    if (own && ok[r]) op.psi[(int64_t)b * op.ld + orig[r]] = S[r];
}

template <bool FIXED, bool F32, bool REAL, int RS, bool REG>
__global__ __launch_bounds__(NT) void k_blk(BlkArgs a) {
  extern __shared__ char s_dyn[];
  double2* s_w = (double2*)s_dyn;   // [lmax] W, the matvec input, at the start of LDS: gathers address it by offset
  __shared__ double2 s_part[RS == 1 ? NWORK * 64 : 1];   // partial sums of parts 1..
  __shared__ BlkShared<FIXED> sh;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* base = a.ws + (int64_t)blockIdx.x * a.wg_bytes;
  int half = 0;
  for (int itm = blockIdx.x; itm < a.nitems; itm += gridDim.x) {
    const int4 item = a.items[itm];
    const SubOp& op = a.ops ? a.ops[item.w] : a.op0;
    if (op.stale && *op.stale == op.call_id) {
      // reused domains that failed their check: the wavepacket is left as it is
      if (threadIdx.x == 0 && op.status) op.status[item.x - op.kcol0] |= RM_STALE_DOMAIN;
      continue;
    }
    if (wv == NWORK)
      blk_control<FIXED>(a, op, item.x, sh, (double2*)(base + a.offG), half);
    else
      blk_work<FIXED, F32, REAL, RS, REG>(a, op, item.x, item.y, item.z, wv, s_dyn, s_w, s_part, sh, (double2*)base,
                                          base, half);
    __syncthreads();   // the next item rewrites LDS and the region after these reads
  }
}

size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

template <int RS, bool REG>
const void* blk_kernel(bool fixed, bool f32, bool real) {
  const void* k[8] = {(const void*)k_blk<false, false, false, RS, REG>, (const void*)k_blk<false, false, true, RS, REG>,
                      (const void*)k_blk<false, true, false, RS, REG>,  (const void*)k_blk<false, true, true, RS, REG>,
                      (const void*)k_blk<true, false, false, RS, REG>,  (const void*)k_blk<true, false, true, RS, REG>,
                      (const void*)k_blk<true, true, false, RS, REG>,   (const void*)k_blk<true, true, true, RS, REG>};
  return k[4 * fixed + 2 * f32 + real];
}

size_t lds_bytes(int64_t lmax) { return sizeof(double2) * (size_t)lmax; }

}  // namespace

int blk_variant(int64_t nslices, bool real) {
  const int rs = nslices <= NWORK ? 1 : nslices <= 2 * NWORK ? 2 : nslices <= 5 * NWORK ? 3 : 0;
  return rs == 0 ? 0 : 2 * rs - (real ? 0 : 1);
}

int blk_part_pairs(int64_t nslices, int64_t maxpairs) {
  if (nslices > NWORK) return INT32_MAX;
  const int64_t G = NWORK / nslices;
  return (int)std::min<int64_t>((maxpairs + G - 1) / G, INT32_MAX);
}

int blk_run(void** ws, size_t* ws_bytes, const SubOp* d_ops, const SubOp* op0, const int4* d_items,
            const std::vector<LongItem>& items, size_t first, size_t count, int variant, int32_t kcap, int32_t fixed_m,
            int32_t maxorder, double tol, bool f32, int n_cu, size_t pre_bytes, hipStream_t s) {
  const int rs = (variant + 1) / 2;   // 1, 2 or 3 (5 slices per wave)
  const bool real = (variant & 1) == 0, fixed = fixed_m > 0;
  // the items come by falling pairs per lane: those that fit the registers last
  size_t mem = 0;
  while (mem < count && items[first + mem].ppairs > BLK_PAIRS(f32, real)) ++mem;
  if (mem > 0 && mem < count) {
    const int rc = blk_run(ws, ws_bytes, d_ops, op0, d_items, items, first, mem, variant, kcap, fixed_m, maxorder, tol,
                           f32, n_cu, pre_bytes, s);
    if (rc) return rc;
    first += mem;
    count -= mem;
    mem = 0;
  }
  const bool reg = mem == 0;
  const void* kern = rs == 1 ? (reg ? blk_kernel<1, true>(fixed, f32, real) : blk_kernel<1, false>(fixed, f32, real))
                             : rs == 2 ? blk_kernel<2, false>(fixed, f32, real) : blk_kernel<5, false>(fixed, f32, real);
  BlkArgs a;
  memset(&a, 0, sizeof(a));
  int64_t lmax = 0, pmax = 0;
  for (size_t i = first; i < first + count; ++i) {
    lmax = std::max<int64_t>(lmax, items[i].item.z);
    if (items[i].nslot > 1) pmax = std::max<int64_t>(pmax, items[i].npairs);
  }
  int64_t q0 = INT64_MAX, q1 = 0;
  for (size_t i = first; i < first + count; ++i) {
    q0 = std::min(q0, items[i].pair0);
    q1 = std::max(q1, items[i].pair0 + items[i].npairs);
  }
  // one job by value: its steps' operators are formed once for all its
  // wavepackets, for as many steps as pre_bytes hold, and the launch is cut
  // there (the state is in psi between launches).  Where one step's do not fit,
  // or the device has no room for them, every workgroup forms its own
  const size_t b_step = (size_t)(f32 ? 8 : 16) * (real ? 1 : 2) * (size_t)std::max<int64_t>(q1 - q0, 1);
  bool pre = !reg && op0 && op0->nslot > 1 && op0->nsteps > 0 && b_step <= pre_bytes;
  const int chunk = pre ? (int)std::min<int64_t>(op0->nsteps, pre_bytes / b_step) : INT32_MAX;
  const size_t lds = lds_bytes(lmax);
  int occ = 0;
  HIPCHK(occupancy(kern, NT, lds, &occ));
  if (occ < 1) return fail(RM_ERR_ARG, "block propagation: a domain of %lld rows does not fit LDS", (long long)lmax);
  const int grid = (int)std::min<int64_t>((int64_t)count, (int64_t)occ * n_cu);
  const size_t b_v = al256(sizeof(double2) * (size_t)kcap * lmax);
  const size_t b_own = al256((f32 ? 8 : 16) * (real ? 1 : 2) * (size_t)std::max<int64_t>(pmax, 1));
  const size_t b_g = fixed ? 0 : al256(sizeof(double2) * ((size_t)kcap * kcap + 2 * (size_t)kcap));
  size_t b_pre = 0;
  auto layout = [&]() {
    const size_t b_a = pre ? 0 : b_own;
    b_pre = pre ? al256(b_step * (size_t)chunk) : 0;
    a.offA = (int64_t)b_v;
    a.offG = (int64_t)(b_v + b_a);
    a.wg_bytes = (int64_t)(b_v + b_a + b_g);
    return b_pre + (size_t)a.wg_bytes * (size_t)grid;
  };
  size_t need = layout();
  if (*ws_bytes < need) {
    if (*ws) {
      HIPCHK(hipDeviceSynchronize());
      HIPCHK(hipFree(*ws));
      *ws = nullptr;
      *ws_bytes = 0;
    }
    hipError_t e = hipMalloc(ws, need);
    if (e == hipErrorOutOfMemory && pre) {
      (void)hipGetLastError();
      pre = false;
      need = layout();
      e = hipMalloc(ws, need);
    }
    if (e != hipSuccess) *ws = nullptr;
    HIPCHK(e);
    *ws_bytes = need;
  }
  a.ops = op0 ? nullptr : d_ops;
  if (op0) a.op0 = *op0;
  a.items = d_items + first;
  a.nitems = (int32_t)count;
  a.ws = (char*)*ws + b_pre;
  a.kcap = kcap;
  a.fixed_m = fixed_m;
  a.maxorder = maxorder;
  a.lmax = (int32_t)lmax;
  a.tol = tol;
  void* args[] = {&a};
  const int nsteps = pre ? op0->nsteps : 1;
  for (int c0 = 0; c0 < nsteps; c0 += chunk) {
    if (pre) {
      const int nc = std::min(chunk, nsteps - c0);
      a.op0.nsteps = nc;
      a.op0.table = op0->table + (int64_t)c0 * op0->nslot;
      a.op0.sflag = op0->sflag + c0;
      if (op0->kused) a.op0.kused = op0->kused + (int64_t)c0 * op0->kused_ld;
      if (op0->expect) a.op0.expect = op0->expect + (int64_t)c0 * op0->expect_ld;
      const dim3 g((unsigned)((q1 - q0 + 255) / 256), (unsigned)((nc + PRE_STEPS - 1) / PRE_STEPS));
      if (f32 && real)
        hipLaunchKernelGGL((k_blk_operators<true, true>), g, dim3(256), 0, s, a.op0, q0, q1 - q0, (float2*)*ws);
      else if (f32)
        hipLaunchKernelGGL((k_blk_operators<true, false>), g, dim3(256), 0, s, a.op0, q0, q1 - q0, (float4*)*ws);
      else if (real)
        hipLaunchKernelGGL((k_blk_operators<false, true>), g, dim3(256), 0, s, a.op0, q0, q1 - q0, (double2*)*ws);
      else
        hipLaunchKernelGGL((k_blk_operators<false, false>), g, dim3(256), 0, s, a.op0, q0, q1 - q0,
                           (PairT<false, false>::T*)*ws);
      HIPCHK(hipGetLastError());
      a.pre = (const char*)*ws - (int64_t)(b_step / (size_t)std::max<int64_t>(q1 - q0, 1)) * q0;
      a.pre_ld = q1 - q0;
    }
    HIPCHK(hipLaunchKernel(kern, dim3((unsigned)grid), dim3(NT), args, lds, s));
  }
  return RM_OK;
}
