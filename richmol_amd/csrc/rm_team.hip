// richmol_amd: a team of T workgroups on each wavepacket, every step of the
// run in one cooperative launch: for a few wavepackets with real operators too
// large for one workgroup's registers (rm_block.hip).
//
// A workgroup holds the entries of its share of the domain's slices in
// registers (several waves per slice, parts of its columns each) and the
// whole Krylov vector in LDS.  Per iteration the workgroups exchange only the
// rows of w = A v: each stores its own rows and reads all of them, and every
// workgroup then takes the sums and updates of the whole vectors itself, in
// the same order, so that all make the same decisions.  That is one exchange
// per iteration in place of two grid-wide sums and a gather of the vector
// from memory.
//
// An exchange carries its own flags: a row's two numbers go to a slot that
// holds LSENT while empty (a signalling-NaN pattern, which no operation
// produces), and its readers poll the slot (agent-scope relaxed atomics).
// Slots come in RING sets taken in turn.  The lane that stores a row is the
// same for the whole run, and so is the lane of each workgroup that reads it.
// Before exchange n the storing lane empties its slot of exchange n - 2: its
// workgroup has read all of exchange n - 1, which the others stored after
// their last read of n - 2.  Every fourth exchange is a release of the storing
// lane and an acquire of the reading one, so one of them lies between that
// emptying and the reuse of the set at n - 2 + RING.  A wait is bounded: past
// SPIN_LIMIT polls the abort flag goes up, nobody waits any more and the
// launch runs to its end, its results marked invalid.
//
// Bound by the latency of the exchange and by its polls, which every wave of
// every workgroup makes: 6.3 us an iteration with 12 workgroups on the device,
// 13 with 192.  Measured against the cooperative form of rm_coop.hip, us a step
// of 4 iterations: one wavepacket on 3 101 rows (370 802 entries) 51 / 63, 1 135
// rows 40 / 51.

#include <algorithm>
#include <climits>

#include "rm_control.h"
#include "rm_team.h"

namespace {

typedef unsigned long long u64;

constexpr int NVL = NWORK * 64;             // lanes that hold the whole vectors
constexpr int RING = 8, SRING = 4;
constexpr int TEAM_MAX = 64;                // workgroups of a team
constexpr unsigned SPIN_LIMIT = 1u << 22;
constexpr u64 LSENT = 0x7FF4DEAD0000BEEFull;
constexpr int R = 4;    // rows of the whole vectors per lane (TEAM_MAX_ROWS)
constexpr int NP = 8;   // pairs of entries a lane holds, within 128 registers beside them

struct TeamArgs {
  const SubOp* ops;        // the jobs, or NULL: the one job is op0
  SubOp op0;
  const int4* items;       // (column, lo, len, op)
  int32_t nitems, team, nteams;
  char* ws;                // per workgroup: basis of its rows [kcap + 1][NVL], Gram matrix and coefficients
  int64_t wg_bytes, offG;
  u64* rows;               // [nitems][RING][lmax][2]
  u64* sums;               // [nitems][SRING][TEAM_MAX][2]
  int32_t* abort_flag;
  int32_t kcap, fixed_m, maxorder, lmax;
  double tol;
};

__device__ __forceinline__ void put(u64* p, double v) {
  __hip_atomic_store(p, (u64)__double_as_longlong(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void empty(u64* p) {
  __hip_atomic_store(p, LSENT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 look(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wait of a wave: take(j) reads value j of this lane's miss set (bits) and
// says whether it was there.
template <int N, typename F>
__device__ __forceinline__ void wait_all(const TeamArgs& a, volatile int* s_ab, int miss, F take) {
  unsigned spins = 0;
  for (;;) {
#pragma unroll
    for (int j = 0; j < N; ++j)
      if ((miss >> j) & 1)
        if (take(j)) miss &= ~(1 << j);
    if (!__any(miss != 0) || *s_ab) break;
    __builtin_amdgcn_s_sleep(1);
    ++spins;
    if ((spins & 255u) == 0 &&
        (spins >= SPIN_LIMIT || __hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
      __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *s_ab = 1;
      break;
    }
  }
}

// Sum over the threads of the team, the same on every one of them; all waves
// of all workgroups call it.  Every sum is a release and an acquire.
template <bool FIXED>
__device__ void team_sum(double (&d)[2], const TeamArgs& a, u64* sums, int t, int& ns, BlkShared<FIXED>& sh, int& half,
                         volatile int* s_ab) {
  blk_sum<2>(d, sh.red, half);
  const int lane = threadIdx.x & 63;
  u64* sl = sums + (size_t)(ns % SRING) * TEAM_MAX * 2;
  if (threadIdx.x == 0) {
    if (ns >= 2) {
      u64* old = sums + (size_t)((ns - 2) % SRING) * TEAM_MAX * 2 + 2 * t;
      empty(old);
      empty(old + 1);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    put(sl + 2 * t, d[0]);
    put(sl + 2 * t + 1, d[1]);
  }
  double2 v = make_double2(0.0, 0.0);
  wait_all<1>(a, s_ab, lane < a.team ? 1 : 0, [&](int) __attribute__((always_inline)) {
    const u64 x = look(sl + 2 * lane), y = look(sl + 2 * lane + 1);
    if (x == LSENT || y == LSENT) return false;
    v = make_double2(__longlong_as_double((long long)x), __longlong_as_double((long long)y));
    return true;
  });
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  ++ns;
  d[0] = wave_allsum(v.x);
  d[1] = wave_allsum(v.y);
}

// The control wave's part of one item (blk_control of rm_block.hip with the
// team's barriers): the metric after vector k runs beside the next matvec.
template <bool FIXED>
__device__ __forceinline__ void team_control(const TeamArgs& a, const SubOp& op, int b, int t, u64* sums,
                                             BlkShared<FIXED>& sh, double2* G2, int& half, volatile int* s_ab) {
  const int lane = threadIdx.x & 63;
  const int kc = a.kcap;
  int ns = 0;
  auto observe = [&](int step) __attribute__((always_inline)) {
    if (op.ow <= 0) return;
    __syncthreads();
    double d[2] = {0.0, 0.0};
    team_sum<FIXED>(d, a, sums, t, ns, sh, half, s_ab);
    if (t == 0 && lane == 0 && op.expect)
      op.expect[(int64_t)step * op.expect_ld + b - op.kcol0] = make_double2(d[0], d[1]);
  };
  for (int step = 0; step < op.nsteps; ++step) {
    if (!step_on(op, step)) {
      if (t == 0 && lane == 0 && op.kused) op.kused[(int64_t)step * op.kused_ld + b - op.kcol0] = 0;
      observe(step);
      continue;
    }
    bool herm = (op.sflags & 1) && op.f.x == 0.0;
    for (int s = 0; s < op.nslot; ++s) herm = herm && op.table[(int64_t)step * op.nslot + s].y == 0.0;
    __syncthreads();
    double2* Gm = sh.gram;
    double2* cv = sh.cv;
    int g_ld = GL, k = 1;
    bool brk = false;
    double conv = 1.0;
    for (int it = 0;; ++it) {
      __syncthreads();   // the parts' sums
      if (!FIXED && it > 0 && !(k < a.maxorder && conv > a.tol)) break;
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
      double bs[1] = {0.0};
      blk_sum<1>(bs, sh.red, half);
      const double beta = sqrt(bs[0]);
      if (lane == 0) sh.beta[k] = beta;
      if (!FIXED) {
        if (it == 0) {
          if (lane == 0) {
            Gm[0] = make_double2(red[2], 0.0);
            cv[g_ld] = make_double2(1.0, 0.0);   // c_prev = [1]
            sh.conv = 1.0;
          }
        } else {
          wave_sync();
          conv = it < 16 ? metric16(it, brk, Gm, g_ld, sh.alpha, sh.beta, op.f, herm, cv, sh.cf)
                         : adaptive_metric<false>(it, brk, Gm, g_ld, sh.alpha, sh.beta, op.f, cv, cv + g_ld);
          if (lane == 0) sh.conv = conv;
        }
        if (k < a.maxorder && conv > a.tol && k == GL) {
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
      brk = !(beta != 0.0);
      if (!brk) continue;
      __syncthreads();   // the metric decides before the restart
      if (!FIXED && !(k < a.maxorder && conv > a.tol)) break;
      for (int j = 0; j <= k; ++j) {
        double d[2] = {0.0, 0.0};
        team_sum<FIXED>(d, a, sums, t, ns, sh, half, s_ab);
      }
      if (!FIXED) {
        // Gram column of the restart vector, explicit dots
        for (int j = 0; j < k; ++j) {
          double d[2] = {0.0, 0.0};
          team_sum<FIXED>(d, a, sums, t, ns, sh, half, s_ab);
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
    if (t == 0 && lane == 0) {
      if (op.kused) op.kused[(int64_t)step * op.kused_ld + b - op.kcol0] = k;
      if (!FIXED && k >= a.maxorder && op.status) op.status[b - op.kcol0] |= RM_NOT_CONVERGED;
    }
    observe(step);
  }
}

// The other waves' part.  A lane owns row `row` of its slice (part 0 of the
// slice's waves: state, basis and exchange of that row) and keeps rows
// vr + NVL j of the whole vectors.
template <bool FIXED>
__device__ __forceinline__ void team_work(const TeamArgs& a, const SubOp& op, int b, int lo, int len, int t, int wv,
                                          double2* s_x, double2* s_part, BlkShared<FIXED>& sh, double2* __restrict__ V,
                                          char* base, u64* slots, u64* sums, int& half, volatile int* s_ab) {
  const int lane = threadIdx.x & 63;
  const double2 zero = make_double2(0.0, 0.0);
  const int ns0 = op.srow[lo], nsl = op.srow[lo + len - 1] - ns0 + 1;   // the domain's slices
  const int s0 = nsl * t / a.team, nown = nsl * (t + 1) / a.team - s0;  // and this workgroup's
  const int G = nown > 0 ? NWORK / nown : 1;                            // parts per slice
  const int part = nown > 0 ? wv / nown : 1;
  const bool act = part < G, own = act && part == 0;
  const int nslot = op.nslot;
  const int si = ns0 + (act ? s0 + wv % nown : 0);
  const int4 sl = op.sslice[si];
  int row = sl.x - lo + lane;
  const bool ok = act && lane < sl.y && row >= 0 && row < len;
  if (!ok) row = 0;
  const bool mine = own && ok;
  const uint32_t cb = (uint32_t)(sl.w - lo) * 0x100010u;
  const int p0 = (int)((int64_t)sl.z * part / G), p1 = (int)((int64_t)sl.z * (part + 1) / G);
  const int np = ok ? p1 - p0 : 0;
  const int64_t e0 = op.soff[si] + (int64_t)p0 * 64 + lane;
  const int orig = op.perm[lo + row];
  const int vl = wv * 64 + lane;   // this lane's basis column and its rows of the whole vectors
  const int lmax = a.lmax;
  double2 S = load_or_zero(mine, op.psi + (int64_t)b * op.ld + orig);
  double2 A[NP];
  uint32_t cc[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    cc[p] = 0;
    A[p] = zero;
    if (p < np) {
      cc[p] = op.scol[e0 + 64 * p] + cb;
      if (nslot == 1) A[p] = pair_load<true>(op, 0, e0 + 64 * p);
    }
  }
  int n = 0, ns = 0, built = -1;
  double2 Vp[R], u[R];
  // this row's part in exchange n (one store per lane and exchange), then every row of it
  auto exchange = [&](double2 v) __attribute__((always_inline)) {
    if (mine) {
      if (n >= 2) {
        u64* old = slots + ((size_t)((n - 2) % RING) * lmax + row) * 2;
        empty(old);
        empty(old + 1);
      }
      if (n % 4 == 0) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      u64* p = slots + ((size_t)(n % RING) * lmax + row) * 2;
      put(p, v.x);
      put(p + 1, v.y);
    }
    const u64* q = slots + ((size_t)(n % RING) * lmax + vl) * 2;
    int miss = 0;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      u[j] = zero;
      if (vl + NVL * j < len) miss |= 1 << j;
    }
    wait_all<R>(a, s_ab, miss, [&](int j) __attribute__((always_inline)) {
      const u64 x = look(q + 2 * NVL * j), y = look(q + 2 * NVL * j + 1);
      if (x == LSENT || y == LSENT) return false;
      u[j] = make_double2(__longlong_as_double((long long)x), __longlong_as_double((long long)y));
      return true;
    });
    if (n % 4 == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    ++n;
  };
  // the exchanged rows as the vector in LDS (its readers are past a barrier)
  auto spread = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (vl + NVL * j < len) s_x[vl + NVL * j] = u[j];
  };
  auto observe = [&](int step) __attribute__((always_inline)) {
    if (op.ow <= 0) return;
    exchange(S);
    spread();
    __syncthreads();
    double d[2] = {0.0, 0.0};
    if (mine) {
      double2 y = zero;
      for (int j = 0; j < op.ow; ++j) {
        const int64_t q = (int64_t)j * op.n + lo + row;
        const int c = op.ocol[q] - lo;
        if (c >= 0 && c < len) y = fmac(op.oval[q], s_x[c], y);
      }
      d[0] = S.x * y.x + S.y * y.y;
      d[1] = S.x * y.y - S.y * y.x;
    }
    team_sum<FIXED>(d, a, sums, t, ns, sh, half, s_ab);   // its barrier: s_x is rewritten only after these reads
  };

  for (int step = 0; step < op.nsteps; ++step) {
    if (!step_on(op, step)) {
      // no field: the expv is skipped (tdse.py:377), phases only
      if (op.phase) S = cmul(cmul(S, op.phase[orig]), op.phase[orig]);
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
        imag = imag || f.y != 0.0;
        same = same && f.x == fb[s].x && f.y == fb[s].y;
      }
      if (!same && !imag) {
        built = step;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          double2 v = zero;
          if (p < np)
            for (int s = 0; s < nslot; ++s) pair_add(v, fp[s], pair_load<true>(op, s, e0 + 64 * p));
          A[p] = v;
        }
      }
    }
    const double2 f0 = nslot == 1 ? fp[0] : make_double2(1.0, 0.0);
    const bool realal = (op.sflags & 1) && op.f.x == 0.0 && !imag && f0.y == 0.0;
    // V_0 = phi = P psi (unnormalised, tdse.py:443-446), the first matvec input
    exchange(op.phase ? cmul(S, op.phase[orig]) : S);
    spread();
#pragma unroll
    for (int j = 0; j < R; ++j) Vp[j] = zero;
    __syncthreads();
    int k = 1;
    double beta = 0.0, ib = 1.0;
    for (int it = 0;; ++it) {
      if (mine) V[(int64_t)it * NVL + vl] = cscale(ib, s_x[row]);
      // this lane's part of w = A (W / beta)
      double2 y = zero;
      if (imag) {
        // complex field products: slot by slot
        for (int s = 0; s < nslot; ++s) {
          double2 acc = zero;
          for (int p = 0; p < np; ++p) {
            const uint32_t c = op.scol[e0 + 64 * p] + cb;
            pair_mac(pair_load<true>(op, s, e0 + 64 * p), s_x[(c & 0xffffu) >> 4], s_x[c >> 20], acc);
          }
          y = fmac(fp[s], acc, y);
        }
      } else {
        double2 acc0 = zero, acc1 = zero;
#pragma unroll
        for (int p = 0; p < NP; ++p) keep(A[p]);
#pragma unroll
        for (int p = 0; p < NP; p += 2) {
          // (the empty asm keeps the columns packed)
          asm volatile("" : "+v"(cc[p]));
          asm volatile("" : "+v"(cc[p + 1]));
          if (p < np) {
            const char* x = (const char*)s_x;
            pair_mac(A[p], *(const double2*)(x + (cc[p] & 0xffffu)), *(const double2*)(x + (cc[p] >> 16)), acc0);
            pair_mac(A[p + 1], *(const double2*)(x + (cc[p + 1] & 0xffffu)), *(const double2*)(x + (cc[p + 1] >> 16)),
                     acc1);
          }
        }
        y = cmul(f0, cadd(acc0, acc1));
      }
      if (act && part > 0) s_part[((part - 1) * nown + wv % nown) * 64 + lane] = y;
      __syncthreads();
      // the metric of the vectors so far (k = it)
      if (!FIXED && it > 0 && !(k < a.maxorder && sh.conv > a.tol)) break;
      if (own)
        for (int g = 1; g < G; ++g) y = cadd(y, s_part[((g - 1) * nown + wv) * 64 + lane]);
      exchange(cscale(ib, y));
      double red[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int j = 0; j < R; ++j)
        if (vl + NVL * j < len) {
          const double2 v = cscale(ib, s_x[vl + NVL * j]);
          red[0] += u[j].x * v.x + u[j].y * v.y;
          red[1] += u[j].x * v.y - u[j].y * v.x;
          red[2] += v.x * v.x + v.y * v.y;
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
      // W = w - alpha V_it - beta V_{it-1}, and |W|^2; every lane its own rows of s_x
      double bs[1] = {0.0};
#pragma unroll
      for (int j = 0; j < R; ++j)
        if (vl + NVL * j < len) {
          const double2 v = cscale(ib, s_x[vl + NVL * j]);
          const double2 w = csub(csub(u[j], cscale(beta, Vp[j])), cmul(al, v));
          Vp[j] = v;
          s_x[vl + NVL * j] = w;
          bs[0] += w.x * w.x + w.y * w.y;
        }
      // beta_k = |W| (tdse.py:453); publishes W, the next matvec input
      blk_sum<1>(bs, sh.red, half);
      beta = sqrt(bs[0]);
      if (beta != 0.0) {
        ib = __builtin_amdgcn_rcp(beta);   // and two Newton steps (within an ulp of the quotient)
        ib = fma(fma(-beta, ib, 1.0), ib, ib);
        ib = fma(fma(-beta, ib, 1.0), ib, ib);
        continue;
      }
      __syncthreads();
      if (!FIXED && !(k < a.maxorder && sh.conv > a.tol)) break;
      // exact breakdown: Gram-Schmidt of ones against the basis (tdse.py:459-465)
      // on the owned rows; the restart vector becomes the next matvec input with ib = 1
      ib = 1.0;
      double2 W = mine ? make_double2(1.0, 0.0) : zero;
      for (int j = 0; j < k; ++j) {
        const double2 vj = load_or_zero(mine, V + (int64_t)j * NVL + vl);
        double d[2] = {vj.x * W.x + vj.y * W.y, vj.x * W.y - vj.y * W.x};
        team_sum<FIXED>(d, a, sums, t, ns, sh, half, s_ab);
        W = csub(W, cmul(make_double2(d[0], d[1]), vj));
      }
      double nv[2] = {W.x * W.x + W.y * W.y, 0.0};
      team_sum<FIXED>(nv, a, sums, t, ns, sh, half, s_ab);
      const double nrm = sqrt(nv[0]);
      // nrm == 0: the basis spans the domain; the reference's restart vector
      // lies outside it and enters with coefficient exactly zero
      W = nrm > 0.0 ? make_double2(W.x / nrm, W.y / nrm) : zero;
      if (!FIXED)   // Gram column of the restart vector, explicit dots
        for (int j = 0; j < k; ++j) {
          const double2 vj = load_or_zero(mine, V + (int64_t)j * NVL + vl);
          double d[2] = {vj.x * W.x + vj.y * W.y, vj.x * W.y - vj.y * W.x};
          team_sum<FIXED>(d, a, sums, t, ns, sh, half, s_ab);
        }
      exchange(W);
      spread();
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
    if (mine) {
      double2 v = zero;
#pragma unroll 4
      for (int j = 0; j < k; ++j) v = fmac(cf[j], V[(int64_t)j * NVL + vl], v);
      S = op.phase ? cmul(v, op.phase[orig]) : v;
    }
    observe(step);
    // the coefficients are rewritten only after the next step's first barrier
  }
  if (mine) op.psi[(int64_t)b * op.ld + orig] = S;
}

template <bool FIXED>
__global__ __launch_bounds__(NT) void k_team(TeamArgs a) {
  extern __shared__ double2 s_x[];   // [lmax] the vector, at the start of LDS: gathers address it by offset
  __shared__ double2 s_part[NWORK * 64];
  __shared__ BlkShared<FIXED> sh;
  __shared__ int s_ab;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // members of a team nteams apart: with nteams a multiple of 8 they share an XCD's L2
  const int t = blockIdx.x / a.nteams;
  char* base = a.ws + (int64_t)blockIdx.x * a.wg_bytes;
  int half = 0;
  if (threadIdx.x == 0) s_ab = 0;
  __syncthreads();
  for (int itm = blockIdx.x % a.nteams; itm < a.nitems; itm += a.nteams) {
    const int4 item = a.items[itm];
    const SubOp& op = a.ops ? a.ops[item.w] : a.op0;
    if (op.stale && *op.stale == op.call_id) {
      // reused domains that failed their check: the wavepacket is left as it is
      if (t == 0 && threadIdx.x == 0 && op.status) op.status[item.x - op.kcol0] |= RM_STALE_DOMAIN;
      continue;
    }
    u64* slots = a.rows + (size_t)itm * RING * a.lmax * 2;
    u64* sums = a.sums + (size_t)itm * SRING * TEAM_MAX * 2;
    if (wv == NWORK)
      team_control<FIXED>(a, op, item.x, t, sums, sh, (double2*)(base + a.offG), half, &s_ab);
    else
      team_work<FIXED>(a, op, item.x, item.y, item.z, t, wv, s_x, s_part, sh, (double2*)base, base, slots, sums,
                          half, &s_ab);
    __syncthreads();   // the next item rewrites LDS after these reads
    if (t == 0 && threadIdx.x == 0 && op.status &&
        (s_ab || __hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
      op.status[item.x - op.kcol0] |= RM_DEVICE_TIMEOUT;
  }
}

__global__ void k_team_reset(u64* slots, int64_t count, int32_t* abort_flag, int32_t abort_preset) {
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i0 == 0) *abort_flag = abort_preset ? 1 : 0;
  for (int64_t i = i0; i < count; i += (int64_t)gridDim.x * blockDim.x) slots[i] = LSENT;
}

size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

// The teams are as large as the device and the domains allow: fewer members
// would hold more entries each but poll less, which was not measured apart.  The
// bound on the launch's workgroups (800 entries of the smallest domain for each)
// lies where the block kernel's step gets shorter.  Measured (water-like top,
// adaptive rule with 4 vectors, us per step, block / team):
//   90 372 entries, 1 wavepacket 56 / 40, 4: 56 / 47, 8: 57 / 64
//  153 186 entries, 1 wavepacket 74 / 43, 4: 75 / 57, 8: 76 / 85
//  370 802 entries, 1 wavepacket 194 / 51, 4: 236 / 87
// (shorter domains: 49 218 entries 38 / 43).
int team_size(const std::vector<LongItem>& items, int n_cu, int32_t max_grid, bool forced) {
  if (items.empty()) return 0;
  if (max_grid > 0) n_cu = std::min<int>(n_cu, max_grid);
  int64_t lo = 2, hi = std::min<int64_t>(TEAM_MAX, n_cu / (int64_t)items.size()), emin = INT64_MAX;
  for (const LongItem& it : items) {
    if (it.item.z <= NVL || it.item.z > TEAM_MAX_ROWS || !it.real) return 0;
    // a workgroup without a slice of every item could not take part in its exchanges
    hi = std::min<int64_t>(hi, it.nslices);
    emin = std::min(emin, it.nent);
  }
  for (const LongItem& it : items) {
    int64_t need = 0;
    for (int64_t t = lo; t <= hi && !need; ++t) {
      const int64_t own = (it.nslices + t - 1) / t;
      if (own <= NWORK && (it.maxpairs + NWORK / own - 1) / (NWORK / own) <= NP) need = t;
    }
    if (!need) return 0;
    lo = std::max(lo, need);
  }
  return forced || hi * (int64_t)items.size() * 800 <= emin ? (int)hi : 0;
}

extern "C" int rm_team_size(int32_t nitems, const int32_t* rows, const int32_t* slices, const int32_t* pairs,
                            const int64_t* entries, int32_t n_cu, int32_t max_grid, int32_t forced) {
  if (nitems < 0 || n_cu < 1 || (nitems > 0 && (!rows || !slices || !pairs || !entries)))
    return fail(RM_ERR_ARG, "rm_team_size: bad arguments");
  std::vector<LongItem> items((size_t)nitems);
  for (int32_t i = 0; i < nitems; ++i) {
    items[i].item = make_int4(i, 0, rows[i], 0);
    items[i].nslices = slices[i];
    items[i].maxpairs = pairs[i];
    items[i].nent = entries[i];
    items[i].real = true;
  }
  return team_size(items, n_cu, max_grid, forced != 0);
}

int team_run(void** ws, size_t* ws_bytes, const SubOp* d_ops, const SubOp* op0, const int4* d_items,
             const std::vector<LongItem>& items, int team, int32_t kcap, int32_t fixed_m, int32_t maxorder, double tol,
             int n_cu, hipStream_t s, int32_t abort_preset) {
  const bool fixed = fixed_m > 0;
  TeamArgs a;
  memset(&a, 0, sizeof(a));
  int64_t lmax = 0;
  for (const LongItem& it : items) lmax = std::max<int64_t>(lmax, it.item.z);
  const void* kern = fixed ? (const void*)k_team<true> : (const void*)k_team<false>;
  const size_t lds = sizeof(double2) * (size_t)lmax;
  int occ = 0;
  HIPCHK(occupancy(kern, NT, lds, &occ));
  const int nteams = (int)std::min<int64_t>((int64_t)items.size(), (int64_t)occ * n_cu / team);
  if (nteams < 1) return fail(RM_ERR_ARG, "team propagation: %d workgroups of %lld rows do not fit", team, (long long)lmax);
  const size_t b_v = al256(sizeof(double2) * (size_t)(kcap + 1) * NVL);
  const size_t b_g = fixed ? 0 : al256(sizeof(double2) * ((size_t)kcap * kcap + 2 * (size_t)kcap));
  const size_t wg = b_v + b_g;
  const size_t n_rows = items.size() * RING * (size_t)lmax * 2, n_sums = items.size() * SRING * TEAM_MAX * 2;
  const size_t b_slots = al256(sizeof(u64) * (n_rows + n_sums));
  const size_t need = b_slots + 256 + wg * (size_t)(nteams * team);
  if (*ws_bytes < need) {
    if (*ws) {
      HIPCHK(hipDeviceSynchronize());
      HIPCHK(hipFree(*ws));
      *ws = nullptr;
      *ws_bytes = 0;
    }
    HIPCHK(hipMalloc(ws, need));
    *ws_bytes = need;
  }
  a.ops = op0 ? nullptr : d_ops;
  if (op0) a.op0 = *op0;
  a.items = d_items;
  a.nitems = (int32_t)items.size();
  a.team = team;
  a.nteams = nteams;
  a.rows = (u64*)*ws;
  a.sums = a.rows + n_rows;
  a.abort_flag = (int32_t*)((char*)*ws + b_slots);
  a.ws = (char*)*ws + b_slots + 256;
  a.wg_bytes = (int64_t)wg;
  a.offG = (int64_t)b_v;
  a.kcap = kcap;
  a.fixed_m = fixed_m;
  a.maxorder = maxorder;
  a.lmax = (int32_t)lmax;
  a.tol = tol;
  hipLaunchKernelGGL(k_team_reset, dim3(grid_for((int64_t)(n_rows + n_sums), 256)), dim3(256), 0, s, a.rows,
                     (int64_t)(n_rows + n_sums), a.abort_flag, abort_preset);
  HIPCHK(hipGetLastError());
  void* args[] = {&a};
  HIPCHK(hipLaunchCooperativeKernel(kern, dim3((unsigned)(nteams * team)), dim3(NT), args, lds, s));
  return RM_OK;
}
