// richmol_amd: arguments of the one-wave kernels (rm_subspace.hip, rm_wave.hip).
#pragma once

#include "rm_common.h"

struct SubArgs {
  const SubOp* ops;        // the jobs, or NULL: the one job is op0
  SubOp op0;               // the job of a single-job launch, by value (no staging)
  const int4* items;       // (column, lo, len, op), one wavepacket each
  int32_t nitems;
  double2* basis;          // per wave kcap * 64R (global-basis variant)
  double2* gram;           // per wave kcap * kcap (adaptive)
  double2* cscr;           // per wave 2 * kcap (adaptive)
  int32_t kcap, fixed_m, maxorder;
  double tol;
  int32_t max_waves;       // > 0: at most this many waves (the launch's workspace holds no more)
  int32_t obs;             // 1: some job reads an observable (k_sub_prop: LDS for the state)
};

// k_wav launch kinds: one or two wavepackets per wave, pairs of entries per
// lane at most, real or complex operator
enum { WAV_S2 = 0, WAV_S32 = 1, WAV_P2 = 2, WAV_P16 = 3, WAV_SC = 4, WAV_PC = 5 };
constexpr int WAV_NP[6] = {2, 32, 2, 16, 32, 16};
inline bool wav_pair(int kind) { return kind == WAV_P2 || kind == WAV_P16 || kind == WAV_PC; }
// elements (double2) per wave: the Krylov basis, the Gram matrices and the
// coefficients beyond what LDS holds
inline size_t wav_basis(int kcap) { return (size_t)kcap * 64; }
inline size_t wav_gram(int kind, int kcap, bool fixed) { return fixed ? 0 : (size_t)kcap * kcap * (wav_pair(kind) ? 2 : 1); }
// (c, c_prev, alpha, and beta as reals)
inline size_t wav_cscr(int kind, int kcap) { return (4 * (size_t)kcap + 1) * (wav_pair(kind) ? 2 : 1); }
// Launches a.items (column, lo, len, op; a pair's items adjacent, column -1: an
// empty half) or, dry, only tells the number of waves.
hipError_t launch_wav(int kind, const SubArgs& a, bool f32, int n_cu, hipStream_t s, int* waves, bool dry);
