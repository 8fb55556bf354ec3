// richmol_amd: the Kronecker-block operator in the primitive symmetric-top
// basis (rm_kprim.hip), used by a plan whose K blocks came with their factors.
#pragma once

#include "rm_common.h"

struct KPrim;

// The M side of one source block (as rm_kplan keeps it).
struct KPrimBlock {
  int32_t J1, J2, ncart, slot0, nsig;
  int32_t sig[5];
  int64_t d_off;   // its diagonals in the plan's mdiag
};

// C: per J (ascending) the (2J+1) x (2J+1) coefficient matrix, complex
// row-major (primitive k, state); P: per block [5][2 J1 + 1] complex, the
// entry (s + 2, k1) multiplying primitive column k1 - s.  mdiag: the plan's
// device array of M diagonals.
int kprim_create(KPrim** out, const std::vector<int32_t>& Js, const std::vector<int64_t>& voff, int64_t n,
                 const std::vector<KPrimBlock>& blk, const double2* mdiag, const double* C, const double* P);
void kprim_free(KPrim* p);
// y = H(F) x (rows of stride ld, the plan's internal order)
int kprim_matvec(KPrim* p, const double2* x, double2* y, int64_t ld, int32_t ncols, const double2* fprod, bool f32,
                 hipStream_t s);
// rm_kplan_propagate on this form; d_fp: the steps' field products on the
// device, fprod: the same on the host.  obs (may be NULL): an observable on
// the same states, d_ofp its products; ex: [nsteps][ncols] values.
int kprim_propagate(KPrim* p, double2* psi, int64_t ld, int32_t ncols, int64_t nsteps, int32_t nslot,
                    const double* fprod, const double2* d_fp, double2 f, const double2* phase, int32_t krylov_fixed,
                    int32_t maxorder, double tol, int32_t* kused, int32_t* status, bool f32, KPrim* obs,
                    const double2* d_ofp, double2* ex, hipStream_t s);
