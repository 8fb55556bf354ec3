"""The block kernel (one workgroup per wavepacket on its invariant subspace,
kernel 'block') against the FP64 oracle (1e-10) and the full-vector kernel
on the same field table (1e-11), at the sizes where its layout changes: one
slice of rows to several per wave, entries in registers or read at every
matvec, operators real or complex, field products complex.
"""
import numpy as np
import pytest

from _fixtures import linear_rotor
from test_gpu_subspace import TOL_PSI, _device_run, _oracle_run
from richmol_amd import ensemble

pytestmark = pytest.mark.gpu

# off-Z fields mix m: two domains per rotor (even and odd J); a Y component makes the operator complex
XZ, XYZ = (0.5, 0.0, 0.8), (0.4, 0.3, 0.8)


def _columns(n, seed):
    """|0,0>, a row on the odd-J domain and a dense row (both domains)."""
    rng = np.random.default_rng(seed)
    X = np.zeros((3, n), dtype=np.complex128)
    X[0, 0] = 1.0
    X[1, 2] = 1.0
    X[2] = rng.normal(size=n) + 1j * rng.normal(size=n)
    X[2] /= np.linalg.norm(X[2])
    return X


@pytest.mark.parametrize("jmax,axis,fixed", [(2, XZ, 0), (8, XZ, 12), (11, XZ, 0), (11, XYZ, 12), (21, XZ, 0),
                                             (30, XYZ, 0), (30, XZ, 20)])
def test_against_oracle(device, jmax, axis, fixed):
    h0, H, cos2, bas = linear_rotor(jmax)
    n = (jmax + 1) ** 2
    X = _columns(n, jmax)
    fields = [[a * c for c in axis] for a in (6e8, 0.0, 1.1e9, 1.1e9)]
    psi_d, k_d, _ = _device_run(h0, H, fields, X, kernel="block", fixed=fixed)
    psi_o, k_o = _oracle_run(h0, H, fields, X, fixed=fixed or None)
    assert np.abs(psi_d - psi_o).max() <= TOL_PSI
    if not fixed:
        assert np.array_equal(k_d, k_o)


@pytest.mark.parametrize("jmax,axis", [(11, XZ), (44, XZ), (50, XYZ), (62, XZ), (63, XZ)])
@pytest.mark.parametrize("factor", [1.0, 0.8 + 0.1j])
@pytest.mark.parametrize("fixed", [0, 9])
def test_against_full_vector_kernel(device, jmax, axis, factor, fixed):
    """Up to 4 096 rows in a domain (several slices per wave); the field
    table also with complex products (real operator entries, slot by slot)."""
    import torch
    h0, H, cos2, bas = linear_rotor(jmax)
    n = (jmax + 1) ** 2
    X = _columns(n, jmax)
    fields = [[a * c for c in axis] for a in (7e8, 1.2e9, 1.2e9)]
    O = ensemble.Ensemble.observable_plan(cos2)
    out = []
    for kern in ("block", "global"):
        H.field(fields[0])
        e = ensemble.Ensemble(H, h0, -0.0019j, X, krylov_fixed=fixed)
        e.set_kernel(kern)
        table = e.prepare(fields) * factor
        ex, _ = e.propagate(None, table=table, obs=O)
        out.append((e.psi.cpu().numpy(), ex.cpu().numpy()))
    (pa, ea), (pb, eb) = out
    assert np.abs(pa - pb).max() <= 1e-11
    assert np.abs(ea - eb).max() <= 1e-11


@pytest.mark.parametrize("jmax", [11, 30])
def test_fp32(device, jmax):
    """FP32 matvecs within 2e-6 of FP64 (registers and memory forms)."""
    h0, H, cos2, bas = linear_rotor(jmax)
    n = (jmax + 1) ** 2
    X = _columns(n, 1)
    fields = [[a * c for c in XZ] for a in (7e8, 1.2e9, 9e8)]
    out = []
    for prec in ("fp64", "fp32"):
        H.field(fields[0])
        e = ensemble.Ensemble(H, h0, -0.0019j, X, krylov_fixed=12)
        e.set_kernel("block")
        e.set_precision(prec)
        e.propagate(fields)
        out.append(e.psi.cpu().numpy())
    assert 0 < np.abs(out[0] - out[1]).max() <= 2e-6


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("fixed", [0, 9])
@pytest.mark.parametrize("kib", [0, 256, 512])
def test_launches_cut_between_steps(device, kib, fixed, prec):
    """Domains of 990 to 2 025 rows whose operators are formed ahead for one or
    two steps a launch, or by every workgroup (0): amplitudes, observable and
    Krylov dimensions bit for bit those of the uncut run.  A zero-field step and
    repeated products come right after a cut."""
    import torch
    h0, H, cos2, bas = linear_rotor(44)
    X = _columns(2025, 44)
    fields = [[a * c for c in XZ] for a in (6e8, 9e8, 0.0, 1.1e9, 1.1e9, 1.1e9, 7e8)]
    H.field(fields[0])
    O = ensemble.Ensemble.observable_plan(cos2)
    out = []
    for k in (kib, 1 << 18):
        e = ensemble.Ensemble(H, h0, -0.0019j, X, krylov_fixed=fixed)
        e.set_kernel("block")
        e.set_precision(prec)
        e.set_tuning(operator_kib=k)
        ku = torch.full((7, 3), -1, dtype=torch.int32, device=device)
        ex, _ = e.propagate(None, table=e.prepare(fields), obs=O, kused=ku)
        out.append((e.psi.cpu().numpy(), ex.cpu().numpy(), ku.cpu().numpy()))
        e.set_tuning()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert np.all((out[0][2] == 0) == (np.arange(7) == 2)[:, None])


@pytest.mark.parametrize("jmax", [8, 14])
def test_fp32_of_one_slot_over_many_steps(device, jmax):
    """One field slot: B_0's entries rounded to FP32 are the same at every step,
    so their error adds up -- to at most steps |f F| 2^-24 times the operator's
    largest row sum (registers and memory forms, 200 steps)."""
    from _fixtures import water
    h0, leaves, bas = water(jmax)
    H = leaves[0]
    n = sum((2 * J + 1) ** 2 for J in range(jmax + 1))
    X = np.zeros((2, n), dtype=np.complex128)
    X[0, 0] = 1.0
    X[1, [0, 1, 5]] = 3.0 ** -0.5
    amp = 3e8 * (1.0 + 0.5 * np.cos(0.1 * np.arange(200)))
    fields = [[a, 0.0, 0.0] for a in amp]
    f = -0.00094j
    out = []
    for prec in ("fp64", "fp32"):
        H.field(fields[0])
        e = ensemble.Ensemble(H, h0, f, X, krylov_fixed=8)
        e.set_kernel("block")
        e.set_precision(prec)
        e.propagate(fields)
        out.append(e.psi.cpu().numpy())
    row = float(abs(H.tomat(form="full", cart="x")).sum(axis=1).max())
    bound = abs(f) * amp.sum() * row * 2.0 ** -24
    err = np.linalg.norm(out[0] - out[1], axis=1).max()
    print(f"J<={jmax}: FP32 error {err:.2e} after 200 steps, bound {bound:.2e}", flush=True)
    assert 0 < err <= bound
