"""The team kernel (several workgroups on each of a few wavepackets with real
operators) against the full-vector kernel on the same field table (1e-11), at
the sizes where its layout and the rule for it change: one or more slices per
workgroup, few and many wavepackets, adaptive and fixed Krylov dimensions,
complex field products, steps whose products are so small that |W|^2
underflows (the restart after a breakdown), an observable, wavepackets on
domains of different lengths side by side without one.
"""
import numpy as np
import pytest
from scipy.sparse import csr_matrix
from scipy.sparse.csgraph import connected_components

from _fixtures import linear_rotor, water, water_fields
from test_gpu_asymtop import DT, _summed
from richmol_amd import ensemble
from richmol_amd.tdse import TDSE

pytestmark = pytest.mark.gpu


def _rows(n, ncols, seed):
    """A row of every basis state, and single basis states."""
    rng = np.random.default_rng(seed)
    X = np.zeros((ncols, n), dtype=np.complex128)
    X[0] = rng.normal(size=n) + 1j * rng.normal(size=n)
    X[0] /= np.linalg.norm(X[0])
    X[np.arange(1, ncols), np.sort(rng.choice(n, size=ncols - 1, replace=False))] = 1.0
    return X


def _compare(H, h0, f, X, table_of, fixed, factor, obs, kernel):
    out = []
    for kern in (kernel, "global"):
        e = ensemble.Ensemble(H, h0, f, X, krylov_fixed=fixed)
        e.set_kernel(kern)
        ex = e.propagate(None, table=table_of(e) * factor, obs=obs)
        out.append((e.psi.cpu().numpy(), ex[0].cpu().numpy() if obs is not None else np.zeros(1)))
    (pa, ea), (pb, eb) = out
    assert np.abs(pa - pb).max() <= 1e-11
    assert np.abs(ea - eb).max() <= 1e-11


@pytest.mark.parametrize("jmax,ncols", [(12, 2), (14, 2), (14, 5), (14, 9), (16, 3), (17, 13)])
@pytest.mark.parametrize("fixed,factor", [(0, 1.0), (9, 1.0), (0, 0.9 + 0.1j)])
def test_asymmetric_top(device, jmax, ncols, fixed, factor):
    h0, leaves, bas = water(jmax)
    n = sum((2 * J + 1) ** 2 for J in range(jmax + 1))
    fields = water_fields(395.0 + DT * np.arange(3))
    f = TDSE(t_end=20.0, dt=DT, t_units="fs").exp_fac
    X = _rows(n, ncols, jmax)[1:]   # both sides of the rule: the team kernel and the block kernel
    _compare(_summed(leaves, fields, 0), h0, f, X, lambda e: e.prepare(fields, per_term=True), fixed, factor, None, "auto")


@pytest.mark.parametrize("jmax", [34, 50])
@pytest.mark.parametrize("fixed", [0, 12])
@pytest.mark.parametrize("kernel", ["coop", "block"])
def test_linear_rotor_observable_and_restart(device, jmax, fixed, kernel):
    h0, H, cos2, bas = linear_rotor(jmax)
    fields = [[0.5 * a, 0.0, 0.8 * a] for a in (7e8, 1.2e9, 1.2e9, 0.0, 1e-165)]
    H.field(fields[0])
    obs = ensemble.Ensemble.observable_plan(cos2)
    X = _rows((jmax + 1) ** 2, 3, jmax)
    _compare(H, h0, -0.0019j, X, lambda e: e.prepare(fields), fixed, 1.0, obs, kernel)


@pytest.mark.parametrize("order", [1, -1])
@pytest.mark.parametrize("fixed", [0, 9])
@pytest.mark.parametrize("kernel", ["auto", "coop"])
def test_unequal_domains(device, order, fixed, kernel):
    """A basis state (18 slices) beside a superposition of two species (36), no
    observable, many exchanges: amplitudes and Krylov dimensions."""
    import torch
    h0, leaves, bas = water(14)
    n = sum((2 * J + 1) ** 2 for J in range(15))
    fields = water_fields(395.0 + DT * np.arange(12))
    f = TDSE(t_end=20.0, dt=DT, t_units="fs").exp_fac
    H = _summed(leaves, fields, 0)
    e = ensemble.Ensemble(H, h0, f, np.eye(1, n, dtype=np.complex128), krylov_fixed=fixed)
    e.prepare(fields, per_term=True)
    arr = e.plan._arrays
    A = csr_matrix((np.ones(arr["nnz"]), arr["col_idx"], arr["row_ptr"]), shape=(n, n))
    _, lab = connected_components(A)
    X = np.zeros((2, n), dtype=np.complex128)
    X[:, np.argmax(lab == 0)] = 1.0
    X[1, np.argmax(lab == 1)] = 1.0
    assert e.plan.domain_sizes(X)[0].tolist() == [1135, 2255]
    X[1] /= np.linalg.norm(X[1])
    out = []
    for kern in (kernel, "global"):
        e = ensemble.Ensemble(H, h0, f, X[::order].copy(), krylov_fixed=fixed)
        e.set_kernel(kern)
        ku = torch.full((12, 2), -1, dtype=torch.int32, device=device)
        e.propagate(None, table=e.prepare(fields, per_term=True), kused=ku)
        out.append((e.psi.cpu().numpy(), ku.cpu().numpy()))
    assert np.abs(out[0][0] - out[1][0]).max() <= 1e-11
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("fixed", [0, 9])
def test_cooperative_form_at_these_sizes(device, fixed):
    """The grid form of the cooperative kernel on domains teams would take
    (kernel 'coop' with coop_max 0): the full-vector kernel's amplitudes."""
    h0, leaves, bas = water(14)
    n = sum((2 * J + 1) ** 2 for J in range(15))
    fields = water_fields(395.0 + DT * np.arange(3))
    f = TDSE(t_end=20.0, dt=DT, t_units="fs").exp_fac
    H = _summed(leaves, fields, 0)
    out = []
    for kern in ("coop", "global"):
        e = ensemble.Ensemble(H, h0, f, _rows(n, 3, 4)[1:], krylov_fixed=fixed)
        e.set_kernel(kern)
        e.set_tuning(coop_max=0 if kern == "coop" else 8)
        e.propagate(None, table=e.prepare(fields, per_term=True))
        out.append(e.psi.cpu().numpy())
        e.set_tuning()
    assert np.abs(out[0] - out[1]).max() <= 1e-11
