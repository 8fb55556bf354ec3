"""The one-wave kernel of short domains (k_wav: the adaptive rule, fixed
dimensions beyond 16, wider operators) against the FP64 oracle: amplitudes to
1e-10 and the adaptive Krylov dimensions, for one and two wavepackets per wave,
real and complex operators; orders beyond what LDS holds against the
full-vector kernel; bits independent of the partner.
"""
import numpy as np
import pytest

from _fixtures import linear_rotor, water
from test_gpu_subspace import TOL_PSI, _basis_columns, _device_run, _oracle_run
from richmol_amd import ensemble

pytestmark = pytest.mark.gpu

Z, XZ, XYZ = (0.0, 0.0, 1.0), (0.5, 0.0, 0.8), (0.4, 0.3, 0.8)


@pytest.mark.parametrize("jmax,axis,fixed,ncols", [(10, Z, 0, 5), (10, Z, 20, 3), (70, Z, 0, 2), (6, XZ, 0, 3),
                                                   (6, XYZ, 0, 3), (6, XYZ, 20, 2), (9, XYZ, 0, 4), (9, XZ, 12, 4),
                                                   (1, XZ, 0, 2)])
def test_against_oracle(device, jmax, axis, fixed, ncols):
    """Chains of 1..36 rows (Z) and mixed domains of 1..55 rows (entries of
    up to 15 per row), a zero-field step, rows of norm other than one."""
    h0, H, cos2, bas = linear_rotor(jmax)
    n = (jmax + 1) ** 2
    X = _basis_columns(n, [0, 2, n - 1, 1, 6][:ncols])
    X[0] *= 1.7
    fields = [[a * c for c in axis] for a in (6e8, 0.0, 1.1e9, 1.1e9)]
    psi_d, k_d, _ = _device_run(h0, H, fields, X, fixed=fixed)
    psi_o, k_o = _oracle_run(h0, H, fields, X, fixed=fixed or None)
    assert np.abs(psi_d - psi_o).max() <= TOL_PSI
    if not fixed:
        assert np.array_equal(k_d, k_o)


@pytest.mark.parametrize("fixed", [0, 30])
@pytest.mark.parametrize("factor", [1.0, 0.7 - 0.2j])
@pytest.mark.parametrize("f", [-0.0019j, -0.03j])
def test_long_recurrences(device, fixed, factor, f):
    """A strong field and a long step need Krylov dimensions beyond 16
    (adaptive), or 30 are asked for; the table also with complex products;
    <cos^2> after every step."""
    h0, H, cos2, bas = linear_rotor(40)
    X = _basis_columns(1681, [0, 2, 6, 12, 20])
    fields = [[0.0, 0.0, a] for a in (6e9, 8e9, 2e9)]
    O = ensemble.Ensemble.observable_plan(cos2)
    out = []
    for kern in ("subspace", "global"):
        H.field(fields[0])
        e = ensemble.Ensemble(H, h0, f, X, krylov_fixed=fixed)
        e.set_kernel(kern)
        table = e.prepare(fields) * factor
        import torch
        ku = torch.zeros((3, 5), dtype=torch.int32, device=device)
        try:
            ex, _ = e.propagate(None, table=table, obs=O, kused=ku)
        except ValueError:   # maxorder reached: the recurrence is not made for a non-Hermitian operator
            assert factor != 1.0 and fixed == 0
            out.append(None)
            continue
        out.append((e.psi.cpu().numpy(), ex.cpu().numpy(), ku.cpu().numpy()))
    a, b = out
    assert (a is None) == (b is None)
    if a is None:
        return
    scale = np.abs(b[0]).max()
    assert np.abs(a[0] - b[0]).max() <= 1e-10 * scale
    assert np.abs(a[1] - b[1]).max() <= 1e-10 * max(1.0, np.abs(b[1]).max())
    assert np.array_equal(a[2], b[2])
    if f == -0.03j and factor == 1.0:
        assert b[2].max() > 16


def test_bits_independent_of_partner(device):
    """Adaptive: every column alone, in a batch and in another order."""
    h0, H, cos2, bas = linear_rotor(20)
    rng = np.random.default_rng(5)
    idx = rng.choice(441, size=9, replace=False)
    X = _basis_columns(441, idx)
    fields = [[0.0, 0.0, a] for a in (6e8, 1.4e9, 1.0e9)]
    full, kf, _ = _device_run(h0, H, fields, X)
    back, _, _ = _device_run(h0, H, fields, X[::-1])
    assert np.array_equal(full, back[::-1])
    for i in range(9):
        one, k1, _ = _device_run(h0, H, fields, X[i:i + 1])
        assert np.array_equal(one[0], full[i]) and np.array_equal(k1[:, 0], kf[:, i])


def test_fp32_and_pairing_choice(device):
    """FP32 matvecs within 2e-6; one wavepacket per wave (pair = 0) to 1e-12."""
    h0, H, cos2, bas = linear_rotor(16)
    X = _basis_columns(289, [0, 2, 3, 7, 30])
    fields = [[0.0, 0.0, a] for a in (6e8, 1.4e9, 1.0e9)]
    ref, kr, _ = _device_run(h0, H, fields, X)
    f32, _, _ = _device_run(h0, H, fields, X, precision="fp32")
    assert 0 < np.abs(f32 - ref).max() <= 2e-6
    H.field(fields[0])
    from richmol_amd.tdse import TDSE
    e = ensemble.Ensemble(H, h0, TDSE(t_end=30.0, dt=10.0, t_units="fs").exp_fac, X)
    e.set_tuning(pair=0)
    e.propagate(fields)
    assert np.abs(e.psi.cpu().numpy() - ref).max() <= 1e-12
