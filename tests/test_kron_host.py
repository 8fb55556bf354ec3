"""Kronecker-block operator builder (richmol_amd.kron) on the CPU: the
vectorised 3j symbols against the exact ones, and the factored operator
against the oracle's block operator (CarTens.vec, field.py:1145-1245) on an
asymmetric top with a dipole and a full polarizability under a general field."""
import numpy as np
import pytest
from scipy.sparse import csr_matrix

from _fixtures import large_top, large_top_tensors
from richmol_amd import kron, rot


def test_wigner3j_array_vs_exact():
    """Racah sum in extended precision vs exact rational arithmetic
    (rot.wigner3j), first angular momenta up to 80 with the second <= 2 as the
    operators use them, plus a brute-force grid of small values."""
    rng = np.random.default_rng(4)
    cases = []
    for _ in range(400):
        j1 = int(rng.integers(0, 81))
        j2 = int(rng.integers(0, 3))
        j3 = int(rng.integers(abs(j1 - j2), j1 + j2 + 1))
        m1 = int(rng.integers(-j1, j1 + 1))
        m2 = int(rng.integers(-j2, j2 + 1))
        cases.append((j1, j2, j3, m1, m2, -m1 - m2))
    for j1 in range(4):
        for j2 in range(3):
            for j3 in range(5):
                for m1 in range(-j1, j1 + 1):
                    for m2 in range(-j2, j2 + 1):
                        cases.append((j1, j2, j3, m1, m2, -m1 - m2))
    c = np.array(cases)
    got = kron.wigner3j_array(*c.T)
    ref = np.array([float(rot.wigner3j(*row)) for row in cases])
    assert np.abs(got - ref).max() <= 1e-14
    # selection rules: m sum, triangle
    assert kron.wigner3j_array(2, 1, 2, 1, 0, 0) == 0.0
    assert kron.wigner3j_array(5, 1, 2, 0, 0, 0) == 0.0


def _oracle_apply(bas, fields, X):
    from oracle.cartens import OracleCarTens, flatten, unflatten
    tens, scales = large_top_tensors()
    Y = np.zeros_like(X)
    for t, s, F in zip(tens, scales, fields):
        O = OracleCarTens.from_attrs(rot.tensor(t, bas) * s)
        O.field(list(F))
        for b in range(len(X)):
            Y[b] += flatten(O, O.vec(unflatten(O, X[b])))
    return Y


@pytest.mark.parametrize("fields", [[(0.3e8, -0.8e8, 0.5e8)] * 2,
                                    [(1e8, 0.0, 0.0), (0.0, 0.7e8, 0.2e8)]])
def test_kron_matvec_equals_oracle(fields):
    """J <= 4 with all m (165 states): the factored matvec, after mapping the
    reference's full-form order to the internal one, equals the oracle's
    block operator to rounding, for the same and for different fields on the
    two tensors."""
    kop, bas = large_top(4)
    assert kop.n == 165
    rng = np.random.default_rng(2)
    Xf = rng.normal(size=(3, kop.n)) + 1j * rng.normal(size=(3, kop.n))
    Yf = _oracle_apply(bas, fields, Xf)
    Xi = np.zeros_like(Xf)
    Xi[:, kop.perm] = Xf
    Yi = kop.matvec(Xi, kop.field_products(fields))
    assert np.abs(Yi[:, kop.perm] - Yf).max() <= 1e-12 * np.abs(Yf).max()


def test_kron_layout_and_energies():
    """perm is a permutation onto the J-blocked (m, k) layout, and the
    internal energies are the field-free Hamiltonian's diagonal."""
    kop, bas = large_top(5)
    assert sorted(kop.perm.tolist()) == list(range(kop.n))
    h0 = rot.hamiltonian(bas).tomat(form="full", cart="0").diagonal().real
    assert np.allclose(kop.energies[kop.perm], h0, rtol=0, atol=1e-12 * np.abs(h0).max())
    for J in kop.Jlist:
        assert kop.off[J] == sum((2 * j + 1) ** 2 for j in kop.Jlist if j < J)


def test_slot_products_order():
    """Slots follow each tensor's Cartesian labels; a product is the field
    components named by the label."""
    kop, _ = large_top(2)
    F = [np.array([[2.0, 3.0, 5.0]]), np.array([[7.0, 11.0, 13.0]])]
    fp = kron.slot_products(kop, F)
    assert fp.shape == (1, sum(len(c) for c in kop.carts))
    vals = dict(zip([f"{li}:{c}" for li, cs in enumerate(kop.carts) for c in cs], fp[0].real))
    assert vals["0:z"] == 5.0 and vals["1:xy"] == 77.0 and vals["1:zz"] == 169.0


def test_from_cartens_equals_builder():
    """The factored form read from richmol-style CarTens blocks (a sum of a
    dipole and a full polarizability, each multiplied with its field) equals
    the builder's factored operator: same matvec on random rows (1e-13
    relative), same layout and permutation."""
    from richmol_amd.field import CarTens  # noqa: F401
    kop, bas = large_top(5)
    tens, scales = large_top_tensors()
    T = [rot.tensor(t, bas) * s for t, s in zip(tens, scales)]
    F = [(0.3e8, -0.8e8, 0.5e8), (1e8, 0.2e8, -0.4e8)]
    for t, f in zip(T, F):
        t.field(list(f))
    H = T[0] + T[1]
    kc, fprods = kron.KronOperator.from_cartens(H)
    assert kc.n == kop.n and np.array_equal(kc.perm, kop.perm)
    rng = np.random.default_rng(9)
    X = rng.normal(size=(2, kop.n)) + 1j * rng.normal(size=(2, kop.n))
    a = kop.matvec(X, kop.field_products(F))
    fp_c = [{c: fp.get(c, 0.0) for c in carts} for fp, carts in zip(fprods, kc.carts)]
    b = kc.matvec(X, fp_c)
    assert np.abs(a - b).max() <= 1e-13 * np.abs(a).max()
    assert np.allclose(kc.slot_row(fprods), kron.slot_products(kop, [np.array([f]) for f in F])[0])


def test_from_cartens_refuses_thresholds_and_partial_m():
    kop, bas = large_top(2)
    t = rot.tensor(np.array([0.0, 0.0, 1.0]), bas)
    t.field([0, 0, 1.0], thresh=1e-3)
    with pytest.raises(ValueError):
        kron.KronOperator.from_cartens(t)
    b0 = rot.asymtop_basis(4.73, 10.36, 9.02, 2, m_filter=lambda J, m: m == 0)
    t0 = rot.tensor(np.array([0.0, 0.0, 1.0]), b0)
    t0.field([0, 0, 1.0])
    with pytest.raises(ValueError):
        kron.KronOperator.from_cartens(t0)


def test_factors_only_to_rounding():
    """The primitive-basis factors are taken where they give K back to rounding
    and the coefficients are unitary to rounding, not a little beyond."""
    bas = rot.asymtop_basis(9.0, 6.0, 4.0, 6)

    def leaf():
        T = rot.tensor(np.array([0.2, 0.3, -0.1]), bas)
        T.field([1e8, 2e8, -3e8])
        return T

    assert kron.KronOperator.from_cartens(leaf())[0].factors is not None
    T = leaf()
    (sym, K), = [(s, d[1]) for s, d in T.kmat[(6, 5)].items() if 1 in d][:1]
    top = max(abs(d[1]).max() for d in T.kmat[(6, 5)].values() if 1 in d)
    K = K.toarray()
    K[0, -1] += 5e-14 * top
    T.kmat[(6, 5)][sym][1] = csr_matrix(K)
    assert kron.KronOperator.from_cartens(T)[0].factors is None
    T = leaf()
    T._kcoef[4] = T._kcoef[4] * (1 + 2e-13)
    assert kron.KronOperator.from_cartens(T)[0].factors is None

    assert kron.KronOperator(bas, [np.array([0.2, 0.3, -0.1])]).factors is not None
    for s, (kp, c) in bas.kfun[4].items():
        bas.kfun[4][s] = (kp, c * (1 + 2e-13))
    assert kron.KronOperator(bas, [np.array([0.2, 0.3, -0.1])]).factors is None
