"""Every route of the invariant-subspace path against the full-vector kernel on
random operators (1e-11): subspaces of 1 to 4 200 rows side by side, narrow and
wide rows, rows that name a column twice, real, complex and non-symmetric
entries, one to four field slots, complex field products, steps without field,
wavepackets on one or on several subspaces, with and without phases and kept
domains, adaptive and fixed Krylov dimensions.
"""
import numpy as np
import pytest

from richmol_amd import plan as _plan

pytestmark = pytest.mark.gpu

SIZES = {"short": [1, 2, 3, 7, 20, 31, 32, 33, 50, 63, 64], "mid": [5, 65, 70, 130, 300, 640],
         "long": [40, 961, 1100, 2500], "longest": [700, 4096, 4200]}


def _operator(rng, sizes, width, nslot, kind, repeat):
    """(arrays of a plan, offsets of the subspaces): Hermitian (or, kind 'skew',
    real non-symmetric) entries of norm ~1 per slot."""
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = int(off[-1])
    label = rng.permutation(n)            # the subspaces interleaved
    rows, cols = [], []
    for lo, size in zip(off, sizes):
        i = np.arange(size)
        a = [i, i[:-1]]
        b = [i, i[1:]]
        for _ in range(width):
            a.append(rng.integers(0, size, size))
            b.append(rng.integers(0, size, size))
        a, b = np.concatenate(a), np.concatenate(b)
        rows += [lo + a, lo + b]
        cols += [lo + b, lo + a]
    key = np.unique(np.concatenate(rows) * n + np.concatenate(cols))
    r, c = key // n, key % n
    up = np.minimum(r, c) * n + np.maximum(r, c)
    _, pos = np.unique(up, return_inverse=True)
    w = 2.0 * width + 3.0
    vals = np.zeros((nslot, r.size), dtype=np.complex128)
    for s in range(nslot):
        x = rng.normal(size=pos.max() + 1)
        v = x[pos] + 0j
        if kind == "complex":
            y = rng.normal(size=pos.max() + 1)
            v = v + 1j * np.sign(c - r) * y[pos]
        if kind == "skew":
            v = v + 0.1 * rng.normal(size=r.size)
        vals[s] = v / w
    if repeat:                            # every entry again, half of it each
        r, c, vals = np.tile(r, 2), np.tile(c, 2), np.tile(0.5 * vals, 2)
    r, c = label[r], label[c]
    order = np.lexsort((c, r))
    r, c, vals = r[order], c[order], vals[:, order]
    nnz = r.size
    ptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int64)
    arr = dict(n=n, n2=n, nnz=nnz, row_ptr=ptr, col_idx=c.astype(np.int32),
               pair_ptr=np.arange(nnz + 1, dtype=np.int64) * nslot,
               pair_term=np.tile(np.arange(nslot, dtype=np.int32), nnz), pair_kval=np.ascontiguousarray(vals.T).ravel(),
               nterm=nslot, term_ptr=np.arange(nslot + 1, dtype=np.int64), term_field=np.arange(nslot, dtype=np.int32),
               term_mval=np.ones(nslot, np.complex128), term_leaf=np.zeros(nslot, np.int32), slots=[["x"] * nslot],
               nfield=nslot, nleaf=1)
    return arr, [label[lo:hi] for lo, hi in zip(off[:-1], off[1:])]


@pytest.mark.parametrize("seed", range(40))
def test_random_operator(device, seed):
    import torch
    rng = np.random.default_rng(1000 + seed)
    group = ["short", "short", "mid", "mid", "long", "longest"][seed % 6]
    sizes = [int(x) for x in rng.permutation(SIZES[group])]
    width, nslot = int(rng.choice([0, 1, 6, 20])), int(rng.choice([1, 1, 2, 4]))
    kind, repeat = str(rng.choice(["real", "real", "complex", "skew"])), rng.random() < 0.25
    arr, subs = _operator(rng, sizes, width, nslot, kind, repeat)
    n = arr["n"]
    ncols = int(rng.integers(2, 12))
    X = np.zeros((ncols, n), dtype=np.complex128)
    for b in range(ncols):
        for q in rng.choice(len(subs), size=1 if b % 3 else min(2, len(subs)), replace=False):
            X[b, rng.choice(subs[q], size=min(len(subs[q]), 1 + b % 4), replace=False)] = 1.0 + 0.3j * b
        X[b] /= np.linalg.norm(X[b])
    nsteps, fixed = 5, int(rng.choice([0, 0, 1, 7, 12, 20]))
    table = rng.normal(size=(nsteps, nslot)) + 0j
    if kind == "real" and rng.random() < 0.3:
        table = table * (1 + 0.05j)
    table[2] = 0.0
    table[4] = table[3]
    phase = np.exp(1j * rng.normal(size=n)) if rng.random() < 0.7 else None
    d = dict(sizes=sizes, width=width, nslot=nslot, kind=kind, repeat=repeat, ncols=ncols, fixed=fixed,
             phases=phase is not None)
    print(f"seed {seed}: {d}", flush=True)
    p = _plan.DevicePlan(None, active=arr["slots"], arrays=arr)
    tab = torch.from_numpy(table).to(device)
    ph = None if phase is None else torch.from_numpy(phase).to(device)

    def run(kernel, calls, **tuning):
        p.set_kernel(kernel)
        p.set_tuning(**tuning)
        psi = torch.from_numpy(X).to(device)
        work = torch.empty_like(psi)
        ku = torch.full((nsteps, ncols), -1, dtype=torch.int32, device=device)
        p.set_domain_reuse(calls > 1)
        for _ in range(calls):
            p.propagate(psi, work, tab, -0.4j, phase=ph, krylov_fixed=fixed, maxorder=60, kused=ku)
        return psi.cpu().numpy(), ku.cpu().numpy()

    for calls in (1, 2):
        ref, kr = run("global", calls)
        for kernel, tuning in (("subspace", {}), ("subspace", {"pair": 0, "fork": 0}), ("block", {}),
                               ("block", {"operator_kib": 0}), ("subspace", {"wave_max_rows": 1024}), ("coop", {})):
            print(f"  {kernel} {tuning} calls={calls}", flush=True)
            got, kg = run(kernel, calls, **tuning)
            assert np.abs(got - ref).max() <= 1e-11 * max(1.0, np.abs(ref).max()), (kernel, tuning)
            assert np.abs(kg - kr).max() <= (0 if fixed else 1), (kernel, tuning)
    p.close()
