"""Host paths of the library on the CPU, in a process whose HIP runtime is
hip_host_stub.cpp: memory is host memory, kernels do not run, launches are
recorded and allocations can be made to fail.  What a plan's launches read after
an allocation failed, and after its arrays were replaced; which operators count
as real and as symmetric; where rows with repeated columns run; a device with no
room for operators formed ahead; as many static jobs as the header allows;
the arrays a call is built from.
"""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
P = ctypes.c_void_p
LONG, SHORT, BAND = 2000, 300, 60   # rows of the two subspaces, half the band


def _matrix():
    """A real band matrix of a long subspace (first) and a short one, two slots."""
    rng = np.random.default_rng(0)
    rows, cols = [], []
    for lo, n in ((0, LONG), (LONG, SHORT)):
        for i in range(n):
            c = np.arange(max(0, i - BAND), min(n, i + BAND + 1))
            rows.append(np.full(c.size, lo + i))
            cols.append(lo + c)
    rows, cols = np.concatenate(rows), np.concatenate(cols)
    return rows, cols.astype(np.int32), rng.normal(size=(2, rows.size))


class Stub:
    def __init__(self, lib_path, stub_path):
        """The library and the stub; plan: a plan of _matrix()."""
        from richmol_amd import _lib
        self.lib, self.stub = ctypes.CDLL(lib_path), ctypes.CDLL(stub_path)
        for name, (res, args) in _lib.SIGNATURES.items():
            if hasattr(self.lib, name):
                getattr(self.lib, name).restype, getattr(self.lib, name).argtypes = res, args
        self.stub.stub_launch.restype = P
        self.batch = P()
        assert self.lib.rm_batch_create(ctypes.byref(self.batch)) == 0
        assert self.lib.rm_batch_set_block_rows(self.batch, 64) == 0
        self.n = n = LONG + SHORT
        self.table, self.flags = np.ones((3, 2), np.complex128), np.ones(3, np.int32)
        self.psi, self.work = np.zeros((1, n), np.complex128), np.zeros((1, n), np.complex128)
        self.rows, self.cols, self.vals = _matrix()
        self.plan = self.make_plan(self.vals)

    def make_plan(self, vals, rows=None, cols=None, n=None):
        """A plan of these values (2, entries) on _matrix()'s pattern or another."""
        from richmol_amd import _lib
        rows, cols, n = (self.rows, self.cols, self.n) if rows is None else (rows, cols, n)
        nnz = rows.size
        i64, i32 = np.int64, np.int32
        ptr = np.zeros(n + 1, i64)
        np.add.at(ptr, rows + 1, 1)
        ptr = np.cumsum(ptr).astype(i64)
        kval = np.ascontiguousarray(np.asarray(vals, dtype=np.complex128).T).view(np.float64)
        a = [ptr, cols, np.arange(nnz + 1, dtype=i64) * 2, np.tile(np.array([0, 1], i32), nnz), kval,
             np.array([0, 1, 2], i64), np.array([0, 1], i32), np.array([1.0, 0.0, 1.0, 0.0]), np.zeros(2, i32)]
        q = [x.ctypes.data_as(t) for x, t in zip(a, _lib.SIGNATURES["rm_plan_create"][1][2:7])]
        t = [x.ctypes.data_as(t) for x, t in zip(a[5:], _lib.SIGNATURES["rm_plan_create"][1][8:12])]
        plan = P()
        assert self.lib.rm_plan_create(n, nnz, *q, 2, *t, 2, 1, ctypes.byref(plan)) == 0
        return plan

    def job_record(self, lo, n):
        from richmol_amd import _lib
        return _lib.RmJob(plan=self.plan, psi=self.psi.ctypes.data, ld=self.n, col=0, lo=lo, len=n,
                          fprod_dev=self.table.ctypes.data, sflag_dev=self.flags.ctypes.data, nsteps=3, f_re=0.0,
                          f_im=-0.1, phase=None, kused=None, status=None)

    def job(self, lo, n):
        """A batch job on one domain; the library's status."""
        j = self.job_record(lo, n)
        self.stub.stub_clear()
        return self.lib.rm_batch_propagate(self.batch, ctypes.byref(j), 1, ctypes.sizeof(j), 6, 100, 1e-15, 0, None)

    def propagate(self):
        self.stub.stub_clear()
        return self.lib.rm_propagate(self.plan, self.psi.ctypes.data, self.work.ctypes.data, self.n, 1, 3,
                                     self.table.ctypes.data, None, 0.0, -0.1, None, 6, 100, 1e-15, None, None, None)

    def launches(self, kernel):
        """(first argument as 64-bit words, second, third) of the recorded launches of a kernel."""
        out = []
        for i in range(self.stub.stub_count()):
            at = self.stub.stub_launch(i)
            if kernel in ctypes.string_at(at).decode():
                w = np.frombuffer(ctypes.string_at(at + 96, 66 * 8), np.uint64)
                out.append(([int(x) for x in w[:64]], int(w[64]), int(w[65])))
        return out

    def check_operator(self, op, lo, n):
        """The sliced operator a launch reads (a SubOp's words: sslice 7, soff 8,
        srow 9, scol 10, sval 11, npairs 13) holds the domain's rows."""
        def arr(word, dtype, count, off=0):
            nb = np.dtype(dtype).itemsize
            return np.frombuffer(ctypes.string_at(op[word] + off * nb, count * nb), dtype)
        npairs = op[13]
        for r in range(lo, lo + n, 7):
            s = int(arr(9, np.int32, 1, r)[0])
            x, rows, z, w = (int(v) for v in arr(7, np.int32, 4, 4 * s))
            e0 = int(arr(8, np.int64, 1, s)[0]) + r - x
            assert 0 <= r - x < rows and 0 <= e0 and e0 + 64 * (z - 1) < npairs
            got = np.zeros((2, self.n))
            for p in range(z):
                c = int(arr(10, np.uint32, 1, e0 + 64 * p)[0])
                for q in range(2):
                    v = arr(11, np.float64, 2, 2 * (q * npairs + e0 + 64 * p))
                    got[q, w + ((c & 0xffff) >> 4)] += v[0]
                    got[q, w + (c >> 20)] += v[1]
            ref = np.zeros((2, self.n))
            sel = self.rows == r
            ref[:, self.cols[sel]] = self.vals[:, sel]
            assert np.array_equal(got, ref), r

    def check_job(self, lo, n):
        (words, _, _), = self.launches("k_blk")
        self.check_operator([int(x) for x in np.frombuffer(ctypes.string_at(words[0], 8 * 14), np.uint64)], lo, n)


def case_failed_allocation(s):
    """Every device allocation of a plan's first long domain fails in turn;
    short domains before, in between and after read their own entries."""
    assert s.job(LONG, SHORT) == 0
    s.check_job(LONG, SHORT)
    failed = 0
    for k in range(1, 20):
        s.stub.stub_fail_in(k)
        rc = s.job(0, LONG)
        s.stub.stub_fail_in(0)
        assert s.job(LONG, SHORT) == 0
        s.check_job(LONG, SHORT)
        if rc == 0:
            break
        failed += 1
    assert rc == 0 and failed >= 1


def case_kept_lists(s):
    """Launch lists kept for domain reuse, then a batch job that replaces the
    plan's slices: the next call's operators are those of its domain."""
    s.psi[0, LONG + 5] = 1.0
    assert s.lib.rm_plan_set_kernel(s.plan, 6) == 0
    assert s.lib.rm_plan_set_domain_reuse(s.plan, 1) == 0

    def check():
        assert s.propagate() == 0
        (op, q0, count), = s.launches("k_blk_operators")
        s0, s1 = (int(np.frombuffer(ctypes.string_at(op[9] + 4 * r, 4), np.int32)[0]) for r in (LONG, s.n - 1))
        off = np.frombuffer(ctypes.string_at(op[8] + 8 * s0, 8 * (s1 - s0 + 2)), np.int64)
        assert (q0, count) == (off[0], off[-1] - off[0])

    check()
    check()
    assert s.job(0, LONG) == 0
    check()
    check()


def case_real_operators(s):
    """An operator runs as a real one, and as a symmetric one, only where the
    rest is rounding: what the caller put there stays, a NaN too."""
    sym = np.empty_like(s.vals)
    for q in range(2):
        A = np.zeros((s.n, s.n))
        A[s.rows, s.cols] = s.vals[q]
        sym[q] = (A + A.T)[s.rows, s.cols]
    one = np.zeros(s.rows.size)
    one[np.flatnonzero((s.rows == LONG + 40) & (s.cols == LONG + 41))] = 1.0
    for vals, real, symmetric in ((sym, True, True), (s.vals, True, False), (sym * (1 + 2.0 ** -51 * 1j), True, True),
                                  (sym * (1 + 2.0 ** -49 * 1j * one), False, False),
                                  (sym + np.where(one > 0, complex(0, np.nan), 0), False, False),
                                  (np.where(one > 0, 1e-25 * (1 + 0.4j), sym), True, False),
                                  (np.where(one > 0, 1e-15 * (1 + 0.4j), sym), False, False),
                                  (sym * (1 + 2.0 ** -50 * one), True, True),
                                  (sym * (1 + 2.0 ** -47 * one), True, False)):
        s.plan = s.make_plan(vals)
        assert s.job(LONG, SHORT) == 0
        kernels = [n for n in (ctypes.string_at(s.stub.stub_launch(i)).decode() for i in range(s.stub.stub_count()))
                   if "k_blkILb" in n]   # k_blk<FIXED, F32, REAL, ...>
        (words, _, _), = s.launches("k_blk")
        flags = int(np.frombuffer(ctypes.string_at(words[0] + 8 * 14, 4), np.int32)[0])
        assert len(kernels) == 1 and ("k_blkILb1ELb0ELb%d" % real) in kernels[0]
        assert flags == (1 if real and symmetric else 0)


def case_repeated_columns(s):
    """20-row domains, in one of which every column of a row is named twice (40
    entries): that one runs on the kernel that reads any number of entries,
    its neighbour on the one that holds 32 per row."""
    r, c = (x.ravel() for x in np.meshgrid(np.arange(20), np.arange(20), indexing="ij"))
    rows, cols = np.concatenate([r, r, 20 + r]), np.concatenate([c, c, 20 + c]).astype(np.int32)
    order = np.lexsort((cols, rows))
    s.plan = s.make_plan(np.ones((2, rows.size)), rows[order], cols[order], 40)
    s.n, s.psi = 40, np.zeros((1, 40), np.complex128)
    for lo, kernel in ((0, "k_sub_prop"), (20, "k_wav")):
        assert s.job(lo, 20) == 0
        assert [k for k in ("k_sub_prop", "k_wav", "k_sub_pair") if s.launches(k)] == [kernel]


def case_no_room_for_operators(s):
    """A device with no room for the operators of all steps: the call runs
    with every workgroup forming its own, as it does when asked to."""
    s.psi[0, LONG + 5] = 1.0
    assert s.lib.rm_plan_set_kernel(s.plan, 6) == 0
    assert s.lib.rm_plan_set_domain_reuse(s.plan, 1) == 0
    # three steps' operators: 937 kB; one workgroup's region with its own: 341 kB
    for kib, limit, ahead in ((0, 0, 0), (1 << 18, 600000, 0), (1 << 18, 0, 1), (0, 0, 0)):
        assert s.lib.rm_plan_set_tuning(s.plan, 6, kib) == 0
        s.stub.stub_limit(ctypes.c_size_t(limit))
        assert s.propagate() == 0, s.lib.rm_last_error()
        assert len(s.launches("k_blk_operators")) == ahead and len(s.launches("k_blkILb")) == 1
    assert s.lib.rm_plan_set_tuning(s.plan, 6, 350) == 0   # one step a launch
    assert s.propagate() == 0
    assert len(s.launches("k_blk_operators")) == 3 and len(s.launches("k_blkILb")) == 3


def case_static_jobs(s):
    """RM_STATIC_MAX_JOBS jobs on short domains, under the adaptive rule and
    with a fixed dimension: every launch form takes them."""
    src = open(os.path.join(os.path.dirname(HERE), "include", "richmol_amd.h")).read()
    count = int(re.search(r"#define RM_STATIC_MAX_JOBS (\d+)", src).group(1))
    r, c = (x.ravel() for x in np.meshgrid(np.arange(20), np.arange(20), indexing="ij"))
    for width in (1, 19):   # banded and full rows
        on = np.abs(r - c) <= width
        s.plan = s.make_plan(np.ones((2, int(on.sum()))), r[on], c[on].astype(np.int32), 20)
        s.n, s.psi = 20, np.zeros((1, 20), np.complex128)
        assert s.lib.rm_plan_subspaces(s.plan, None, None) >= 0
        jobs = (type(s.job_record(0, 20)) * count)(*[s.job_record(0, 20)] * count)
        for fixed in (0, 9, 20):
            rc = s.lib.rm_batch_propagate_static(ctypes.byref(jobs), count, ctypes.sizeof(jobs[0]), fixed, 100, 1e-15,
                                                 0, None)
            assert rc == 0, s.lib.rm_last_error()


def case_arrays_of_a_call(s):
    """A mid-size domain's block launch is built without the CSR arrays that only
    the cooperative kernels read; the cooperative form on the same plan gets them."""
    on = s.rows >= LONG
    s.plan = s.make_plan(s.vals[:, on], s.rows[on] - LONG, s.cols[on] - LONG, SHORT)
    s.n, s.psi, s.work = SHORT, np.zeros((1, SHORT), np.complex128), np.zeros((1, SHORT), np.complex128)
    s.psi[0, 3] = 1.0
    for kernel, launch, csr in ((6, "k_blkILb", False), (5, "k_longILi", True)):
        assert s.lib.rm_plan_set_kernel(s.plan, kernel) == 0
        assert s.propagate() == 0 and len(s.launches(launch)) == 1
        assert s.job(0, SHORT) == 0
        (words, _, _), = s.launches("k_blkILb")
        rp = int(np.frombuffer(ctypes.string_at(words[0] + 8 * 2, 8), np.uint64)[0])
        assert (rp != 0) == csr


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_host_stub.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-I/opt/rocm/include", "-o", so,
                    os.path.join(HERE, "hip_host_stub.cpp")], check=True)
    return so


@pytest.mark.parametrize("case", ["failed_allocation", "kept_lists", "real_operators", "repeated_columns",
                                  "no_room_for_operators", "static_jobs", "arrays_of_a_call"])
def test_host_path(stub, case):
    from richmol_amd import _build
    if not os.path.exists(_build.LIB_PATH):
        _build.build()
    env = dict(os.environ, LD_PRELOAD=":".join(filter(None, [stub, os.environ.get("LD_PRELOAD")])))
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case, _build.LIB_PATH, stub], env=env,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]


if __name__ == "__main__":
    sys.path.insert(0, os.path.dirname(HERE))
    globals()["case_" + sys.argv[1]](Stub(sys.argv[2], sys.argv[3]))
