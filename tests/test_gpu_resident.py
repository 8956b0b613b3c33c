"""GPU tests of the on-chip CG (csrc/cg_resident.hip).

A Jacobi (or unpreconditioned) CG whose system fits the registers and LDS of
the chip runs its iterations in one launch; TFLOWS_CG_RESIDENT=0 runs one
launch per kernel.  The two differ only in the order in which the dot
products are summed, so capped solves agree to rounding and converged ones
as the parity tests of the kernel-per-phase form do with the oracle.

Sizes sit at the edges of the form: one block and two, a last block of one
slice, rows of a thread (512 threads), one-step and two-step
synchronisation, offsets shorter and longer than a block, the locality order
(no shared offsets), and the largest system of each kind.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _residuals_agree(s, a, b):
    """r = b - A x up to the rounding of its recurrence in both forms, so
    r_a - r_b is -A (x_a - x_b) and that rounding: at most a few eps of
    |A| |x| per iteration, 100 eps over a dozen or two."""
    norm_a = abs(s.matrix.to_scipy()).sum(axis=1).max()
    bound = norm_a * (np.linalg.norm(a[1] - b[1]) + 100 * 2.2e-16 * np.linalg.norm(b[1]))
    return np.linalg.norm(a[2] - b[2]) <= bound


def _solve(pkg, cuda, s, prec, cap, tol, method="cg"):
    import torch
    ds = pkg.krylov.DeviceSystem(s.matrix)
    x = torch.zeros(s.matrix.n, dtype=torch.float64, device=cuda)
    r = torch.from_numpy(s.b.copy()).to(cuda)
    res = ds.solve(method, prec, x, r, cap, tol)
    torch.cuda.synchronize()
    ds.close()
    return res, x.cpu().numpy(), r.cpu().numpy()


SHAPES = {"one_slice": (4, 4, 4), "one_slice_short": (5, 3, 4), "rows_513": (3, 9, 19), "one_block_full": (16, 16, 16),
          "two_blocks": (17, 241, 1), "last_block_short": (19, 16, 17), "line": (9000, 1, 1),
          "blocks_64": (40, 40, 41), "blocks_64_full": (64, 64, 32), "two_step": (65, 64, 32),
          "two_step_ragged": (67, 53, 59)}


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("prec", [0, 1])
def test_capped_iterations_match(pkg, oracle, cuda, monkeypatch, shape, prec):
    """12 iterations: the rounding of 24 sums of n terms, summed in blocks in
    both forms (each good to about 1e-15), enters alfa and beta and grows by
    the 12 recurrences; 1e-12 leaves two orders."""
    s = pkg.meshgen.pressure_system(SHAPES[shape], seed=3)
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        out[mode] = _solve(pkg, cuda, s, prec, 12, 0.0)
    a, b = out["1"], out["0"]
    assert a[0][0] == b[0][0] == 13 and a[0][1] == b[0][1]
    assert _rel(a[1], b[1]) <= 1e-12 and _residuals_agree(s, a, b)
    assert a[0][2] == pytest.approx(np.linalg.norm(a[2]), rel=1e-12)
    if s.matrix.n < 20000:
        ref = oracle.run("cg", s.matrix, s.b, prec=prec, niter=12, tol=0.0)
        assert _rel(a[1], ref["x"]) <= 1e-11


@pytest.mark.parametrize("case", ["natural", "locality", "nonsymmetric", "rows_8_per_thread", "locality_largest",
                                  "beyond"])
def test_layouts_match(pkg, cuda, monkeypatch, case):
    """The matrix forms a block can hold (shared offsets with symmetric and
    with full values, columns per entry) at 20 iterations, and a system too
    large for the form, which must give the same bits either way."""
    mg = pkg.meshgen
    s = {"natural": lambda: mg.pressure_system(20, seed=5),
         "locality": lambda: mg.pressure_system((41, 37, 33), seed=6, perm_seed=2),
         "nonsymmetric": lambda: mg.momentum_system(14, seed=7),
         "rows_8_per_thread": lambda: mg.pressure_system((101, 99, 98), seed=8),
         "locality_largest": lambda: mg.pressure_system((81, 80, 78), seed=9, perm_seed=3),
         "beyond": lambda: mg.pressure_system((105, 103, 101), seed=10)}[case]()
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        out[mode] = _solve(pkg, cuda, s, 1, 20, 0.0)
    a, b = out["1"], out["0"]
    assert a[0][0] == b[0][0] == 21
    if case == "beyond":
        assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
    assert _rel(a[1], b[1]) <= 1e-11 and _residuals_agree(s, a, b)


def test_shared_offsets_beyond_the_window(pkg, oracle, cuda, monkeypatch):
    """Two boxes of different lines in one system: each slice's offsets are
    shared, but the system has more of them than a block's halo allows, so
    the rows are read from the CSR arrays every iteration."""
    import scipy.sparse as sp
    mg = pkg.meshgen
    parts = [mg.pressure_system((16, 4, 8), seed=15), mg.pressure_system((13, 7, 9), seed=16),
             mg.pressure_system((40, 40, 41), seed=17)]
    for some in (parts[:2], [parts[0], parts[2]]):
        A = sp.block_diag([q.matrix.to_scipy() for q in some], format="csr")
        s = mg.LinearSystem(mg.from_scipy(A), np.concatenate([q.b for q in some]), np.zeros(A.shape[0]), 1e-8, 1, 100, {})
        out = {}
        for mode in ("1", "0"):
            monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
            ds = pkg.krylov.DeviceSystem(s.matrix)
            assert ds.fp64_layout()["shared"]
            ds.close()
            out[mode] = _solve(pkg, cuda, s, 1, 12, 0.0)
        assert out["1"][0][0] == out["0"][0][0] == 13
        assert _rel(out["1"][1], out["0"][1]) <= 1e-12 and _residuals_agree(s, out["1"], out["0"])


@pytest.mark.parametrize("n", [2, 514, 9000])
@pytest.mark.parametrize("op", ["sliced", "csr"])
def test_breakdown_reports_what_the_kernels_do(pkg, cuda, monkeypatch, n, op):
    """(p, A p) = 0 exactly: alfa, x and FinRes become infinite; the threads
    past the last row must not turn the norm into NaN."""
    import scipy.sparse as sp
    A = sp.csr_matrix((np.ones(2 * n), (np.repeat(np.arange(n), 2), (np.arange(n)[:, None] // 2 * 2 + [0, 1]).ravel())),
                      shape=(n, n))
    A.data[:] = np.tile([0.0, 1.0, -1.0, 0.0], n // 2)
    s = pkg.meshgen.LinearSystem(pkg.meshgen.from_scipy(A), np.ones(n), np.zeros(n), 0.0, 0, 1, {})
    if op == "csr":
        monkeypatch.setenv("TFLOWS_FP64_OP", "csr")
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        out[mode] = _solve(pkg, cuda, s, 0, 1, 0.0)
    a, b = out["1"], out["0"]
    assert a[0] == b[0] and a[0][2] == np.inf
    assert np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2]) and np.isinf(a[1]).all()


@pytest.mark.parametrize("method", ["cg", "cgs"])
@pytest.mark.parametrize("renumber", [False, True])
def test_new_values_after_a_solve_that_ends_at_once(pkg, cuda, method, renumber):
    """A solve that is over before its first iteration (b = 0) does not fill
    new values into the operator; the next one does."""
    import torch
    s = pkg.meshgen.momentum_system((25, 24, 23), seed=9, renumber=renumber)
    n, b = s.matrix.n, torch.from_numpy(s.b.copy()).to(cuda)
    values = torch.from_numpy(s.matrix.aval.copy()).to(cuda)

    def run(ds, rhs, cap=8):
        x, r = torch.zeros(n, dtype=torch.float64, device=cuda), rhs.clone()
        res = ds.solve(method, 1, x, r, cap, 0.0 if cap else 1e-9)
        return res, x.cpu().numpy(), r.cpu().numpy()

    ds = pkg.krylov.DeviceSystem(s.matrix)
    run(ds, b)
    want = {}
    for scale in (3.0, 0.25):
        ds.set_values(values * scale)
        want[scale] = run(ds, b)
    for scale in (3.0, 0.25):
        ds.set_values(values * scale)
        x, r = torch.zeros(n, dtype=torch.float64, device=cuda), torch.zeros(n, dtype=torch.float64, device=cuda)
        assert ds.solve(method, 1, x, r, 8, 1e-9)[0] == 0 and not x.any()
        assert run(ds, b, 0)[0][0] == 1             # a cap of 0 ends before the first iteration, too
        got = run(ds, b)
        assert got[0] == want[scale][0] and np.array_equal(got[1], want[scale][1])
        assert np.array_equal(got[2], want[scale][2])
    ds.close()


def _graph(pkg, n, offsets, rows=None, seed=3):
    """Symmetric diagonally dominant matrix: entries i, i + d for the offsets,
    and for a few rows i, i + 2, i + 5, ... (`rows`: how many more)."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    A = sp.diags([rng.uniform(0.5, 1.0, n - d) for d in offsets], offsets, shape=(n, n), format="csr")
    if rows:
        r = np.repeat(rng.choice(n - 100, n // 20, replace=False), rows)
        A = A + sp.csr_matrix((np.full(len(r), 0.01), (r, r + np.tile(2 + 3 * np.arange(rows), n // 20))), shape=(n, n))
    A = A + A.T
    A = (sp.diags(np.asarray(A.sum(axis=1)).ravel() * 1.01) - A).tocsr()
    A.sort_indices()
    m = pkg.meshgen.from_scipy(A)
    return pkg.meshgen.LinearSystem(m, rng.standard_normal(n), np.zeros(n), 1e-8, 1, 100, {})


@pytest.mark.parametrize("case", ["rows_9", "rows_27", "rows_199_one_block", "dense_row"])
def test_long_rows_keep_the_kernels(pkg, cuda, monkeypatch, case):
    """Rows longer than a mesh's run one launch per kernel either way: the
    same bits (a thread of the on-chip form reads its row entry by entry,
    which takes up to 25 times as long as the kernels on such rows)."""
    import scipy.sparse as sp
    if case == "dense_row":
        A = _graph(pkg, 20000, [1, 50, 2500]).matrix.to_scipy().tolil()
        A[10000, :4000] = -1e-3
        A[:4000, 10000] = -1e-3
        m = pkg.meshgen.from_scipy(sp.csr_matrix(A))
        s = pkg.meshgen.LinearSystem(m, np.ones(m.n), np.zeros(m.n), 1e-8, 1, 100, {})
    else:
        s = {"rows_9": lambda: _graph(pkg, 20000, [1, 50, 2500, 2501]),
             "rows_27": lambda: _graph(pkg, 20000, [1, 29, 30, 31, 869, 870, 871, 899, 900, 901, 929, 930, 931]),
             "rows_199_one_block": lambda: _graph(pkg, 4000, list(range(1, 100)))}[case]()
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        out[mode] = _solve(pkg, cuda, s, 1, 12, 0.0)
    a, b = out["1"], out["0"]
    assert a[0] == b[0] and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])


@pytest.mark.parametrize("n", [3000, 20000, 90000])
def test_rows_of_a_refined_mesh(pkg, cuda, monkeypatch, n):
    """Rows of 7 with some of up to 12 entries: on the chip, their rows read
    every iteration."""
    s = _graph(pkg, n, [1, 40, 1600], rows=2)
    assert 8 <= np.diff(s.matrix.to_scipy().indptr).max() <= 12
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        out[mode] = _solve(pkg, cuda, s, 1, 12, 0.0)
    a, b = out["1"], out["0"]
    assert a[0][0] == b[0][0] == 13 and _rel(a[1], b[1]) <= 1e-12 and _residuals_agree(s, a, b)
    assert not np.array_equal(a[2], b[2])      # the on-chip form's own sums


@pytest.mark.parametrize("shape", [(2500, 1, 1), (9000, 1, 1)])
def test_iterations_past_one_launch(pkg, cuda, monkeypatch, shape):
    """A launch runs at most 1024 iterations; the next one goes on from its
    x, r and p (one block, and several that read each other's p).  CG needs
    about as many iterations as a line has cells, so both forms run past a
    launch; each must reach the tolerance with its true residual, which the
    recurrence's follows to the rounding of that many updates of x."""
    s = pkg.meshgen.pressure_system(shape, seed=4)
    A = s.matrix.to_scipy()
    norm_a = abs(A).sum(axis=1).max()
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        (it, ini, fin), x, r = _solve(pkg, cuda, s, 1, 60000, s.tol)
        assert 1100 < it < 60000 and fin < s.tol
        assert np.linalg.norm(s.b - A @ x) <= s.tol + it * 2.2e-16 * norm_a * np.linalg.norm(x)


@pytest.mark.parametrize("case", ["one_block", "last_block_short", "locality", "two_step", "locality_largest"])
@pytest.mark.parametrize("prec", [0, 1])
def test_cgs_matches(pkg, oracle, cuda, monkeypatch, case, prec):
    """CGS on the chip: 6 iterations against one launch per kernel (its
    squared polynomial amplifies the rounding of the dot products; the
    parity bar of a capped CGS is 1e-9), and the converged solve's true
    residual."""
    mg = pkg.meshgen
    s = {"one_block": lambda: mg.momentum_system((15, 13, 11), seed=61, renumber=False),
         "last_block_short": lambda: mg.momentum_system((19, 16, 17), seed=62),
         "locality": lambda: mg.momentum_system((41, 37, 33), seed=63),
         "two_step": lambda: mg.momentum_system((67, 53, 59), seed=64, renumber=False),
         "locality_largest": lambda: mg.momentum_system((80, 80, 78), seed=65)}[case]()
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        out[mode] = (_solve(pkg, cuda, s, prec, 6, 0.0, "cgs"), _solve(pkg, cuda, s, prec, 600, s.tol, "cgs"))
    (a, ac), (b, bc) = out["1"], out["0"]
    assert a[0][0] == b[0][0] == 7 and a[0][1] == b[0][1]
    assert _rel(a[1], b[1]) <= 1e-9
    if case == "one_block":            # keeps one launch per kernel
        assert ac[0] == bc[0] and np.array_equal(ac[1], bc[1]) and np.array_equal(ac[2], bc[2])
    if s.matrix.n < 10000:
        assert _rel(a[1], oracle.run("cgs", s.matrix, s.b, prec=prec, niter=6, tol=0.0)["x"]) <= 1e-9
    if bc[0][0] <= 600:                # it converges without the on-chip form, too
        # (the count is not compared: a CGS residual rises and falls by orders
        # from one iteration to the next, so rounding decides which one first
        # falls below tol; what its peaks lose, both forms lose alike)
        A = s.matrix.to_scipy()
        true = [np.linalg.norm(s.b - A @ v) for v in (ac[1], bc[1])]
        assert ac[0][0] <= 600 and ac[0][2] < s.tol and true[0] < 10 * max(s.tol, true[1])


@pytest.mark.parametrize("shape", [(17, 17, 17), (25, 24, 23), (31, 30, 29)])
@pytest.mark.parametrize("renumber", [False, True])
def test_cgs_count_of_momentum_matrices(pkg, oracle, cuda, shape, renumber):
    """The velocity matrices CGS is run on converge in a few dozen iterations,
    in which rounding shifts the last one by one at most: the on-chip count is
    the reference loop's.  (On pressure matrices of these sizes, hundreds of
    iterations, either form's count is up to 6 % from it, by rounding.)"""
    for seed in (1, 2, 3):
        s = pkg.meshgen.momentum_system(shape, seed=seed, renumber=renumber)
        res = _solve(pkg, cuda, s, 1, 2000, s.tol, "cgs")[0]
        ref = oracle.run("cgs", s.matrix, s.b, prec=1, niter=2000, tol=s.tol)
        assert abs(res[0] - ref["niter"]) <= 1 and res[2] < s.tol


@pytest.mark.parametrize("boxes", [[(16, 16, 16)] * 8, [(40, 40, 41)] * 2, [(70, 60, 25)] * 3, [(40, 40, 41)]])
def test_cgs_of_boxes_numbered_one_after_another(pkg, cuda, monkeypatch, boxes):
    """A block's halo is loaded whole: rows of a zone's last plane lack the
    entry whose rows are loaded, and so do the empty blocks at the end, so it
    goes beyond the blocks that the columns reach and has to wait for those,
    too (tests/resident_window_check.cpp shows which).  What a solve that
    ended in NaN has left in the workspace must not enter the next one."""
    import scipy.sparse as sp
    import torch
    mg = pkg.meshgen
    parts = [mg.momentum_system(b, seed=70 + q, renumber=False) for q, b in enumerate(boxes)]
    A = mg.from_scipy(sp.block_diag([q.matrix.to_scipy() for q in parts], format="csr"))
    b = np.concatenate([q.b for q in parts])
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        ds = pkg.krylov.DeviceSystem(A)
        assert ds.fp64_layout()["shared"]
        got = []
        for _ in range(3):
            x = torch.zeros(A.n, dtype=torch.float64, device=cuda)
            r = torch.full((A.n,), float("nan"), dtype=torch.float64, device=cuda)
            ds.solve("cgs", 1, x, r, 2, 0.0)
            assert torch.isnan(x).all()
            x.zero_()
            r.copy_(torch.from_numpy(b))
            res = ds.solve("cgs", 1, x, r, 6, 0.0)
            got.append((res, x.cpu().numpy(), r.cpu().numpy()))
        ds.close()
        for g in got[1:]:
            assert g[0] == got[0][0] and np.array_equal(g[1], got[0][1]) and np.array_equal(g[2], got[0][2])
        out[mode] = got[0]
    a, k = out["1"], out["0"]
    assert a[0][0] == k[0][0] == 7 and np.isfinite(a[1]).all()
    assert _rel(a[1], k[1]) <= 1e-9


@pytest.mark.parametrize("method", ["cg", "cgs"])
def test_wait_bound_falls_back(pkg, cuda, monkeypatch, capfd, method):
    """A synchronisation that waits beyond TFLOWS_BARRIER_WAIT_MS is given up
    by every block, and the solve runs one launch per kernel from its inputs,
    to that form's bits.  With 0 the first poll that finds a post missing
    gives up: some block's does, as not all of several blocks post before any
    of them polls."""
    mg = pkg.meshgen
    s = (mg.pressure_system((40, 40, 41), seed=11) if method == "cg"
         else mg.momentum_system((40, 40, 41), seed=66, renumber=False))
    monkeypatch.setenv("TFLOWS_CG_RESIDENT", "0")
    want = _solve(pkg, cuda, s, 1, 40, 0.0, method)
    monkeypatch.setenv("TFLOWS_CG_RESIDENT", "1")
    monkeypatch.setenv("TFLOWS_BARRIER_WAIT_MS", "0")
    got = _solve(pkg, cuda, s, 1, 40, 0.0, method)
    assert capfd.readouterr().err.count("gave up waiting") == 1
    assert got[0] == want[0] and np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2])


def test_mixed_wait_bound_falls_back(pkg, cuda, monkeypatch, capfd):
    import torch
    s = pkg.meshgen.pressure_system((40, 40, 41), seed=14)
    b = torch.from_numpy(s.b.copy()).to(cuda)
    out = {}
    for mode, wait in (("0", "2000"), ("1", "0"), ("1", "2000")):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        monkeypatch.setenv("TFLOWS_BARRIER_WAIT_MS", wait)
        ds = pkg.krylov.DeviceSystem(s.matrix)
        for _ in range(2):             # the second call keeps the form
            x = torch.from_numpy(np.random.default_rng(9).standard_normal(s.matrix.n)).to(cuda)
            r = torch.zeros_like(x)
            res = ds.solve_mixed_reliable(1, x, b, 120, 0.0, interval=40, r_out=r)
            torch.cuda.synchronize()
            out.setdefault((mode, wait), []).append((res, x.cpu().numpy(), r.cpu().numpy()))
        ds.close()
        assert capfd.readouterr().err.count("gave up waiting") == (wait == "0")
    for g in out["1", "0"] + out["0", "2000"]:
        w = out["0", "2000"][0]
        assert g[0] == w[0] and np.array_equal(g[1], w[1]) and np.array_equal(g[2], w[2])
    assert not np.array_equal(out["1", "2000"][0][1], out["0", "2000"][0][1])   # the on-chip form's own bits


@pytest.mark.parametrize("case", ["natural", "one_block", "locality", "csr_rows", "cgs", "cgs_locality"])
def test_fallback_restores_every_row(pkg, cuda, monkeypatch, capfd, case):
    """Blocks that start after another has given up (a bound below 0 raises
    the fault word before the launch) still save their x and r, so that the
    fallback starts from the inputs and not from an earlier solve's."""
    import torch
    mg = pkg.meshgen
    method = "cgs" if case.startswith("cgs") else "cg"
    s = {"natural": lambda: mg.pressure_system((40, 40, 41), seed=11),
         "one_block": lambda: mg.pressure_system((16, 16, 16), seed=11),
         "locality": lambda: mg.pressure_system((41, 37, 33), seed=6, perm_seed=2),
         "csr_rows": lambda: mg.pressure_system((40, 40, 41), seed=11),
         "cgs": lambda: mg.momentum_system((40, 40, 41), seed=66, renumber=False),
         "cgs_locality": lambda: mg.momentum_system((41, 37, 33), seed=63)}[case]()
    if case == "csr_rows":
        monkeypatch.setenv("TFLOWS_FP64_OP", "csr")
    rng = np.random.default_rng(5)
    starts = [rng.standard_normal(s.matrix.n) for _ in range(2)]
    rhs = [s.b, s.b + rng.standard_normal(s.matrix.n) * np.abs(s.b).max()]
    out = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        monkeypatch.delenv("TFLOWS_BARRIER_WAIT_MS", raising=False)
        ds = pkg.krylov.DeviceSystem(s.matrix)
        for q in range(2):
            x, r = torch.from_numpy(starts[q]).to(cuda), torch.from_numpy(rhs[q]).to(cuda)
            res = ds.solve(method, 1, x, r, 6, 0.0)
            torch.cuda.synchronize()
            monkeypatch.setenv("TFLOWS_BARRIER_WAIT_MS", "-1")
        ds.close()
        out[mode] = (res, x.cpu().numpy(), r.cpu().numpy())
        assert ("gave up waiting" in capfd.readouterr().err) == (mode == "1")
    a, k = out["1"], out["0"]
    assert a[0] == k[0] and np.array_equal(a[1], k[1]) and np.array_equal(a[2], k[2])


def test_two_threads(pkg, cuda):
    """Solves from two host threads on their own streams, each a launch that
    needs many CUs at once, give what they give alone."""
    import torch
    mg = pkg.meshgen
    systems = [mg.pressure_system((67, 53, 59), seed=12), mg.pressure_system((64, 64, 32), seed=13)]
    alone = [_solve(pkg, cuda, s, 1, 60, 0.0) for s in systems]
    got = [[], []]

    def work(q):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(5):
                got[q].append(_solve(pkg, cuda, systems[q], 1, 60, 0.0))

    ts = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for q in range(2):
        assert len(got[q]) == 5
        for g in got[q]:
            assert g[0] == alone[q][0] and np.array_equal(g[1], alone[q][1]) and np.array_equal(g[2], alone[q][2])


def test_batch_beside_small_systems(pkg, cuda, capfd):
    """An on-chip batch whose launch has about as many blocks as the chip, no
    multiple of the XCDs', beside solves of five blocks from another thread:
    neither waits for CUs that the other holds, and both give what they give
    alone."""
    import torch
    mg = pkg.meshgen
    shapes = [(61, 60, 59), (61, 59, 47), (53, 51, 49)] + [(17, 241, 1)] * 9
    systems = [mg.pressure_system(s, seed=110 + q) for q, s in enumerate(shapes)]
    k = len(systems)
    B = pkg.krylov.DeviceBatch([s.matrix for s in systems])
    b = torch.from_numpy(np.concatenate([s.b for s in systems])).to(cuda)
    small = mg.pressure_system((17, 17, 17), seed=96)
    want = _solve(pkg, cuda, small, 1, 40, 0.0)
    runs = {"batch": [], "small": []}

    def batch():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(8):
                x, r = torch.zeros_like(b), b.clone()
                torch.cuda.current_stream().synchronize()
                B.solve("cg", 1, x, r, np.full(k, 60, np.int32), np.zeros(k))
                runs["batch"].append(x.cpu().numpy())

    def singles():
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                runs["small"].append(_solve(pkg, cuda, small, 1, 40, 0.0))

    batch()
    assert B.config("cg", 1)["form"] == 3
    ts = [threading.Thread(target=f) for f in (batch, singles)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    B.close()
    assert "gave up" not in capfd.readouterr().err
    assert len(runs["batch"]) == 16 and len(runs["small"]) == 30
    assert all(np.array_equal(x, runs["batch"][0]) for x in runs["batch"])
    assert all(g[0] == want[0] and np.array_equal(g[1], want[1]) for g in runs["small"])


def test_kernel_form_batch_leaves_the_chip_to_others(pkg, cuda):
    """A batch whose kernels do not wait for each other (form 1) does not hold
    the CUs: an on-chip solve of another thread ends while the batch, 100 times
    as long, still runs, and both give what they give alone."""
    import time
    import torch
    mg = pkg.meshgen
    systems = [mg.pressure_system((40, 40, 41), seed=90 + q) for q in range(4)]
    caps, tols = np.full(4, 6000, np.int32), np.zeros(4)
    single = mg.pressure_system((32, 32, 32), seed=95)
    want = _solve(pkg, cuda, single, 1, 60, 0.0)
    B = pkg.krylov.DeviceBatch([s.matrix for s in systems])
    B.set_form(1)
    x = torch.zeros(B.rows, dtype=torch.float64, device=cuda)
    b = torch.from_numpy(np.concatenate([s.b for s in systems])).to(cuda)
    ends, xs = {}, []

    def batch():
        with torch.cuda.stream(torch.cuda.Stream()):
            xx, rr = x.clone(), b.clone()
            torch.cuda.current_stream().synchronize()
            B.solve("cg", 1, xx, rr, caps, tols)
            ends["batch"] = time.perf_counter()
            xs.append(xx.cpu().numpy())

    batch()                            # tuned, and the graph captured
    t = threading.Thread(target=batch)
    t.start()
    time.sleep(0.01)
    with torch.cuda.stream(torch.cuda.Stream()):
        got = _solve(pkg, cuda, single, 1, 60, 0.0)
    ends["single"] = time.perf_counter()
    t.join()
    assert ends["single"] < ends["batch"]
    assert got[0] == want[0] and np.array_equal(got[1], want[1])
    assert np.array_equal(xs[0], xs[1], equal_nan=True)
    B.close()


@pytest.mark.parametrize("shape", ["one_slice_short", "last_block_short", "blocks_64", "two_step_ragged", "rows_16"])
def test_mixed_matches(pkg, cuda, monkeypatch, shape):
    """The FP32 iterations of the reliable-update solve: both forms reach the
    FP64 tolerance in about the same count, and their x agree as two solutions
    with residuals below tol do (bounded here by their difference's residual)."""
    import torch
    mg = pkg.meshgen
    s = mg.pressure_system((129, 127, 115) if shape == "rows_16" else SHAPES[shape], seed=14)
    A = s.matrix.to_scipy()
    cap = 150 if shape == "rows_16" else 3000
    out = {}
    for mode in ("1", "0"):
        monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
        ds = pkg.krylov.DeviceSystem(s.matrix)
        x = torch.zeros(s.matrix.n, dtype=torch.float64, device=cuda)
        b = torch.from_numpy(s.b.copy()).to(cuda)
        res = ds.solve_mixed_reliable(1, x, b, cap, s.tol, interval=40)
        torch.cuda.synchronize()
        out[mode] = (res, x.cpu().numpy())
        ds.close()
    a, b = out["1"], out["0"]
    assert a[0][1] == pytest.approx(b[0][1], rel=1e-12)
    if shape == "rows_16":             # capped: FP32 rounding over 150 iterations
        assert a[0][0] == b[0][0] == cap + 1 and _rel(a[1], b[1]) <= 1e-4
        return
    assert a[0][2] < s.tol and b[0][2] < s.tol
    assert abs(a[0][0] - b[0][0]) <= 0.05 * b[0][0] + 3
    assert np.linalg.norm(A @ (a[1] - b[1])) <= 2 * s.tol


def test_mixed_error_against_64_bits(pkg, cuda, monkeypatch):
    """Capped mixed solves against FP64 CG of the same cap.  Both forms round
    the same FP32 vectors and the on-chip one adds its blocks' sums in FP64, so
    its mean error is no larger; single solves scatter (a factor of 1.8 either way, so
    the mean of 16 by about 15 %, and 1.25 is the ratio's bar)."""
    import torch
    mg = pkg.meshgen
    mean = {"1": 0.0, "0": 0.0}
    for q, shape in enumerate([(64, 64, 64), (83, 61, 47), (70, 72, 51), (96, 64, 32)] * 4):
        s = mg.pressure_system(shape, seed=80 + q)
        ds = pkg.krylov.DeviceSystem(s.matrix)
        b = torch.from_numpy(s.b.copy()).to(cuda)
        want, r = torch.zeros_like(b), b.clone()
        ds.solve("cg", 1, want, r, 220, 0.0)
        for mode in mean:
            monkeypatch.setenv("TFLOWS_CG_RESIDENT", mode)
            x = torch.zeros_like(b)
            ds.solve_mixed_reliable(1, x, b, 220, 0.0, interval=50)
            mean[mode] += float((x - want).norm() / want.norm()) / 16
        monkeypatch.delenv("TFLOWS_CG_RESIDENT")
        ds.close()
    print(f"mean error on the chip {mean['1']:.2e}, one launch per kernel {mean['0']:.2e}", flush=True)
    assert mean["1"] <= 1.25 * mean["0"]


def _batch(pkg, cuda, systems, form, caps, tols, prec=1, b=None):
    import torch
    B = pkg.krylov.DeviceBatch([s.matrix for s in systems])
    B.set_form(form)
    x = torch.zeros(B.rows, dtype=torch.float64, device=cuda)
    r = torch.from_numpy(np.concatenate([s.b for s in systems] if b is None else b)).to(cuda)
    out = []
    for _ in range(2):                 # twice: the posts and the state carry over
        xx, rr = x.clone(), r.clone()
        res = B.solve("cg", prec, xx, rr, caps, tols, fin_in=np.full(len(systems), 0.5))
        torch.cuda.synchronize()
        out.append((res, [v.cpu().numpy() for v in B.split(xx)], [v.cpu().numpy() for v in B.split(rr)]))
    out.append(B.config("cg", prec))
    B.configure(*(out[-1][k] for k in ("grid", "lanes", "chunk")))    # what it reports may be set again
    assert B.config("cg", prec) == out[-1]
    B.close()
    return out


@pytest.mark.parametrize("prec", [0, 1])
def test_batch_matches_kernel_form(pkg, cuda, prec):
    """Systems of one row to several blocks, in one launch: converged, capped
    and early-exit ones, against one launch per kernel (form 1)."""
    import scipy.sparse as sp
    mg = pkg.meshgen
    one = mg.LinearSystem(mg.from_scipy(sp.csr_matrix(np.array([[4.0]]))), np.array([2.0]), np.zeros(1), 1e-8, 1, 100, {})
    shapes = [(7, 5, 3), (16, 16, 16), (17, 241, 1), (40, 40, 41), (13, 11, 17), (9000, 1, 1), (64, 64, 32)]
    systems = [mg.pressure_system(sh, seed=20 + q) for q, sh in enumerate(shapes)] + [one]
    caps = np.array([3000, 12, 12, 3000, 3000, 15, 3000, 10], np.int32)
    tols = np.array([s.tol for s in systems])
    b = [s.b.copy() for s in systems]
    b[4][:] = 0.0                      # ||b|| < tol: the early exit
    got = _batch(pkg, cuda, systems, 0, caps, tols, prec, b)
    ref = _batch(pkg, cuda, systems, 1, caps, tols, prec, b)
    assert got.pop() == dict(grid=0, lanes=0, chunk=0, rebalances=0, form=3, groups=1)
    assert ref.pop()["form"] == 1
    ref = ref[0]
    for a in got:
        assert np.array_equal(a[0]["niter"], got[0][0]["niter"])
        for q, s in enumerate(systems):
            assert np.array_equal(a[1][q], got[0][1][q]) and np.array_equal(a[2][q], got[0][2][q])
            assert abs(int(a[0]["niter"][q]) - int(ref[0]["niter"][q])) <= 1, q
            if a[0]["niter"][q] <= caps[q] and q != 4:
                assert a[0]["fin_res"][q] < tols[q]
                assert np.linalg.norm(s.b - s.matrix.to_scipy() @ a[1][q]) < 10 * tols[q]
            elif q != 4:               # capped after a dozen iterations
                assert _rel(a[1][q], ref[1][q]) <= 1e-12
        assert a[0]["niter"][4] == 0 and a[0]["fin_res"][4] == 0.5 and not np.any(a[1][4])


def test_batch_of_several_launches(pkg, cuda):
    """More rows than the chip holds: the systems are dealt out to several
    launches."""
    mg = pkg.meshgen
    systems = [mg.pressure_system((61, 60, 59), seed=30 + q) for q in range(6)] + [mg.pressure_system(9, seed=40)]
    caps, tols = np.full(7, 12, np.int32), np.zeros(7)
    a, ref = _batch(pkg, cuda, systems, 0, caps, tols)[0], _batch(pkg, cuda, systems, 1, caps, tols)[0]
    for q in range(7):
        assert a[0]["niter"][q] == ref[0]["niter"][q] == 13
        assert _rel(a[1][q], ref[1][q]) <= 1e-12


@pytest.mark.parametrize("larger", [0, 1])
def test_batch_of_more_small_systems_than_blocks(pkg, cuda, larger):
    """More one-block systems than the chip holds blocks, of two rows to the
    most of a block: one launch, each stopping by itself; systems of several
    blocks beside them have launches of their own."""
    mg = pkg.meshgen
    rng = np.random.default_rng(8)
    shapes = [tuple(int(v) for v in rng.integers(2, 9, 3)) for _ in range(297)] + [(16, 16, 16), (2, 1, 1), (64, 8, 1)]
    shapes += [(40, 40, 41), (19, 16, 17)] * larger
    systems = [mg.pressure_system(sh, seed=100 + q) for q, sh in enumerate(shapes)]
    caps = np.full(len(shapes), 500, np.int32)
    caps[::7] = 3
    caps[300:] = 12
    tols = np.array([s.tol for s in systems])
    got = _batch(pkg, cuda, systems, 0, caps, tols)
    ref = _batch(pkg, cuda, systems, 1, caps, tols)[0]
    cfg = got.pop()
    assert cfg["form"] == 3 and cfg["groups"] == 1 + larger      # launches
    for a in got:
        assert np.array_equal(a[0]["niter"], got[0][0]["niter"])
        for q, s in enumerate(systems):
            assert np.array_equal(a[1][q], got[0][1][q]) and np.array_equal(a[2][q], got[0][2][q])
            assert abs(int(a[0]["niter"][q]) - int(ref[0]["niter"][q])) <= 1, q
            if a[0]["niter"][q] <= caps[q]:
                assert np.linalg.norm(s.b - s.matrix.to_scipy() @ a[1][q]) < 10 * tols[q]
            else:                      # capped after three or twelve iterations
                assert _rel(a[1][q], ref[1][q]) <= 1e-12


def test_batch_of_small_systems_keeps_its_memory(pkg, cuda):
    """Systems of one block post nothing: the first solve of 2,000 of them
    takes their tables (250 bytes a system), not posts (278 KB each)."""
    import torch
    s = pkg.meshgen.pressure_system((5, 4, 3), seed=60)
    B = pkg.krylov.DeviceBatch([s.matrix] * 2000)
    x = torch.zeros(B.rows, dtype=torch.float64, device=cuda)
    r = torch.from_numpy(np.tile(s.b, 2000)).to(cuda)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    res = B.solve("cg", 1, x, r, np.full(2000, 8, np.int32), np.zeros(2000))
    assert free - torch.cuda.mem_get_info()[0] < 64 << 20
    assert np.all(res["niter"] == 9)
    B.close()


def test_batch_wait_bound_falls_back(pkg, cuda, monkeypatch, capfd):
    mg = pkg.meshgen
    systems = [mg.pressure_system((40, 40, 41), seed=50), mg.pressure_system((41, 39, 38), seed=51)]
    caps, tols = np.full(2, 30, np.int32), np.zeros(2)
    whole = _batch(pkg, cuda, systems, 0, caps, tols)[0]
    monkeypatch.setenv("TFLOWS_BARRIER_WAIT_MS", "0")
    got, _, cfg = _batch(pkg, cuda, systems, 0, caps, tols)
    assert capfd.readouterr().err.count("gave up waiting") == 1 and cfg["form"] in (1, 2)
    for q in range(2):
        assert got[0]["niter"][q] == 31 and _rel(got[1][q], whole[1][q]) <= 1e-11
