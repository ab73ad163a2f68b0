"""CG with all iterations in one launch (onchip_cg.hip) against the kernel-per-step modes, bit for bit."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NOT_RUN, RAN, GAVE_UP = 0, 1, 2


def band(n, offsets, values, seed=0):
    """Symmetric diagonally dominant band matrix in CSR: offsets > 0 given, `values` distinct numbers
    on every diagonal (0: all different)."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    M = sp.csr_matrix((n, n))
    for o in offsets:
        if o < n:
            v = -rng.uniform(0.5, 1.0, n - o) if values == 0 else -1.0 / (1.0 + np.arange(n - o) % values)
            D = sp.diags(v, o, shape=(n, n))
            M = M + D + D.T
    top = float(np.asarray(abs(M).sum(axis=1)).max()) if M.nnz else 1.0
    d = top + 0.05 + (rng.uniform(0, 1, n) if values == 0 else (np.arange(n) % values) * 0.5)
    M = sp.csr_matrix(M + sp.diags(d))
    M.sort_indices()
    return M.indptr.astype(np.uint32), M.indices.astype(np.uint32), M.data.astype(np.float64)


def run(vh, A, b, dtype, **kw):
    db, dx = vh.DeviceArray.from_numpy(b.astype(dtype)), vh.DeviceArray.zeros(b.size, dtype)
    hist = np.zeros(kw["max_iters"])
    vh.lib().onchip_cg_last()
    res = vh.cg(A, db, dx, history=hist, **kw)
    return dx.to_numpy(), res, hist, vh.lib().onchip_cg_last()


def check(vh, A, b, dtype, want, **kw):
    x0, r0, h0, mode = run(vh, A, b, dtype, **kw)
    x1, r1, h1, other = run(vh, A, b, dtype, variant=1, **kw)
    assert mode == want and other == NOT_RUN
    assert r0.iters == r1.iters and np.array_equal(r0.error, r1.error, equal_nan=True) and r0.converged == r1.converged
    assert r0.kernels_per_iter in (1, r1.kernels_per_iter)
    assert np.array_equal(x0, x1, equal_nan=True) and np.array_equal(h0, h1, equal_nan=True)
    return r0


# rows: the edges of tiles, of one owner per chunk (65536), of the workgroup's share (131072), of the
# chunk length (524288) and of the value dictionary (262144); offsets: inside a workgroup's rows, just
# around them, and far (read from memory from two rows per lane on).
CASES = {
    "one_row": (1, [], 1, True), "tile_edge_255": (255, [1], 1, True), "tile_edge_257": (257, [1, 16], 0, True),
    "owners_65535": (65535, [1, 255], 0, True), "owners_65536": (65536, [1, 256], 0, True),
    "owners_65537": (65537, [1, 256], 0, True), "two_tiles_131073": (131073, [1, 300, 6000], 0, True),
    "coded_262144": (262144, [1, 64, 4096], 1, True), "two_values_262145": (262145, [1, 64, 4096], 2, True),
    "regs_300001": (300001, [1, 547], 0, True), "halo_524289": (524289, [1, 80, 6400], 0, True),
    "halo_one_value": (700001, [1, 88, 7744], 1, True), "halo_codes": (700003, [1, 88, 7744], 3, True),
    "halo_wide": (1048577, [1, 101, 10201], 0, True), "halo_wide_one_value": (1500001, [1, 114, 13000], 1, True),
    # a tile per chunk, unequal numbers of chunks per workgroup and a reach of many workgroups: the stencils
    # of 1300 x 19 x 16, 1281 x 62 x 5, 1132 x 37 x 11 and 1568 x 63 x 4 (more workgroups than it waits for)
    "unequal_stored": (395200, [1, 1300, 24700], 0, True), "unequal_one_value": (397110, [1, 1281, 79422], 1, True),
    "unequal_codes": (460724, [1, 1132, 41884], 3, True), "unequal_too_far": (395136, [1, 1568, 98784], 0, False),
    "far_middle": (700001, [1, 7000, 7744], 1, False), "eight_diagonals": (70001, [1, 3, 40, 900], 0, False),
}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("precond", [0, 1])
@pytest.mark.parametrize("case", list(CASES))
def test_equals_the_kernel_per_step_modes(dev, vh, case, precond, dtype):
    """x, iterations, error and history of the one-launch solve equal those of the launched modes bit
    for bit: every partial sum is formed in the same order.  Systems it does not take run launched."""
    n, offsets, values, fits = CASES[case]
    rp, col, val = band(n, offsets, values, seed=n)
    A = vh.CsrMatrix(rp, col, val, dtype=dtype)
    tol = 1e-9 if dtype == np.float64 else 1e-4
    r = check(vh, A, vh.random_uniform(4, n), dtype, RAN if fits else NOT_RUN, precond=precond, tol=tol, max_iters=400)
    assert r.converged


def test_nonsymmetric_reach(dev, vh):
    """Diagonals on one side only (an upper band; CG does not converge on it): the same iterates up to
    the limit."""
    import scipy.sparse as sp
    n = 600001
    M = sp.csr_matrix(sp.diags([np.full(n, 4.0), -np.ones(n - 1), -np.ones(n - 7000)], [0, 1, 7000]))
    A = vh.CsrMatrix(M.indptr.astype(np.uint32), M.indices.astype(np.uint32), M.data)
    check(vh, A, vh.random_uniform(6, n), np.float64, RAN, tol=1e-30, max_iters=37)


def test_more_iterations_than_one_launch_runs(dev, vh):
    """A launch ends after 4096 iterations and the next one goes on: 1-D and 2-D systems (exchanged rows
    of the operator's product, and of the direction) beyond that, and ends at 4096 exactly."""
    for n, offsets in ((9001, [1]), (525001, [1, 6000])):
        rp, col, val = band(n, offsets, 1)
        rows = np.repeat(np.arange(n), np.diff(rp.astype(np.int64)))
        val[col.astype(np.int64) == rows] -= 0.05 - 1e-9  # nearly singular: thousands of iterations
        A = vh.CsrMatrix(rp, col, val)
        for limit in (4095, 4096, 4097, 4610):
            r = check(vh, A, vh.random_uniform(8, n), np.float64, RAN, tol=0.0, max_iters=limit)
            assert r.iters == limit


def test_values_that_are_not_finite(dev, vh):
    """NaN and infinity in the right-hand side spread as in the launched modes."""
    rp, col, val = band(140001, [1, 375], 0)
    A = vh.CsrMatrix(rp, col, val)
    for bad in (np.nan, np.inf):
        b = vh.random_uniform(2, 140001)
        b[70000] = bad
        for pc in (0, 1):
            check(vh, A, b, np.float64, RAN, precond=pc, tol=1e-9, max_iters=9)


def test_gives_up_when_its_workgroups_do_not_meet(dev, vh):
    """With a wait limit of zero every first unsuccessful look gives up: the launched modes take over
    from the start, with their results."""
    limit = vh.lib().onchip_cg_wait_limit
    limit.argtypes = [ctypes.c_double]
    for n, offsets in ((65536, [1, 256]), (700001, [1, 88, 7744])):
        rp, col, val = band(n, offsets, 1)
        A = vh.CsrMatrix(rp, col, val)
        b = vh.random_uniform(3, n)
        limit(0.0)
        try:
            check(vh, A, b, np.float64, GAVE_UP, tol=1e-9, max_iters=400)
        finally:
            limit(-1.0)
        check(vh, A, b, np.float64, RAN, tol=1e-9, max_iters=400)


@pytest.mark.parametrize("case", ["ghost", "halo"])
def test_workgroups_that_start_after_others_gave_up(dev, vh, case):
    """256 workgroups at a wait limit of zero, again and again: the first to look gives up while others
    are still starting, which then leave at once, all waves of a workgroup together.  Every solve ends
    and the launched modes take over with their results."""
    limit = vh.lib().onchip_cg_wait_limit
    limit.argtypes = [ctypes.c_double]
    n, offsets, values = {"ghost": (300001, [1, 547], 0), "halo": (700001, [1, 88, 7744], 3)}[case]
    rp, col, val = band(n, offsets, values, seed=n)
    A, b = vh.CsrMatrix(rp, col, val), vh.random_uniform(3, n)
    want, _, _, _ = run(vh, A, b, np.float64, variant=1, tol=1e-9, max_iters=40)
    limit(0.0)
    try:
        for _ in range(25):
            x, res, _, mode = run(vh, A, b, np.float64, tol=1e-9, max_iters=40)
            assert mode == GAVE_UP and np.array_equal(x, want)
    finally:
        limit(-1.0)


@pytest.mark.parametrize("case", ["whole_device", "quarters", "mixed_sizes"])
def test_solves_of_several_threads_take_turns(dev, vh, case):
    """Solves of host threads on streams of their own: each waits for the compute units it needs and runs on
    chip (none is left to the launched modes, beside which it would hardly progress), one after the other
    or together where they fit, over several launches too; all give what they give alone."""
    whole, quarter = (300001, [1, 547], 0), (60001, [1, 245], 0)
    systems = {"whole_device": [whole, whole], "quarters": [quarter] * 6, "mixed_sizes": [whole, quarter, quarter]}[case]
    made = {s[0]: band(*s, seed=s[0]) for s in systems}
    reps, kw = 6, dict(tol=0.0, max_iters=5000 if case == "mixed_sizes" else 300)
    mats = [vh.CsrMatrix(*made[s[0]]) for s in systems]
    arrays = [(vh.DeviceArray.from_numpy(vh.random_uniform(7, s[0])), vh.DeviceArray.zeros(s[0], np.float64)) for s in systems]
    want = []
    for A, (b, x) in zip(mats, arrays):
        vh.cg(A, b, x, **kw)
        want.append(x.to_numpy())
    streams = [vh.Stream() for _ in systems]
    vh.call("vclhip_device_synchronize")
    modes, got = [[] for _ in systems], [None] * len(systems)

    def work(i):
        for _ in range(reps):
            vh.lib().onchip_cg_last()
            vh.cg(mats[i], *arrays[i], stream=streams[i].handle, **kw)
            modes[i].append(vh.lib().onchip_cg_last())
        got[i] = arrays[i][1].to_numpy(streams[i].handle)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not any(t.is_alive() for t in threads)
    assert all(m == [RAN] * reps for m in modes), modes
    assert all(np.array_equal(g, w, equal_nan=True) for g, w in zip(got, want))
    for s in streams:
        s.close()


def test_leaves_the_device_to_another_threads_launched_solve(dev, vh):
    """Beside a BiCGStab solve of another thread a CG that would take the whole device runs launched, one
    that takes a quarter of it on chip; both on chip again afterwards.  The results are the same."""
    rp, col, val = vh.convection_diffusion(40, 40, 40)
    C, cb, cx = vh.CsrMatrix(rp, col, val), vh.DeviceArray.from_numpy(vh.random_uniform(2, 64000)), vh.DeviceArray.zeros(64000, np.float64)
    solves = [(vh.CsrMatrix(*band(n, o, 0)), vh.random_uniform(3, n), mode)
              for n, o, mode in ((300001, [1, 547], NOT_RUN), (60001, [1, 245], RAN))]
    kw, stream = dict(tol=1e-9, max_iters=400), vh.Stream()
    want = [run(vh, A, b, np.float64, **kw) for A, b, _ in solves]
    vh.call("vclhip_device_synchronize")
    beside, stop = threading.Event(), threading.Event()

    @vh.MONITOR
    def going_on(x, rel, user):
        beside.set()
        return 1 if stop.is_set() else 0

    t = threading.Thread(target=lambda: vh.bicgstab(C, cb, cx, tol=0.0, max_iters=1000000, monitor=going_on, stream=stream.handle))
    t.start()
    try:
        assert beside.wait(30)
        got = [run(vh, A, b, np.float64, **kw) for A, b, _ in solves]
    finally:
        stop.set()
        t.join(timeout=60)
    assert not t.is_alive()
    for (x, _, h, mode), (x0, _, h0, mode0), (_, _, expected) in zip(got, want, solves):
        assert mode0 == RAN and mode == expected and np.array_equal(x, x0) and np.array_equal(h, h0)
    for A, b, _ in solves:
        assert run(vh, A, b, np.float64, **kw)[3] == RAN
    stream.close()


@pytest.mark.parametrize("precond", [0, 1])
def test_solution_over_the_right_hand_side(dev, vh, precond):
    """b and x in one array: the launched modes read b before they write x.  The one-launch solve gives the
    same, and so does a solve that gives up and starts over in the launched modes."""
    limit = vh.lib().onchip_cg_wait_limit
    limit.argtypes = [ctypes.c_double]
    rp, col, val = band(70001, [1, 265], 0)
    A, b = vh.CsrMatrix(rp, col, val), vh.random_uniform(3, 70001)
    kw = dict(precond=precond, tol=1e-9, max_iters=400)
    want, _, _, _ = run(vh, A, b, np.float64, variant=1, **kw)
    for microseconds, mode in ((-1.0, RAN), (0.0, GAVE_UP)):
        x = vh.DeviceArray.from_numpy(b)
        limit(microseconds)
        try:
            res = vh.cg(A, x, x, **kw)
        finally:
            limit(-1.0)
        assert vh.lib().onchip_cg_last() == mode and res.converged
        assert np.array_equal(x.to_numpy(), want)


@pytest.mark.parametrize("case", ["diffusion_small", "diffusion_halo", "laplace_one_value", "sixteen_rows_a_lane", "limit"])
def test_mixed_inner_iterations(dev, vh, case):
    """The mixed solver's FP32 inner iterations between two FP64 corrections in one launch: x, counts,
    error and history equal those of the launched ones bit for bit."""
    k = lambda n, s: np.exp(s * vh.random_normal(3, n))
    rp, col, val = {"diffusion_small": lambda: vh.diffusion(31, 29, 23, k(31 * 29 * 23, 1.0)),
                    "diffusion_halo": lambda: vh.diffusion(95, 91, 89, k(95 * 91 * 89, 1.0)),
                    "laplace_one_value": lambda: vh.laplace_3d(120, 118, 110),
                    "sixteen_rows_a_lane": lambda: vh.diffusion(161, 159, 150, k(161 * 159 * 150, 0.3)),
                    "limit": lambda: vh.fdm_laplace_2d(300, 301)}[case]()
    n = rp.size - 1
    A, b = vh.CsrMatrix(rp, col, val), vh.random_uniform(5, n)
    kw = dict(tol=1e-10, max_iters=150 if case == "limit" else 4000, mixed_mode=1)
    out = []
    for variant in (0, 1):
        db, dx, hist = vh.DeviceArray.from_numpy(b), vh.DeviceArray.zeros(n, np.float64), np.zeros(kw["max_iters"])
        vh.lib().onchip_cg_last()
        res = vh.mixed_cg(A, db, dx, variant=variant, history=hist, **kw)
        out.append((dx.to_numpy(), hist, res, vh.lib().onchip_cg_last()))
    (x0, h0, r0, m0), (x1, h1, r1, m1) = out
    assert (m0, m1) == (RAN, NOT_RUN)
    assert r0.iters == r1.iters and r0.restarts == r1.restarts and r0.error == r1.error and r0.converged == r1.converged
    assert np.array_equal(x0, x1) and np.array_equal(h0, h1)
    assert r0.converged == (case != "limit") and r0.restarts >= 1
