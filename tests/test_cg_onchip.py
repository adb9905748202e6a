"""The one-launch CG (vectors on the chip) against the sweeps, bit for bit."""
import ctypes

import numpy as np
import pytest

from maze_poisson_amd import driver, workloads as W

D = np.ctypeslib.ndpointer(dtype=np.float64, flags="C_CONTIGUOUS")
FIT_MAX = 128  # the largest grid whose vectors fit


def _solve(hip_raw, b, x, tol, n, reductions, onchip, coef=None):
    f = hip_raw.maze_test_conj_grad_form
    P = ctypes.c_void_p
    f.restype = ctypes.c_int
    f.argtypes = [D, D, ctypes.c_double, ctypes.c_int, P, P, P, P, ctypes.c_int, ctypes.c_int]
    ptrs = [None] * 4 if coef is None else [c.ctypes.data for c in coef]
    return f(b, x, tol, n, *ptrs, reductions, onchip)


def _problem(n, seed):
    g = np.random.default_rng(seed)
    b = g.normal(size=(n, n, n))
    return b - b.mean(), g.normal(size=(n, n, n)) * 1e-3


# Slab heights 1 to 16, one to four tiles per work-group, partly filled last
# tiles and slabs, windows that wrap onto themselves.
@pytest.mark.gpu
@pytest.mark.parametrize("reductions", [1, 2])
@pytest.mark.parametrize("n", [2, 5, 16, 23, 31, 32, 48, 57, 64, 73, 81, 100, 113, 126, 127,
                               FIT_MAX])
def test_onchip_cg_equals_sweeps(hip_raw, n, reductions):
    b, x0 = _problem(n, n)
    tol = 1e-7 * np.abs(b).max()
    xs, xo = x0.copy(), x0.copy()
    i_s = _solve(hip_raw, b, xs, tol, n, reductions, 0)
    i_o = _solve(hip_raw, b, xo, tol, n, reductions, 1)
    assert i_o == i_s and i_s >= 0
    assert np.array_equal(xo, xs)


@pytest.mark.gpu
@pytest.mark.parametrize("reductions", [1, 2])
@pytest.mark.parametrize("n", [16, 48, 73, 100, FIT_MAX])
def test_onchip_pb_cg_equals_sweeps(hip_raw, n, reductions):
    b, x0 = _problem(n, n)
    g = np.random.default_rng(7)
    coef = [g.uniform(2.0, 80.0, (n, n, n)) for _ in range(3)] + [g.uniform(0.0, 0.1, (n, n, n))]
    tol = 1e-7 * np.abs(b).max()
    xs, xo = x0.copy(), x0.copy()
    i_s = _solve(hip_raw, b, xs, tol, n, reductions, 0, coef)
    i_o = _solve(hip_raw, b, xo, tol, n, reductions, 1, coef)
    assert i_o == i_s and i_s >= 0
    assert np.array_equal(xo, xs)


# Grids whose x and halo stay in memory: last slabs whole and merged with the one
# before, last work-groups that are nearly full and far smaller than a row, rows that
# start at every offset to a work-group's range.
STREAM_MAX = 161


@pytest.mark.gpu
@pytest.mark.parametrize("pb", [0, 1])
@pytest.mark.parametrize("n", [130, 131, 134, 143, 145, 160, STREAM_MAX])
def test_streaming_cg_equals_sweeps(hip_raw, n, pb):
    b, x0 = _problem(n, n)
    g = np.random.default_rng(7)
    coef = [g.uniform(2.0, 80.0, (n, n, n)) for _ in range(3)] + [g.uniform(0.0, 0.1, (n, n, n))]
    coef = coef if pb else None
    tol = 1e-4 * np.abs(b).max()
    xs, xo = x0.copy(), x0.copy()
    i_s = _solve(hip_raw, b, xs, tol, n, 2, 0, coef)
    i_o = _solve(hip_raw, b, xo, tol, n, 2, 1, coef)
    assert i_o == i_s and i_s >= 0
    assert np.array_equal(xo, xs)


# The one-reduction recurrence against the two-reduction one: the same iterates up to
# rounding.  A relative difference of 1e-16 per sum stays within 1e-10 of the solution
# over a solve of under 300 iterations.
@pytest.mark.gpu
@pytest.mark.parametrize("n", [16, 48, 81, FIT_MAX])
def test_one_reduction_equals_two(hip_raw, n):
    b, x0 = _problem(n, n)
    tol = 1e-6 * np.abs(b).max()
    x1, x2 = x0.copy(), x0.copy()
    i1 = _solve(hip_raw, b, x1, tol, n, 1, 0)
    i2 = _solve(hip_raw, b, x2, tol, n, 2, 0)
    assert i1 == i2
    assert np.linalg.norm(x1 - x2) <= 1e-10 * np.linalg.norm(x2)


@pytest.mark.gpu
@pytest.mark.parametrize("reductions", [1, 2])
def test_onchip_cg_limits(hip_raw, reductions):
    n = (FIT_MAX if reductions == 1 else STREAM_MAX) + 2
    b, x = _problem(n, 1)
    assert _solve(hip_raw, b, x, 1.0, n, reductions, 1) == -2
    # A zero residual stops before the first direction, with x unchanged.
    n = 20
    z, x = np.zeros((n, n, n)), np.full((n, n, n), 3.0)
    assert _solve(hip_raw, z, x, 1e-9, n, reductions, 1) == 0 and (x == 3.0).all()
    # An unreachable tolerance ends at the iteration cap n^2.
    n = 6
    b, x = _problem(n, 2)
    xs = x.copy()
    assert _solve(hip_raw, b, xs, 0.0, n, reductions, 0) == _solve(hip_raw, b, x, 0.0, n, reductions, 1)
    assert np.array_equal(x, xs)


# A launch that finds its solve abandoned leaves x alone, and the sweeps run it.
@pytest.mark.gpu
@pytest.mark.parametrize("n,reductions", [(64, 1), (64, 2), (134, 2)])
def test_abandoned_launch_falls_back(hip_raw, n, reductions):
    b, x0 = _problem(n, 3)
    tol = 1e-6 * np.abs(b).max()
    xs, xo = x0.copy(), x0.copy()
    assert _solve(hip_raw, b, xs, tol, n, reductions, 0) >= 0
    assert _solve(hip_raw, b, xo, tol, n, reductions, 2) == -3
    assert np.array_equal(xo, xs)


# FP64 solves run with one reduction per iteration where their vectors fit the chip, else
# with two, which as sweeps are the faster ones.
@pytest.mark.gpu
@pytest.mark.parametrize("n,reductions", [(64, 1), (FIT_MAX, 1), (FIT_MAX + 1, 2), (136, 2)])
def test_fp64_reductions(hip_raw, n, reductions):
    b, x0 = _problem(n, 6)
    tol = 1e-4 * np.abs(b).max()
    x, xr = x0.copy(), x0.copy()
    assert hip_raw.maze_test_conj_grad(b, x, tol, n) == _solve(hip_raw, b, xr, tol, n, reductions, 0)
    assert np.array_equal(x, xr)
    xr = x0.copy()
    _solve(hip_raw, b, xr, tol, n, 3 - reductions, 0)
    assert not np.array_equal(x, xr)


# Per-kernel timing times the kernels of a run without it.
@pytest.mark.gpu
def test_timing_keeps_the_path(hip, hip_raw):
    s = W.nacl_system(216, 32, seed=1)
    out = []
    for timing in (0, 1):
        driver.initialize(hip, s, driver.RunConfig(tol=W.poisson_tol(s)))
        driver.bootstrap(hip)
        hip_raw.maze_prof_reset()
        hip_raw.maze_prof_enable(timing)
        for _ in range(3):
            hip.solver_md_loop_iter()
        count = {}
        for name in ("cg_onchip", "cg_dir", "cg_update"):
            ms, k = ctypes.c_double(), ctypes.c_long()
            assert hip_raw.maze_prof_get(name.encode(), ctypes.byref(ms), ctypes.byref(k)) == 0
            count[name] = k.value
            assert (ms.value > 0) == (k.value > 0)
        hip_raw.maze_prof_enable(0)
        assert count == {"cg_onchip": 3 * timing, "cg_dir": 0, "cg_update": 0}
        out.append(driver.snapshot(hip, s)["fcs_tot"])
        hip.solver_finalize()
    assert np.array_equal(out[0], out[1])


# One abandoned solve is counted, and solves go on the chip again after a pause.
@pytest.mark.gpu
def test_abandoned_launch_is_tried_again(hip_raw, capfd):
    b, _ = _problem(16, 5)
    f = hip_raw.maze_test_onchip_pause
    I = np.ctypeslib.ndpointer(dtype=np.int32, flags="C_CONTIGUOUS")
    f.restype, f.argtypes = ctypes.c_int, [D, ctypes.c_double, ctypes.c_int, ctypes.c_int, I]
    on_chip = np.full(260, -1, dtype=np.int32)
    assert f(b, 1e-3 * np.abs(b).max(), 16, len(on_chip), on_chip) == 1
    assert (on_chip[:257] == 0).all() and (on_chip[257:] == 1).all()
    assert capfd.readouterr().err.count("waited 0.2 s") == 1


# The first solve after the epochs have run out.
@pytest.mark.gpu
@pytest.mark.parametrize("n,reductions", [(48, 1), (48, 2), (131, 2)])
def test_epochs_start_anew(hip_raw, n, reductions):
    b, x0 = _problem(n, 4)
    tol = 1e-6 * np.abs(b).max()
    xs, xo = x0.copy(), x0.copy()
    i_s = _solve(hip_raw, b, xs, tol, n, reductions, 0)
    assert _solve(hip_raw, b, xo, tol, n, reductions, 3) == i_s >= 0
    assert np.array_equal(xo, xs)


# No launch uses an epoch that may be in the words already, whatever the solves before
# it: a long one (its span is its own cap) followed by short ones among them.
def test_epochs_never_repeat(hip):
    f = hip.lib.maze_test_next_epoch
    f.restype, f.argtypes = ctypes.c_uint, [ctypes.c_uint] * 3
    top = 2 ** 32 - 1
    assert f(top - 100, 49158, 36) == 0
    assert f(top - 72, 36, 36) == top - 36 and f(top - 71, 36, 36) == 0
    g = np.random.default_rng(0)
    epoch, used, low = 1, 6, 1
    for span in (2 ** g.uniform(3, 31, 5000)).astype(np.uint64):
        span = int(span)
        e = f(epoch, used, span)
        assert e == 0 or (e >= epoch + used >= low and e + span <= top)
        epoch, used, low = (e, span, e) if e else (1, span, 1)


# ---- the exchange of sums, as a model ----------------------------------------------
# Every work-group puts its slot of an exchange and waits for the totals; the first
# work-group of a group of slots folds them into the group's sum; where the halo is
# exchanged too, another wave waits for the neighbours' slots.  A wait is for the exact
# epoch, so a word must not move on before everyone who looks for it has seen it.
WGS, PER_GROUP, EXCHANGES = 6, 2, 8


def _waves(w, form, exchange_set):
    """The waves of work-group w as lists of ("put" | "wait", words, epoch) and "meet"."""
    groups = WGS // PER_GROUP
    w0, w1, w2 = [], [], []
    for e in range(1, EXCHANGES + 1):
        s = exchange_set(e)
        halo = form == 1 or e % 2 == 0
        w0.append(("put", [("slot", s, w)], e))
        if halo:
            w1.append(("wait", [("slot", s, (w + d) % WGS) for d in (1, WGS - 1)], e))
        if w < groups:
            w2.append(("wait", [("slot", s, PER_GROUP * w + q) for q in range(PER_GROUP)], e))
            w2.append(("put", [("sum", s, w)], e))
        totals = ("wait", [("sum", s, g) for g in range(groups)], e)
        if halo:  # the totals are taken once the neighbours' values are there
            for x in (w0, w1, w2):
                x.append("meet")
        w0.append(totals)
        for x in (w0, w1, w2):
            x.append("meet")
    return [w0, w1, w2]


def _lost_waits(form, exchange_set):
    """Waits that never end if their wave is held up until all others are stuck."""
    progs = {(w, v): p for w in range(WGS) for v, p in enumerate(_waves(w, form, exchange_set))}
    lost = []
    for victim, prog in progs.items():
        for stop in [i for i, op in enumerate(prog) if op != "meet" and op[0] == "wait"]:
            at, mem, moved = dict.fromkeys(progs, 0), {}, True
            while moved:
                moved = False
                for a, p in progs.items():
                    if at[a] == len(p) or (a == victim and at[a] == stop):
                        continue
                    op = p[at[a]]
                    if op == "meet":  # all three waves of a work-group have come to it
                        if all(at[b] < len(progs[b]) and progs[b][at[b]] == "meet" and
                               progs[b][:at[b]].count("meet") == p[:at[a]].count("meet")
                               for b in progs if b[0] == a[0]):
                            for b in progs:
                                at[b] += b[0] == a[0]
                            moved = True
                    elif op[0] == "put":
                        mem.update({x: op[2] for x in op[1]})
                        at[a] += 1
                        moved = True
                    elif all(mem.get(x) == op[2] for x in op[1]):
                        at[a] += 1
                        moved = True
            if at[victim] == stop and any(mem.get(x) != prog[stop][2] for x in prog[stop][1]):
                lost.append((victim, prog[stop]))
    return lost


@pytest.mark.parametrize("form", [1, 2])
def test_no_exchange_is_missed(hip, form):
    f = hip.lib.maze_test_exchange_set
    f.restype, f.argtypes = ctypes.c_int, [ctypes.c_uint]
    assert _lost_waits(form, f) == []
    assert _lost_waits(form, lambda e: 0)  # one set of words: a late look finds them gone


# A second grid without finalize gives the memory of the first one back.
@pytest.mark.gpu
def test_second_grid_frees_the_first(hip):
    free_now, total = ctypes.c_size_t(), ctypes.c_size_t()
    small, large = W.nacl_system(216, 32, seed=1), W.nacl_system(216, 128, seed=1)
    free = []
    for systems in ([small], [large, small]):
        for s in systems:
            driver.initialize(hip, s, driver.RunConfig(tol=W.poisson_tol(s)))
            driver.bootstrap(hip)
        assert hip.lib.hipMemGetInfo(ctypes.byref(free_now), ctypes.byref(total)) == 0
        free.append(free_now.value)
        hip.solver_finalize()
    assert free[0] - free[1] < 16 << 20  # the first grid's arrays take 150 MB
