"""The direct Poisson solve and the mixed mode that uses it at tight tolerances."""
import ctypes

import numpy as np
import pytest

from maze_poisson_amd import driver, workloads as W

D = np.ctypeslib.ndpointer(dtype=np.float64, flags="C_CONTIGUOUS")


def _fft_solve(b):
    n = b.shape[0]
    lam = 2 * np.cos(2 * np.pi * np.arange(n) / n) - 2
    l3 = lam[:, None, None] + lam[None, :, None] + lam[None, None, :n // 2 + 1]
    l3[0, 0, 0] = 1.0
    f = np.fft.rfftn(b) / l3
    f[0, 0, 0] = 0.0
    return np.fft.irfftn(f, s=b.shape, axes=(0, 1, 2))


# Half sizes below, at and past whole 16-wide tiles, odd halves, line groups that
# end in the middle of a plane, the largest size.  Both solves round at 2^-53 per
# term of sums of n terms with eigenvalue ratios up to (n / pi)^2: 1e-11 of the
# largest value covers n = 256 with room.
@pytest.mark.gpu
@pytest.mark.parametrize("n", [4, 6, 14, 16, 30, 32, 34, 48, 66, 82, 102, 128, 130, 222, 256])
def test_direct_solve(hip_raw, n):
    g = np.random.default_rng(n)
    b = g.normal(size=(n, n, n))
    b -= b.mean()
    x = np.zeros_like(b)
    f = hip_raw.maze_test_spectral
    f.restype, f.argtypes = ctypes.c_int, [D, D, ctypes.c_int]
    assert f(b, x, n) == n
    ref = _fft_solve(b)
    assert np.abs(x - ref).max() <= 1e-11 * np.abs(ref).max()


@pytest.mark.gpu
def test_direct_solve_sizes(hip_raw):
    f = hip_raw.maze_test_spectral
    f.restype, f.argtypes = ctypes.c_int, [D, D, ctypes.c_int]
    z = np.zeros((1,))
    assert f(z, z, 33) == -1 and f(z, z, 258) == -1 and f(z, z, 2) == -1


def _run(hip, s, rtol, precision, steps=5):
    cfg = driver.RunConfig(tol=W.poisson_tol(s, rtol))
    driver.initialize(hip, s, cfg)
    hip.solver_set_precision(precision)
    driver.bootstrap(hip)
    its = [driver.md_step(hip)[0] for _ in range(steps)]
    passes = hip.solver_get_last_passes(np.zeros(16, dtype=np.int32), 16)
    out = driver.snapshot(hip, s)
    y = np.zeros((s.n_grid,) * 3)
    hip.get_y(y)
    hip.solver_finalize()
    return its, passes, out, y


@pytest.mark.gpu
@pytest.mark.parametrize("n_ions,n_grid", [(216, 48), (512, 66)])
def test_tight_mixed_runs_direct(hip, n_ions, n_grid):
    """Below the multigrid pass's reach the mixed mode solves directly: no inner
    iteration, forces at the FP64 multigrid-free limit; above it nothing changes."""
    s = W.nacl_system(n_ions, n_grid, seed=5)
    its, passes, out, _ = _run(hip, s, 1e-10, 2)
    assert its == [0] * 5 and passes == 0
    _, _, ref, _ = _run(hip, s, 1e-12, 0)
    rms = np.sqrt(((out["fcs_tot"] - ref["fcs_tot"]) ** 2).mean() / (ref["fcs_tot"] ** 2).mean())
    assert rms <= 1e-7  # the FP64 start-up solves at rtol 1e-10 on one side
    its, passes, _, _ = _run(hip, s, 1e-8, 2)
    assert min(its) >= 1 and passes >= 1
