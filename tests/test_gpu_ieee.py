"""The box kernel (choices 51, 52) in IEEE arithmetic beside the cell-per-thread
kernel (choice 11), whose forms are the reference's: no further from 64 bits."""
import numpy as np
import pytest

from drnum_amd import configs, hip, solver
from oracle import oracle as O
from test_gpu_parity import make

pytestmark = pytest.mark.gpu

N = 32  # the spacing 1/32 and its powers are exact in both types


def flow(mach, pressure, rough, seed):
    """smooth in all directions, with noise of `rough` times its amplitude"""
    rng = np.random.default_rng(seed)
    x = 2.0 * np.pi * (np.arange(N) + 0.5) / N

    def f():
        out = rough * rng.standard_normal((N, N, N))
        for _ in range(4):
            s = [np.sin(rng.integers(1, 4) * x + rng.uniform(0.0, 6.0)) for _ in range(3)]
            out = out + rng.uniform(0.3, 1.0) * s[0][:, None, None] * s[1][None, :, None] * s[2][None, None, :]
        return out

    p, rho = pressure * (1.0 + 0.05 * f()), 1.0 + 0.05 * f()
    vel = [mach * np.sqrt(1.4 * pressure) * (0.3 + 0.5 * f()) for _ in range(3)]
    return np.stack([rho, *(rho * v for v in vel), p * (717.5 / 287.2) + 0.5 * rho * sum(v * v for v in vel)])


def residuals(w, U, choices, dtype):
    """drn_stage on a base field of zeros with factor dV gives the residual itself"""
    gg = solver.GpuGrid(w, dtype)
    gg.ctx.set_arith(hip.DRN_ARITH_IEEE)
    gg.ctx.upload(0, 0, U)
    gg.ctx.upload(0, 1, np.zeros_like(U))
    out = []
    for c in choices:
        gg.ctx.set_tiling(c)
        gg.ctx.stage(0, 1, 2, 1.0 / N ** 3)
        out.append(gg.ctx.download(0, 2))
    gg.close()
    return out


@pytest.mark.parametrize("recon", [configs.RECON_UPWIND1, configs.RECON_UPWIND2])
@pytest.mark.parametrize("mach,pressure,rough", [(0.3, 1.0 / 1.4, 0.0), (0.3, 1.0 / 1.4, 0.3), (1.2, 1.0 / 1.4, 0.0),
                                                 (0.1, 1.0e5, 0.0), (0.5, 1.0e5, 0.3)])
def test_rounding_error_of_the_residual(gpu, recon, mach, pressure, rough):
    """FP32 residuals against the oracle's FP64 residual of the same FP32 state: the
    rms error per variable of the box kernel is at most the cell kernel's.  Both
    round the same formulas; over 3 x 32,768 cells the two rms values of equal
    error sources differ by sampling alone, 1 / sqrt(2 x 98,304) = 0.23 %, of
    which 1 % is more than four times."""
    w = configs.sod(n=N)
    w.recon = recon
    err = np.zeros((3, 5))
    for seed in range(3):
        U = flow(mach, pressure, rough, seed).reshape(5, -1).astype(np.float32)
        og = O.OracleGrid(w, np.float64, threads=8)
        og.field(0, 0)[:] = U
        exact = og.residual(0)
        err += [((g.astype(np.float64) - exact) ** 2).mean(1) for g in residuals(w, U, (11, 51, 52), np.float32)]
    err = np.sqrt(err)
    print("rms error", recon, mach, pressure, rough, err[0], err[1] / err[0], flush=True)
    assert np.isfinite(err).all()
    assert (err[1:] <= 1.01 * err[0]).all()


@pytest.mark.parametrize("power", [30, 45, 52, 60, 84, 110])
def test_large_states(gpu, power):
    """FP32 states times a power of two, up to where their squares leave the type's
    range: the residual is homogeneous of degree one, and with differences that are
    zero or above nonZero's 1e-10 every value of it scales exactly."""
    w = configs.sod(n=N)
    U = flow(0.3, 1.0 / 1.4, 0.3, 9).reshape(5, -1).astype(np.float32)
    scale = np.float32(2.0) ** power
    for small, large in zip(residuals(w, U, (51, 52), np.float32), residuals(w, U * scale, (51, 52), np.float32)):
        assert np.isfinite(large).all()
        assert np.array_equal(large, small * scale)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("arith", [hip.DRN_ARITH_IEEE, hip.DRN_ARITH_FAST])
def test_non_finite_values_spread_as_in_the_cell_kernel(gpu, dtype, arith):
    """Residuals around single NaN and infinite values and a negative energy: the
    same values are finite as in choice 11, so that the count of non-finite
    values that a program watches is the same."""
    w = configs.sod(n=N)
    U = flow(0.3, 1.0 / 1.4, 0.0, 5).reshape(5, -1).astype(dtype)
    n = 0
    for v in range(5):
        for x in (np.nan, np.inf, -np.inf):
            U[v, 37 + 2111 * n] = x
            n += 1
    U[4, 37 + 2111 * n] = -1.0
    gg = solver.GpuGrid(w, dtype)
    gg.ctx.set_arith(arith)
    gg.ctx.upload(0, 0, U)
    gg.ctx.upload(0, 1, np.zeros_like(U))
    out = []
    for c in (11, 51, 52):
        gg.ctx.set_tiling(c)
        gg.ctx.stage(0, 1, 2, 1.0 / N ** 3)
        out.append(np.isfinite(gg.ctx.download(0, 2)))
    gg.close()
    print("non-finite", dtype.__name__, arith, [int((~o).sum()) for o in out], flush=True)
    assert not out[0].all()
    for o in out[1:]:
        assert np.array_equal(o, out[0])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("arith", [hip.DRN_ARITH_IEEE, hip.DRN_ARITH_FAST])
def test_non_finite_values_after_a_step(gpu, dtype, arith):
    """The same on patches with exchange receivers after one RK step, for all cells:
    boxes, and the sweep (53) in FP32 fast arithmetic, beside choice 11"""
    w = configs.jet(core=24, blocks=2)
    rng = np.random.default_rng(8)
    states = [w.initial_state(p, dtype) for p in range(len(w.patches))]
    for U in states:
        for v in range(5):
            U.reshape(5, -1)[v, rng.integers(0, U.reshape(5, -1).shape[1])] = rng.choice([np.nan, np.inf, -np.inf])
    masks = []
    for choice in (11, 51, 52, 53):
        _, gg = make(w, dtype)
        gg.ctx.set_arith(arith)
        gg.ctx.set_tiling(choice)
        gg.upload_state(states)
        gg.rk_step()
        masks.append([np.isfinite(U) for U in gg.state(0)])
        gg.close()
    print("non-finite after a step", dtype.__name__, arith, [sum(int((~a).sum()) for a in m) for m in masks], flush=True)
    assert not all(a.all() for a in masks[0])
    for m in masks[1:]:
        for a, b in zip(masks[0], m):
            assert np.array_equal(a, b)
