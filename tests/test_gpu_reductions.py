"""The reductions finished on the device (core sums, diagnostics, CFL over the
axes, variable difference) against numpy, on grids with fewer and with more
plane chunks than the workgroups of a reduction, one-cell axes and several
patches.  Sums run in FP64: at most 2^-53 per addition of the summed magnitudes,
so 1e-11 of their sum covers the 10^5 cells here; extrema and counts are exact."""
import numpy as np
import pytest

from drnum_amd import configs, hip

pytestmark = pytest.mark.gpu

GRIDS = [[(1, 1, 1)], [(3, 2, 5)], [(17, 16, 16), (1, 300, 2)], [(700, 9, 31)], [(40, 41, 43), (2, 2, 2), (90, 60, 7)]]


def grid(shapes, dtype, seed):
    ctx = hip.Context(dtype)
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    rng = np.random.default_rng(seed)
    h, seeks, fields = (0.5, 0.25, 0.125), [], []
    for n in shapes:
        seek = [1 if m > 3 else 0 for m in n for _ in (0, 1)]
        ctx.add_patch(*n, seek, h, [configs.BC_SLIP] * 6, np.zeros((6, configs.NPAR)))
        seeks.append(seek)
    ctx.layout()
    for p, n in enumerate(shapes):
        c = int(np.prod(n))
        rho = 1.0 + rng.random(c)
        vel = rng.standard_normal((3, c))
        U = np.stack([rho, *(rho * vel), rho * (2.0 + 0.5 * (vel ** 2).sum(0))]).astype(dtype)
        ctx.upload(p, 0, U)
        ctx.upload(p, 1, (U * dtype(1.125)).astype(dtype))
        fields.append(U)
    return ctx, h, seeks, fields


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("shapes", GRIDS)
def test_reductions_against_numpy(gpu, dtype, shapes):
    ctx, h, seeks, fields = grid(shapes, dtype, 5)
    dt = 0.01
    sums, mags, cfl_x, cfl_3 = np.zeros(5), np.zeros(5), 0.0, 0.0
    for n, s, U in zip(shapes, seeks, fields):
        V = U.astype(np.float64).reshape((5,) + n)
        core = V[:, s[0]:n[0] - s[1], s[2]:n[1] - s[3], s[4]:n[2] - s[5]] * (h[0] * h[1] * h[2])
        sums += core.reshape(5, -1).sum(1)
        mags += np.abs(core).reshape(5, -1).sum(1)
        vel = V[1:4] / V[0]
        a = np.sqrt(1.4 * 287.2 * (V[4] / V[0] - 0.5 * (vel ** 2).sum(0)) / 717.5)
        cfl_x = max(cfl_x, np.maximum(np.abs(vel[0] + a), np.abs(vel[0] - a)).max() * dt / h[0])
        cfl_3 = max([cfl_3] + [(np.abs(vel[d]) + a).max() * dt / h[d] for d in range(3)])
    assert np.all(np.abs(ctx.core_sums(0) - sums) <= 1e-11 * mags)
    assert np.array_equal(ctx.core_sums(0), ctx.core_sums(0))
    d = ctx.diagnostics(0, dt)
    rho = np.concatenate([U[0] for U in fields]).astype(np.float64)
    assert (d["rho_min"], d["rho_max"], d["nonfinite"]) == (rho.min(), rho.max(), 0)
    # 1/rho, three products, the energy, the root, the product and the quotient: ten roundings
    assert d["cfl"] == pytest.approx(cfl_x, rel=10 * np.finfo(dtype).eps)
    assert ctx.cfl_axes(0, dt) == pytest.approx(cfl_3, rel=1e-14)
    assert ctx.diagnostics(0, -dt)["cfl"] == 0.0
    for p, U in enumerate(fields):
        sq = ((U[4] * dtype(1.125)).astype(dtype) - U[4]) ** 2
        mx, l2 = ctx.variable_difference(p, 0, 4, 1, 4)
        assert mx == float(np.sqrt(sq.max()))
        assert l2 == pytest.approx(np.sqrt(sq.astype(np.float64).sum()), rel=1e-11)
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_non_finite_values_are_counted_and_left_out(gpu, dtype):
    ctx, h, _, fields = grid([(9, 8, 70), (5, 5, 5)], dtype, 6)
    U = fields[0].copy()
    U[4, 3], U[4, 77], U[1, 200] = np.inf, -np.inf, np.nan
    ctx.upload(0, 0, U)
    d = ctx.diagnostics(0, 0.01)
    assert d["nonfinite"] == 3 and np.isfinite(d["cfl"]) and d["cfl"] > 0
    assert np.isfinite(ctx.cfl_axes(0, 0.01))
    ctx.close()
