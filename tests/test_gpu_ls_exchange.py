"""The exchange before a stage that follows a level-set fill copies only the
receivers the fill can have touched (filled cells and receivers of filled
donors).  Every stored cell must come out as with full exchanges called one by
one, for spheres that lie across patch overlaps, in steps, in the graph, after
other calls between the steps and after the tables are set anew."""
import numpy as np
import pytest

from drnum_amd import configs, hip, host

pytestmark = pytest.mark.gpu

ALPHA = [0.25, 0.5, 1.0]


def workload(blocks, where):
    w = configs.levelset_spheres(core=16, blocks=blocks, n_spheres=1, r_range=(3.0, 3.5))
    w.spheres = np.array([[x / 16.0, y / 16.0, z / 16.0, 4.2 / 16.0] for x, y, z in where])
    return w


def setup(w, dtype):
    hg = host.HostGrid.from_workload(w, fp64_geometry=True)
    hg.compute_dependencies(w.periodic)
    ctx = hip.Context(dtype)
    ctx.set_operator(w.recon, w.limiter)
    hg.to_device(ctx)
    hg.upload_exchange(ctx)
    hg.levelset_spheres(w.spheres, w.ls_inner_layers, 0, w.ls_min_inner_rel)
    hg.upload_levelset(ctx)
    for p in range(len(w.patches)):
        ctx.upload(p, 0, w.initial_state(p, dtype))
    return hg, ctx


def by_hand(ctx, dt, steps):
    for _ in range(steps):
        ctx.exchange(0)
        ctx.copy_field(0, 1)
        for s, a in enumerate(ALPHA):
            if s:
                ctx.exchange(0)
            ctx.stage(0, 1, 2, a * dt)
            ctx.swap_fields(0, 2)
            ctx.exchange(0)
            ctx.levelset_fill(0)


def states(ctx, w):
    return [ctx.download(p, 0) for p in range(len(w.patches))]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("blocks,where", [((2, 1, 1), [(16.0, 8.0, 8.0)]), ((2, 2, 2), [(16.0, 15.0, 17.0)]),
                                          ((2, 2, 1), [(8.0, 8.0, 8.0)]), ((3, 2, 2), [(16.0, 9.0, 8.0), (30.0, 16.0, 16.0)])])
def test_touched_receivers_suffice(gpu, dtype, blocks, where):
    w = workload(blocks, where)
    _, ref = setup(w, dtype)
    hg, got = setup(w, dtype)

    def same(what):
        for p, (a, b) in enumerate(zip(states(ref, w), states(got, w))):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b), (what, p)

    by_hand(ref, w.dt, 3)
    for _ in range(3):
        got.rk_step(w.dt, ALPHA)
    same("steps")
    by_hand(ref, w.dt, 5)
    got.rk_graph_run(w.dt, ALPHA, 5)
    same("graph")
    # writes and fills between the steps
    U = states(ref, w)[0] * np.asarray(1.01, dtype)
    for ctx in (ref, got):
        ctx.upload(0, 0, U)
        ctx.levelset_fill(0)
        ctx.levelset_fill(0)
    by_hand(ref, w.dt, 1)
    got.rk_step(w.dt, ALPHA)
    same("after an upload and two fills")
    got.rk_graph_run(w.dt, ALPHA, 4)
    by_hand(ref, w.dt, 4)
    same("graph again")
    # the same tables committed anew, in both orders
    hg.upload_levelset(got)
    hg.upload_exchange(got)
    got.rk_step(w.dt, ALPHA)
    by_hand(ref, w.dt, 1)
    same("tables anew")
    got.close()
    ref.close()
