"""The work-list choices as drn_get_tiling, drn_autotune and the launches show them
(CPU: the launches are recorded, not carried out)."""
import numpy as np
import pytest

import fakedev
from fakedev import run_child


def context(w, viscous=None, dtype=np.float32):
    from drnum_amd import hip, host

    hg = host.HostGrid.from_workload(w, fp64_geometry=True)
    hg.compute_dependencies(w.periodic)
    ctx = hip.Context(dtype)
    ctx.set_operator(w.recon, w.limiter, w.viscous if viscous is None else viscous)
    hg.to_device(ctx)
    hg.upload_exchange(ctx)
    return hg, ctx


def stage_lists(call):
    """(kernel, work list) of the stage launches of a call, in order"""
    fakedev.clear()
    call()
    return [(c[0], c[3]) for c in fakedev.launches("k_stage")]


def autotune_child():
    """With the viscous or the flagged operator every choice runs the same list inside
    the RK step: the autotuner times drn_stage's lists, each once."""
    from drnum_amd import configs

    w = configs.viscous_shear(core=9, blocks=(2, 2, 2))
    for viscous in (True, False):
        hg, ctx = context(w, viscous)
        if not viscous:
            flags = np.zeros(w.patches[0].cells, np.uint8)
            flags[::5] = 1
            ctx.set_cell_flags(0, flags)
        for launch in (0, 1):
            np_ = len(w.patches) if launch else 1
            runs = stage_lists(lambda: ctx.autotune(launch))
            tried = [tuple(runs[q:q + np_]) for q in range(0, len(runs), np_)]
            # a warm-up and three timed stages per candidate
            assert len(tried) % 4 == 0 and all(len(set(tried[q:q + 4])) == 1 for q in range(0, len(tried), 4))
            lists = tried[::4]
            assert len(lists) > 1 and len(set(lists)) == len(lists), (viscous, launch, len(lists), len(set(lists)))
            best = ctx.get_tiling(launch)
            alone = stage_lists(lambda: ctx.stage(0, 1, 2, 0.0, launch))
            assert tuple(alone) in lists, (viscous, launch, best)
        ctx.close()


def sweep_fallback_child():
    """Where the sweep does not run (FP64, IEEE, rows too long for its tile, no receivers)
    it is no candidate beside the box kernel that stands in for it."""
    from drnum_amd import configs, hip

    long_rows = configs.Workload("rows", configs.block_grid([6, 6, 500], [1, 1, 2], [1.0] * 3, 2, [True] * 3,
                                                            [configs.BC_SLIP] * 6), configs.RECON_UPWIND2,
                                 configs.LIM_VANALBADA, [1.0] * 3, [1.0], 1e-3, None)
    for w, dtype, arith in ((configs.jet(core=9, blocks=2), np.float64, None),
                            (configs.jet(core=9, blocks=2), np.float32, hip.DRN_ARITH_IEEE),
                            (long_rows, np.float32, None), (configs.sod(n=16), np.float32, None)):
        hg, ctx = context(w, dtype=dtype)
        if arith is not None:
            ctx.set_arith(arith)
        for launch in (0, 1):
            np_ = len(w.patches) if launch else 1
            runs = [k for k, _ in stage_lists(lambda: ctx.autotune(launch)) if k.startswith("k_stage_box")]
            # one and four planes per item: a warm-up and three timed stages each
            assert len(runs) == 2 * 4 * np_ and len(set(runs)) == 2, (w.name, dtype, launch, len(runs), set(runs))
        ctx.close()


def fusion_child():
    """drn_get_tiling answers the choice whose kernel runs, with the exchange fusion on
    and off (then the RK step runs on whole patches, which the sweep does not)"""
    from drnum_amd import configs

    w = configs.jet(core=40, blocks=5)
    names = {51: "k_stage_box<float, 1, 0, true, 1>", 52: "k_stage_box<float, 1, 0, true, 4>",
             53: "k_stage_sweep<float, 1, 0, true, 168, 4>"}
    hg, ctx = context(w)
    seen = []
    for on in (True, False, True):
        ctx.set_exchange_fusion(on)
        kernels = {c[0] for c in stage_lists(lambda: ctx.rk_step(w.dt, w.alpha))}
        assert kernels == {names[ctx.get_tiling()]}, (on, ctx.get_tiling(), kernels)
        seen.append(ctx.get_tiling())
    assert seen == [53, 52, 53], seen
    ctx.close()


@pytest.mark.parametrize("child", ["autotune_child", "sweep_fallback_child", "fusion_child"])
def test_choices(tmp_path, child):
    run_child(tmp_path, "test_tiling_rules", child)
