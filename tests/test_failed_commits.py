"""A table commit that runs out of device memory returns an error and leaves a
context whose steps launch on complete lists only: every device allocation and
copy of the commit fails once, and the stages, the exchange and the fill after it are looked
over (CPU: the launches are recorded, not carried out)."""
import ctypes as C

import numpy as np
import pytest

import fakedev
from fakedev import run_child


def _context(w, choice, viscous):
    from drnum_amd import hip, host

    hg = host.HostGrid.from_workload(w, fp64_geometry=True)
    hg.compute_dependencies(w.periodic)
    ctx = hip.Context(np.float32)
    ctx.set_operator(w.recon, w.limiter, viscous)
    hg.to_device(ctx)
    if choice is not None:
        for launch in (0, 1):
            ctx.set_tiling(choice, launch)
    return hg, ctx


def _step(ctx, w, launch):
    fakedev.clear()
    ctx.rk_step(w.dt, w.alpha, launch)
    return fakedev.launches()


def _check(calls, np_, n_stage, what):
    """the stage launches of a step: complete work lists in device memory"""
    stages = [c for c in calls if c[0].startswith("k_stage")]
    assert stages, what
    for name, grid, pds, tiles in stages:
        assert fakedev.fake.fake_is_device(pds) and fakedev.fake.fake_is_device(tiles), (what, name)
        per = 16  # TileCell and TileMarch: patch and three more 32-bit values
        patches = np.ctypeslib.as_array(C.cast(tiles, C.POINTER(C.c_int32)), (grid * per // 4,)).reshape(grid, 4)[:, 0]
        assert patches.min() >= 0 and patches.max() < np_, (what, name)
    assert sum(c[1] for c in stages) in n_stage, (what, sum(c[1] for c in stages), n_stage)
    for name, n, a0, a1 in calls:
        if name.startswith("k_ls_access"):
            assert fakedev.fake.fake_is_device(a1), (what, name)


def exchange_child():
    from drnum_amd import configs

    fail = fakedev.fake.fake_fail_after
    for w, choice, viscous in ((configs.jet(core=8, blocks=2), None, False), (configs.jet(core=8, blocks=2), 52, False),
                               (configs.jet(core=8, blocks=2), 53, False), (configs.jet(core=8, blocks=2), 47, False),
                               (configs.viscous_shear(core=6, blocks=(2, 1, 2)), None, True)):
        np_ = len(w.patches)
        for launch in (0, 1):
            hg, ctx = _context(w, choice, viscous)
            whole = {sum(c[1] for c in _step(ctx, w, launch) if c[0].startswith("k_stage"))}
            hg.upload_exchange(ctx)
            box = {sum(c[1] for c in _step(ctx, w, launch) if c[0].startswith("k_stage"))}
            ctx.set_tiling(52, launch)
            box.add(sum(c[1] for c in _step(ctx, w, launch) if c[0].startswith("k_stage")))
            ctx.close()
            k = 0
            while True:
                hg, ctx = _context(w, choice, viscous)
                fail(k)
                failed = False
                try:
                    hg.upload_exchange(ctx)
                except Exception:
                    failed = True
                fail(-1)
                _check(_step(ctx, w, launch), np_, whole | box, (w.name, choice, launch, k))
                if failed:  # the same tables commit once there is memory again
                    hg.upload_exchange(ctx)
                    _check(_step(ctx, w, launch), np_, box, (w.name, choice, launch, k, "again"))
                ctx.close()
                if not failed:
                    break
                k += 1
            assert k > 10


def levelset_child():
    from drnum_amd import configs

    fail = fakedev.fake.fake_fail_after
    w = configs.levelset_spheres(core=16, blocks=(2, 1, 1), n_spheres=1, r_range=(3.0, 3.5))
    k = 0
    while True:
        hg, ctx = _context(w, None, False)
        hg.upload_exchange(ctx)
        hg.levelset_spheres(w.spheres, w.ls_inner_layers, 0, w.ls_min_inner_rel)
        fail(k)
        failed = False
        try:
            hg.upload_levelset(ctx)
        except Exception:
            failed = True
        fail(-1)
        calls = _step(ctx, w, 0)
        _check(calls, len(w.patches), {sum(c[1] for c in calls if c[0].startswith("k_stage"))}, k)
        if failed:
            hg.upload_levelset(ctx)
        calls = _step(ctx, w, 0)
        assert any(c[0].startswith("k_ls_access") for c in calls)
        _check(calls, len(w.patches), {sum(c[1] for c in calls if c[0].startswith("k_stage"))}, k)
        ctx.close()
        if not failed:
            break
        k += 1
    assert k > 4


@pytest.mark.parametrize("child", ["exchange_child", "levelset_child"])
def test_every_allocation_and_copy_may_fail(tmp_path, child):
    run_child(tmp_path, "test_failed_commits", child)
