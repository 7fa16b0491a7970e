"""The bytes that bench.py prices the kernels at, against the grid and against the
lists that the device library launches (CPU: the launches are recorded, not carried
out)."""
import importlib.util
import os

import numpy as np

import fakedev
from fakedev import ROOT, run_child


def bench():
    spec = importlib.util.spec_from_file_location("bench_mod", os.path.join(ROOT, "bench.py"))
    b = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(b)
    return b


def _grid(w):
    from drnum_amd import host

    hg = host.HostGrid.from_workload(w, fp64_geometry=True)
    hg.compute_dependencies(w.periodic)
    return hg


def test_stage_bytes_of_the_jet():
    """16,777,216 of 19,248,832 cells are no receivers; 786,432 receivers are fused"""
    from drnum_amd import configs

    b, w = bench(), configs.jet(core=64, blocks=4)
    hg = _grid(w)
    assert b.stage_cells(hg, w, 49, 786_432) == (19_248_832,) * 3
    cells = b.stage_cells(hg, w, 53, 786_432)
    assert cells == (19_248_832, 16_777_216, 16_777_216 + 786_432)
    # three stages: 5 values of 4 B each
    assert b.stage_bytes_per_step(cells, 4, 3) == 20 * (3 * 19_248_832 + 2 * 16_777_216 + 3 * 17_563_648)
    assert b.stage_bytes_per_step((7, 7, 7), 4, 3) == 7 * 40 * 4


def test_stage_bytes_of_the_viscous_box():
    from drnum_amd import configs

    w = configs.viscous_shear(core=6, blocks=(2, 2, 2))
    n = 8 * 6 * 6 * 10  # the planes and rows without receivers, whole along z
    assert bench().stage_cells(_grid(w), w, 35, 0) == (8 * 1000, n, n)


def test_the_default_choice_of_the_jet_has_a_profile():
    """the traffic and VALU entries of the bench line need the running choice's counters"""
    b = bench()
    for choice in (52, 53):
        row = b.sweep_profile(choice)
        # no more than twice the bytes that the launch cannot do without
        assert 0.9e9 < row["traffic"] < 2.0e9 and 1e8 < row["instructions"] < 1e9
        assert 87_629_568 <= row["exchange"] < 2 * 87_629_568
    assert b.sweep_profile(11) is None
    assert b.profile_hash(b.SWEEP_TABLE) is not None


def touched_child():
    from drnum_amd import configs, hip

    b = bench()
    w = configs.levelset_spheres(core=16, blocks=(2, 2, 1), n_spheres=1, r_range=(3.0, 3.5))
    w.spheres = np.array([[1.0, 15.0 / 16.0, 0.5, 4.2 / 16.0]])
    hg = _grid(w)
    ctx = hip.Context(np.float32)
    ctx.set_operator(w.recon, w.limiter)
    hg.to_device(ctx)
    hg.upload_exchange(ctx)
    hg.levelset_spheres(w.spheres, w.ls_inner_layers, 0, w.ls_min_inner_rel)
    hg.upload_levelset(ctx)
    ctx.rk_step(w.dt, w.alpha)
    fakedev.clear()
    ctx.rk_step(w.dt, w.alpha)
    calls = fakedev.launches()
    # the exchange before each stage: the launches that are followed by a stage kernel
    before = [calls[q][2] for q in range(len(calls) - 1) if calls[q + 1][0].startswith("k_stage")]
    n_rec, n_pairs = b.touched_receivers(hg, w)
    assert n_rec > 0 and before == [n_rec] * 3, (before, n_rec)
    assert n_pairs >= n_rec and b.touched_bytes(hg, w, 4) == 24 * n_rec + 28 * n_pairs
    ctx.close()


def test_touched_receivers_are_those_of_the_device_list(tmp_path):
    run_child(tmp_path, "test_bench_bytes", "touched_child")
