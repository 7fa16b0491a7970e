"""The box kernel (tiling choices 51 and 52) and the sweep over the same positions
(53, FP32 fast arithmetic in the RK step): one thread per cell of the patch's box,
which in the RK step leaves out the planes, rows and z layers whose cells
are all exchange receivers.  Against the oracle where its lanes, planes and
boxes can go wrong: row lengths around its 62 positions per wavefront, plane
counts around its 4 planes per item, whole patches (drn_stage alone), thin
patches, every limiter; and bit for bit between one and four planes, launch
forms, with the boxes switched off, and in FP32 with choice 11."""
import copy

import numpy as np
import pytest

from drnum_amd import configs, hip
from test_gpu_fused_exchange import run as run_fused
from test_gpu_fused_exchange import setup as setup_fused
from test_gpu_parity import TOL, make, rel_linf
from test_gpu_thin import SHAPES, thin

pytestmark = pytest.mark.gpu

B, PP = hip.DRN_LAUNCH_BATCHED, hip.DRN_LAUNCH_PER_PATCH
CHOICES = (51, 52, 53)


def wave(nx, zc, bc=None):
    """Two patches along z of nx x 5 x zc core cells, periodic (or with face
    functors bc on a closed box), smooth in all directions, Mach about 0.4."""
    patches = configs.block_grid([nx, 5, 2 * zc], [1, 1, 2], [1.0] * 3, 2, [bc is None] * 3,
                                 bc or [configs.BC_SLIP] * 6)

    def init(x, y, z):
        p = configs.P_AMB * (1.0 + 0.05 * np.sin(2.0 * np.pi * z))
        T = p / ((1.0 + 0.1 * np.cos(2.0 * np.pi * (x + z))) * configs.gas.R)
        return np.stack([p, T, 0.2 * np.sin(2.0 * np.pi * z), 0.1 * np.cos(2.0 * np.pi * x),
                         0.1 + 0.2 * np.sin(2.0 * np.pi * y)])

    dt = 0.4 * (1.0 / max(nx, 2 * zc)) / 1.5
    return configs.Workload("wave%dx%d" % (nx, zc), patches, configs.RECON_UPWIND2, configs.LIM_VANALBADA,
                            [1.0 if bc is None else 0.0] * 3, [0.25, 0.5, 1.0], dt, init)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nx,zc", [(3, 2), (4, 29), (5, 59), (6, 60), (7, 61), (8, 62), (4, 63), (5, 124),
                                   (9, 70), (19, 65), (3, 197)])
@pytest.mark.parametrize("walls", [False, True])
def test_lanes_planes_and_rows(gpu, dtype, nx, zc, walls):
    w = wave(nx, zc, [configs.BC_TRANSMISSIVE, configs.BC_SLIP] * 3 if walls else None)
    og, _ = make(w, dtype)
    for _ in range(4):
        og.rk_step()
    for choice in CHOICES:
        _, gg = make(w, dtype)
        gg.ctx.set_tiling(choice, B)
        gg.ctx.set_tiling(choice, PP)
        for s in range(4):
            gg.rk_step(B if s % 2 == 0 else PP)
        err = rel_linf(gg.state(0), og)
        print("box", w.name, walls, choice, np.dtype(dtype).name, err, flush=True)
        assert err <= TOL[dtype]
        gg.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_stage_alone_covers_the_whole_patch(gpu, dtype):
    """drn_stage updates every stored cell, seek layers included"""
    w = configs.jet(core=9, blocks=2)
    for choice in CHOICES:
        og, gg = make(w, dtype)
        gg.ctx.set_tiling(choice)
        og.copy_field(0, 1)
        og.compute(0.25 * w.dt)
        gg.ctx.copy_field(0, 1)
        gg.ctx.stage(0, 1, 2, 0.25 * w.dt)
        assert rel_linf(gg.state(2), og) <= TOL[dtype]
        gg.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("cells,blocks", SHAPES)
def test_thin_patches(gpu, dtype, cells, blocks):
    w = thin(cells, blocks)
    og, _ = make(w, dtype)
    for _ in range(4):
        og.rk_step()
    for choice in CHOICES:
        for launch in (B, PP):
            _, gg = make(w, dtype)
            gg.ctx.set_tiling(choice, launch)
            for _ in range(4):
                gg.rk_step(launch=launch)
            assert rel_linf(gg.state(0), og) <= TOL[dtype], (choice, launch)
            gg.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("recon,limiter", [(configs.RECON_UPWIND1, configs.LIM_VANALBADA),
                                           (configs.RECON_UPWIND2, configs.LIM_MINMOD),
                                           (configs.RECON_UPWIND2, configs.LIM_SECONDORDER)])
@pytest.mark.parametrize("arith", [hip.DRN_ARITH_IEEE, hip.DRN_ARITH_FAST])
def test_limiters_and_arithmetic(gpu, dtype, recon, limiter, arith):
    w = copy.copy(wave(6, 33))
    w.recon, w.limiter = recon, limiter
    og, _ = make(w, dtype)
    for _ in range(3):
        og.rk_step()
    for choice in CHOICES:
        _, gg = make(w, dtype)
        gg.ctx.set_arith(arith)
        gg.ctx.set_tiling(choice)
        for _ in range(3):
            gg.rk_step()
        assert rel_linf(gg.state(0), og) <= TOL[dtype], choice
        gg.close()


@pytest.mark.parametrize("arith", [hip.DRN_ARITH_IEEE, hip.DRN_ARITH_FAST])
@pytest.mark.parametrize("choice", CHOICES)
def test_sod_stays_uniform(gpu, choice, arith):
    """no transverse momentum, uniform planes, exactly (as test_sod_keeps_mirror_symmetry)"""
    n = 16
    _, gg = make(configs.sod(n=n), np.float32)
    gg.ctx.set_tiling(choice)
    gg.ctx.set_arith(arith)
    for _ in range(10):
        gg.rk_step()
    G = gg.state(0)[0].reshape(5, n, n, n)
    assert np.isfinite(G).all()
    assert np.count_nonzero(G[2]) == 0 and np.count_nonzero(G[3]) == 0
    for v in (0, 1, 4):
        assert np.array_equal(G[v], np.broadcast_to(G[v][:, :1, :1], G[v].shape)), v
    gg.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("make_w", [lambda: configs.jet(core=23, blocks=2), lambda: configs.kelvin_helmholtz(core=9, blocks=1),
                                    lambda: configs.kelvin_helmholtz(core=2, blocks=2),
                                    lambda: configs.uneven_batch(n_patches=30, size_range=(12, 24)),
                                    lambda: configs.rotated_star(core=16, tilt_deg=7.0),
                                    lambda: configs.levelset_spheres(core=24, r_range=(3.0, 6.0))],
                         ids=["jet", "kh1", "kh_thin", "uneven", "star", "spheres"])
def test_boxes_change_no_bit(gpu, dtype, make_w):
    """Every stored cell after three steps: one and four planes per item, both
    launch forms, and the boxes off (drn_set_exchange_fusion(0): whole patches);
    in FP32 fast arithmetic also the cell-per-thread kernel (choice 11)."""
    w = make_w()
    ref, _ = run_fused(w, dtype, False, 51, B)
    forms = [(True, 51, B), (True, 52, B), (True, 51, PP), (True, 52, PP), (False, 52, B), (True, 53, B),
             (True, 53, PP)]
    if dtype == np.float32:
        forms.append((True, 11, B))
    for fuse, choice, launch in forms:
        got, _ = run_fused(w, dtype, fuse, choice, launch)
        for p, (a, b) in enumerate(zip(ref, got)):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b), (fuse, choice, launch, p)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("viscous", [False, True])
@pytest.mark.parametrize("launch", [B, PP])
def test_boxes_of_the_flagged_and_the_viscous_operator(gpu, dtype, viscous, launch):
    """The z-shared cell kernel, which these operators run, on the boxes' planes
    and rows: every stored cell as with whole patches (boxes off), for row
    lengths that end an item inside and beyond the box."""
    for core in (5, 13, 18):
        w = configs.viscous_shear(core=core, blocks=(2, 1, 2))
        outs = []
        for fuse in (False, True):
            hg, ctx = setup_fused(w, dtype, fuse)
            ctx.set_operator(w.recon, w.limiter, viscous)
            if not viscous:
                for p, P in enumerate(w.patches):
                    flags = np.zeros(P.cells, np.uint8)
                    flags[::7] = 1
                    flags[3::11] |= 2
                    ctx.set_cell_flags(p, flags)
            for _ in range(3):
                ctx.rk_step(w.dt, w.alpha, launch)
            outs.append([ctx.download(p, 0) for p in range(len(w.patches))])
            ctx.close()
        for a, b in zip(*outs):
            assert np.isfinite(a).all()
            assert np.array_equal(a, b), core
