"""The exchange of the receivers that a level-set fill can touch writes no cell that
the full exchange does not write: cells that occur in the donors' receiver lists
but not among the patch's unique receivers stay as they are (CPU: the receiver
counts of the launches after a fill, on a table with one such cell)."""
import numpy as np
import pytest

import fakedev
from fakedev import run_child


def tables(n):
    """Two donors of patch 0 serve patch 1: cell 0 from cell 200, cells 1 and 2 from
    cells 201 and 202; cell 2 is in the donors' lists only (and not among the unique
    receivers)."""
    return dict(receivers=[0, 1], donors=[(0, 1, 1, 0, 0), (0, 2, 1, 1, 1)], rec_concat=[0, 1, 2],
                donor_index=[200, 201, 202], donor_weight=[1.0, 0.5, 0.25])


def levelset():
    """two layer cells of patch 0, donor cells of the table's last two receivers"""
    cells = np.array([201, 202])
    donors = np.tile(np.arange(300, 308), (2, 1))
    return cells, np.tile([1.0, 0.0, 0.0], (2, 1)), donors, np.full((2, 8), 0.125)


def grid(dtype, hip, configs):
    ctx = hip.Context(dtype)
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    for _ in range(2):
        ctx.add_patch(8, 8, 8, [0] * 6, (1.0, 1.0, 1.0), [configs.BC_TRANSMISSIVE] * 6, np.zeros((6, configs.NPAR)))
    ctx.layout()
    ctx.set_exchange(1, tables(8))
    ctx.commit_exchange()
    ctx.set_levelset(0, *levelset())
    ctx.commit_levelset()
    return ctx


def child():
    from drnum_amd import configs, hip

    ctx = grid(np.float32, hip, configs)
    ctx.rk_step(1e-4, [0.5, 1.0])
    fakedev.clear()
    ctx.rk_step(1e-4, [0.5, 1.0])
    lists = [c[2] for c in fakedev.launches("k_exchange_multi")]
    # before each stage the exchange of the touched receivers: cell 1 alone
    assert lists == [1, 1], lists
    ctx.close()


def test_touched_receivers_are_unique_receivers(tmp_path):
    run_child(tmp_path, "test_ls_receivers", "child")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_step_equals_the_separate_calls(gpu, dtype):
    """states after steps with the short exchange and after full exchanges, bit for bit"""
    from drnum_amd import configs, hip

    rng = np.random.default_rng(2)
    states = []
    for _ in range(2):
        rho = 1.0 + 0.1 * rng.random(512)
        vel = 20.0 * rng.standard_normal((3, 512))
        states.append(np.stack([rho, *(rho * vel), 2.5e5 * rho + 0.5 * rho * (vel ** 2).sum(0)]).astype(dtype))
    outs = []
    for by_hand in (False, True):
        ctx = grid(dtype, hip, configs)
        for p, U in enumerate(states):
            ctx.upload(p, 0, U)
        for _ in range(3):
            if not by_hand:
                ctx.rk_step(1e-5, [0.5, 1.0])
                continue
            ctx.exchange(0)
            ctx.copy_field(0, 1)
            for s, a in enumerate((0.5, 1.0)):
                if s:
                    ctx.exchange(0)
                ctx.stage(0, 1, 2, a * 1e-5)
                ctx.swap_fields(0, 2)
                ctx.exchange(0)
                ctx.levelset_fill(0)
        outs.append([ctx.download(p, 0) for p in range(2)])
        ctx.close()
    for a, b in zip(*outs):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
