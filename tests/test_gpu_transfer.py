"""drn_patch_upload / drn_patch_download and drn_post_variables through the
pinned staging memory: byte for byte, for value counts that do and do not
divide into 16-byte lanes, patches below and above a staging half (8 MiB), and
several patches and fields behind each other."""
import numpy as np
import pytest

from drnum_amd import configs, hip

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 1, 3), (3, 1, 1), (4, 5, 7), (16, 16, 16), (33, 35, 37), (74, 75, 76), (80, 81, 83), (120, 121, 64)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_round_trip_is_exact(gpu, dtype):
    ctx = hip.Context(dtype)
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    for n in SHAPES:
        ctx.add_patch(*n, [0] * 6, (1.0, 1.0, 1.0), [configs.BC_SLIP] * 6, np.zeros((6, configs.NPAR)))
    ctx.layout()
    rng = np.random.default_rng(3)
    for field in (0, 2):
        states = [rng.standard_normal((5, int(np.prod(n)))).astype(dtype) for n in SHAPES]
        for p, U in enumerate(states):
            ctx.upload(p, field, U)
        for p in reversed(range(len(SHAPES))):
            assert np.array_equal(ctx.download(p, field), states[p]), SHAPES[p]
    rho = ctx.post_variables(7, ("rho",), field=2)["rho"]
    assert np.array_equal(rho, states[7][0])
    ctx.close()
