"""drn_patch_upload / drn_patch_download and drn_post_variables through the
pinned staging memory: byte for byte, for value counts that do and do not
divide into 16-byte lanes, patches below and above a staging half (8 MiB), and
several patches and fields behind each other."""
import ctypes as C

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


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_odd_counts_over_several_pieces(gpu, dtype):
    """the one-value lanes of k_host_copy across variables and reused halves"""
    ctx = hip.Context(dtype)
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    for n in ((81, 81, 81), (95, 93, 91)):
        ctx.add_patch(*n, [0] * 6, (1.0, 1.0, 1.0), [configs.BC_SLIP] * 6, np.zeros((6, configs.NPAR)))
    ctx.layout()
    rng = np.random.default_rng(4)
    states = [rng.standard_normal((5, ctx.patch_cells(p))).astype(dtype) for p in range(2)]
    for p, U in enumerate(states):
        ctx.upload(p, 1, U)
    for p, U in enumerate(states):
        assert np.array_equal(ctx.download(p, 1), U)
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_post_variables_over_several_pieces(gpu, dtype):
    """all eight quantities, more than a staging half, as one by one"""
    ctx = hip.Context(dtype)
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    ctx.add_patch(73, 75, 77, [0] * 6, (1.0, 1.0, 1.0), [configs.BC_SLIP] * 6, np.zeros((6, configs.NPAR)))
    ctx.layout()
    rng = np.random.default_rng(5)
    n = ctx.patch_cells(0)
    rho = 1.0 + 0.1 * rng.random(n)
    vel = 50.0 * rng.standard_normal((3, n))
    ctx.upload(0, 0, np.stack([rho, *(rho * vel), rho * (2.2e5 + 0.5 * (vel ** 2).sum(0))]).astype(dtype))
    together = ctx.post_variables(0)
    for name in ctx.POST_NAMES:
        assert np.array_equal(together[name], ctx.post_variables(0, (name,))[name]), name
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_pinned_buffers(gpu, dtype):
    """buffers in pinned memory, which go past the staging memory"""
    ctx = hip.Context(dtype)
    rt = C.CDLL("libamdhip64.so.7")  # the runtime the library is linked against
    rt.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    rt.hipHostFree.argtypes = [C.c_void_p]
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    shapes = [(3, 1, 1), (5, 7, 9), (33, 35, 37), (80, 81, 83)]
    for n in shapes:
        ctx.add_patch(*n, [0] * 6, (1.0, 1.0, 1.0), [configs.BC_SLIP] * 6, np.zeros((6, configs.NPAR)))
    ctx.layout()
    rng = np.random.default_rng(6)
    for p, n in enumerate(shapes):
        U = rng.standard_normal((5, int(np.prod(n)))).astype(dtype)
        h = C.c_void_p()
        assert rt.hipHostMalloc(C.byref(h), U.nbytes, 0) == 0
        a = np.frombuffer((C.c_char * U.nbytes).from_address(h.value), dtype).reshape(U.shape)
        a[:] = U
        ctx._chk(ctx.L.drn_patch_upload(ctx.h, p, 0, h), "drn_patch_upload")
        a[:] = 0
        ctx._chk(ctx.L.drn_patch_download(ctx.h, p, 0, h), "drn_patch_download")
        assert np.array_equal(a, U), n
        rt.hipHostFree(h)
    ctx.close()
