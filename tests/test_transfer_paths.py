"""drn_patch_upload / drn_patch_download / drn_post_variables beyond the pageable
buffer on one thread: buffers that HIP can copy from or to directly, no pinned
memory left, several threads on one context, and the caller's buffer changed
right after the call (CPU: k_host_copy is carried out by the stand-in runtime when
the host waits for it)."""
import ctypes as C
import threading

import numpy as np
import pytest

import fakedev
from fakedev import run_child

# value counts that divide into 16-byte lanes and not, below and above a staging half of 8 MiB
SHAPES = [(3, 1, 1), (5, 7, 9), (40, 40, 40), (75, 75, 75), (90, 91, 93)]


def _grid(dtype, shapes=SHAPES):
    from drnum_amd import configs, hip

    ctx = hip.Context(dtype)
    ctx.set_operator(configs.RECON_UPWIND2, configs.LIM_VANALBADA)
    for n in shapes:
        ctx.add_patch(*n, [0] * 6, (1.0, 1.0, 1.0), [configs.BC_SLIP] * 6, np.zeros((6, configs.NPAR)))
    ctx.layout()
    return ctx, [np.random.default_rng(7 + p).standard_normal((5, int(np.prod(n)))).astype(dtype)
                 for p, n in enumerate(shapes)]


def _at(address, like):
    """an array over the memory at `address`"""
    buf = (C.c_char * like.nbytes).from_address(address)
    return np.frombuffer(buf, like.dtype).reshape(like.shape)


def _call(ctx, name, p, field, address):
    ctx._chk(getattr(ctx.L, name)(ctx.h, p, field, C.c_void_p(address)), name)


def pageable_child():
    for dtype in (np.float32, np.float64):
        ctx, states = _grid(dtype)
        for p, U in enumerate(states):
            a = U.copy()
            ctx.upload(p, 0, a)
            a[:] = 0
        for p, U in enumerate(states):
            assert np.array_equal(ctx.download(p, 0), U), SHAPES[p]
        ctx.close()


def direct_child():
    """pinned and device buffers are copied as they are, without staging or helper copies"""
    for dtype in (np.float32, np.float64):
        ctx, states = _grid(dtype)
        for alloc in (fakedev.fake.fake_pinned_alloc, fakedev.fake.fake_device_alloc):
            for p, U in enumerate(states):
                a, b = alloc(C.c_size_t(U.nbytes)), alloc(C.c_size_t(U.nbytes))
                _at(a, U)[:] = U
                fakedev.clear()
                _call(ctx, "drn_patch_upload", p, 1, a)
                _at(a, U)[:] = 0
                _call(ctx, "drn_patch_download", p, 1, b)
                assert np.array_equal(_at(b, U), U), SHAPES[p]
                assert not fakedev.launches("k_host_copy"), SHAPES[p]
                assert sum(c[1] for c in fakedev.launches("memcpy")) == 2 * U.nbytes
        ctx.close()


def no_pinned_child():
    for dtype in (np.float32, np.float64):
        ctx, states = _grid(dtype)
        fakedev.fake.fake_fail_pinned(1)
        for p, U in enumerate(states):
            ctx.upload(p, 0, U)
        for p, U in enumerate(states):
            assert np.array_equal(ctx.download(p, 0), U), SHAPES[p]
        ctx.post_variables(1, ("rho", "p"))
        fakedev.fake.fake_fail_pinned(0)
        ctx.close()


def threads_child():
    for dtype in (np.float32, np.float64):
        shapes = [(60, 61, 63), (75, 75, 75), (90, 91, 93), (80, 80, 80)]
        ctx, states = _grid(dtype, shapes)
        for _ in range(5):
            bad = []

            def work(p):
                ctx.upload(p, 0, states[p])
                if not np.array_equal(ctx.download(p, 0), states[p]):
                    bad.append(shapes[p])

            ts = [threading.Thread(target=work, args=(p,)) for p in range(len(shapes))]
            for t in ts:
                t.start()
            for t in ts:
                t.join()
            assert not bad, bad
        ctx.close()


@pytest.mark.parametrize("child", ["pageable_child", "direct_child", "no_pinned_child", "threads_child"])
def test_transfers(tmp_path, child):
    run_child(tmp_path, "test_transfer_paths", child)
