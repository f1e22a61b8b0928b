"""A state's way to the device and back (``fds_set_state``, ``fds_get_state``) around the sizes
where it changes: the runtime's copies with the conversion on the host below 2^20 values, chunks
of 2^18 through pinned memory with the conversion on the device from there on.  The roundings are
IEEE's, so every bit is known."""
import ctypes as ct

import numpy as np
import pytest

from pyfds_amd import _native as nat

pytestmark = pytest.mark.gpu

DP = ct.POINTER(ct.c_double)


def _values(n):
    rng = np.random.default_rng(n)
    v = rng.standard_normal(n) * 10.0 ** rng.integers(-60, 60, n)
    special = [0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40, -1e-45, 1e-50, 3.5e38, 1 + 2.0 ** -24]
    for at in (0, n // 2, n - len(special)):
        v[at:at + len(special)] = special
    return v


@pytest.mark.parametrize('form', ['fp64', 'fp32', 'fp32_kahan'])
@pytest.mark.parametrize('nx, ny', [(37, 3), (1 << 10, (1 << 10) - 1), (1 << 10, 1 << 10),
                                    (1031, 1021), (1 << 11, 3 << 8), (2049, 1537)])
def test_state_round_trip_rounds_like_ieee(form, nx, ny):
    lib = nat.load()
    n = nx * ny
    v = _values(n)
    got = np.empty(n)
    ctx = ct.c_void_p()
    nat.check(lib.fds_create(ct.byref(ctx), nat.ACOUSTIC2D, nat.FORMS[form], nx, ny, 0))
    try:
        for _ in range(2):                  # new buffers, then the same again
            nat.check(lib.fds_set_state(ctx, 0, v.ctypes.data_as(DP), n))
            got[:] = 7.0
            nat.check(lib.fds_get_state(ctx, 0, got.ctypes.data_as(DP), n))
            want = v
            if form != 'fp64':
                with np.errstate(over='ignore', invalid='ignore'):
                    x = v.astype(np.float32)
                    want = x.astype(np.float64)
                    if form == 'fp32_kahan':
                        c = (want - v).astype(np.float32)
                        want = want - c.astype(np.float64)
            np.testing.assert_array_equal(got, want)
            np.testing.assert_array_equal(np.signbit(got[want == 0]), np.signbit(want[want == 0]))
    finally:
        lib.fds_destroy(ctx)


def test_large_contexts_share_the_transfer_workspace():
    """A context's first large transfer takes no device memory of its own once another's has been,
    and the last context's end gives the workspace back.  (The first round loads the kernels, which
    the runtime keeps.)"""
    import torch
    lib = nat.load()
    nx = ny = 1 << 10
    v = np.random.default_rng(0).standard_normal(nx * ny)
    got = np.empty_like(v)

    def free():
        torch.cuda.synchronize()
        return torch.cuda.mem_get_info()[0]

    for _ in range(2):
        ctxs, before = [], free()
        try:
            for i in range(4):
                ctx = ct.c_void_p()
                nat.check(lib.fds_create(ct.byref(ctx), nat.ACOUSTIC2D, nat.FORMS['fp32'], nx, ny,
                                         0))
                ctxs.append(ctx)
                held = free()
                nat.check(lib.fds_set_state(ctx, 0, v.ctypes.data_as(DP), v.size))
                nat.check(lib.fds_get_state(ctx, 0, got.ctypes.data_as(DP), v.size))
                np.testing.assert_array_equal(got, v.astype(np.float32))
                if i:
                    assert held - free() < 4 << 20
        finally:
            for ctx in ctxs:
                lib.fds_destroy(ctx)
    assert before - free() < 4 << 20


def test_large_transfers_of_several_threads():
    import threading
    lib = nat.load()
    nx, ny = 1031, 1021
    errors = []

    def work(seed, form):
        try:
            v = np.random.default_rng(seed).standard_normal(nx * ny)
            got = np.empty_like(v)
            ctx = ct.c_void_p()
            nat.check(lib.fds_create(ct.byref(ctx), nat.ACOUSTIC2D, nat.FORMS[form], nx, ny, 0))
            for _ in range(3):
                nat.check(lib.fds_set_state(ctx, 0, v.ctypes.data_as(DP), v.size))
                nat.check(lib.fds_get_state(ctx, 0, got.ctypes.data_as(DP), v.size))
                np.testing.assert_array_equal(got, v if form == 'fp64' else v.astype(np.float32))
            lib.fds_destroy(ctx)
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i, ('fp64', 'fp32')[i % 2])) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
