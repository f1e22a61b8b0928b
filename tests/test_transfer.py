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
