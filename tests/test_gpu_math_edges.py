"""The paired exp and erfc of the flux where their ranges end.

The pair evaluates both sides of a face without branches, the special values by
selects: each element of the pair equals the host's scalar functions (bit for
bit, NaN where they are NaN) at zeros, subnormals, infinities, NaN, the largest
values, and on both sides of every bound of either precision, whatever the
other element holds.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUNDS = {np.float64: (-745.1332191019412, -708.3964185322641, 709.782712893384, 27.5, -27.5, 1.0, -1.0),
          np.float32: (-104.0, -103.97, -87.34, 88.72284, 89.0, 10.1, -10.1, 1.0, -1.0)}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_pairs(afar, dtype):
    from afar_cudaeuler2dmixo3rk3solver_amd._lib import check, lib, ptr
    info = np.finfo(dtype)
    x = [0.0, -0.0, np.inf, -np.inf, np.nan, info.max, -info.max, info.tiny, -info.tiny, info.smallest_subnormal,
         710.0, -746.0, 1e4, -1e4]
    for b in BOUNDS[dtype]:
        b = dtype(b)
        x += [b, np.nextafter(b, dtype(np.inf)), np.nextafter(b, dtype(-np.inf))]
    rng = np.random.default_rng(1)
    # every value at even and odd places, beside every kind of partner
    x = np.concatenate([rng.permutation(np.array(x, dtype)) for _ in range(200)])
    print("case: paired exp and erfc, %s, %d arguments" % (dtype.__name__, len(x)), flush=True)
    dev, host = np.zeros((len(x), 4), dtype), np.zeros((len(x), 4), dtype)
    ct = C.c_double if dtype is np.float64 else C.c_float
    suffix = "" if dtype is np.float64 else "_f32"
    check(getattr(lib(), "afar_selftest_math" + suffix)(ptr(x, ct), ptr(dev, ct), len(x)))
    check(getattr(lib(), "afar_host_math" + suffix)(ptr(x, ct), ptr(host, ct), len(x)))
    u = np.uint64 if dtype is np.float64 else np.uint32
    same = (dev.view(u) == host.view(u)) | (np.isnan(dev) & np.isnan(host))
    assert same[:, :2].all(), (x[~same[:, :2].all(1)][:5], dev[~same[:, :2].all(1)][:5], host[~same[:, :2].all(1)][:5])
