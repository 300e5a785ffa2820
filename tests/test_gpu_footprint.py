"""The served solves' estimate of a solver's device memory against the memory
pool's own count: never below it, and at most a tenth (and a MiB) above."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

USED_NOW = 7  # hipMemPoolAttrUsedMemCurrent


def _pool_used():
    L = C.CDLL("libamdhip64.so.7", mode=C.RTLD_GLOBAL)  # the runtime the library is linked against
    pool, used = C.c_void_p(), C.c_uint64()
    assert L.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    assert L.hipMemPoolGetAttribute(pool, USED_NOW, C.byref(used)) == 0
    return used.value


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["quads", "triangles and quads", "periodic triangles"])
def test_estimate(afar, kind, precision):
    print("case: device memory of %s, %s" % (kind, precision), flush=True)
    from afar_cudaeuler2dmixo3rk3solver_amd import cases
    from afar_cudaeuler2dmixo3rk3solver_amd.serve import footprint_bytes
    mesh, W0 = (cases.corner_case(nx=400, ny=200) if kind == "quads" else
                cases.riemann_case(n=250) if kind == "triangles and quads" else cases.vortex_case(n=200))
    sc = afar.schemes(cOrder=7, fOrder=2, precision=precision)
    mesh.precompute(sc, gpu=True)
    before = _pool_used()
    gpu = afar.BasicCUDASolver(mesh, sc, W0)
    gpu.evolve_auto(1)
    gpu.conserved()
    gpu.write_field()
    used = _pool_used() - before
    gpu.close()
    estimate = footprint_bytes(mesh, precision)
    print("  used %.2f MiB, estimated %.2f MiB" % (used / 2 ** 20, estimate / 2 ** 20), flush=True)
    assert used <= estimate <= 1.1 * used + (1 << 20)
