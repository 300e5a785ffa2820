"""Flat cells across a periodic seam, whose temperatures the BVD test forms.

A blast beside the seam of a periodic mesh: limited cells on one side of it see
flat neighbours on the other, whose centres are shifted, and flat cells within
a flagged extended stencil are limited themselves.  Steps equal the oracle bit
for bit.
"""
import numpy as np
import pytest

from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("x0", [0.1, 9.95])
def test_blast_at_the_seam(afar, lanes, x0):
    print("case: blast at x = %g of a periodic mesh, lanes %d" % (x0, lanes), flush=True)
    from afar_cudaeuler2dmixo3rk3solver_amd import cases
    mesh, _ = cases.vortex_case(n=40, split_p=0.0)
    sc = afar.schemes(cOrder=7, fOrder=2, maxCo=0.4, reconLanes=lanes)
    mesh.precompute(sc)
    xy = np.zeros((mesh.nc, 2))
    xy[mesh.permutation()] = mesh.cells()[0][:mesh.nc]
    W0 = np.empty((mesh.nc, 4))
    W0[:] = (1.0, 0.0, 0.0, 1.4)
    W0[np.hypot(xy[:, 0] - x0, xy[:, 1] - 5.0) < 1.3] = (8.0, 0.2, 0.0, 4.0)
    gpu = afar.BasicCUDASolver(mesh, sc, W0)
    orc = O.OracleState(mesh.reference_arrays(sc, W0), sc.R, sc.Cv)
    for _ in range(20):
        dt = gpu.set_delta_t()
        assert dt == orc.adjust_time_step(sc.maxCo)
        gpu.evolve(dt)
        orc.evolve(dt)
    assert np.array_equal(gpu.conserved()[mesh.permutation()], orc.U)
    gpu.close()
