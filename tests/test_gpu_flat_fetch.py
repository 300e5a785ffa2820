"""Face states and limiters fetched after plain steps hold every cell.

The FP64 reconstruction leaves out the face states and limiters of cells of
uniform temperature, which the face pass forms itself; fetch completes the
arrays with what the last reconstruction started from.  A twin solver takes
the last step stage by stage, where everything is stored: after host and
device time steps, a device step past the end time, a time step asked for,
a profile and a restart in between, both
arrays equal the twin's bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _pulse(xy):
    W = np.empty((len(xy), 4))
    W[:] = (1.0, 0.2, 0.0, 1.4)
    W[np.hypot(xy[:, 0] - 0.3, xy[:, 1] - 0.5) < 0.15] = (2.5, 0.3, 0.0, 2.0)
    return W


def _arrays(gpu, mesh):
    nf = mesh.sizes()["nf"]
    return gpu.fetch("fv", np.float64, (nf, 2, 4)), gpu.fetch("lim", np.float64, (mesh.nc, 4))


@pytest.mark.parametrize("first_order", [False, True])
@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("how", ["host", "device", "past the end", "past the end, then dt", "device, then dt",
                                 "residual", "profile", "restart"])
def test_fetch_after_steps(afar, how, lanes, first_order):
    print("case: fv and lim after %s, lanes %d, first-order boundary %s" % (how, lanes, first_order), flush=True)
    from afar_cudaeuler2dmixo3rk3solver_amd import cases
    mesh, _ = cases.riemann_case(n=33)
    sc = afar.schemes(cOrder=7, fOrder=2, maxCo=0.4, boundaryFirstOrder=first_order, reconLanes=lanes)
    mesh.precompute(sc)
    xy = np.zeros((mesh.nc, 2))
    xy[mesh.permutation()] = mesh.cells()[0][:mesh.nc]
    W0 = _pulse(xy)
    gpu, twin = afar.BasicCUDASolver(mesh, sc, W0), afar.BasicCUDASolver(mesh, sc, W0)
    U0 = gpu.conserved()
    gpu.evolve_auto(4)
    twin.evolve_auto(4)
    # the last reconstruction: the third stage of a fifth step, or one more on the state as it is
    if how in ("host", "device", "device, then dt", "restart"):
        dt = twin.set_delta_t()
        if how == "host":
            gpu.evolve(gpu.set_delta_t())
        else:
            gpu.evolve_auto(1)
        for s in range(3):
            twin.run_stage(3, dt, s)
    else:
        if how.startswith("past the end"):
            gpu.set_time(1.0, 1.0)
            gpu.evolve_auto(2)
        elif how == "residual":
            gpu.residual_norm()
        else:
            gpu.profile(2)
        twin.run_stage(2)
    if how.endswith("then dt"):
        assert gpu.set_delta_t() > 0.0
    if how == "restart":
        gpu.set_conserved(U0)
    fv, lim = _arrays(gpu, mesh)
    fv1, lim1 = _arrays(twin, mesh)
    T = twin.fetch("W", np.float64, (mesh.nc + twin.nb, 4))[:mesh.nc, 3]
    assert 0 < (np.abs(T - 1.4) < 1e-12).sum() < mesh.nc
    assert np.array_equal(lim, lim1)
    assert np.array_equal(fv, fv1)
    gpu.close()
    twin.close()
