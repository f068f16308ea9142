"""GPU: the two-level iteration's chunks (update with restriction, coarse
product, direction by chunks of an aggregate's nodes) at their edges: one
aggregate, and aggregates below, at and above one workgroup's 256 nodes.

The solution does not depend on the preconditioner: bar 1e-8 against the
oracle's direct solve (solves to a relative residual of 1e-12).  The
Drucker-Prager material keeps the assembled matrix, where the update kernel
works by chunks; the elastic one takes the matrix-free operator, where it
does not.
"""
import ctypes

import numpy as np
import pytest

from oracle import HEX8 as O8, fem

pytestmark = pytest.mark.gpu


def limits(dev, chunks):
    from amaru_amd import _lib
    f = _lib.lib().amr_test_limits
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int]
    _lib.check(f(dev.handle, 0, chunks))


@pytest.mark.parametrize("plastic", [True, False])
@pytest.mark.parametrize("target", [40, 255, 256, 300, 700, 100000])
@pytest.mark.parametrize("precision", ["fp64", "mixed64acc"])
def test_chunks_match_direct(amaru, plastic, target, precision):
    am = amaru
    mesh = am.Mesh(am.Block([[0, 0, 0], [2.0, 1.0, 1.0]], nx=13, ny=9, nz=8, cellshape="HEX8"))
    prm = (50e6, 0.3, 0.23094, 24000.0, 0.0)
    mat = (am.DruckerPrager(E=prm[0], nu=prm[1], alpha=prm[2], kappa=prm[3], H=prm[4]) if plastic
           else am.LinearElastic(E=prm[0], nu=prm[1]))
    model = am.FEModel(mesh, [("all", am.MechSolid, mat)])
    bcs = {"x==0": dict(ux=0, uy=0, uz=0), "x==2": dict(tz=-1e3)}
    model.configure_dofs([(f, am.SurfaceBC(**c)) for f, c in bcs.items()])
    om = fem.Model(mesh.coords, mesh.conn, O8, [("LinearElastic", prm[:2])])
    om.configure_dofs([(f, fem.SurfaceBC(**c)) for f, c in bcs.items()])
    Uo, Fo = model.bc_vals([(f, am.SurfaceBC(**c)) for f, c in bcs.items()])
    U, F = Uo.copy(), Fo.copy()
    fem.solve_system(om.mount_K().tocsr(), Uo, Fo, om.nu)
    dev = am.DeviceModel(model)
    dev.set_coarse(target)
    dev.assemble()
    r = dev.solve_system(U, F, rtol=1e-12, precision=precision, precond="two_level")
    assert r["converged"]
    assert np.linalg.norm(U - Uo) <= 1e-8 * np.linalg.norm(Uo)
    assert np.linalg.norm(F - Fo) <= 1e-8 * np.linalg.norm(Fo)
    dev.close()


# chunks: the slots of their partials (0: 1,024); fewer slots than the
# aggregates have chunks of 256 nodes make chunks of 512 (1100, 8), 768 and
# 2,816 nodes, which a workgroup takes in several passes
@pytest.mark.parametrize("target,chunks", [(3, 0), (64, 0), (256, 0), (257, 0), (1100, 0), (100000, 0), (1100, 8),
                                           (1100, 4), (100000, 4), (100000, 1)])
def test_restrictions_agree(amaru, target, chunks):
    """The restriction's own kernel (elastic models) against the chunks of the
    update kernel (Drucker-Prager, not yet plastic: the same K), with
    aggregates below, at and above a workgroup's 256 nodes and, at the last,
    above the 2,048 it holds in flight.  The two iterations differ by rounding
    only, so their lengths differ by a few iterations at most; a node left out
    of a restriction costs many."""
    am = amaru
    mesh = am.Mesh(am.Block([[0, 0, 0], [2.0, 1.0, 1.0]], nx=19, ny=11, nz=10, cellshape="HEX8"))
    its, Us = [], []
    for mat in (am.LinearElastic(E=50e6, nu=0.3),
                am.DruckerPrager(E=50e6, nu=0.3, alpha=0.23094, kappa=24000.0, H=0.0)):
        model = am.FEModel(mesh, [("all", am.MechSolid, mat)])
        bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)), ("x==2", am.SurfaceBC(tz=-1e3))]
        model.configure_dofs(bcs)
        U, F = model.bc_vals(bcs)
        dev = am.DeviceModel(model)
        limits(dev, chunks)
        dev.set_coarse(target)
        dev.assemble()
        r = dev.solve_system(U, F, rtol=1e-10, precond="two_level")
        assert r["converged"]
        its.append(r["iterations"])
        Us.append(U)
        dev.close()
    assert abs(its[0] - its[1]) <= 4, its
    assert np.linalg.norm(Us[0] - Us[1]) <= 1e-8 * np.linalg.norm(Us[1])
