"""GPU: a model that has no room for its matrix-free operator does without.

The operator's element data are the model's to give back: an allocation that
finds no memory (``amr_test_model_bytes``: a limit on the bytes of one model)
takes them, at creation and later, and the solves go on with the assembled
matrix.  The limits lie 100 kB below what the model would hold with the
element data (more than 200 kB here, and each operation needs more than 100 kB
after they are there), so that each operation fails without giving back.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHORT = 100_000


@pytest.fixture
def limit():
    from amaru_amd import _lib
    f = _lib.lib().amr_test_model_bytes
    f.argtypes, f.restype = [ctypes.c_int64], None
    yield f
    f(-1)


def problem(am):
    mesh = am.Mesh(am.Block([[0, 0, 0], [1.8, 1.0, 0.8]], nx=14, ny=9, nz=8, cellshape="HEX8"))
    model = am.FEModel(mesh, [("all", am.MechSolid(rho=2000.0), am.LinearElastic(E=50e6, nu=0.3))])
    bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)), ("x==1.8", am.SurfaceBC(tz=-1e3))]
    model.configure_dofs(bcs)
    return model, bcs


def solve(dev, model, bcs, assembled=False, **kw):
    dev.assemble()
    if assembled:
        dev.assemble_M(0.0)
        dev.combine_KM(1.0, 0.0)
    U, F = model.bc_vals(bcs)
    assert dev.solve_system(U, F, **kw)["converged"]
    return U


def two_level(dev, model, bcs):
    dev.set_coarse(40)
    solve(dev, model, bcs, precond="two_level")


OPS = {"two_level": two_level,
       "mass": lambda dev, model, bcs: dev.assemble_M(0.0),
       "recovery": lambda dev, model, bcs: dev.nodal_values()}


def test_creation(amaru, limit):
    model, bcs = problem(amaru)
    free = amaru.DeviceModel(model)
    with_mf = free.device_bytes()
    matrix_free, assembled = solve(free, model, bcs), solve(free, model, bcs, assembled=True)
    assert not np.array_equal(matrix_free, assembled)
    limit(with_mf - SHORT)
    dev = amaru.DeviceModel(model)
    assert dev.device_bytes() < with_mf - 2 * SHORT
    assert np.array_equal(solve(dev, model, bcs), assembled)
    dev.close()
    # far too little memory is still refused
    limit(with_mf // 4)
    with pytest.raises(amaru_error()) as e:
        amaru.DeviceModel(model)
    assert e.value.code == -7
    limit(-1)
    assert np.array_equal(solve(free, model, bcs), matrix_free)
    free.close()


def amaru_error():
    from amaru_amd import _lib
    return _lib.AmaruError


@pytest.mark.parametrize("op", sorted(OPS))
def test_later_allocation(amaru, limit, op):
    model, bcs = problem(amaru)
    free = amaru.DeviceModel(model)
    before = free.device_bytes()
    OPS[op](free, model, bcs)
    total = free.device_bytes()
    assert total - before > SHORT
    dev = amaru.DeviceModel(model)
    limit(total - SHORT)
    OPS[op](dev, model, bcs)
    assert dev.device_bytes() <= total - SHORT
    limit(-1)
    # the assembled matrix from now on
    assert np.array_equal(solve(dev, model, bcs), solve(free, model, bcs, assembled=True))
    dev.close()
    free.close()
