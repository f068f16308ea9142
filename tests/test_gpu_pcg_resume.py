"""GPU: a PCG whose stop the true residual refuses goes on from where it was.

The recursion of a member that forms its direction inside the operator (one
level: matrix-free, or assembled up to 16,384 nodes) can stop inside a step,
before the next direction is stored.  Resumed on the spent one (orthogonal to
the residual) it diverges.

``early`` asks for stops that the check of the true residual refuses
(``amr_test_early_stops``): the k-th at 1e-3^k of the right-hand side, then
the tolerance.  check_every 256 puts every stop inside the one step, 1 at a
step's end.

Bars.  Exact arithmetic gives the uninterrupted iteration: the replaced
residual differs from the recursive one by about 1e-15 of the right-hand
side, 1e-9 of itself at 1e-6, so the counts differ by rounding at the last
threshold: 3 iterations.  A change of the operator restarts the direction,
which costs at most a fresh solve: twice the count.  Solutions: relative
residual 1e-12 on a well-conditioned block, 1e-8.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def early(dev, n, rtol=1e-3):
    from amaru_amd import _lib
    f = _lib.lib().amr_test_early_stops
    f.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_double]
    _lib.check(f(dev.handle, n, rtol))


def block(am, n=(9, 5, 4)):
    mesh = am.Mesh(am.Block([[0, 0, 0], [1.8, 1.0, 0.8]], nx=n[0], ny=n[1], nz=n[2], cellshape="HEX8"))
    model = am.FEModel(mesh, [("all", am.MechSolid, am.LinearElastic(E=50e6, nu=0.3))])
    bcs = [("x==0", am.SurfaceBC(ux=0, uy=0, uz=0)), ("x==1.8", am.SurfaceBC(tz=-1e3, ty=4e2))]
    model.configure_dofs(bcs)
    return model, bcs


def solve(dev, model, bcs, **kw):
    U, F = model.bc_vals(bcs)
    r = dev.solve_system(U, F, **dict(dict(rtol=RTOL, maxiter=5000), **kw))
    assert r["converged"]
    return r, U


@pytest.mark.parametrize("operator", ["matrix_free", "assembled"])
@pytest.mark.parametrize("precond", ["jacobi", "block_jacobi", "two_level"])
@pytest.mark.parametrize("check", [1, 7, 256])
def test_refused_stops(amaru, operator, precond, check):
    model, bcs = block(amaru)
    dev = amaru.DeviceModel(model)
    dev.set_coarse(40)
    dev.assemble()
    if operator == "assembled":
        dev.assemble_M(0.0)
        dev.combine_KM(1.0, 0.0)   # the same K, handed to the assembled matrix
    kw = dict(precond=precond, check_every=check)
    r0, U0 = solve(dev, model, bcs, **kw)
    assert r0["replacements"] == 1 and not r0["fallback"]
    for n in (1, 2):
        early(dev, n)
        r, U = solve(dev, model, bcs, **kw)
        assert r["replacements"] == n + 1
        # the second refused stop ends the use of the matrix-free operator
        changed = operator == "matrix_free" and n == 2
        assert r["fallback"] == changed
        if changed:
            assert r["iterations"] <= 2 * r0["iterations"]
        else:
            assert abs(r["iterations"] - r0["iterations"]) <= 3
        assert np.linalg.norm(U - U0) <= 1e-8 * np.linalg.norm(U0)
    early(dev, 0)
    r, U = solve(dev, model, bcs, **kw)
    assert r["iterations"] == r0["iterations"] and np.array_equal(U, U0)
    dev.close()


@pytest.mark.parametrize("graphs", [False, True])
def test_change_of_operator_in_a_pool(amaru, graphs):
    """Members that leave the matrix-free operator while others go on: the
    launches' lists follow (tiles, partials, chunks); every member ends as
    alone, bit for bit."""
    from amaru_amd import pool as P
    specs = [("jacobi", 2, (9, 5, 4)), ("two_level", 2, (13, 7, 6)), ("jacobi", 0, (17, 6, 5)),
             ("two_level", 0, (9, 5, 4)), ("block_jacobi", 1, (11, 5, 4)), ("two_level", 1, (8, 8, 7))]
    devs = []
    for precond, n, size in specs:
        model, bcs = block(amaru, size)
        dev = amaru.DeviceModel(model)
        dev.set_coarse(40)
        early(dev, n)
        U, F = model.bc_vals(bcs)
        dev.stage_begin(U, F)
        devs.append((dev, dev.opts(rtol=RTOL, precond=precond, maxiter=5000, check_every=16)))
    alone = []
    for dev, o in devs:
        dev.increment_begin(1.0, 1.0, False)
        r = dev.nr_iteration(1, o)
        assert r["status"] == 0
        alone.append((r["pcg_iterations"], r["replacements"], r["fallback"], dev.stage_get(last=True)))
        dev.increment_reject()
    pool = P.Pool(max_members=len(devs), check_every=16)
    pool.set_graphs(graphs)
    for dev, o in devs:
        dev.increment_begin(1.0, 1.0, False)
        dev.nr_prepare(1)
        pool.attach(dev)
        pool.add(dev, o)
    fin = {}
    for _ in range(2000):
        fin.update(pool.step())
        if len(fin) == len(devs):
            break
    for (dev, o), (its, rep, fb, (dU, dF)) in zip(devs, alone):
        si = fin[dev.handle.value]
        assert si.converged and si.iterations == its and si.refinements == rep and bool(si.fallback) == fb
        dev.nr_finish(si)
        gU, gF = dev.stage_get(last=True)
        assert np.array_equal(gU, dU) and np.array_equal(gF, dF)
    assert [a[2] for a in alone] == [True, True, False, False, False, False]
    for dev, o in devs:
        dev.close()
    pool.close()
