"""The CG iteration's fused kernels at the sizes where they can go wrong: equations around the ends
of the dots' 2048-entry chunks, tiles cut by the lattice's end, tied and general batches (whose
product and dot stay apart), and more chunks than a workgroup reduces by itself.

A fixed number of iterations is compared with the oracle's CG in the same dot order (lanes 64):
both sides round differently only inside the operator, 1e-15 per product, and CG carries such a
difference on with a factor of about the iteration count squared: 1e-11 of the largest entry
after 12 iterations is a wide bound.
"""
import numpy as np
import pytest

from femorax_amd import core
from femorax_amd import synthetic as S
from oracle import fxo
from tests import meshes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = core.Context(0)
    yield c
    c.close()


def box(nx, ny, nz, layers=1):
    xyz, conn, ek = S.grid(nx, ny, nz, 1.0, 0.9, 1.1)
    params = [dict(E=3e7 * (1 + g), nu=0.3, rho=2000.0, b=(0.0, 0.0, -2e4), mass_type=0) for g in range(layers)]
    return dict(nnode=len(xyz), xyz=xyz, nelem=len(conn), conn=conn,
                group=np.minimum(ek * layers // nz, layers - 1).astype(np.int32), fix=S.fixed_base(nx, ny),
                tie=np.zeros((0, 3), np.int32), params=params, grid=(nx, ny, nz), h=(1.0, 0.9, 1.1))


CASES = {
    "one_element": lambda: box(1, 1, 1),                # 12 equations: one partial chunk
    "one_tile_and_a_cell": lambda: box(9, 8, 4, 2),     # one shared plane, a cut tile
    "chunk_less_3": lambda: box(10, 2, 62),             # 6138 equations: six short of three chunks
    "chunk_plus": lambda: box(13, 9, 13, 3),            # 5460: the last chunk partly shared equations
    "tied": lambda: meshes.column(10),                  # tied sets behind the shared equations
    "general": lambda: meshes.distorted_box(6),
    "rows_of_tiles": lambda: box(33, 17, 25, 2),        # edges and corners of 4 and 8 tiles
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_fixed_iterations_match_oracle(ctx, name):
    model = CASES[name]()
    pm = core.Mesh(model)
    params = pm.params_for(model)
    batch = core.Batch(ctx, pm, params)
    om, op = fxo.OracleMesh(model), fxo.elastic_params(params)
    b = meshes.random_vector(pm.neq, 5)
    db, dx = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq)
    for its in (1, 2, 12):
        dx.zero()
        r = batch.cg(db, dx, rtol=0.0, max_it=its)
        xo, ro = om.cg(op, b, rtol=0.0, max_it=its, lanes=64)
        assert r["iterations"] == ro["iterations"]
        got = dx.get()
        assert np.max(np.abs(got - xo)) <= 1e-11 * np.max(np.abs(xo)), name
        assert abs(r["final_residual"] - ro["final_residual"]) <= 1e-10 * r["rhs_norm"]
    batch.close()


def test_totals_by_their_own_launch(ctx):
    """More chunk partials than every workgroup adds up by itself (kInlineParts = 1024)."""
    model = box(89, 88, 89)
    pm = core.Mesh(model)
    assert pm.neq > 1024 * 2048
    params = pm.params_for(model)
    batch = core.Batch(ctx, pm, params, tune=False)
    om, op = fxo.OracleMesh(model, coloring=False), fxo.elastic_params(params)
    b = np.resize(meshes.random_vector(10007, 3), pm.neq)
    db, dx = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq)
    dx.zero()
    r = batch.cg(db, dx, rtol=0.0, max_it=3)
    xo, ro = om.cg(op, b, rtol=0.0, max_it=3, lanes=64, nthreads=8)
    assert r["iterations"] == ro["iterations"] == 3
    assert np.max(np.abs(dx.get() - xo)) <= 1e-12 * np.max(np.abs(xo))
    batch.close()


def test_stop_is_seen_without_iterations_to_spare(ctx):
    """The host stops launching once the device reports the stop: solves that need 0, 1 and many
    iterations, one after another on the same batch, each with its own counts."""
    model = box(9, 8, 4, 2)
    pm = core.Mesh(model)
    batch = core.Batch(ctx, pm, pm.params_for(model))
    b = meshes.random_vector(pm.neq, 5)
    db, dx, zero = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq), core.DeviceArray(ctx, pm.neq)
    zero.zero()
    dx.zero()
    r = batch.cg(db, dx, rtol=1e-10)
    assert r["converged"] and r["iterations"] > 20
    again = batch.cg(db, dx, rtol=1e-9)  # starts at the solution
    assert again["converged"] and again["iterations"] == 0
    dx.zero()
    assert batch.cg(zero, dx)["iterations"] == 0  # b = 0
    dx.zero()
    assert batch.cg(db, dx, rtol=0.0, max_it=0)["iterations"] == 0
    dx.zero()
    assert batch.cg(db, dx, rtol=0.0, max_it=1)["iterations"] == 1
    dx.zero()
    assert batch.cg(db, dx, rtol=1e-10)["iterations"] == r["iterations"]
    batch.close()


@pytest.mark.parametrize("name", ["one_element", "chunk_plus", "tied", "general", "rows_of_tiles"])
def test_gmres_steps_match_oracle(ctx, name):
    """The Arnoldi steps kept on the device: the first steps, a whole cycle, one step past it, and a
    stop inside a cycle with steps still queued (the same counts and residuals as the oracle's
    host loop, whose dots have the same order). Two Gram-Schmidt passes keep the basis orthogonal
    to rounding, so x moves by about the condition number of the projected system times 1e-16."""
    model = CASES[name]()
    pm = core.Mesh(model)
    params = pm.params_for(model)
    batch = core.Batch(ctx, pm, params, gmres=True)
    om, op = fxo.OracleMesh(model), fxo.elastic_params(params)
    b = meshes.random_vector(pm.neq, 5)
    db, dx = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq)
    for its in (1, 2, 30, 31, 37):
        if its > pm.neq:
            continue
        dx.zero()
        r = batch.gmres(db, dx, rtol=1e-12, max_it=its)
        xo, ro = om.gmres(op, b, rtol=1e-12, max_it=its)
        assert r["iterations"] == ro["iterations"] and r["converged"] == ro["converged"]
        assert np.max(np.abs(dx.get() - xo)) <= 1e-9 * np.max(np.abs(xo)), (name, its)
    dx.zero()
    r = batch.gmres(db, dx, rtol=0.3)
    _, ro = om.gmres(op, b, rtol=0.3)
    assert r["converged"] and r["iterations"] == ro["iterations"]
    batch.close()
