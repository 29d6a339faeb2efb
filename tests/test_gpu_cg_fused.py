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


def graded(model):
    """The planes in z moved apart towards the top: a rectilinear lattice."""
    z = model["xyz"][:, 2]
    model["xyz"][:, 2] = z * (1.0 + 0.4 * z / z.max())
    return model


def form_of(form, model):
    """Three layers with stiffness and mass damping, the second with lumped mass, and the element."""
    model = graded(model) if form == "graded" else model
    model["region"] = model["group"].copy()
    model["rayleigh"] = [(0.6 + 0.1 * g, 5.8e-4, 1e-4 * (g % 2), 2e-5) for g in range(3)]
    for g, p in enumerate(model["params"]):
        p["mass_type"] = g % 2
    pm = core.Mesh(model)
    element = "SSPbrick" if form == "ssp" else "stdBrick"
    return model, pm, [dict(p, element=element) for p in pm.params_for(model)], element


# every group of the product's instantiations: uniform stdBrick (16-deep tiles take the direction
# given), SSPbrick and rectilinear, at each tile depth; 19 x 10 x 21 cells cut the last tiles of
# every axis and depth
FORMS = [("box", 4), ("box", 8), ("box", 16), ("ssp", 4), ("ssp", 8), ("graded", 4), ("graded", 8)]
OPERATORS = {"K": (1.0, 0.0, 0.0), "KCM": (1.0, 20.0, 4e4)}


@pytest.mark.parametrize("op_name", sorted(OPERATORS))
@pytest.mark.parametrize("form,depth", FORMS)
def test_every_form_matches_oracle(ctx, form, depth, op_name):
    model, pm, params, element = form_of(form, box(19, 10, 21, 3))
    batch = core.Batch(ctx, pm, params, element=element, tile_depth=depth, tune=False)
    assert batch.info()["lattice"] == 1 and batch.info()["tiles"] == 6 * -(-21 // depth)
    om, op = fxo.OracleMesh(model), fxo.elastic_params(params)
    k = OPERATORS[op_name]
    b = meshes.random_vector(pm.neq, 5)
    db, dx = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq)
    for its in (1, 2, 12):
        dx.zero()
        r = batch.cg(db, dx, rtol=0.0, max_it=its, k=core.coeffs(*k))
        xo, ro = om.cg(op, b, rtol=0.0, max_it=its, lanes=64, k=fxo.coeffs(*k))
        assert r["iterations"] == ro["iterations"] == its
        assert np.max(np.abs(dx.get() - xo)) <= 1e-11 * np.max(np.abs(xo)), its
    batch.close()


@pytest.mark.parametrize("op_name", sorted(OPERATORS))
@pytest.mark.parametrize("form,depth", FORMS)
def test_every_form_in_fp32(ctx, form, depth, op_name):
    """The inner solve of the mixed CG stopped after a few iterations, before it can correct itself: an
    FP32 product is within 2e-6 of its largest entry (the operator tests' bound), carried on with the
    iteration count squared. A wrong direction entry is of the order of x."""
    model, pm, params, element = form_of(form, box(19, 10, 21, 3))
    batch = core.Batch(ctx, pm, params, element=element, tile_depth=depth, tune=False, fp32=True)
    om, op = fxo.OracleMesh(model), fxo.elastic_params(params)
    k = OPERATORS[op_name]
    b = meshes.random_vector(pm.neq, 5)
    db, dx = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq)
    for its in (1, 2, 5):
        dx.zero()
        r = batch.cg_mixed(db, dx, rtol=1e-30, inner_rtol=1e-20, max_it=its, k=core.coeffs(*k))
        assert r["iterations"] == its and r["outer_iterations"] == 1
        xo, _ = om.cg(op, b, rtol=0.0, max_it=its, lanes=64, k=fxo.coeffs(*k))
        assert np.max(np.abs(dx.get() - xo)) <= 2e-6 * its * its * np.max(np.abs(xo)), its
    batch.close()


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_direction_by_its_own_pass(ctx, fp32):
    """More chunks than the tiles form the direction for (600), few enough that the pass adds their
    partials up itself."""
    model = box(70, 70, 90)
    pm = core.Mesh(model)
    assert 600 * 2048 < pm.neq < 1024 * 2048
    params = pm.params_for(model)
    batch = core.Batch(ctx, pm, params, tune=False, fp32=fp32)
    om, op = fxo.OracleMesh(model, coloring=False), fxo.elastic_params(params)
    b = np.resize(meshes.random_vector(10007, 3), pm.neq)
    db, dx = core.DeviceArray.from_host(ctx, b), core.DeviceArray(ctx, pm.neq)
    dx.zero()
    if fp32:
        r = batch.cg_mixed(db, dx, rtol=1e-30, inner_rtol=1e-20, max_it=3)
    else:
        r = batch.cg(db, dx, rtol=0.0, max_it=3)
    xo, _ = om.cg(op, b, rtol=0.0, max_it=3, lanes=64, nthreads=8)
    assert r["iterations"] == 3
    assert np.max(np.abs(dx.get() - xo)) <= (2e-6 * 9 if fp32 else 1e-12) * np.max(np.abs(xo))
    batch.close()
