"""The work a program has this library do, as cases that can be timed and compared: operator
products on structured and distorted meshes, Krylov solves, internal forces, explicit and
implicit steps, and the pool of soil columns, each through the public calls of femorax_amd.core.

A program keeps its vectors as GPU tensors (Vec hands their addresses to the library), one
context, and one batch per model. The operator products are stream-ordered, as a caller that
queues kernels of its own runs them; every other call is blocking.

Kinds of case:
  apply     y = K_eff x on an elastic batch (box, graded box or distorted box; stdBrick or
            SSPbrick; FP64 or FP32)
  solve     K_eff x = b by CG + Jacobi, FP32 CG in FP64 refinement, or GMRES(30) + Jacobi
  force     the elastic internal force with Rayleigh damping on the tied soil column
  explicit  CentralDifference steps of a box with Lysmer dashpots and a point source
  pimy      one Newton iteration's element work on a multi-surface soil: the force with the
            return map and damping at (u, v), the tangents kept, one product on them
  newmark   Newmark + Newton + CG steps of a 3D multi-surface soil column under a base record
  columns   a round of site-response columns: admitted, run to their end, fetched, removed
"""
import functools
import math

import numpy as np
import torch

from femorax_amd import core
from femorax_amd import synthetic as S

DEV = "cuda:0"


def listed():
    return [
        # the headline product: the layered 128^3 soil box (6.4 M equations), stiffness only
        dict(name="apply box 128", kind="apply", mesh="box", nx=128, ny=128, nz=128, element="stdBrick", bits=64,
             mass=False),
        # a mesh that follows terrain or a structure: no element is a box; the dynamic operator
        # K + C + M of an implicit step with consistent mass
        dict(name="apply distorted 72", kind="apply", mesh="distorted", nx=72, ny=72, nz=72, element="stdBrick", bits=64,
             mass=True),
        # the smallest solve a server admits often: the 16^3 static block to rtol 1e-8 (latency)
        dict(name="solve block 16", kind="solve", method="cg", nx=16, ny=16, nz=16, layers=1, rtol=1e-8, max_it=10000),
        # the largest static block a server admits
        dict(name="solve block 48", kind="solve", method="cg", nx=48, ny=48, nz=48, layers=1, rtol=1e-8, max_it=10000),
        # CG on the large layered box, a fixed number of iterations of its 2,000
        dict(name="solve box 128", kind="solve", method="cg", nx=128, ny=128, nz=128, layers=8, rtol=0.0, max_it=25),
        # the mixed-precision solve of a mid-size layered box to rtol 1e-8
        dict(name="solve mixed 40", kind="solve", method="mixed", nx=40, ny=40, nz=40, layers=8, rtol=1e-8,
             max_it=100000),
        # GMRES(30) on the Newmark operator of the tied 40^3 column, 20 iterations
        dict(name="gmres column 40", kind="solve", method="gmres", nx=40, ny=40, nz=40, layers=0, rtol=0.0, max_it=20),
        # the elastic force with damping of an explicit step on the tied 40^3 column
        dict(name="force column 40", kind="force", n=40),
        # explicit wave propagation, a batch of time steps between two outputs
        dict(name="explicit box 100", kind="explicit", nx=100, ny=100, nz=50, steps=20),
        # a Newton iteration's element work on the 40^3 multi-surface soil column, yielding
        dict(name="pimy column 40", kind="pimy", n=40),
        # two implicit steps of a small 3D soil column (the per-model analysis)
        dict(name="newmark column 8", kind="newmark", n=8, nz=16, steps=2),
        # one round of 256 site-response columns of 20 to 400 m
        dict(name="columns 256", kind="columns", ncol=256, steps=20, nmin=20, nmax=400, mixed=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box_size(rng, lo, hi):
    """nx, ny, nz with lo..hi^3 cells in all, each side within a factor 2 of the others."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    f, g = (math.exp(rng.uniform(-0.35, 0.35)) for _ in range(2))
    side = [max(2, int(n * f)), max(2, int(n * g)), max(2, int(n / (f * g)))]
    while side[0] * side[1] * side[2] > hi ** 3:
        side[side.index(max(side))] -= 1
    return dict(nx=side[0], ny=side[1], nz=side[2])


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "solve", "solve", "solve", "force", "explicit", "pimy", "newmark",
                       "columns"])
    if kind == "apply":
        mesh = rng.choice(["box", "box", "graded", "distorted"])
        element = "SSPbrick" if mesh != "graded" and rng.random() < 0.25 else "stdBrick"
        size = _box_size(rng, 8, 72 if mesh == "distorted" else 112)
        return dict(kind=kind, mesh=mesh, element=element, bits=rng.choice([64, 64, 32]), mass=rng.random() < 0.5, **size)
    if kind == "solve":
        method = rng.choice(["cg", "cg", "mixed", "gmres"])
        if method == "gmres":
            n = _log_int(rng, 6, 40)
            return dict(kind=kind, method=method, nx=n, ny=n, nz=n, layers=0, rtol=0.0, max_it=rng.randint(5, 35))
        if method == "cg" and rng.random() < 0.4:
            return dict(kind=kind, method=method, layers=rng.randint(1, 8), rtol=0.0, max_it=rng.randint(5, 25),
                        **_box_size(rng, 48, 112))
        return dict(kind=kind, method=method, layers=rng.choice([1, 3]), rtol=1e-8, max_it=100000,
                    **_box_size(rng, 8, 40 if method == "mixed" else 48))
    if kind == "force":
        return dict(kind=kind, n=_log_int(rng, 4, 40))
    if kind == "explicit":
        return dict(kind=kind, steps=rng.randint(3, 20), **_box_size(rng, 10, 79))
    if kind == "pimy":
        return dict(kind=kind, n=_log_int(rng, 4, 40))
    if kind == "newmark":
        return dict(kind=kind, n=rng.randint(1, 8), nz=rng.randint(8, 24), steps=rng.randint(1, 3))
    return dict(kind=kind, ncol=_log_int(rng, 8, 256), steps=rng.randint(5, 20), nmin=20, nmax=rng.randint(40, 400),
                mixed=rng.random() < 0.3)


# ---- models ----------------------------------------------------------------------------------


class Vec:
    """A program's GPU vector: a tensor whose address the library's calls take."""

    def __init__(self, tensor):
        self.t = tensor
        self.n = tensor.numel()
        self.ptr = tensor.data_ptr()

    def zero(self):
        core._check(core.lib().fx_memset0(context().h, self.ptr, self.t.numel() * self.t.element_size()), context())


def vec(a, dtype=torch.float64):
    return Vec(torch.as_tensor(a).to(device=DEV, dtype=dtype).contiguous())


def zeros(n, dtype=torch.float64):
    return Vec(torch.zeros(n, device=DEV, dtype=dtype))


@functools.lru_cache(maxsize=None)
def context():
    ctx = core.Context(0)
    ctx.set_stream_ordered(True)
    return ctx


def _layers(nz, layers):
    return np.minimum(np.arange(nz) * layers // nz, layers - 1).astype(np.int32)


@functools.lru_cache(maxsize=3)
def _box(mesh, nx, ny, nz, layers):
    """A box of 1 m cells, its base fixed, and its compiled mesh; graded: the heights grow with
    depth; distorted: the interior nodes moved by up to 0.2 m."""
    xyz, conn, ek = S.grid(nx, ny, nz, 1.0, 1.0, 1.0)
    if mesh == "graded":
        h = 1.0 + 0.5 * np.linspace(1.0, 0.0, nz)
        z = np.concatenate([[0.0], np.cumsum(h)])
        xyz[:, 2] = z[np.rint(xyz[:, 2]).astype(np.int64)]
    if mesh == "distorted":
        inner = np.all((xyz > 0) & (xyz < np.array([nx, ny, nz])), axis=1)
        rng = np.random.default_rng(nx + 1000 * ny + 1000000 * nz)
        xyz[inner] += 0.2 * rng.uniform(-1.0, 1.0, size=(int(inner.sum()), 3))
    model = dict(nnode=len(xyz), xyz=xyz, nelem=len(conn), conn=conn, group=_layers(nz, layers)[ek],
                 fix=S.fixed_base(nx, ny), tie=np.zeros((0, 3), np.int32), grid=(nx, ny, nz), h=(1.0, 1.0, 1.0))
    return model, core.Mesh(model)


@functools.lru_cache(maxsize=3)
def _column(n, lumped):
    """The tied soil column n^3 of the operator benchmarks (two Rayleigh regions)."""
    model = S.reference_column(n, lumped=lumped)
    return model, core.Mesh(model)


@functools.lru_cache(maxsize=3)
def _soil(n, nz):
    """A tied column n x n x nz of 1 m cells in up to ten layers."""
    model = S.soil_column(nz, 1.0, nx=n, ny=n, layer_of=lambda ek: _layers(nz, min(10, nz))[ek])
    return model, core.Mesh(model)


@functools.lru_cache(maxsize=2)
def _wave_box(nx, ny, nz):
    """The explicit box of 5 m cells, 10 layers, free on top, Lysmer dashpots elsewhere."""
    model = S.config_c3(nx, ny, nz)
    return model, core.Mesh(model)


def _soil_params(rng, layers, mass=False):
    """E log-uniform in 20-200 MPa, nu in 0.25-0.45 per layer; with damping for dynamic operators."""
    out = []
    for _ in range(layers):
        p = dict(E=float(np.exp(rng.uniform(np.log(20e6), np.log(200e6)))), nu=float(rng.uniform(0.25, 0.45)), rho=2000.0,
                 b=(0.0, 0.0, -2000.0 * 9.81), mass_type=0)
        if mass:
            p["rayleigh"] = (0.6, 5.8e-4, 0.0, 0.0)
        out.append(p)
    return out


def _column_params(rng, model, mesh):
    """Per parameter set, the column's materials with moduli within 20% of the benchmark's."""
    params = [dict(p, E=p["E"] * float(rng.uniform(0.8, 1.2))) for p in model["params"]]
    return [params[g] for g in mesh.param_group]


def _field(rng, model, mesh, amplitude, wave):
    """A smooth displacement-like field of random phases at the equations: amplitude in m, wave in m."""
    x = model["xyz"]
    out = np.zeros(mesh.neq)
    eqs = mesh.node_eq.reshape(-1, 3)[mesh.node_rank]
    for d in range(3):
        ph = rng.uniform(0.0, 2.0 * np.pi, 3)
        k = 2.0 * np.pi / wave * rng.uniform(0.7, 1.3, 3)
        f = amplitude * np.sin(k[2] * x[:, 2] + ph[2]) * (1.0 + 0.3 * np.sin(k[0] * x[:, 0] + ph[0]) *
                                                         np.sin(k[1] * x[:, 1] + ph[1]))
        m = eqs[:, d] >= 0
        out[eqs[m, d]] = f[m]
    return out


def _coeffs(case):
    """The operator's coefficients (stiffness, damping, mass)."""
    if case["kind"] == "apply":
        return (1.0, 2e3, 1.6e7) if case["mass"] else (1.0, 0.0, 0.0)
    if case["kind"] == "solve" and case["method"] == "gmres":  # Newmark, dt = 1e-3
        return (1.0, 2e3, 4e6)
    return (1.0, 0.0, 0.0)


def _inputs(case, seed):
    """model, mesh, parameters and host input arrays of an elastic case (from the seed alone)."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "apply":
        layers = min(8, case["nz"])
        model, mesh = _box(case["mesh"], case["nx"], case["ny"], case["nz"], layers)
        params = [dict(p, element=case["element"]) for p in _soil_params(rng, layers, case["mass"])]
        x = rng.standard_normal(mesh.neq)
        return model, mesh, params, dict(x=x.astype(np.float32) if case["bits"] == 32 else x)
    if kind == "solve" and case["layers"] == 0:
        model, mesh = _column(case["nx"], False)
        return model, mesh, _column_params(rng, model, mesh), dict(b=rng.uniform(0.5, 1.5, mesh.neq))
    if kind == "solve":
        model, mesh = _box("box", case["nx"], case["ny"], case["nz"], case["layers"])
        t = 1e4 * (1.0 + 0.5 * rng.uniform(-1.0, 1.0, (case["ny"] + 1) * (case["nx"] + 1)))
        return model, mesh, _soil_params(rng, case["layers"]), dict(b=mesh.to_equations(_traction(model, t)))
    if kind == "force":
        model, mesh = _column(case["n"], True)
        return model, mesh, _column_params(rng, model, mesh), dict(u=_field(rng, model, mesh, 1e-4, 10.0),
                                                             v=_field(rng, model, mesh, 1e-3, 10.0))
    model, mesh = _wave_box(case["nx"], case["ny"], case["nz"])
    params = [dict(p, E=p["E"] * float(rng.uniform(0.8, 1.0))) for p in mesh.params_for(model)]
    um = _field(rng, model, mesh, 1e-3, 60.0)
    return model, mesh, params, dict(u=um, um=0.999 * um, dash=mesh.to_equations(model["dashpots"]),
                                     load=1e6 * rng.standard_normal(case["steps"]))


def _traction(model, t):
    """Consistent nodal loads of the traction t (per top node, downwards) on the top face."""
    nx, ny, nz = model["grid"]
    F = np.zeros((model["nnode"], 3))
    q = t.reshape(ny + 1, nx + 1)
    quad = 0.25 * (q[:-1, :-1] + q[:-1, 1:] + q[1:, :-1] + q[1:, 1:])
    f = np.zeros_like(q)
    for a in (slice(0, ny), slice(1, ny + 1)):
        for b in (slice(0, nx), slice(1, nx + 1)):
            f[a, b] -= 0.25 * quad
    F[(nx + 1) * (ny + 1) * nz:, 2] = f.ravel()
    return F


def _explicit_dt(model):
    """Half of a safe step: 0.3 h / Vp of the fastest layer."""
    vp = max(v for v in model["vs"]) * math.sqrt(3.5)
    return 0.3 * model["h"][0] / vp


def _source_eq(model, mesh):
    return int(mesh.node_eq[3 * mesh.node_rank[model["source_node"]] + 2])


def prepare(case, seed):
    kind = case["kind"]
    ctx = context()
    st = dict(case=case, ctx=ctx)
    if kind in ("apply", "solve", "force", "explicit"):
        model, mesh, params, inp = _inputs(case, seed)
        if kind == "apply":
            t = torch.float32 if case["bits"] == 32 else torch.float64
            st.update(batch=core.Batch(ctx, mesh, params, fp32=case["bits"] == 32, element=case["element"]),
                      x=vec(inp["x"], t), y=zeros(mesh.neq, t))
        elif kind == "solve":
            st.update(batch=core.Batch(ctx, mesh, params, fp32=case["method"] == "mixed", gmres=case["method"] == "gmres"),
                      b=vec(inp["b"]), x=zeros(mesh.neq))
        elif kind == "force":
            st.update(batch=core.Batch(ctx, mesh, params), u=vec(inp["u"]), v=vec(inp["v"]), f=zeros(mesh.neq))
        else:
            st.update(batch=core.Batch(ctx, mesh, params), dt=_explicit_dt(model), dash=vec(inp["dash"]),
                      load_eq=np.array([_source_eq(model, mesh)], np.int32), load=inp["load"], u0=vec(inp["u"]),
                      um0=vec(inp["um"]), u=zeros(mesh.neq), um=zeros(mesh.neq), v=zeros(mesh.neq), a=zeros(mesh.neq))
        st["k"] = core.coeffs(*_coeffs(case))
    elif kind == "pimy":
        rng = np.random.default_rng(seed)
        model, mesh = _column(case["n"], False)
        params = _column_params(rng, model, mesh)
        keep = []
        mats = [core.pimy_material(p["rho"], p["E"] / (2.0 * (1.0 + p["nu"])), p["E"] / (3.0 * (1.0 - 2.0 * p["nu"])), 30.0,
                                   0.1, 0.0, 100.0, 0.0, nsurf=20, b=p["b"], mass_type=0, keep=keep) for p in params]
        batch = core.Batch.pimy(ctx, mesh, mats, rayleigh=[p["rayleigh"] for p in params])
        batch.set_stage(1)
        st.update(batch=batch, u=vec(_field(rng, model, mesh, 4e-3, 10.0)), v=vec(_field(rng, model, mesh, 1e-2, 10.0)),
                  x=vec(rng.standard_normal(mesh.neq)), f=zeros(mesh.neq), y=zeros(mesh.neq),
                  k=core.coeffs(*S.REFERENCE_COLUMN_COEFFS))
    elif kind == "newmark":
        model, mesh = _soil(case["n"], case["nz"])
        rng = S.Lcg(seed)
        mats = core.pimy_materials(S.soil_layers(rng, int(model["group"].max()) + 1))
        batch = core.Batch.pimy(ctx, mesh, [mats[g] for g in mesh.param_group])
        batch.set_stage(1)
        # the strong part of a 0.3 g record: the columns yield from the first pass on
        st.update(batch=batch, record=S.ground_motion(1024, 0.005, seed)[200:], step=0,
                  vecs=[zeros(mesh.neq) for _ in range(4)])
    else:
        rng = S.Lcg(seed)
        heights = np.random.default_rng(case["ncol"]).integers(case["nmin"], case["nmax"] + 1, case["ncol"])
        cols = []
        for n in heights.tolist():
            cols.append((core.pimy_materials(S.soil_layers(rng, 10)), S.column_layer_of(n, 10)))
        record = S.ground_motion(1024, 0.005, seed)[200:200 + case["steps"]]
        total = sum(len(c[1]) for c in cols)
        pool = core.ColumnPool(ctx, max_elements=total + 1024, max_columns=case["ncol"], dt=0.005,
                               max_materials=10 * case["ncol"], max_record=case["ncol"] * 10 * case["steps"] + 1024,
                               mixed=case["mixed"])
        st.update(pool=pool, cols=cols, record=np.ascontiguousarray(record))
    torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "apply":
        if case["bits"] == 32:
            st["batch"].apply_f32(st["x"], st["y"], st["k"])
        else:
            st["batch"].apply(st["x"], st["y"], st["k"])
        return st["y"].t
    if kind == "solve":
        st["x"].zero()
        solve = {"cg": st["batch"].cg, "mixed": functools.partial(st["batch"].cg_mixed, inner_rtol=1e-6),
                 "gmres": st["batch"].gmres}[case["method"]]
        solve(st["b"], st["x"], rtol=case["rtol"], max_it=case["max_it"], k=st["k"])
        return st["x"].t
    if kind == "force":
        st["batch"].force(st["u"], st["f"], st["v"])
        return st["f"].t
    if kind == "explicit":
        # the time loop starts from the displacements of the last two steps
        for a, b in (("u0", "u"), ("um0", "um")):
            core.copy(st["ctx"], st[a], st[b])
        for a in ("v", "a"):
            st[a].zero()
        st["batch"].explicit_cd(st["dt"], case["steps"], st["u"], st["um"], st["v"], st["a"], dash=st["dash"],
                                load_eq=st["load_eq"], load_hist=st["load"])
        return [st[a].t for a in ("u", "um", "v", "a")]
    if kind == "pimy":
        st["batch"].force(st["u"], st["f"], st["v"])
        st["batch"].store_tangents(st["u"])
        st["batch"].apply(st["x"], st["y"], st["k"])
        return [st["f"].t, st["y"].t]
    if kind == "newmark":
        # the next steps of the stage: the record is walked on from pass to pass
        n, i = case["steps"], st["step"]
        if i + n > len(st["record"]):
            i = 0
        st["batch"].newmark(*st["vecs"], 0.005, n, ground_dir=0, ground_accel=st["record"][i:i + n])
        st["step"] = i + n
        # the fourth vector, the solver's last increment, is below Newton's tolerance: rounding
        return [v.t for v in st["vecs"][:3]]
    pool = st["pool"]
    ids = [pool.add(mats, mat_of, case["steps"], st["record"]) for mats, mat_of in st["cols"]]
    while pool.run(8):
        pass
    got = [pool.fetch(i) for i in ids]
    for i in ids:
        pool.remove(i)
    return {k: np.concatenate([g[k] for g in got]) for k in ("u", "v", "a", "history")}


# ---- what a pass cannot do without --------------------------------------------------------------


def _sizes(case):
    """equations, elements, nodes (to within the ties and fixed nodes)."""
    kind = case["kind"]
    if kind in ("apply", "solve", "explicit"):
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
    else:
        nx = ny = case["n"]
        nz = case.get("nz", case["n"])
    nodes = (nx + 1) * (ny + 1) * (nz + 1)
    free = nodes if kind == "explicit" else (nx + 1) * (ny + 1) * nz
    if kind in ("force", "pimy", "newmark") or case.get("layers") == 0:
        free = nz * ((nx - 1) * (ny - 1) + 1)
    return 3 * free, nx * ny * nz, nodes


def _operator_work(neq, nel, nodes, w, flops):
    """x read, y written, connectivity and parameter index, coordinates, node to equation map."""
    return 2 * w * neq + 36 * nel + 3 * w * nodes + 12 * nodes, flops * nel


def work(case):
    kind = case["kind"]
    if kind == "columns":
        elems = case["ncol"] * (case["nmin"] + case["nmax"]) / 2
        # three Newton iterations a step: the moved part of a point's history read and written
        return {"bytes": 3 * case["steps"] * elems * 860.0, "flops": 3 * case["steps"] * elems * 2000.0}
    neq, nel, nodes = _sizes(case)
    if kind == "apply":
        b, f = _operator_work(neq, nel, nodes, case["bits"] // 8, 1900 if case["mesh"] == "distorted" else 250)
        return {"bytes": b, "flops": f}
    if kind == "solve":
        its = case["max_it"] if case["rtol"] == 0.0 else 15.0 * max(case["nx"], case["ny"], case["nz"]) * (
            1.6 if case["method"] == "mixed" else 1.0)
        b, f = _operator_work(neq, nel, nodes, 4 if case["method"] == "mixed" else 8, 300)
        vectors = 10 if case["method"] != "gmres" else 8 + 2 * min(30, case["max_it"])
        moved = b + (4 if case["method"] == "mixed" else 8) * vectors * neq
        # an iteration whose data fit the 256 MB last-level cache need not read HBM again
        return {"bytes": moved * (its if moved > 256e6 else 1.0), "flops": its * f}
    if kind == "force":
        b, f = _operator_work(neq, nel, nodes, 8, 400)
        return {"bytes": b + 16 * neq, "flops": f}
    if kind == "explicit":
        return {"bytes": case["steps"] * (6 * 8 * neq + 16 * nodes), "flops": case["steps"] * 260.0 * nel}
    # per Gauss point: half of the history read and written twice (force, tangents), the tangent
    # written and read
    points = 8 * nel
    per = points * (4 * 95 * 8 + 2 * 21 * 8)
    if kind == "pimy":
        return {"bytes": per, "flops": points * 4000.0}
    return {"bytes": case["steps"] * 3 * per, "flops": case["steps"] * 3 * points * 4000.0}


def tolerance(case):
    # about four times the larger of the distance to exact() and the change under inputs moved by
    # rounding, both measured on the listed and some drawn cases
    kind = case["kind"]
    if kind == "apply":
        return {"rel": 7e-6} if case["bits"] == 32 else {"rel": 3e-14}
    if kind == "solve":
        if case["rtol"] == 0.0:
            return {"rel": 1e-11}
        # the stop at rtol 1e-8 leaves x 1e-9 (CG) to 4e-9 (mixed) from the solution
        return {"rel": 3e-8} if case["method"] == "mixed" else {"rel": 1e-8}
    if kind == "force":
        return {"rel": 5e-14}
    if kind == "explicit":
        return {"rel": 3e-13}
    if kind == "newmark":
        return {"rel": 1e-6}  # the accelerations of the Newton steps' stop: 1e-7 under moved inputs
    return {"rel": 1e-11}  # the return map's branches


# ---- the same in plain torch, 64 bits -----------------------------------------------------------

_CORNER = torch.tensor([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1],
                        [-1, 1, 1]], dtype=torch.float64)


def _gauss(X):
    """Per Gauss point of hex8 elements X [E, 8, 3]: N [8], dN/dx [E, 8, 3], the weight dV [E]."""
    c = _CORNER.to(X.device)
    for g in _CORNER / math.sqrt(3.0):
        g = g.to(X.device)
        one = 1.0 + c * g
        N = 0.125 * one[:, 0] * one[:, 1] * one[:, 2]
        dN = 0.125 * torch.stack([c[:, 0] * one[:, 1] * one[:, 2], c[:, 1] * one[:, 0] * one[:, 2],
                                  c[:, 2] * one[:, 0] * one[:, 1]], 1)  # [8, 3]
        J = [[(X[:, :, d] * dN[:, k]).sum(1) for d in range(3)] for k in range(3)]  # dx_d / dxi_k
        cof = [[J[(k + 1) % 3][(d + 1) % 3] * J[(k + 2) % 3][(d + 2) % 3] -
                J[(k + 1) % 3][(d + 2) % 3] * J[(k + 2) % 3][(d + 1) % 3] for d in range(3)] for k in range(3)]
        det = sum(J[0][d] * cof[0][d] for d in range(3))
        G = torch.stack([sum(dN[None, :, k] * (cof[k][d] / det)[:, None] for k in range(3)) for d in range(3)], 2)
        yield N, G, det


class _Exact:
    """The assembled elastic operator f K + m M on vectors in equation numbering."""

    def __init__(self, model, mesh, params):
        eqs = mesh.node_eq.reshape(-1, 3)[mesh.node_rank]
        conn = np.asarray(model["conn"], np.int64)
        self.n = mesh.neq
        self.eq = torch.from_numpy(np.where(eqs >= 0, eqs, mesh.neq).astype(np.int64)[conn]).to(DEV)  # [E, 8, 3]
        self.xyz = torch.from_numpy(np.asarray(model["xyz"])[conn]).to(DEV)
        by_element = np.empty(mesh.nelem, np.int64)
        by_element[mesh.elem_order] = mesh.param[:mesh.nelem]
        self.param = torch.from_numpy(by_element).to(DEV)
        self.params = params

    def per_element(self, f):
        return torch.tensor([float(f(p)) for p in self.params], dtype=torch.float64, device=DEV)[self.param]

    def damping(self, p):
        return p.get("rayleigh", (0.0, 0.0, 0.0, 0.0))

    def setup(self, k):
        """Element matrices' action for K_eff of the coefficients k: the factors per element."""
        cK, cC, cM = k
        self.fD = self.per_element(lambda p: cK + cC * sum(self.damping(p)[1:]))
        lam = self.per_element(lambda p: p["E"] * p["nu"] / ((1.0 + p["nu"]) * (1.0 - 2.0 * p["nu"])))
        mu = self.per_element(lambda p: p["E"] / (2.0 * (1.0 + p["nu"])))
        self.lam, self.mu = self.fD * lam, self.fD * mu
        self.rho = self.per_element(lambda p: (cM + cC * self.damping(p)[0]) * p["rho"])
        self.lumped = self.per_element(lambda p: p.get("mass_type", 0)) != 0
        return self

    def apply(self, x):
        xe = torch.cat([x.to(torch.float64), torch.zeros(1, dtype=torch.float64, device=DEV)])
        y = torch.zeros(self.n + 1, dtype=torch.float64, device=DEV)
        for s in range(0, len(self.eq), 1 << 19):
            at = slice(s, s + (1 << 19))
            v, lam, mu, rho, lumped = xe[self.eq[at]], self.lam[at], self.mu[at], self.rho[at], self.lumped[at]
            out = torch.zeros_like(v)
            for N, G, dv in _gauss(self.xyz[at]):
                H = [[(G[:, :, d] * v[:, :, c]).sum(1) for c in range(3)] for d in range(3)]  # du_c / dx_d
                tr = lam * (H[0][0] + H[1][1] + H[2][2])
                u = (N[None, :, None] * v).sum(1)
                m = rho * dv
                for c in range(3):
                    sig = [dv * ((tr if d == c else 0.0) + mu * (H[d][c] + H[c][d])) for d in range(3)]
                    out[:, :, c] += sum(G[:, :, d] * sig[d][:, None] for d in range(3))
                    mass = torch.where(lumped[:, None], v[:, :, c], u[:, c][:, None].expand(-1, 8))
                    out[:, :, c] += m[:, None] * N * mass
            y.index_add_(0, self.eq[at].reshape(-1), out.reshape(-1))
        return y[:self.n]

    def body(self):
        """F_body: b times the nodal weights."""
        f = torch.zeros(self.n + 1, dtype=torch.float64, device=DEV)
        b = torch.stack([self.per_element(lambda p, c=c: p.get("b", (0.0, 0.0, 0.0))[c]) for c in range(3)], 1)
        out = sum(N[None, :, None] * dv[:, None, None] for N, _, dv in _gauss(self.xyz)) * b[:, None, :]
        f.index_add_(0, self.eq.reshape(-1), out.reshape(-1))
        return f[:self.n]

    def lumped_mass(self):
        m = torch.zeros(self.n + 1, dtype=torch.float64, device=DEV)
        rho = self.per_element(lambda p: p["rho"])
        out = sum(N[None, :] * dv[:, None] for N, _, dv in _gauss(self.xyz)) * rho[:, None]
        m.index_add_(0, self.eq.reshape(-1), out[:, :, None].expand(-1, -1, 3).reshape(-1))
        return m[:self.n]

    def matrix_diagonal(self):
        """diag(K_eff): each equation's entry, cross terms of tied DOFs inside an element included."""
        d = torch.zeros(self.n + 1, dtype=torch.float64, device=DEV)
        flat = self.eq.reshape(len(self.eq), 24)
        for s in range(0, len(self.eq), 1 << 16):
            at = slice(s, s + (1 << 16))
            X, q = self.xyz[at], flat[at]
            Ke = torch.zeros(len(X), 24, 24, dtype=torch.float64, device=DEV)
            for N, G, dv in _gauss(X):
                lam, mu, m = self.lam[at] * dv, self.mu[at] * dv, self.rho[at] * dv
                gg = (G[:, :, None, :] * G[:, None, :, :]).sum(3) * mu[:, None, None]
                NN = torch.where(self.lumped[at][:, None, None], torch.diag(N)[None], (N[:, None] * N[None, :])[None])
                for c in range(3):
                    for e in range(3):
                        blk = (lam[:, None, None] * G[:, :, None, c] * G[:, None, :, e] +
                               mu[:, None, None] * G[:, :, None, e] * G[:, None, :, c])
                        if c == e:
                            blk = blk + gg + m[:, None, None] * NN
                        Ke[:, c::3, e::3] += blk
            same = q[:, :, None] == q[:, None, :]
            d.index_add_(0, q.reshape(-1), (Ke * same).sum(2).reshape(-1))
        return d[:self.n]


def _exact_cg(A, b, rtol, max_it):
    inv = 1.0 / A.matrix_diagonal()
    x, r = torch.zeros_like(b), b.clone()
    z = inv * r
    p, rz, stop = z.clone(), torch.dot(r, z), rtol * torch.linalg.norm(b)
    for i in range(max_it):
        Ap = A.apply(p)
        alpha = rz / torch.dot(p, Ap)
        x += alpha * p
        r -= alpha * Ap
        if rtol > 0.0 and i % 8 == 7 and torch.linalg.norm(r) <= stop:
            break
        z = inv * r
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
    return x


def _exact_gmres(A, b, restart, max_it):
    inv = 1.0 / A.matrix_diagonal()
    x, done = torch.zeros_like(b), 0
    while done < max_it:
        r = b - A.apply(x)
        beta = torch.linalg.norm(r)
        m = min(restart, max_it - done)
        V, H = [r / beta], torch.zeros(m + 1, m, dtype=torch.float64)
        for j in range(m):
            w = A.apply(inv * V[j])
            for _ in range(2):
                for i in range(j + 1):
                    h = torch.dot(V[i], w)
                    w = w - h * V[i]
                    H[i, j] += float(h)
            H[j + 1, j] = float(torch.linalg.norm(w))
            V.append(w / H[j + 1, j].item())
        g = torch.zeros(m + 1, 1, dtype=torch.float64)
        g[0, 0] = float(beta)
        y = torch.linalg.lstsq(H, g).solution[:, 0]
        for j in range(m):
            x = x + y[j].item() * inv * V[j]
        done += m
    return x


def exact(case, seed):
    """None for the kinds with the multi-surface return map, for SSPbrick, and for the solves too
    long for plain torch."""
    kind = case["kind"]
    if kind not in ("apply", "solve", "force", "explicit") or case.get("element") == "SSPbrick":
        return None
    neq, nel, _ = _sizes(case)
    if kind == "solve" and case["rtol"] > 0.0 and nel > 20000:
        return None
    model, mesh, params, inp = _inputs(case, seed)
    A = _Exact(model, mesh, params)
    t = {k: torch.as_tensor(v).to(DEV, torch.float64) for k, v in inp.items()}
    if kind == "apply":
        return A.setup(_coeffs(case)).apply(t["x"])
    if kind == "solve":
        A.setup(_coeffs(case))
        if case["method"] == "gmres":
            return _exact_gmres(A, t["b"], 30, case["max_it"])
        return _exact_cg(A, t["b"], 1e-13 if case["rtol"] > 0.0 else 0.0, 5000 if case["rtol"] > 0.0 else case["max_it"])
    if kind == "force":
        return A.setup((1.0, 0.0, 0.0)).apply(t["u"]) + A.setup((0.0, 1.0, 0.0)).apply(t["v"]) - A.body()
    dt, m = _explicit_dt(model), A.lumped_mass()
    c2, c3 = 0.5 / dt, 1.0 / (dt * dt)
    u, um, v, a = t["u"].clone(), t["um"].clone(), torch.zeros_like(t["u"]), torch.zeros_like(t["u"])
    A.setup((1.0, 0.0, 0.0))
    src = _source_eq(model, mesh)
    for k in range(case["steps"]):
        f = A.apply(u) + t["dash"] * (-c2 * um)
        f[src] -= t["load"][k]
        new = (-f - m * c3 * (um - 2.0 * u)) / (m * c3 + t["dash"] * c2)
        rate = c2 * (3.0 * new - 4.0 * u + um)
        a = (rate - v) / dt
        v, um, u = rate, u, new
    return [u, um, v, a]
