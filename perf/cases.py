"""The work that users of rainbow_amd wait for, as cases to be timed.

Each case goes through the public entry points: ``api.simulate`` on an engine,
the device context of ``rainbow_amd.native`` (the binding of include/rbh.h:
scenes kept on the device, stepped alone or as a batch), the continuous-batching
server, and the signed-distance build of a new shape.  The workloads are those
of ``rainbow_amd/scenes.py`` (box stack, sphere rain, mixed drop, serving
requests, meshes of about 10^4 triangles, hinge chains), in the regime that
costs the most in use: bodies that have landed and lie in contact.  Bodies are
therefore placed in contact from the start, on jittered lattices, instead of
being dropped for hundreds of steps.  (Two bodies give a contact only where a
point of one lies half a length unit inside the other's grid, as in the
reference, so settled neighbours overlap deeply.)

A pass starts from the prepared state each time: the state is set, a few steps
are taken, and state, contacts and solver records are read back.

Kinds (case["kind"]):

* "engine"   one engine, ``api.simulate`` for some steps: what a script written
             against the reference does.  Host-side state in and out each call.
* "scene"    one scene resident on the device, ``Context.step`` for some steps.
* "batch"    many scenes stepped together, one graph replay per step.
* "serve"    requests of different sizes and lengths through ``Server.run``:
             admission, steps with a shrinking batch, read-back, release.
* "sdf"      the signed-distance grid of a mesh (``Context.sdf_build``), which
             every new shape needs.

Values of 64 bits: ``exact`` gives them for the signed-distance grids.  The
steps have none of their own outside this package: the order in which contacts
are solved follows the package's seeded colouring, and the sweeps stop at a
fixed count, long before the solution no longer depends on that order.
"""
import math
import random

import numpy as np
import torch

from rainbow_amd import api as API
from rainbow_amd import math3 as Q
from rainbow_amd import mesh as MESH
from rainbow_amd import native
from rainbow_amd import scenes
from rainbow_amd import serving
from rainbow_amd.stepper import engine_desc, gather_state, upload_hinges

SPHERE_TRIS, BOX_TRIS, MESH_TRIS = 448, 12, 9840     # create_sphere(0.5, 16, 16), create_box, mean of the two meshes


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the reference's own hinge scene, one step per call: nothing but latency and launches
        dict(name="hinge_chain", kind="engine", scene="chain", n=5, iterations=100, steps=1, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # a script's stack of 64 boxes, a few steps per call, 100 sweeps a step
        dict(name="box_stack", kind="engine", scene="boxes", n=64, iterations=100, steps=4, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # the double-precision build with the options of the soft-body simulator: anisotropic friction, post-stabilisation
        dict(name="boxes_fp64", kind="engine", scene="boxes", n=27, iterations=50, steps=2, precision="fp64",
             scheme="parallel_gauss_seidel", friction="anisotropic", post=True),
        # the headline workload: 4096 spheres, most still falling, some landed, neighbours sunk into each other
        dict(name="rain_4096", kind="scene", scene="rain", n=4096, iterations=50, steps=5, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # a settled pile: islands of up to several hundred contacts, too large for a workgroup's LDS
        dict(name="pile_1500", kind="scene", scene="pile", n=1500, iterations=50, steps=3, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # a Jacobi scheme on a middle-sized pile, an odd count
        dict(name="pile_333_jacobi", kind="scene", scene="pile", n=333, iterations=60, steps=4, precision="fp32",
             scheme="parallel_jacobi_hybrid", friction="isotropic", post=False),
        # meshes of ten thousand triangles with 64^3 grids pressed together: the narrow phase
        dict(name="meshes_48", kind="scene", scene="meshes", n=48, iterations=50, steps=4, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # a batch of environments: more scenes than compute units, boxes and spheres, landed
        dict(name="batch_320", kind="batch", scene="mixed", n=24, scenes=320, iterations=30, steps=20, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # a small batch of larger scenes
        dict(name="batch_24", kind="batch", scene="mixed", n=180, scenes=24, iterations=30, steps=8, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # requests of 8 to 300 bodies and different lengths served together
        dict(name="serve_16", kind="serve", scene="rain", n=300, scenes=16, iterations=50, steps=24, precision="fp32",
             scheme="parallel_gauss_seidel", friction="isotropic", post=False),
        # a simple shape's grid, and a scanned object's
        dict(name="sdf_sphere_32", kind="sdf", mesh="sphere", tess=16, resolution=32),
        dict(name="sdf_knot_64", kind="sdf", mesh="knot", tess=25, resolution=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ranges: sizes spread evenly over their logarithm."""
    def step_case(kind, scene, n, iterations, steps, **kw):
        c = dict(kind=kind, scene=scene, n=n, iterations=iterations, steps=steps, precision="fp32",
                 scheme="parallel_gauss_seidel", friction="isotropic", post=False)
        c.update(kw)
        return c

    family = rng.choice(["chain", "boxes", "rain", "pile", "meshes", "batch", "serve", "sdf", "sdf"])
    if family == "chain":
        return step_case("engine", "chain", _log_int(rng, 2, 48), rng.choice([50, 100]), rng.randint(1, 4))
    if family == "boxes":
        return step_case("engine", "boxes", _log_int(rng, 1, 125), rng.choice([30, 50, 100]), rng.randint(1, 4),
                         precision=rng.choice(["fp32", "fp32", "fp64"]),
                         scheme=rng.choice(["gauss_seidel", "parallel_gauss_seidel", "parallel_jacobi"]),
                         friction=rng.choice(["isotropic", "anisotropic"]), post=rng.random() < 0.3)
    if family == "rain":
        return step_case("scene", "rain", _log_int(rng, 60, 4096), rng.choice([30, 50]), rng.randint(2, 5))
    if family == "pile":
        return step_case("scene", "pile", _log_int(rng, 20, 1500), rng.choice([30, 50]), rng.randint(1, 3),
                         scheme=rng.choice(["parallel_gauss_seidel", "parallel_gauss_seidel", "parallel_jacobi_hybrid"]),
                         post=rng.random() < 0.25)
    if family == "meshes":
        return step_case("scene", "meshes", _log_int(rng, 2, 48), rng.choice([30, 50]), rng.randint(1, 4))
    if family == "batch":
        count = _log_int(rng, 3, 320)
        return step_case("batch", "mixed", max(4, min(180, int(6000 / count))), 30, rng.randint(4, 10), scenes=count)
    if family == "serve":
        return step_case("serve", "rain", _log_int(rng, 40, 300), rng.choice([30, 50]), rng.randint(8, 24),
                         scenes=_log_int(rng, 3, 16))
    shape = rng.choice(["sphere", "box", "ico", "knot"])
    return dict(kind="sdf", mesh=shape, tess=_log_int(rng, 5, 22), resolution=_log_int(rng, 12, 64))


# ------------------------------------------------------------------ scenes
def _bank(resolution):
    return scenes.ShapeBank(resolution=resolution)


def _params(case, seed, time_step):
    return dict(time_step=time_step, max_iterations=case["iterations"], absolute_tolerance=0.0, relative_tolerance=0.0,
                proximal_solver=case["scheme"], friction_model=case["friction"], precision=case["precision"],
                use_post_stabilization=case["post"], coloring_seed=seed)


def _random_quaternion(rng):
    q = rng.normal(size=4)
    return q / np.linalg.norm(q)


def _lattice(rng, n, columns, pitch, layer, jitter, occupancy, y0):
    """n positions: layers of columns x columns sites, a share of them taken at random."""
    out = []
    k = 0
    while len(out) < n:
        sites = np.array([(i, j) for i in range(columns) for j in range(columns)], dtype=np.float64)
        sites = (sites - 0.5 * (columns - 1)) * pitch
        sites = sites[rng.uniform(size=len(sites)) < occupancy][: n - len(out)]
        for x, z in sites:
            d = rng.uniform(-jitter, jitter, 3)
            out.append((x + d[0], y0 + k * layer + abs(d[1]), z + d[2]))
        k += 1
    return np.array(out)


def _world(case, bank, seed, time_step, mu, backend="hip"):
    eng = scenes.new_engine(bank, _params(case, seed, time_step), backend)
    if case["friction"] == "anisotropic":
        eng.surfaces_interactions.storage[("default", "default")].mu = np.array([mu, 0.6 * mu, 0.1 * mu])
    else:
        scenes.set_friction(eng, mu)
    API.create_gravity_force(eng, "gravity", 9.81, np.array([0.0, 1.0, 0.0]))
    scenes.add_ground(eng, bank)
    return eng


def _engine(case, bank, seed, n=None):
    """The engine of one scene, its bodies in contact."""
    n = case["n"] if n is None else n
    rng = np.random.default_rng(seed)
    if case["scene"] == "chain":
        eng = scenes.cube_hinge_chain(bank, n=n, params=_params(case, seed, 0.01))
        for b in eng.bodies.values():
            if not b.is_fixed:
                b.v, b.w = rng.normal(0.0, 0.3, 3), rng.normal(0.0, 0.1, 3)
        return eng
    if case["scene"] == "boxes":
        eng = _world(case, bank, seed, 0.01, 0.5)
        box = bank.get("box_shape", lambda: MESH.create_box(1.0, 1.0, 1.0))
        side = max(1, int(math.ceil(n ** (1.0 / 3.0) - 1e-9)))
        for i, p in enumerate(_lattice(rng, n, side, 1.05, 0.68, 0.01, 2.0, 0.48)):
            scenes.add_body(eng, "box_%d" % i, box, p, q=Q.identity(), v=rng.normal(0.0, 0.05, 3))
        return eng
    if case["scene"] == "mixed":
        eng = _world(case, bank, seed, 0.01, float(rng.uniform(0.1, 0.8)))
        shapes = (bank.get("box_shape", lambda: MESH.create_box(1.0, 1.0, 1.0)),
                  bank.get("sphere_shape", lambda: MESH.create_sphere(0.5, 16, 16)))
        side = max(2, int(math.ceil((n / 3.0) ** 0.5)))
        for i, p in enumerate(_lattice(rng, n, side, 0.74, 0.7, 0.03, 0.9, 0.47)):
            scenes.add_body(eng, "body_%d" % i, shapes[int(rng.integers(2))], p, q=Q.Ry(rng.uniform(-0.03, 0.03)),
                            v=rng.normal(0.0, 0.1, 3))
        return eng
    if case["scene"] == "meshes":
        eng = _world(case, bank, seed, 0.005, 0.4)
        shape_rng = np.random.default_rng(seed + 1)
        kinds = (scenes._unit_shape(bank, "ico", lambda: MESH.create_noisy_icosphere(shape_rng, 22)),
                 scenes._unit_shape(bank, "knot", MESH.create_torus_knot))
        side = max(1, int(math.ceil(n ** (1.0 / 3.0))))
        for i, p in enumerate(_lattice(rng, n, side, 0.72, 0.68, 0.04, 2.0, 0.56)):
            scenes.add_body(eng, "body_%d" % i, kinds[i % 2], p, q=_random_quaternion(rng), v=rng.normal(0.0, 0.2, 3))
        return eng
    # spheres: "rain" (falling, some landed; loose) or "pile" (landed; every neighbour touches)
    eng = _world(case, bank, seed, 0.005, 0.3)
    sphere = bank.get("sphere_shape", lambda: MESH.create_sphere(0.5, 16, 16))
    if case["scene"] == "rain":
        side = max(2, min(20, int(math.ceil(n ** 0.4))))
        P = _lattice(rng, n, side, 0.95, 1.0, 0.13, 0.45, 0.0)
        P[:, 1] += 0.46 + rng.uniform(0.0, 0.55, n)
        V = rng.normal(0.0, 0.5, (n, 3)) - np.outer(rng.uniform(0.0, 8.0, n) * (P[:, 1] > 2.0), (0.0, 1.0, 0.0))
    else:
        side = max(2, int(math.ceil(n ** (1.0 / 3.0) * 1.2)))
        P = _lattice(rng, n, side, 0.73, 0.71, 0.05, 0.9, 0.47)
        V = rng.normal(0.0, 0.2, (n, 3))
    for i in range(n):
        scenes.add_body(eng, "sphere_%d" % i, sphere, P[i], q=Q.identity(), v=V[i], w=rng.normal(0.0, 0.3, 3))
    return eng


def _sdf_mesh(case, seed):
    """(V, T) of the mesh, with a size and a pose that follow from the seed."""
    rng = np.random.default_rng(seed)
    t = case["tess"]
    if case["mesh"] == "sphere":
        V, T = MESH.create_sphere(0.5, t, t)
    elif case["mesh"] == "box":
        V, T = MESH.create_box(1.0, 0.5, 0.25)
    elif case["mesh"] == "ico":
        V, T = MESH.create_noisy_icosphere(rng, t)
    else:
        V, T = MESH.create_torus_knot(segments=8 * t, sides=t)
    q = _random_quaternion(rng)
    V = np.array([Q.rotate(q, v) for v in V]) * rng.uniform(0.9, 1.1, 3)
    return np.ascontiguousarray(V), np.ascontiguousarray(T, dtype=np.int32)


def _sdf_box(V):
    """The grid's corners as api.create_shape sets them (a tenth of the largest extent around the mesh)."""
    lo, hi = V.min(axis=0), V.max(axis=0)
    pad = max(0.1 * float((hi - lo).max()), 0.2)
    return lo - pad, hi + pad


# ------------------------------------------------------------------ prepare and run
class _Resident:
    """Scenes kept on a device context of their own, with the states a pass starts from."""

    def __init__(self, case, engines):
        self.ctx = native.Context(0, case["precision"])
        self.ids, self.starts, self.sizes = [], [], []
        for eng in engines:
            desc, keep = engine_desc(eng, self.ctx)
            sid = self.ctx.scene_create(desc)
            del keep
            if eng.hinges:
                upload_hinges(self.ctx, sid, eng)
            self.ids.append(sid)
            self.starts.append(gather_state(list(eng.bodies.values())))
            self.sizes.append(len(eng.bodies))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "sdf":
        V, T = _sdf_mesh(case, seed)
        lo, hi = _sdf_box(V)
        return dict(case=case, ctx=native.Context(0, "fp64"), V=V, T=T, lo=lo, hi=hi)
    bank = _bank(64 if case["scene"] == "meshes" else 32)
    if kind == "engine":
        eng = _engine(case, bank, seed)
        bodies = list(eng.bodies.values())
        return dict(case=case, engine=eng, start=[(b.r.copy(), b.q.copy(), b.v.copy(), b.w.copy()) for b in bodies])
    if kind == "scene":
        return dict(case=case, world=_Resident(case, [_engine(case, bank, seed)]))
    # sizes of a batch's scenes and of the requests: spread over their logarithm, the same for every seed
    rng = random.Random(case["scenes"] * 1009 + case["n"])
    if kind == "batch":
        sizes = [max(4, min(4 * case["n"], int(case["n"] * math.exp(rng.uniform(-1.4, 1.0)))))
                 for _ in range(case["scenes"])]
        return dict(case=case, world=_Resident(case, [_engine(case, bank, seed * 1000 + i, n)
                                                      for i, n in enumerate(sizes)]))
    server = serving.Server(native.Context(0, case["precision"]), budget=8 << 30)
    requests = []
    for i in range(case["scenes"]):
        n = case["n"] if i == 0 else _log_int(rng, 8, case["n"])
        req = serving.Request(i, _engine(case, bank, seed * 1000 + i, n), max(1, case["steps"] - 2 * (i % 8)))
        requests.append(server.prepare(req))
    return dict(case=case, server=server, requests=requests)


def _contact_buffers(case, contacts):
    """The contacts in buffers of a fixed length (zero past the last one), as a viewer or a logger keeps them."""
    per_body, more = {"chain": (8, 64), "boxes": (8, 64), "rain": (4, 1024), "pile": (40, 1024),
                      "meshes": (128, 4096)}[case["scene"]]
    cap = per_body * case["n"] + more
    out = {}
    for key, a in contacts.items():
        if len(a) > cap:
            raise RuntimeError("more contacts than the buffers hold: %d" % len(a))
        out[key] = np.zeros((cap,) + a.shape[1:], a.dtype)
        out[key][:len(a)] = a
    return out


def _stacked(states):
    """The states of many scenes, body after body."""
    return dict(zip("rqvw", (np.concatenate(f) for f in zip(*states))))


def _scene_outputs(case, ctx, sid, n):
    log = ctx.get_log(sid, case["iterations"])
    out = dict(zip("rqvw", ctx.get_state(sid, n)))
    out.update(_contact_buffers(case, ctx.get_contacts(sid)))
    out["residuals"] = log["residuals"].copy()
    for key in ("contact_points", "iterations", "exitcode", "rejects", "colors"):
        out[key] = int(log[key])
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "sdf":
        r = case["resolution"]
        return state["ctx"].sdf_build(state["V"], state["T"], state["lo"], state["hi"], r, r, r)
    if kind == "engine":
        eng = state["engine"]
        bodies = list(eng.bodies.values())
        for b, (r, q, v, w) in zip(bodies, state["start"]):
            b.r, b.q, b.v, b.w = r, q, v, w
        eng.step_index = 0
        API.simulate(eng, case["steps"] * eng.params.time_step)
        out = dict(zip("rqvw", gather_state(bodies)))
        out.update(_contact_buffers(case, eng.contact_points.arrays))
        return out
    if kind == "serve":
        state["server"].run(state["requests"])
        return _stacked(req.state for req in state["requests"])
    world = state["world"]
    ctx = world.ctx
    for sid, start in zip(world.ids, world.starts):
        ctx.set_state(sid, *start)
        ctx.set_step_index(sid, 0)
    if kind == "scene":
        ctx.step(world.ids, case["steps"])
        return _scene_outputs(case, ctx, world.ids[0], world.sizes[0])
    ctx.step(world.ids, case["steps"], 0.0, native.STEP_GRAPH)
    return _stacked(ctx.get_state(sid, n) for sid, n in zip(world.ids, world.sizes))


# ------------------------------------------------------------------ work
def _mesh_triangles(case):
    t = case["tess"]
    return {"sphere": 2 * t * (t - 2), "box": 12, "ico": 20 * t * t, "knot": 16 * t * t}[case["mesh"]]


def work(case):
    """Bytes and operations one pass cannot do without.

    A grid: the mesh read and the values written; per node one closest triangle
    and one sign (about 200 operations).  Steps: state in and out, the shapes'
    meshes and grids once, the contacts out; per step and body its boxes, per
    contact and sweep one projection of its four rows (about 250 operations).
    Contacts per body are what these placements give."""
    if case["kind"] == "sdf":
        n = case["resolution"] ** 3
        return dict(bytes=8 * n + 36 * _mesh_triangles(case), flops=200 * n)
    bodies = case["n"] * case.get("scenes", 1)
    if case["kind"] == "serve":
        bodies = bodies * 0.35
    word = 8 if case["precision"] == "fp64" else 4
    contacts = {"chain": 1.0, "boxes": 2.3, "rain": 1.7, "pile": 12.0, "mixed": 10.0, "meshes": 45.0}[case["scene"]]
    tris = {"chain": 12, "boxes": 12, "rain": 448, "pile": 448, "mixed": 230, "meshes": 9840}[case["scene"]]
    grid = 64 ** 3 if case["scene"] == "meshes" else 32 ** 3
    steps = case["steps"] * (0.7 if case["kind"] == "serve" else 1.0)
    data = 2 * bodies * 13 * word + 2 * (grid + 3 * tris) * word + contacts * bodies * 15 * word
    ops = steps * bodies * (30 * tris + 250 * contacts * case["iterations"])
    return dict(bytes=int(data), flops=int(ops))


# ------------------------------------------------------------------ exact values
def _point_triangle_sq(P, a, b, c):
    """Squared distances (points x triangles): the nearest of the plane's foot, where it falls inside, and the edges."""
    def dot(x, y):
        return (x * y).sum(-1)

    ab, ac, bc = b - a, c - a, c - b
    p = P[:, None, :] - a[None]
    d00, d01, d11 = dot(ab, ab), dot(ab, ac), dot(ac, ac)
    d20, d21 = dot(p, ab[None]), dot(p, ac[None])
    den = d00 * d11 - d01 * d01
    v, w = (d11 * d20 - d01 * d21) / den, (d00 * d21 - d01 * d20) / den
    normal = torch.linalg.cross(ab, ac)
    h2 = dot(p, normal[None]) ** 2 / dot(normal, normal)
    best = torch.where((v >= 0) & (w >= 0) & (v + w <= 1), h2, torch.full_like(h2, math.inf))
    for o, e in ((a, ab), (a, ac), (b, bc)):
        x = P[:, None, :] - o[None]
        t = (dot(x, e[None]) / dot(e, e)).clamp(0.0, 1.0)
        y = x - t[..., None] * e[None]
        best = torch.minimum(best, dot(y, y))
    return best


def _solid_angle(P, a, b, c):
    x, y, z = a[None] - P[:, None], b[None] - P[:, None], c[None] - P[:, None]
    lx, ly, lz = x.norm(dim=-1), y.norm(dim=-1), z.norm(dim=-1)
    det = (x * torch.linalg.cross(y, z)).sum(-1)
    den = lx * ly * lz + (x * y).sum(-1) * lz + (y * z).sum(-1) * lx + (z * x).sum(-1) * ly
    return 2.0 * torch.atan2(det, den)


def exact(case, seed):
    if case["kind"] != "sdf":
        return None
    V, T = _sdf_mesh(case, seed)
    lo, hi = _sdf_box(V)
    r = case["resolution"]
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    if r ** 3 * len(T) > (4e9 if dev.type == "cuda" else 4e7):
        return None
    axes = [lo[i] + (hi[i] - lo[i]) / (r - 1) * np.arange(r) for i in range(3)]
    k, j, i = np.meshgrid(axes[2], axes[1], axes[0], indexing="ij")     # i runs fastest
    P = torch.tensor(np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1), dtype=torch.float64, device=dev)
    corners = torch.tensor(V[T], dtype=torch.float64, device=dev)
    a, b, c = corners[:, 0], corners[:, 1], corners[:, 2]
    out = torch.empty(len(P), dtype=torch.float64, device=dev)
    chunk = max(1, int((4e6 if dev.type == "cuda" else 1e5) / len(T)))
    for s in range(0, len(P), chunk):
        p = P[s:s + chunk]
        dist = _point_triangle_sq(p, a, b, c).min(dim=1).values.sqrt()
        winding = _solid_angle(p, a, b, c).sum(dim=1) / (4.0 * math.pi)
        out[s:s + chunk] = torch.where(winding.abs() > 0.5, -dist, dist)
    return out.cpu().numpy()
