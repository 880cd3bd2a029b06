"""What a user of warp_psr_amd has it do, as cases that can be timed.

Five kinds of work, each through the public entry points:

* ``recon``: reconstruct() of one oriented cloud, then the field at query points
  (the inputs and uniform points of the bounding cube), from a few hundred
  points to the 800,000-point depth-9 scan, in float32, float64 and mixed
  precision, screened, exactly interpolating and unscreened.
* ``batch``: reconstruct_batch() of independent clouds of 5,000-200,000 points,
  then each field at its cloud's points.
* ``query``: evaluate() of a field in hand at many points (``grad`` outputs too).
* ``field``: a LevelField over the caller's own keys and coefficients (a field
  that was stored and is loaded again) at many points.
* ``mesh``: extract_mesh() of a float32 reconstruction in hand.
* ``backward``: reconstruct_differentiable(), a field loss and its gradients to
  positions, normals and queries.

Sizes are those of the repository's workloads and fixtures: a 512-point sphere
at depth 4, the 20,000-point sphere at depth 6, the noisy torus at depth 8, the
six-ellipsoid union at depth 9, the 64-cloud batch and the displaced sphere at
depth 7.  Clouds are drawn on the GPU from the seed; a shape's parameters do not
depend on it, so that another seed is another scan of the same object.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "warp-psr_amd"))

from warp_psr_amd import LevelField, reconstruct, reconstruct_batch, reconstruct_differentiable, synthetic  # noqa: E402
from warp_psr_amd.meshing import extract_mesh  # noqa: E402

DEVICE = "cuda:0"
DTYPES = {"float32": torch.float32, "float64": torch.float64, "mixed": torch.float64}

# basis functions of one level per 4^level on the workloads' surfaces, while the points still fill the level
ROWS_PER_CELL = 30.0
# basis functions of one level per input point once they no longer do
ROWS_PER_POINT = 4.5


def listed():
    return [
        # a cloud picked in an interactive tool: latency, launches and host reads are all of it
        dict(name="recon_512_d4_float32", kind="recon", shape="sphere", points=512, queries=200, depth=4, full_depth=2,
             dtype="float32", point_weight=2.0, exact=False, iters=8),
        # a small scan with the default full depth
        dict(name="recon_20k_d6_float32", kind="recon", shape="sphere", points=20000, queries=5000, depth=6, full_depth=3,
             dtype="float32", point_weight=2.0, exact=False, iters=8),
        # an ordinary object in double precision without screening (PSR), an odd count
        dict(name="recon_60001_d7_float64_psr", kind="recon", shape="torus", points=60001, queries=5000, depth=7, full_depth=4,
             dtype="float64", point_weight=0.0, exact=False, iters=8),
        # a noisy scan with uneven sampling and zeroed normals
        dict(name="recon_250k_d8_float32", kind="recon", shape="torus", points=250000, queries=20000, depth=8, full_depth=4,
             dtype="float32", point_weight=2.0, exact=False, iters=8),
        # the large scan the throughput is quoted on
        dict(name="recon_800k_d9_mixed", kind="recon", shape="union", points=800000, queries=12000, depth=9, full_depth=4,
             dtype="mixed", point_weight=2.0, exact=False, iters=8),
        # the same scan in double precision throughout, interpolating its points exactly
        dict(name="recon_800k_d9_float64_exact", kind="recon", shape="union", points=800000, queries=12000, depth=9, full_depth=4,
             dtype="float64", point_weight=4.0, exact=True, iters=8),
        # many independent objects in one call
        dict(name="batch_12_mixed", kind="batch", clouds=12, smallest=5000, largest=200000, full_depth=4, dtype="mixed",
             point_weight=2.0, iters=8),
        # residuals of a large scan: the field and its gradient at every input point and around it
        dict(name="query_812k_d9_float64", kind="query", shape="union", points=800000, queries=812000, depth=9, full_depth=4,
             dtype="float64"),
        # a stored field loaded again and probed by a renderer's rays
        dict(name="field_100k_d8_float64", kind="field", queries=100003, depth=8, dtype="float64"),
        # a mesh for viewing
        dict(name="mesh_256_d8_float32", kind="mesh", shape="torus", points=250000, depth=8, full_depth=4, resolution=256),
        # a point-cloud optimisation step: loss at targets, gradients to every position and normal
        dict(name="backward_100k_d7_float64", kind="backward", shape="displaced", points=100000, queries=50000, depth=7, full_depth=4,
             dtype="float64", point_weight=2.0, positions=True),
        # a light step on a small cloud: normals only, unscreened, single precision
        dict(name="backward_5k_d5_float32", kind="backward", shape="torus", points=5000, queries=2000, depth=5, full_depth=3,
             dtype="float32", point_weight=0.0, positions=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _depth_for(rng, points, lo, hi):
    """A scan's depth: about the level at which its points fill the surface's cells."""
    return max(lo, min(hi, int(round(math.log(points, 4) + rng.uniform(-1.7, 0.0)))))


def draw(rng):
    kind = rng.choice(["recon"] * 5 + ["batch", "query", "field", "mesh", "backward", "backward"])
    shape = rng.choice(["sphere", "torus", "union", "displaced"])
    if kind == "recon":
        points = _log_int(rng, 500, 800000)
        depth = _depth_for(rng, points, 4, 9)
        weight = rng.choice([0.0, 2.0, 2.0, 4.0])
        return dict(kind=kind, shape=shape, points=points, queries=_log_int(rng, 100, 20000), depth=depth,
                    full_depth=rng.randint(2, min(4, depth)), dtype=rng.choice(["float32", "float64", "mixed"]), point_weight=weight,
                    exact=weight > 0 and rng.random() < 0.25, iters=rng.choice([4, 8, 8]))
    if kind == "batch":
        return dict(kind=kind, clouds=rng.randint(3, 12), smallest=_log_int(rng, 2000, 5000), largest=_log_int(rng, 50000, 200000),
                    full_depth=rng.randint(3, 4), dtype=rng.choice(["float32", "mixed"]), point_weight=2.0, iters=8)
    if kind == "query":
        points = _log_int(rng, 5000, 800000)
        return dict(kind=kind, shape=shape, points=points, queries=_log_int(rng, 1000, 812000), depth=_depth_for(rng, points, 5, 9),
                    full_depth=rng.randint(3, 4), dtype=rng.choice(["float32", "float64"]))
    if kind == "field":
        return dict(kind=kind, queries=_log_int(rng, 1000, 500000), depth=rng.randint(5, 8), dtype=rng.choice(["float32", "float64"]))
    if kind == "mesh":
        points = _log_int(rng, 5000, 250000)
        return dict(kind=kind, shape=shape, points=points, depth=_depth_for(rng, points, 5, 8), full_depth=rng.randint(3, 4),
                    resolution=rng.randint(48, 256))
    points = _log_int(rng, 2000, 100000)
    return dict(kind=kind, shape=shape, points=points, queries=_log_int(rng, 500, 50000), depth=_depth_for(rng, points, 5, 7),
                full_depth=rng.randint(3, 4), dtype=rng.choice(["float32", "float64"]), point_weight=rng.choice([0.0, 2.0]),
                positions=rng.random() < 0.5)


# -- inputs ---------------------------------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _uniform(gen, shape, lo=0.0, hi=1.0):
    return torch.rand(shape, generator=gen, dtype=torch.float64, device=DEVICE) * (hi - lo) + lo


def _directions(gen, count):
    d = torch.randn((count, 3), generator=gen, dtype=torch.float64, device=DEVICE)
    return d / d.norm(dim=1, keepdim=True)


def _torus(gen, count, R=0.6, r=0.2):
    """Torus, x > 0 half sampled 4x denser, position noise 0.002, 1% of the normals zeroed."""
    m = 4 * count + 4096
    u, v = _uniform(gen, m, 0, 2 * math.pi), _uniform(gen, m, 0, 2 * math.pi)
    ring = R + r * v.cos()
    accept = ring / (R + r) * torch.where(u.cos() > 0, 1.0, 0.25)
    keep = (_uniform(gen, m) < accept).nonzero()[:count, 0]
    u, v, ring = u[keep], v[keep], ring[keep]
    n = torch.stack([v.cos() * u.cos(), v.cos() * u.sin(), v.sin()], 1)
    p = torch.stack([ring * u.cos(), ring * u.sin(), r * v.sin()], 1)
    p = p + 0.002 * torch.randn(p.shape, generator=gen, dtype=torch.float64, device=DEVICE)
    n[_uniform(gen, len(n)) < 0.01] = 0
    return p, n


def _union(gen, count, noise=0.001):
    """Smooth union of six ellipsoids, sampling density varying 10x, position noise, exact normals."""
    s = synthetic.EllipsoidUnion()
    on = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEVICE)  # noqa: E731
    centers, axes, rot, lattice = on(s.centers), on(s.axes), on(s.rot), on(s.lattice)

    def value_and_gradient(x):
        f, g = [], []
        for k in range(len(s.centers)):
            scaled = ((x - centers[k]) @ rot[k]) / axes[k]
            rad = scaled.norm(dim=1)
            f.append(rad - 1)
            g.append(((scaled / axes[k]) @ rot[k].T) / rad.clamp_min(1e-12)[:, None])
        f, g = torch.stack(f, 1), torch.stack(g, 1)
        w = torch.softmax(-f / s.smooth, 1)
        return -s.smooth * torch.logsumexp(-f / s.smooth, 1), (w[:, :, None] * g).sum(1)

    def density(x):
        t = ((x + 1) * 4).clamp(0, 7.999)
        i = t.floor().long()
        f = t - i
        f = f * f * (3 - 2 * f)
        out = torch.zeros(len(x), dtype=torch.float64, device=DEVICE)
        for c in range(8):
            o = [(c >> 2) & 1, (c >> 1) & 1, c & 1]
            w = torch.ones_like(out)
            for a in range(3):
                w = w * (f[:, a] if o[a] else 1 - f[:, a])
            out += w * lattice[i[:, 0] + o[0], i[:, 1] + o[1], i[:, 2] + o[2]]
        lo, hi = float(s.lattice.min()), float(s.lattice.max())
        return 0.1 + 0.9 * (out - lo) / (hi - lo)

    pts, nrm, have = [], [], 0
    while have < count:
        m = 3 * (count - have) + 4096
        k = torch.randint(0, len(s.centers), (m,), generator=gen, device=DEVICE)
        x = centers[k] + torch.bmm(rot[k], (axes[k] * _directions(gen, m))[:, :, None])[:, :, 0]
        for _ in range(10):
            v, g = value_and_gradient(x)
            x = x - (v / (g * g).sum(1).clamp_min(1e-20))[:, None] * g
        v, g = value_and_gradient(x)
        ok = (v.abs() < 1e-9) & (_uniform(gen, m) < density(x))
        pts.append(x[ok])
        nrm.append(g[ok] / g[ok].norm(dim=1, keepdim=True))
        have += len(pts[-1])
    p, n = torch.cat(pts)[:count], torch.cat(nrm)[:count]
    return p + noise * torch.randn(p.shape, generator=gen, dtype=torch.float64, device=DEVICE), n


def _displaced(gen, count, amplitude=0.05):
    """Unit sphere displaced radially by amplitude sin(6 theta) cos(4 phi), analytic normals."""
    d = _directions(gen, count)
    theta, phi = d[:, 2].clamp(-1, 1).acos(), torch.atan2(d[:, 1], d[:, 0])
    r = 1 + amplitude * (6 * theta).sin() * (4 * phi).cos()
    rt, rp = 6 * amplitude * (6 * theta).cos() * (4 * phi).cos(), -4 * amplitude * (6 * theta).sin() * (4 * phi).sin()
    et = torch.stack([theta.cos() * phi.cos(), theta.cos() * phi.sin(), -theta.sin()], 1)
    ep = torch.stack([-phi.sin(), phi.cos(), torch.zeros_like(phi)], 1)
    n = r[:, None] * d - rt[:, None] * et - (rp / theta.sin().clamp_min(1e-12))[:, None] * ep
    return d * r[:, None], n / n.norm(dim=1, keepdim=True)


def _cloud(shape, gen, count):
    if shape == "sphere":
        n = _directions(gen, count)
        return n.clone(), n
    return {"torus": _torus, "union": _union, "displaced": _displaced}[shape](gen, count)


def _cube_points(gen, p, count, scale=1.1):
    """Uniform points of the bounding cube."""
    lo, hi = p.amin(0), p.amax(0)
    return (_uniform(gen, (count, 3)) - 0.5) * ((hi - lo).max() * scale) + (hi + lo) / 2


def _options(case):
    return dict(depth=case["depth"], full_depth=case["full_depth"], point_weight=case.get("point_weight", 2.0),
                exact_interpolation=case.get("exact", False), iters=case.get("iters", 8), mixed=case.get("dtype") == "mixed")


def _field_arrays(depth, seed):
    """Sorted keys d<<48|x<<32|y<<16|z and coefficients of an octree field: levels 0..4 complete, then the corners of the
    cells near a sphere (float64, on the CPU)."""
    gen = torch.Generator().manual_seed(int(seed))
    radius = 0.3 + 0.05 * float(torch.rand(1, generator=gen, dtype=torch.float64))
    keys = []
    for d in range(depth + 1):
        n = 1 << d
        if d <= 4:
            axis = torch.arange(n + 1)
            c = torch.cartesian_prod(axis, axis, axis)
        else:
            dirs = torch.randn((24 << (2 * d), 3), generator=gen, dtype=torch.float64)
            cells = ((0.5 + radius * dirs / dirs.norm(dim=1, keepdim=True)) * n).floor().long()
            code = torch.unique((cells[:, 0] << 32) | (cells[:, 1] << 16) | cells[:, 2])
            offsets = torch.cartesian_prod(*[torch.tensor([0, 1])] * 3)
            code = torch.unique((code[:, None] + ((offsets[:, 0] << 32) | (offsets[:, 1] << 16) | offsets[:, 2])[None]).reshape(-1))
            c = torch.stack([code >> 32, (code >> 16) & 0xFFFF, code & 0xFFFF], 1)
        keys.append((d << 48) | (c[:, 0] << 32) | (c[:, 1] << 16) | c[:, 2])
    keys = torch.cat(keys)
    level = (keys >> 48).double()
    coefficients = torch.randn(len(keys), generator=gen, dtype=torch.float64) * torch.exp2(-level)
    cumulative = torch.randn(len(keys), generator=gen, dtype=torch.float64)
    queries = torch.rand((1 << 19, 3), generator=gen, dtype=torch.float64)
    queries[::2] = 0.5 + radius * (2 * queries[::2] - 1) / (2 * queries[::2] - 1).norm(dim=1, keepdim=True)
    # multiples of 2^-20: single precision maps them into the cube without rounding, so no query changes its cell
    queries = (queries * 2.0 ** 20).round() / 2.0 ** 20
    return keys, coefficients, cumulative, queries


def _field_linear(seed):
    """Model -> cube: a permuted similarity, as reconstruct() gives."""
    s = 0.5 ** (1 + int(seed) % 3)
    return np.array([0, s, 0, 0, 0, s, s, 0, 0], dtype=np.float64), np.array([0.125, 0.25, 0.0625])


def _field_queries(cube, linear, translation, dtype):
    """Model-space queries of cube points (the inverse of the permuted similarity)."""
    s = linear[1]
    q = (cube - torch.from_numpy(translation)) / s
    return q[:, [2, 0, 1]].to(dtype)


def prepare(case, seed):
    gen = _generator(seed)
    kind = case["kind"]
    if kind == "field":
        dtype = DTYPES[case["dtype"]]
        keys, coefficients, cumulative, cube = _field_arrays(case["depth"], seed)
        linear, translation = _field_linear(seed)
        q = _field_queries(cube[:case["queries"]], linear, translation, dtype).to(DEVICE)
        f = LevelField(keys.to(DEVICE), coefficients.to(dtype).to(DEVICE), linear, translation, case["depth"], 0.5,
                       cumulative=cumulative.to(dtype).to(DEVICE))
        return dict(kind=kind, field=f, queries=q.contiguous())
    if kind == "batch":
        dtype = DTYPES[case["dtype"]]
        clouds, options = [], []
        for i in range(case["clouds"]):
            # sizes spread over the range in the same way for each seed; shapes and depths alternate
            t = (i * 0.61803398875) % 1.0
            count = int(round(math.exp(math.log(case["smallest"]) * (1 - t) + math.log(case["largest"]) * t)))
            p, n = _cloud(("sphere", "torus", "union")[i % 3], gen, count)
            p = p * (0.2 + 1.8 * ((i * 0.7548776662) % 1.0)) + _uniform(gen, (1, 3), -5.0, 5.0)
            clouds.append((p.to(dtype).contiguous(), n.to(dtype).contiguous()))
            options.append(dict(depth=7 + (i % 2), full_depth=case["full_depth"], point_weight=case["point_weight"], iters=case["iters"],
                                mixed=case["dtype"] == "mixed"))
        return dict(kind=kind, clouds=clouds, options=options)
    dtype = DTYPES[case.get("dtype", "float32")]
    p, n = _cloud(case["shape"], gen, case["points"])
    if kind == "mesh":
        lo, hi = p.amin(0), p.amax(0)
        pad = 0.02 * (hi - lo)
        result = reconstruct(p.to(dtype).contiguous(), n.to(dtype).contiguous(), **_options(case))
        # a viewer's buffers of a fixed capacity: the draw call takes their size, so what a mesh leaves free is zero
        return dict(kind=kind, result=result, resolution=case["resolution"],
                    bounds=(tuple((lo - pad).tolist()), tuple((hi + pad).tolist())),
                    vertices=torch.zeros((8 * case["resolution"] ** 2, 3), dtype=torch.float32, device=DEVICE),
                    indices=torch.zeros(48 * case["resolution"] ** 2, dtype=torch.int32, device=DEVICE))
    extra = _cube_points(gen, p, case["queries"])
    if kind == "query":
        # half of the queries on the surface, half in the cube around it
        half = min(case["queries"] // 2, len(p))
        q = torch.cat([p[:half], extra[half:]]).to(dtype).contiguous()
        result = reconstruct(p.to(dtype).contiguous(), n.to(dtype).contiguous(), **_options(case))
        return dict(kind=kind, result=result, queries=q)
    p, n = p.to(dtype).contiguous(), n.to(dtype).contiguous()
    if kind == "recon":
        return dict(kind=kind, points=p, normals=n, queries=torch.cat([p, extra.to(dtype)]).contiguous(), options=_options(case))
    k = torch.randint(0, len(p), (case["queries"],), generator=gen, device=DEVICE)
    targets = (p[k] + 0.02 * torch.randn((len(k), 3), generator=gen, dtype=torch.float64, device=DEVICE).to(dtype)).contiguous()
    return dict(kind=kind, points=p, normals=n, queries=targets, options=_options(case), positions=case["positions"])


# -- one pass -------------------------------------------------------------------------------------------------------


def run(state):
    kind = state["kind"]
    if kind == "recon":
        result = reconstruct(state["points"], state["normals"], **state["options"])
        values, gradients, valid = result.evaluate(state["queries"])
        return dict(values=values, gradients=gradients, valid=valid, iso_value=result.iso_value)
    if kind == "batch":
        results = reconstruct_batch(state["clouds"], per_cloud=state["options"])
        return [[r.evaluate(p)[0], r.iso_value] for r, (p, _) in zip(results, state["clouds"])]
    if kind == "query":
        values, gradients, valid = state["result"].evaluate(state["queries"])
        return dict(values=values, gradients=gradients, valid=valid)
    if kind == "field":
        values, gradients, valid = state["field"].evaluate(state["queries"])
        return dict(values=values, gradients=gradients, valid=valid)
    if kind == "mesh":
        mesh = extract_mesh(state["result"], resolution=state["resolution"], bounds=state["bounds"])
        vertices, indices = state["vertices"], state["indices"]
        for buffer, new in ((vertices, mesh.vertices), (indices, mesh.indices)):
            buffer[:len(new)] = new
            buffer[len(new):] = 0
        return dict(vertices=vertices, indices=indices, counts=[len(mesh.vertices), len(mesh.indices)])
    normals = state["normals"].detach().requires_grad_(True)
    points = state["points"].detach().requires_grad_(state["positions"])
    queries = state["queries"].detach().requires_grad_(state["positions"])
    recon = reconstruct_differentiable(points, normals, **state["options"])
    values, gradients, _ = recon.evaluate(queries, centered=True)
    loss = (values * values).sum() + 1e-3 * (gradients * gradients).sum()
    loss.backward()
    out = dict(values=values.detach(), gradients=gradients.detach(), grad_normals=normals.grad)
    if state["positions"]:
        out.update(grad_points=points.grad, grad_queries=queries.grad)
    return out


# -- sizes ----------------------------------------------------------------------------------------------------------


def _rows(points, depth, full_depth):
    """About how many basis functions each level has: the complete grid down to full_depth, then the smaller of what
    the surface's cells and what the points give."""
    return [(2 ** d + 1) ** 3 if d <= full_depth else min((2 ** d + 1) ** 3, ROWS_PER_CELL * 4 ** d, ROWS_PER_POINT * points)
            for d in range(depth + 1)]


def _recon_work(points, depth, full_depth, iters, value, operator):
    """One reconstruction: points and normals in, one key, coefficient and cumulative coefficient per basis function out.
    Operations: `iters` relaxation sweeps of 27-point rows (a product and a sum a slot) and their assembly (a few sums of
    products a slot).  Bytes beyond the inputs and outputs: each level's operator written and read once."""
    rows = sum(_rows(points, depth, full_depth))
    return (2 * 3 * value * points + rows * (8 + 2 * value) + rows * 27 * operator * 2,
            rows * 27 * (2 * iters + 2 * 16))


def _query_work(queries, value, grads=True):
    """27 coefficients of three levels are blended; queries in, values, gradients and validity out."""
    return queries * (3 * value + value + (3 * value if grads else 0) + 4), queries * 3 * 8 * 20


def work(case):
    kind = case["kind"]
    value = 8 if case.get("dtype") in ("float64", "mixed") else 4
    operator = 8 if case.get("dtype") == "float64" else 4
    if kind == "recon":
        a = _recon_work(case["points"], case["depth"], case["full_depth"], case["iters"], value, operator)
        b = _query_work(case["points"] + case["queries"], value)
    elif kind == "batch":
        a, b = (0, 0), (0, 0)
        for i in range(case["clouds"]):
            t = (i * 0.61803398875) % 1.0
            count = math.exp(math.log(case["smallest"]) * (1 - t) + math.log(case["largest"]) * t)
            x = _recon_work(count, 7 + i % 2, case["full_depth"], case["iters"], value, operator)
            y = _query_work(count, value, grads=False)
            a, b = (a[0] + x[0], a[1] + x[1]), (b[0] + y[0], b[1] + y[1])
    elif kind == "query":
        a, b = (0, 0), _query_work(case["queries"], value)
    elif kind == "field":
        a, b = (0, 0), _query_work(case["queries"], value)
    elif kind == "mesh":
        # every node's value decides its cells; about six crossing cells per res^2, two triangles and a vertex each
        nodes, crossing = case["resolution"] ** 3, 6 * case["resolution"] ** 2
        a, b = (crossing * (12 + 24), 0), (nodes / 8, nodes * 3 * 8 * 8)
    else:
        a = _recon_work(case["points"], case["depth"], case["full_depth"], 8, value, operator)
        b = _query_work(case["queries"], value)
        # the reverse of every step once more, gradients of each input out; with positions the matrices' side too
        again = 3 if case["positions"] and case["point_weight"] > 0 else 2
        a, b = (again * a[0], again * a[1]), (2 * b[0], 2 * b[1])
    return {"bytes": float(a[0] + b[0]), "flops": float(a[1] + b[1])}


# -- what the results are held to -----------------------------------------------------------------------------------


def tolerance(case):
    """About four times the largest difference between a cloud and the same cloud with its points in another order, whose
    group sums, and all that follows from them, round differently: over these cases and 24 drawn ones.  Single precision
    loses about a bit a level.  Mixed precision rounds the operators to 32 bits, so a last bit of 64 now and then becomes
    one of 32."""
    kind, dtype = case["kind"], case.get("dtype", "float32")
    if kind == "field":
        return {"rel": 1e-14} if dtype == "float64" else {"rel": 3e-7}
    if kind == "backward":
        if dtype == "float64":
            return {"rel": 1.5e-13, "max": 2e-12}
        rel = 2e-5 * 2.0 ** (case["depth"] - 5)
        return {"rel": rel, "max": 12 * rel}
    if dtype == "float64":
        return {"rel": 2e-13, "max": 5e-12}
    if dtype == "mixed":
        return {"rel": 4e-11, "max": 1e-8}
    rel = 2.5e-6 * 2.0 ** (case.get("depth", 8) - 4)
    return {"rel": rel, "max": 15 * rel}


def exact(case, seed):
    """A stored field's values and gradients in 64 bits from its arrays.  A reconstruction's stages (sorted sums, an octree
    chosen by them, a cascadic solve) have no short plain form: None."""
    if case["kind"] != "field":
        return None
    dtype, depth = DTYPES[case["dtype"]], case["depth"]
    keys, coefficients, cumulative, cube = _field_arrays(depth, seed)
    linear, translation = _field_linear(seed)
    q = _field_queries(cube[:case["queries"]], linear, translation, dtype).double()
    coefficients, cumulative = coefficients.to(dtype).double(), cumulative.to(dtype).double()
    L = torch.from_numpy(linear).reshape(3, 3)
    p = q @ L.T + torch.from_numpy(translation)
    valid = ((p >= 0) & (p <= 1)).all(1)

    def find(d, c):
        key = (d << 48) | (c[:, 0] << 32) | (c[:, 1] << 16) | c[:, 2]
        at = torch.searchsorted(keys, key).clamp_max(len(keys) - 1)
        return torch.where(keys[at] == key, at, -1)

    def cell(d):
        return (torch.ceil(p * (1 << d)).long() - 1).clamp(0, (1 << d) - 1)

    leaf = torch.zeros(len(p), dtype=torch.long)
    for d in range(depth + 1):
        leaf = torch.where(find(d, cell(d)) >= 0, d, leaf)
    p = torch.where(p == 0, 1e-6, torch.where(p == 1, 1.0 - 1e-6, p))

    def level(values, d):
        """Trilinear blend of level d's values at the corners of each query's cell: value and cube-space gradient."""
        n, c, out = 1 << d, cell(d), torch.zeros((len(p), 4), dtype=torch.float64)
        t = p * n - torch.floor(p * n)
        base = torch.floor(p * n).long()
        for corner in range(8):
            node = c + torch.tensor([corner // 4, corner // 2 % 2, corner % 2])
            at = find(d, node)
            v = torch.where((at >= 0) & (node >= base).all(1), values[at.clamp_min(0)], 0.0)
            up = node > base
            h, g = torch.where(up, t, 1 - t), torch.where(up, float(n), -float(n))
            out[:, 0] += v * h[:, 0] * h[:, 1] * h[:, 2]
            out[:, 1] += v * g[:, 0] * h[:, 1] * h[:, 2]
            out[:, 2] += v * h[:, 0] * g[:, 1] * h[:, 2]
            out[:, 3] += v * h[:, 0] * h[:, 1] * g[:, 2]
        return out

    total = torch.zeros((len(p), 4), dtype=torch.float64)
    for d in range(depth + 1):
        total += torch.where((leaf == d)[:, None], level(coefficients, d), 0.0)
        total += torch.where((leaf == d + 1)[:, None], level(cumulative, d), 0.0)
        if d:
            total += torch.where((leaf == d - 1)[:, None], level(coefficients, d), 0.0)
    total[~valid] = math.nan
    return dict(values=total[:, 0], gradients=total[:, 1:] @ L, valid=None)
