"""The measured workloads of the SES mesh path: what a program asks of this library, from the
smallest molecule to a million atoms, one at a time, batched, served, and from host arrays.

Molecules come from the library's seeded generator: atoms uniform in a ball at 0.05 atoms/A^3 (or
in a spherical shell) with 1.2 A minimum distance, radii drawn from the C/O/N/H/S mix.  Inputs are
float32, as every entry point takes them; the mesh is float32 vertices, int32 triangles and int32
atom ids.  The library's result arrays are valid until its next call, so the program keeps a mesh
by copying it to arrays of its own, which have room for more than the mesh (the rest stays zero).
A case is one call sequence of one kind:

  device    qs_compute_device: atoms in device memory, mesh left there
  noalloc   qs_compute_device_noalloc: the same, written to the program's arrays by the library
  normals   qs_compute_device, then qs_vertex_normals_device for shading
  host      API_computeSES: host arrays in and out
  batch     qs_compute_batch_device: molecules of different sizes in one launch sequence
  frames    the same for frames of a trajectory (one molecule, coordinates jittered by 0.3 A)
  serve     a Server: requests of mixed sizes and voxel sizes submitted together, each polled for
            its device-resident mesh and released
"""
import math

import numpy as np
import torch

import quickses_amd as qs
from quickses_amd import hipmem

PROBE = 1.4
SERVED_VOXELS = (0.3, 0.5, 1.0)
TRAJECTORY_SIGMA = 0.3


def listed():
    return [
        # a peptide in a coarse preview: launches and latency are all there is
        dict(name="device_300_1.0A", kind="device", atoms=300, voxel=1.0, smooth=1),
        # a small protein at the tool's default voxel size, the common interactive call
        dict(name="device_2000_0.5A", kind="device", atoms=2000, voxel=0.5, smooth=1),
        # a serving loop that owns its buffers and may not allocate
        dict(name="noalloc_5003_0.5A", kind="noalloc", atoms=5003, voxel=0.5, smooth=0),
        # a viewer: surface and normals of a mid-size protein at an odd grid size
        dict(name="normals_10007_0.4A", kind="normals", atoms=10007, voxel=0.4, smooth=0),
        # a plugin on the C interface: host arrays both ways
        dict(name="host_3000_0.5A", kind="host", atoms=3000, voxel=0.5, smooth=1),
        # the benchmark: a large complex at high resolution
        dict(name="device_50000_0.2A", kind="device", atoms=50000, voxel=0.2, smooth=1),
        # a virus capsid part, unsmoothed
        dict(name="device_200000_0.3A", kind="device", atoms=200000, voxel=0.3, smooth=0),
        # the same size as an overview
        dict(name="device_200000_1.0A", kind="device", atoms=200000, voxel=1.0, smooth=1),
        # a capsid shell of a million atoms, two smoothing passes
        dict(name="device_shell_1M_0.5A", kind="device", atoms=1000000, inner=120.0, voxel=0.5, smooth=2),
        # a library of molecules meshed in one sequence
        dict(name="batch_256_0.5A", kind="batch", molecules=256, lo=500, hi=20000, size_seed=4, voxel=0.5, mixed=False, smooth=1),
        # a trajectory
        dict(name="frames_100x10000_0.5A", kind="frames", frames=100, atoms=10000, voxel=0.5, smooth=1),
        # a burst of requests at a server
        dict(name="serve_16", kind="serve", requests=16, lo=1000, hi=50000, size_seed=5, smooth=1),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _ball_radius(atoms, inner=0.0):
    return (atoms / 0.05 * 3.0 / (4.0 * math.pi) + inner ** 3) ** (1.0 / 3.0)


def _voxels(atoms, voxel, inner=0.0):
    """Grid points of a ball's (or shell's) grid, by the grid rule."""
    return math.ceil((2.0 * _ball_radius(atoms, inner) + 2.0 * 1.8 + 4.0 * PROBE) / voxel) ** 3


def draw(rng):
    """One more case of the listed ranges; at most the largest listed grids and atom counts."""
    kind = rng.choice(["device"] * 6 + ["noalloc", "normals", "host", "batch", "frames"])
    voxel = rng.choice([0.2, 0.25, 0.3, 0.37, 0.4, 0.5, 0.5, 0.75, 1.0])
    smooth = rng.choice([0, 1, 1, 2])
    if kind == "batch":
        voxel = rng.choice([0.5, 0.75, 1.0])
        return dict(kind=kind, molecules=_log_uniform(rng, 2, 200), lo=500, hi=15000, size_seed=rng.randrange(1 << 16), voxel=voxel,
                    mixed=rng.random() < 0.3, smooth=smooth)
    if kind == "frames":
        atoms = _log_uniform(rng, 500, 12000)
        return dict(kind=kind, frames=min(_log_uniform(rng, 2, 120), max(2, int(2.5e8 / _voxels(atoms, 0.5)))), atoms=atoms, voxel=0.5,
                    smooth=smooth)
    budget = {"device": 3.0e8, "noalloc": 1.2e7, "normals": 6.0e7, "host": 6.0e7}[kind]
    largest = {"device": 600000, "noalloc": 20000, "normals": 100000, "host": 100000}[kind]
    hollow = rng.choice([0.0, 0.0, 0.0, 0.5, 0.9]) if kind == "device" else 0.0  # of the same atoms' ball radius
    lo, hi = 300, largest
    while hi > lo and _voxels(hi, voxel, hollow * _ball_radius(hi)) > budget:
        hi = max(lo, int(hi * 0.95))
    case = dict(kind=kind, atoms=_log_uniform(rng, lo, hi), voxel=voxel, smooth=smooth)
    if hollow:
        case["inner"] = round(hollow * _ball_radius(case["atoms"]), 1)
    return case


# ------------------------------------------------------------------------------------------ #
# inputs


def _molecule(case, seed):
    inner = case.get("inner", 0.0)
    if not inner:
        return qs.synth_ball(seed, case["atoms"])
    return qs.synth_shell(seed, case["atoms"], inner, _ball_radius(case["atoms"], inner))


def _items(case, seed):
    """Molecules and voxel sizes of a batch, a trajectory or a burst of requests."""
    if case["kind"] == "frames":
        base, rad = qs.synth_ball(seed, case["atoms"])
        items = [(qs.synth_jitter(seed + 1 + f, base, TRAJECTORY_SIGMA), rad) for f in range(case["frames"])]
        return items, [case["voxel"]] * len(items)
    count = case["molecules"] if case["kind"] == "batch" else case["requests"]
    sizes = qs.synth_sizes(case["size_seed"], count, case["lo"], case["hi"])
    items = [qs.synth_ball(1000 * seed + i, int(n)) for i, n in enumerate(sizes)]
    if case["kind"] == "serve" or case["mixed"]:
        return items, [float(v) for v in np.random.default_rng(case["size_seed"]).choice(SERVED_VOXELS, size=count)]
    return items, [case["voxel"]] * count


def _surface_vertices(case):
    """About the vertices of a case's meshes: v dx^2 / atom of the generator's balls."""
    def one(atoms, voxel):
        return atoms / (voxel * voxel) * (2.4 + 48.0 * atoms ** (-1.0 / 3.0))

    if case["kind"] in ("batch", "serve"):
        n = case["molecules"] if case["kind"] == "batch" else case["requests"]
        mean = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        return n * mean, n * one(mean, case.get("voxel", 0.5))
    if case["kind"] == "frames":
        return case["frames"] * case["atoms"], case["frames"] * one(case["atoms"], case["voxel"])
    return case["atoms"], one(case["atoms"], case["voxel"])


_server = None


def _the_server():
    """The program's one server (a process has at most one)."""
    global _server
    if _server is None:
        _server = qs.Server(hbm_budget_bytes=16 << 30, result_bytes=4 << 30, workers=2)
    return _server


def _room(case):
    """Vertices that the program's arrays hold (twice as many triangles)."""
    return int(2.0 * _surface_vertices(case)[1]) + 4096


def _arrays(case, room):
    names = dict(vertices=((room, 3), torch.float32), triangles=((2 * room, 3), torch.int32), atom_ids=((room,), torch.int32))
    if case["kind"] == "normals":
        names["normals"] = ((room, 3), torch.float32)
    where = "cpu" if case["kind"] == "host" else "cuda"
    return {k: torch.zeros(shape, dtype=dtype, device=where) for k, (shape, dtype) in names.items()}


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case=case, mesh=_arrays(case, _room(case)))
    if kind in ("batch", "frames", "serve"):
        items, voxels = _items(case, seed)
    if kind == "serve":
        state.update(server=_the_server(), items=items, voxels=voxels)
        return state
    if kind in ("batch", "frames"):
        pos = np.concatenate([p for p, _ in items])
        rad = np.concatenate([r for _, r in items])
        state.update(counts=[len(r) for _, r in items], voxels=np.array(voxels, dtype=np.float32))
    else:
        pos, rad = _molecule(case, seed)
    if kind == "host":
        state.update(pos=pos, rad=rad)
        state["mesh"] = {k: v.numpy() for k, v in state["mesh"].items()}
        return state
    state.update(pos=torch.from_numpy(pos).cuda(), rad=torch.from_numpy(rad).cuda(), atoms=len(rad))
    torch.cuda.synchronize()
    return state


def _keep(mesh, nvert, ntri, vert, tri, atom, v0=0, t0=0):
    """Copies a library-owned mesh to the program's arrays, from vertex v0 and triangle t0 on."""
    if v0 + nvert > len(mesh["vertices"]) or t0 + ntri > len(mesh["triangles"]):
        raise RuntimeError("the mesh has no room")
    copy = hipmem.hip().hipMemcpy
    bad = copy(mesh["vertices"].data_ptr() + 12 * v0, vert, 12 * nvert, hipmem.D2D)
    bad |= copy(mesh["triangles"].data_ptr() + 12 * t0, tri, 12 * ntri, hipmem.D2D)
    bad |= copy(mesh["atom_ids"].data_ptr() + 4 * v0, atom, 4 * nvert, hipmem.D2D)
    if bad:
        raise RuntimeError("the mesh was not copied")


def run(state):
    case, mesh = state["case"], state["mesh"]
    kind = case["kind"]
    if kind == "host":
        v, t, a = qs.compute_ses(state["pos"], state["rad"], case["voxel"], case["smooth"], copy=False)
        mesh["vertices"][:len(v)], mesh["triangles"][:len(t)], mesh["atom_ids"][:len(a)] = v, t, a
        return dict(mesh, counts=[len(v), len(t)])
    if kind == "serve":
        server = state["server"]
        ids = [server.submit(p, r, v, case["smooth"]) for (p, r), v in zip(state["items"], state["voxels"])]
        counts, v0, t0 = [], 0, 0
        for rid in ids:
            got = server.poll(rid)
            _keep(mesh, got["nvert"], got["ntri"], got["d_vert"], got["d_tri"], got["d_atom"], v0, t0)
            v0, t0 = v0 + got["nvert"], t0 + got["ntri"]
            counts.append([got["nvert"], got["ntri"]])
        hipmem.synchronize()  # the results are copied: their memory may go
        for rid in ids:
            server.release(rid)
        return dict(mesh, counts=np.array(counts))
    pos, rad = state["pos"].data_ptr(), state["rad"].data_ptr()
    if kind == "noalloc":
        v, t, a = mesh["vertices"], mesh["triangles"], mesh["atom_ids"]
        nv, ni = qs.compute_device_noalloc(pos, rad, state["atoms"], case["voxel"], case["smooth"], v.data_ptr(), v.shape[0], t.data_ptr(),
                                           t.shape[0], a.data_ptr())
        return dict(mesh, counts=[nv, ni // 3])
    if kind in ("batch", "frames"):
        vo, to, v, t, a = qs.compute_batch_device(pos, rad, state["counts"], state["voxels"], case["smooth"])
        _keep(mesh, int(vo[-1]), int(to[-1]), v, t, a)
        counts = np.stack([vo, to]).astype(np.int64)
    else:
        nv, ni, v, t, a = qs.compute_device(pos, rad, state["atoms"], case["voxel"], case["smooth"])
        _keep(mesh, nv, ni // 3, v, t, a)
        counts = [nv, ni // 3]
        if kind == "normals":
            qs.vertex_normals_device(mesh["normals"].data_ptr())
    hipmem.synchronize()  # the library's next call may overwrite its arrays
    return dict(mesh, counts=counts)


def work(case):
    """Atoms read once (16 B) and the mesh written once: 16 B a vertex, two triangles of 12 B a
    vertex (and 12 B of normal); a distance, an edge's crossing and the closest atom a vertex."""
    atoms, verts = _surface_vertices(case)
    per_vertex = 40 + (12 if case["kind"] == "normals" else 0)
    return dict(bytes=16.0 * atoms + per_vertex * verts, flops=100.0 * verts)


# ------------------------------------------------------------------------------------------ #
# 64-bit values


def _labels(pos, rad, voxel):
    """Grid origin and the voxel labels' outside and shell masks.  A label is a decision in single
    precision by the method's definition, so it is made in single precision; every number that is
    computed from the labels is in 64 bits."""
    f = np.float32
    voxel, probe = f(voxel), f(PROBE)
    lo, hi, rmax = pos.min(axis=0), pos.max(axis=0), rad.max()
    dist = f(f((hi - lo).max() + f(f(2) * rmax)) + f(f(4) * probe))
    origin = (lo - rmax) - probe
    g, r = int(np.ceil(dist / voxel)), int(np.ceil(probe / voxel))
    d_pos, d_rad = torch.from_numpy(pos).cuda(), torch.from_numpy(rad).cuda()
    axis = [torch.from_numpy(origin[a] + np.arange(g, dtype=f) * voxel).cuda() for a in range(3)]
    near = torch.zeros(g * g * g, dtype=torch.bool, device="cuda")
    inside = torch.zeros_like(near)
    half = int(math.ceil((float(rmax) + PROBE) / float(voxel))) + 1
    span = torch.arange(-half, half + 1, device="cuda")
    step = max(1, int(1.6e7) // len(span) ** 3)
    for s in range(0, len(rad), step):
        p, q = d_pos[s:s + step], d_rad[s:s + step]
        at, sq = [], []
        for a in range(3):
            i = (((p[:, a].double() - float(origin[a])) / float(voxel)).floor().long()[:, None] + span[None, :])
            e = p[:, a, None] - axis[a][i.clamp(0, g - 1)]
            sq.append(torch.where((i >= 0) & (i < g - 1), e * e, torch.full_like(e, 1e9)))
            at.append(i.clamp(0, g - 1))
        d = (sq[0][:, :, None, None] + sq[1][:, None, :, None]) + sq[2][:, None, None, :]
        d = d.double().sqrt().float()
        lin = (at[0][:, :, None, None] * g + at[1][:, None, :, None]) * g + at[2][:, None, None, :]
        near[lin[d < (q + float(probe))[:, None, None, None]]] = True
        inside[lin[d < (q - float(voxel))[:, None, None, None]]] = True
    outside, shell = (~near).view(g, g, g), (near & ~inside).view(g, g, g)
    return origin, g, r, outside, shell


def _window_norm(outside, r):
    """Smallest squared integer distance to an outside point within r along every axis."""
    n = torch.where(outside, 0, 10000).to(torch.int16)
    for axis in range(3):
        best = n.clone()
        size = n.shape[axis]
        for s in range(1, min(r, size - 1) + 1):
            for a, b in ((0, s), (s, 0)):
                part = best.narrow(axis, a, size - s)
                torch.minimum(part, n.narrow(axis, b, size - s) + s * s, out=part)
        n = best
    return n


def _vertices64(pos, rad, voxel, normals):
    """Unsmoothed vertices (and unit field gradients) in (grid point, axis) order, or None where
    field values of exactly zero make the vertices' number a matter of rounding."""
    dx, probe = float(np.float32(voxel)), float(np.float32(PROBE))
    if abs((PROBE / voxel) ** 2 - round((PROBE / voxel) ** 2)) < 1e-3:
        return None, None
    origin, g, r, outside, shell = _labels(pos, rad, voxel)
    n = _window_norm(outside, r)
    field = torch.where(outside, probe, -dx).double()
    reach = shell & (n < 10000)
    field[reach] = probe - dx * n[reach].double().sqrt()
    del n, reach, shell, outside
    neg = field < 0
    ids, axes = [], []
    for a in range(3):
        cut = torch.zeros_like(neg)
        cut.narrow(a, 0, g - 1).copy_(neg.narrow(a, 0, g - 1) ^ neg.narrow(a, 1, g - 1))
        ids.append(cut.view(-1).nonzero()[:, 0])
        axes.append(torch.full_like(ids[-1], a))
    key, order = (torch.cat(ids) * 4 + torch.cat(axes)).sort()
    point, a = key // 4, key % 4
    stride = torch.tensor([g * g, g, 1], device="cuda")
    other = point + stride[a]
    flat = field.view(-1)
    t = -flat[point] / (flat[other] - flat[point])
    cell = torch.stack([point // (g * g), point // g % g, point % g], 1)
    unit = torch.nn.functional.one_hot(a, 3).double()
    vert = torch.from_numpy(origin.astype(np.float64)).cuda() + (cell.double() + t[:, None] * unit) * dx
    if not normals:
        return vert, None

    def gradient(at, c):
        parts = []
        for k in range(3):
            up, down = (c[:, k] < g - 1).long(), (c[:, k] > 0).long()
            parts.append((flat[at + up * stride[k]] - flat[at - down * stride[k]]) / ((up + down).double() * dx))
        return torch.stack(parts, 1)

    grad = (1 - t)[:, None] * gradient(point, cell) + t[:, None] * gradient(other, cell + unit.long())
    return vert, grad / grad.norm(dim=1, keepdim=True)


def exact(case, seed):
    """Unsmoothed vertices and normals have values in 64 bits; a smoothed vertex is a mean over a
    neighbour list that the case table's triangles define, and has none here."""
    if case["smooth"] or case["kind"] in ("batch", "frames", "serve"):
        return None
    vert, normal = _vertices64(*_molecule(case, seed), case["voxel"], case["kind"] == "normals")
    if vert is None:
        return None
    out = dict(triangles=None, atom_ids=None, counts=None)
    for name, v in (("vertices", vert), ("normals", normal)):
        if v is not None:
            out[name] = torch.zeros((_room(case), 3), dtype=torch.float64, device="cuda")
            out[name][:len(v)] = v
    return out
