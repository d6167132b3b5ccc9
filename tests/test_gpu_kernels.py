"""Kernels at the sizes and inputs where their rules change, against the CPU oracle (bit for bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _same(a, b):
    return (a[0].shape == b[0].shape and a[1].shape == b[1].shape and np.array_equal(a[1], b[1])
            and np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32)) and np.array_equal(a[2], b[2]))


def _closest_case(qs, kind):
    pos, rad = qs.synth_ball(61, 400)
    if kind == "every atom twice":  # equal distances at every vertex: the first in (cell, index) order wins
        return np.repeat(pos, 2, axis=0), np.repeat(rad, 2)
    if kind == "far from the origin":  # coordinates in steps of 2^-9 A: many sums and roots agree
        return pos + np.float32(20000.0), rad
    if kind == "two atoms":  # a grid of a few cells, every column next to a clamped one
        return np.array([[0, 0, 0], [3, 0, 0]], np.float32), np.array([1.7, 1.7], np.float32)
    ax = np.arange(-2, 3, dtype=np.float32) * np.float32(2.5)  # mirror planes on grid planes
    return np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3), np.full(125, 1.6, np.float32)


@pytest.mark.parametrize("kind", ["every atom twice", "far from the origin", "two atoms", "mirror planes"])
@pytest.mark.parametrize("reso", [0.25, 0.5])
def test_closest_atom_ties_and_clamps(qs, orc, kind, reso):
    pos, rad = _closest_case(qs, kind)
    print("case closest atom: %s reso=%.2f" % (kind, reso), flush=True)
    assert _same(qs.compute_ses(pos, rad, reso, 0), orc.compute_ses(pos, rad, reso, 0))


def _far_cells_case(qs, kind):
    rng = np.random.default_rng(11)
    if kind == "two large atoms":  # 7 A from their vertices: past the octant's cells on every side
        return np.array([[0, 0, 0], [3, 0, 0]], np.float32), np.full(2, 7.0, np.float32)
    if kind == "mixed radii":  # large empty cells beside crowded ones
        return (rng.random((60, 3)) * 40).astype(np.float32), np.where(rng.random(60) < 0.1, 6.0, 0.9).astype(np.float32)
    n, step = 9, np.float32(3.25)  # every atom on a cell boundary (cell size 3.25), 1000 A off the origin
    ax = np.arange(n, dtype=np.float32) * step + np.float32(1000.0)
    pos = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
    return pos[rng.random(len(pos)) < 0.4], np.full(n ** 3, 1.85, np.float32)


@pytest.mark.parametrize("kind", ["two large atoms", "mixed radii", "cell boundaries"])
@pytest.mark.parametrize("reso", [0.3, 0.5])
def test_closest_atom_beyond_the_octant(qs, orc, kind, reso):
    """The closest atom in a cell of the far side, in none, and on the boundary of two."""
    pos, rad = _far_cells_case(qs, kind)
    rad = rad[:len(pos)]
    print("case far cells: %s reso=%.2f" % (kind, reso), flush=True)
    assert _same(qs.compute_ses(pos, rad, reso, 0), orc.compute_ses(pos, rad, reso, 0))


def _noise_field(g, kind):
    rng = np.random.default_rng(100 * g + len(kind))
    f = rng.standard_normal((g, g, g)).astype(np.float32)  # nearly every cube polygonised
    if kind == "noise with zeros":
        f[rng.random(f.shape) < 0.2] = 0.0
    elif kind == "sheet":  # words of a few cubes beside words without vertices, zeros on the sheet
        x, y, z = np.meshgrid(*[np.arange(g, dtype=np.float32)] * 3, indexing="ij")
        f = (z - np.float32(0.75 * g) + np.float32(0.5) * (x % 3)).astype(np.float32)
    return f.ravel()


@pytest.mark.parametrize("kind", ["noise", "noise with zeros", "sheet"])
@pytest.mark.parametrize("g", [2, 5, 63, 64, 65, 66, 130])
def test_mesh_of_any_field(qs, orc, g, kind):
    """Emission over whole words of cubes, cubes across two row words, and zero grid points."""
    s = orc._Grid()
    s.g, s.gn, s.r, s.reso, s.dx_n = g, 1, 3, 0.5, 3.2
    G = orc.Grid(s)
    fld = _noise_field(g, kind)
    for lim in (g - 1, max(1, g - 3)):
        print("case mesh of a field: %s g=%d lim=%d" % (kind, g, lim), flush=True)
        V, T = qs.stage_mesh(G.params(lim), fld)
        Vo, To = orc.edge_weld(G, lim, fld)
        assert np.array_equal(T, To)
        assert np.array_equal(V.view(np.uint32), Vo.view(np.uint32))


@pytest.mark.parametrize("reso,n", [(0.16, 60), (0.2, 300), (0.28, 300), (0.35, 400), (0.5, 800), (0.7, 800), (1.0, 1500), (1.4, 1500),
                                    (1.6, 1500)])
@pytest.mark.parametrize("offset", [0.0, 30000.0])
def test_field_values_left_out_and_completed(qs, orc, reso, n, offset):
    """A mesh whose field pass stored only the values it reads equals the oracle's, the field asked
    for afterwards is whole, and the mesh after a normals call (which stores every value) is the same."""
    pos, rad = qs.synth_ball(78, n)
    pos = pos + np.float32(offset)
    print("case field left out: reso=%.2f offset=%g" % (reso, offset), flush=True)
    ref = orc.compute_ses(pos, rad, reso, 1)
    first = qs.compute_ses(pos, rad, reso, 1)
    assert _same(first, ref)
    g = qs.last_grid()["g"]
    whole = qs.fetch("field", np.float32, g ** 3)
    assert np.array_equal(whole.view(np.uint32), orc.field(pos, rad, reso)[6].view(np.uint32))
    a = qs.compute_ses(pos, rad, reso, 1)
    normals = qs.vertex_normals(len(a[0]))
    b = qs.compute_ses(pos, rad, reso, 1)
    assert np.array_equal(qs.vertex_normals(len(b[0])).view(np.uint32), normals.view(np.uint32))
    assert _same(a, ref) and _same(b, ref)


@pytest.mark.parametrize("n", [3, 6])
def test_mesh_beyond_the_expected_size(qs, orc, n):
    """Separate spheres have several times the surface that a launch expects of so many atoms: the
    pools are grown and the launches' blocks take more than one block of items."""
    ax = np.arange(n, dtype=np.float32) * np.float32(7.0)
    pos = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3)
    rad = np.full(len(pos), 1.7, np.float32)
    print("case separate spheres n=%d" % len(rad), flush=True)
    for _ in range(2):  # with the pools of the start, then with grown ones
        assert _same(qs.compute_ses(pos, rad, 0.5, 1), orc.compute_ses(pos, rad, 0.5, 1))


@pytest.mark.parametrize("n", [1278, 1279])
def test_dropped_triangles_with_and_without_the_count_scan(qs, orc, n):
    """Degenerate triangles dropped (a probe of seven whole voxels gives zero grid points) from pools
    of 2,047 and 2,049 blocks: up to 2,048 each block adds up the counts before it itself."""
    pos, rad = qs.synth_ball(5, n)
    print("case dropped triangles: n=%d" % n, flush=True)
    assert _same(qs.compute_ses(pos, rad, 0.2, 1), orc.compute_ses(pos, rad, 0.2, 1))


@pytest.mark.parametrize("n", [5, 1025, 4097, 8191, 8192, 8193])
def test_bounding_box_on_the_device(qs, n):
    """The box found by one block (up to 8,192 atoms) or several is the host's: the same mesh."""
    from quickses_amd import hipmem

    pos, rad = qs.synth_ball(17, n)
    pos[n // 2] += np.float32(9.0)  # one atom alone sets three faces
    dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(rad)
    print("case device box: n=%d" % n, flush=True)
    nv, ni, pv, pt, pa = qs.compute_device(dp.ptr, dr.ptr, n, 1.0, 0)
    got = (hipmem.download(pv, (nv, 3), np.float32), hipmem.download(pt, (ni // 3, 3), np.int32), hipmem.download(pa, (nv,), np.int32))
    assert nv > 0 and _same(got, qs.compute_ses(pos, rad, 1.0, 0))


def _cells_fetch(qs, what, n, dtype):
    import ctypes

    out = np.empty(n, dtype)
    got = qs.lib().qs_fetch(what, ctypes.c_void_p(out.ctypes.data), ctypes.c_int64(out.nbytes))
    assert got == out.nbytes
    return out


@pytest.mark.parametrize("sizes,box", [
    ([2], 0), ([1023], 0), ([1025], 0), ([4096], 0), ([4097], 0), ([12288], 0), ([12289], 0),
    ([1, 700, 0, 4096, 64, 2, 1024, 3000], 0), ([24576, 1, 5000, 0, 64, 2, 1024, 3000], 0), ([24577, 1, 5000, 0, 64, 2, 1024, 3000], 0),
    ([200], 104.0), ([200], 110.0)])
def test_cells_in_one_block_or_several_launches(qs, sizes, box):
    """The cell order (cell, then index) and the cells' ranges at the sizes where one block takes over:
    atoms gathered in the same launch up to 4,096, one molecule up to 12,288 atoms, a batch up to
    24,576, and 49,152 cells (a box of 104 A has 36^3 cells, of 110 A 38^3)."""
    rng = np.random.default_rng(len(sizes) + sum(sizes))
    mols = []
    for k, n in enumerate(sizes):
        if box:
            pos = (rng.random((n, 3)) * box).astype(np.float32)
            pos[0], pos[1] = 0.0, box
            mols.append((pos, np.full(n, 1.8, np.float32)))
        else:
            mols.append(qs.synth_ball(30 + k, n) if n else (np.zeros((0, 3), np.float32), np.zeros(0, np.float32)))
    print("case cells: %s box=%g" % (sizes, box), flush=True)
    qs.compute_batch(mols, 2.0, 0)
    perm, cells, at = [], [], 0
    for k, (pos, rad) in enumerate(mols):
        G = qs.batch_grid(k)
        gn, c = G["gn"], np.zeros(len(rad), np.int64)
        for a in range(3):
            e = ((pos[:, a] - np.float32(G["origin"][a])) / np.float32(G["dxn"])).astype(np.int64)
            c = c * gn + np.clip(e, 0, gn - 1)
        perm.append(at + np.argsort(c, kind="stable"))
        lo = np.searchsorted(np.sort(c), np.arange(gn ** 3 + 1))
        ranges = np.stack([at + lo[:-1], at + lo[1:]], -1)
        ranges[lo[:-1] == lo[1:]] = 2 ** 31 - 2  # the marker of an empty cell
        cells.append(ranges)
        at += len(rad)
    perm, cells = np.concatenate(perm), np.concatenate(cells)
    assert np.array_equal(_cells_fetch(qs, b"perm", at, np.int32), perm)
    assert np.array_equal(_cells_fetch(qs, b"cells", cells.size, np.int32).reshape(-1, 2), cells)


@pytest.mark.parametrize("reso", [0.216, 0.22])
def test_smoothing_staged_and_gathered(qs, orc, reso):
    """Above and below the expected size from which a block stages its triangles and vertices; two
    passes, so the second reads what the first wrote."""
    pos, rad = qs.synth_ball(23, 4000)
    print("case smoothing staged: reso=%.3f" % reso, flush=True)
    assert _same(qs.compute_ses(pos, rad, reso, 2), orc.compute_ses(pos, rad, reso, 2))


@pytest.mark.parametrize("shift", [0, 4, 8])
def test_mesh_copied_to_any_alignment(qs, shift):
    """The caller's arrays at 16-byte boundaries and off them; nothing past their ends is written."""
    from quickses_amd import hipmem

    pos, rad = qs.synth_ball(31, 900)
    want = qs.compute_ses(pos, rad, 0.5, 1)
    nv, nt = len(want[0]), len(want[1])
    dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(rad)
    outs = [hipmem.DeviceArray(np.full(n + 8, -7, np.int32)) for n in (3 * nv, 3 * nt, nv)]
    print("case mesh copy: shift=%d" % shift, flush=True)
    qs.compute_device_noalloc(dp.ptr, dr.ptr, len(rad), 0.5, 1, outs[0].ptr + shift, nv, outs[1].ptr + shift, nt, outs[2].ptr + shift)
    for buf, ref in zip(outs, (want[0].view(np.int32), want[1], want[2])):
        got, k = hipmem.download(buf.ptr, (ref.size + 8,), np.int32), shift // 4
        assert np.array_equal(got[k:k + ref.size], ref.ravel())
        assert (got[:k] == -7).all() and (got[k + ref.size:] == -7).all()


@pytest.mark.parametrize("n,smooth", [(2, 1), (5, 1), (5, 2), (7, 1)])
def test_triangles_filtered_beside_smoothing(qs, orc, n, smooth):
    """A lattice whose mesh has triangles to drop: below the pool size up to which the
    first of the passes filters them, and above it (n = 7); the next run reads what this one left."""
    ax = np.arange(n, dtype=np.float32) * np.float32(2.5) - np.float32(2.5 * (n // 2))
    pos, rad = np.stack(np.meshgrid(ax, ax, ax, indexing="ij"), -1).reshape(-1, 3), np.full(n ** 3, 1.6, np.float32)
    G, _, _, _, _, _, fld = orc.field(pos, rad, 0.1)
    tri = orc.edge_weld(G, G.g - 1, fld)[1]
    want = orc.compute_ses(pos, rad, 0.1, smooth)
    assert len(tri) > len(want[1])
    for run in range(2):
        print("case filter beside smoothing: n=%d smooth=%d run=%d" % (n, smooth, run), flush=True)
        assert _same(qs.compute_ses(pos, rad, 0.1, smooth), want)


@pytest.mark.parametrize("sizes", [[7692], [7693], [24000] + [1000] * 7, [12000] * 10, [12000] * 11, [10000, 9000, 500, 30000], [2] * 300, [24576] * 18, [24576] * 19])
def test_cells_on_both_sides_of_the_block_rule(qs, sizes):
    """A block per molecule or launches over the device, by the largest molecule's atoms and the run's."""
    test_cells_in_one_block_or_several_launches(qs, sizes, 0)


def test_cells_of_one_large_molecule_in_a_batch(qs):
    """A batch does not wait for one block that sorts its largest molecule (55 us, where the molecule
    alone takes 24 over the device)."""
    small = [qs.synth_ball(95 + k, 1000) for k in range(7)]
    large = qs.synth_ball(94, 24000)
    times = {}
    qs.set_option("timing", 1)
    try:
        for name, mols in (("alone", [large]), ("with small ones", [large] + small)):
            print("case cells: one large molecule %s" % name, flush=True)
            rows = []
            for _ in range(12):
                qs.compute_batch(mols, 2.0, 0)
                rows.append(qs.stage_times()["cells"])
            times[name] = float(np.median(rows[2:]))
    finally:
        qs.set_option("timing", 0)
    assert times["with small ones"] < 1.8 * times["alone"], times
