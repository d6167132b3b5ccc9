"""What one call leaves for the next: results of calls that stopped early, of other molecules and of
optional passes asked for afterwards."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FETCHES = ("labels", "field", "shellm", "perm", "cells", "vert_unsmoothed", "tri_all")


def _fetch(qs, what, nbytes):
    out = np.zeros(nbytes, np.uint8)
    return qs.lib().qs_fetch(what.encode(), ctypes.c_void_p(out.ctypes.data), ctypes.c_int64(nbytes))


def _refused(qs, kind):
    """A call of `kind` that the library refuses after a run of another shape."""
    pos, rad = qs.synth_ball(91, 900)
    if kind == "second molecule's voxel size":
        with pytest.raises(qs.QuickSESError):
            qs.compute_batch([(pos, rad), (pos[:50], rad[:50])], [0.5, 0.0], 1)
    elif kind == "first molecule's coordinates":
        with pytest.raises(qs.QuickSESError):
            qs.compute_batch([(pos + np.float32(2e5), rad), (pos, rad)], 0.5, 1)
    elif kind == "voxel size":
        with pytest.raises(qs.QuickSESError):
            qs.compute_ses(pos, rad, -1.0, 1)
    else:  # a larger grid that no x-slab of 1 MiB holds
        qs.set_option("slab_mb", 1)
        try:
            with pytest.raises(qs.QuickSESError, match="x-slab"):
                qs.compute_ses(pos, rad, 0.2, 1)
        finally:
            qs.set_option("slab_mb", 0)


@pytest.mark.parametrize("kind", ["second molecule's voxel size", "first molecule's coordinates", "voxel size", "slab memory"])
def test_fetch_after_a_refused_call(qs, orc, kind):
    """Nothing is read (and no field pass is run) through the records of a call that did not finish."""
    pos, rad = qs.synth_ball(90, 300)
    print("case refused call: %s" % kind, flush=True)
    qs.compute_ses(pos, rad, 0.5, 1)
    _refused(qs, kind)
    for what in FETCHES:
        assert _fetch(qs, what, 64 << 20) == -1, what
    assert qs.last_slab_count() == 0
    qs.compute_ses(pos, rad, 0.5, 1)
    g = qs.last_grid()["g"]
    assert _fetch(qs, "field", 4 * g ** 3 - 1) == -1
    assert np.array_equal(qs.fetch("field", np.float32, g ** 3).view(np.uint32), orc.field(pos, rad, 0.5)[6].view(np.uint32))


def test_emission_of_more_surface_than_a_packed_ball(qs):
    """Sixty separate atoms of 6 A have as many vertices as 3,000 packed ones: a launch must have blocks
    for them, not for sixty packed atoms (blocks that looped took six times the packed mesh's time)."""
    rng = np.random.default_rng(1)
    apart = ((rng.random((60, 3)) * 40).astype(np.float32), np.full(60, 6.0, np.float32))
    packed = qs.synth_ball(92, 3000)
    times = {}
    qs.set_option("timing", 1)
    try:
        for name, (pos, rad) in (("apart", apart), ("packed", packed)):
            print("case emission time: %s" % name, flush=True)
            rows = []
            for _ in range(12):
                V = qs.compute_ses(pos, rad, 0.5, 1)[0]
                t = qs.stage_times()
                rows.append(t["mc_emit"] + t.get("closest_atom", 0.0) + t["smooth"])
            times[name] = float(np.median(rows[2:])) / len(V)
    finally:
        qs.set_option("timing", 0)
    assert times["apart"] < 2.5 * times["packed"], times


def _overwrite_field(qs, orc, g):
    """Every value of a field of up to g^3 points replaced by 7 (a caller's field without a surface)."""
    s = orc._Grid()
    s.g, s.gn, s.r, s.reso, s.dx_n = g, 1, 3, 0.5, 3.2
    V, T = qs.stage_mesh(orc.Grid(s).params(g - 1), np.full(g ** 3, 7.0, np.float32))
    assert len(V) == 0 and len(T) == 0


def test_fetch_after_a_mesh_of_a_callers_field(qs, orc):
    """A caller's field comes without masks: an earlier run's, of another grid, are not read as its."""
    qs.compute_ses(*qs.synth_ball(98, 50), 1.0, 0)
    print("case fetch after a stage call", flush=True)
    _overwrite_field(qs, orc, 200)
    for what in ("labels", "shellm"):
        assert _fetch(qs, what, 64 << 20) == -1, what
    assert _fetch(qs, "field", 4 * 200 ** 3) == 4 * 200 ** 3


@pytest.mark.parametrize("reso,n", [(0.16, 60), (0.2, 300), (0.28, 300), (0.3, 300), (0.35, 400), (0.4, 400), (0.5, 800), (0.7, 800),
                                    (1.0, 1500), (1.4, 1500), (1.6, 1500)])
@pytest.mark.parametrize("offset", [0.0, 30000.0])
def test_normals_read_stored_values_only(qs, orc, reso, n, offset):
    """The mesh, its normals and the field read no value that their own field pass did not store: in
    between, the field is another's.  Normals after the mesh, and from the run after (which stores what
    they read at once), are those of the whole field."""
    pos, rad = qs.synth_ball(93, n)
    pos = pos + np.float32(offset)
    print("case stored values: reso=%.2f offset=%g" % (reso, offset), flush=True)
    want = orc.compute_ses(pos, rad, reso, 1)
    qs.compute_ses(pos, rad, reso, 1)
    g = qs.last_grid()["g"]
    field = orc.field(pos, rad, reso)[6].view(np.uint32)
    assert np.array_equal(qs.fetch("field", np.float32, g ** 3).view(np.uint32), field)
    whole = qs.vertex_normals(len(want[0])).view(np.uint32)
    qs.compute_ses(pos, rad, reso, 1)  # (the last run whose field pass is that of a run with normals)
    for _ in range(2):  # after an ordinary run, then after a run with normals
        _overwrite_field(qs, orc, g)
        V, T, A = qs.compute_ses(pos, rad, reso, 1)
        assert np.array_equal(T, want[1]) and np.array_equal(A, want[2])
        assert np.array_equal(V.view(np.uint32), want[0].view(np.uint32))
        assert np.array_equal(qs.vertex_normals(len(V)).view(np.uint32), whole)
    assert np.array_equal(qs.fetch("field", np.float32, g ** 3).view(np.uint32), field)


class _SmallMemory:
    """All of the device's free memory taken but for the given MiB."""

    def __init__(self, mib):
        self.mib, self.taken = mib, []

    def __enter__(self):
        from quickses_amd import hipmem

        self.free, free, total = hipmem.free, ctypes.c_size_t(), ctypes.c_size_t()
        while True:
            assert hipmem.hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            left = free.value - (self.mib << 20)
            if left < (8 << 20):
                return self
            try:
                self.taken.append(hipmem.alloc(min(left, 32 << 30)))
            except RuntimeError:  # (the rest is in smaller pieces)
                hipmem.hip().hipGetLastError()
                return self

    def __exit__(self, *exc):
        for p in self.taken:
            self.free(p)


def test_slabs_where_the_grid_is_held_but_the_mesh_is_not(qs):
    """A grid whose arrays an earlier run left, and pools that the free memory does not hold: the
    molecule is meshed in x-slabs, as it is when nothing is held."""
    rng = np.random.default_rng(4)
    pos = (rng.random((60000, 3)) * 60).astype(np.float32)
    pos[0], pos[1] = 0.0, 60.0
    rad = np.full(len(pos), 1.7, np.float32)
    print("case held grid, small memory", flush=True)
    qs.compute_ses(pos[:8], rad[:8], 0.2, 1)  # the same grid (41 M points), a small mesh
    with _SmallMemory(380):  # (the grid takes 245 MB, the pools 1 GB)
        tight = qs.compute_ses(pos, rad, 0.2, 1)
    whole = qs.compute_ses(pos, rad, 0.2, 1)
    assert len(whole[1]) > 0 and np.array_equal(tight[1], whole[1]) and np.array_equal(tight[2], whole[2])
    assert np.array_equal(tight[0].view(np.uint32), whole[0].view(np.uint32))


def test_call_after_one_that_ran_out_of_memory(qs, orc):
    """The failed call's error is not reported by the next one."""
    n = 8 << 20  # (100 MB of positions)
    print("case out of memory, then an ordinary call", flush=True)
    with _SmallMemory(64):
        with pytest.raises(qs.QuickSESError, match="memory"):
            qs.compute_ses(np.zeros((n, 3), np.float32), np.full(n, 1.7, np.float32), 0.5, 1)
    small = qs.synth_ball(96, 300)
    got, want = qs.compute_ses(*small, 0.5, 1), orc.compute_ses(*small, 0.5, 1)
    assert np.array_equal(got[1], want[1]) and np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32))


def test_server_reserves_what_its_batches_use(qs):
    """A worker's workspace at its start: 25.2 bytes per grid point of a budget that counts 24 (every
    buffer has as much headroom), with no buffer that nothing on the served path reads."""
    from quickses_amd import hipmem

    before, after, total = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    budget, result = 6 << 30, 64 << 20
    print("case server workspace", flush=True)
    qs.compute_ses(*qs.synth_ball(97, 100), 0.5, 1)  # (the library's code and its own buffers are loaded)
    assert hipmem.hip().hipMemGetInfo(ctypes.byref(before), ctypes.byref(total)) == 0
    with qs.Server(hbm_budget_bytes=budget, result_bytes=result, workers=1):
        assert hipmem.hip().hipMemGetInfo(ctypes.byref(after), ctypes.byref(total)) == 0
    used = before.value - after.value - result
    assert 0.9 * budget < used < 1.08 * budget, used / budget
