"""The bounds of the field passes as the library evaluates them (qs_rule_*), against the voxels that a
mesh and its normals read, and against the float predicates they stand for."""
import ctypes

import numpy as np
import pytest

from test_band import _band, _shifted, _window_norm
from test_intervals import _root, _sample

F = np.float32
MESH, NORMALS, WHOLE = 0, 1, 2


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _rule_band(qs, r, dx, coord_max, keep):
    out = (ctypes.c_int * 4)()
    assert qs.lib().qs_rule_band(r, ctypes.c_float(dx), ctypes.c_float(coord_max), keep, out) == 0
    return out[0], out[1], bool(out[2]), bool(out[3])


@pytest.mark.parametrize("dx", [0.155, 0.16, 0.175, 0.2, 0.233, 0.28, 0.3, 0.35, 0.4, 0.47, 0.5, 0.7, 0.75, 1.0, 1.4, 1.5, 2.0, 4.0])
@pytest.mark.parametrize("coord_max", [16.0, 256.0, 32768.0, 131072.0])
def test_band_is_the_stated_rule(qs, dx, coord_max):
    r = int(np.ceil(F(1.4) / F(dx)))
    lo, hi, edge, everything = _band(r, float(F(dx)), coord_max)
    everything = everything or 3 * r * r >= 255  # (half-widths above 9 have kernels that store every shell voxel)
    got = _rule_band(qs, r, dx, coord_max, MESH)
    assert got[3] == everything
    if not everything:
        assert got[:3] == (lo, hi, edge)
        assert _rule_band(qs, r, dx, coord_max, NORMALS)[0] <= lo
    for keep in (NORMALS, WHOLE):
        assert _rule_band(qs, r, dx, coord_max, keep)[1:] == (255, False, True)
    assert _rule_band(qs, r, dx, coord_max, WHOLE)[0] == -1


@pytest.mark.parametrize("reso,n", [(0.175, 40), (0.2, 60), (0.28, 120), (0.3, 150), (0.4, 250), (0.5, 400), (0.7, 500), (1.0, 700),
                                    (1.4, 900), (1.6, 900)])
@pytest.mark.parametrize("offset", [0.0, 30000.0])
def test_voxels_that_mesh_and_normals_read_are_stored(qs, orc, reso, n, offset):
    pos, rad = qs.synth_ball(77, n)
    pos = pos + F(offset)
    G, _, _, _, _, lab, fld = orc.field(pos, rad, reso)
    g, r = G.g, G.r
    lab, fld = lab.reshape(g, g, g), fld.reshape(g, g, g)
    cmax = 1.0
    while cmax < max(np.abs(G.origin).max(), np.abs(G.origin + g * G.dx).max(), g * float(G.dx)):
        cmax *= 2.0
    out, shell = lab == 0, lab == 1
    norm, neg = _window_norm(out, r), fld < 0
    ends = np.zeros_like(neg)
    for a in range(3):
        cut = neg.take(range(g - 1), a) != neg.take(range(1, g), a)
        i, j = [slice(None)] * 3, [slice(None)] * 3
        i[a], j[a] = slice(0, g - 1), slice(1, g)
        ends[tuple(i)] |= cut
        ends[tuple(j)] |= cut
    around = ends | np.logical_or.reduce([_shifted(ends, a, s) for a in range(3) for s in (-1, 1)])
    for keep, read in ((MESH, ends), (NORMALS, around)):
        lo, hi, edge, everything = _rule_band(qs, r, reso, cmax, keep)
        far = (norm >= hi) & (not everything)
        stored = shell & (norm > lo) & ~far
        if edge:
            stored |= shell & far & np.logical_or.reduce([_shifted(out, a, s) for a in range(3) for s in (-(r + 1), r + 1)])
        left = shell & ~stored
        assert not (read & left).any()
        assert np.array_equal(neg[left], norm[left] > lo)


@pytest.mark.parametrize("dx", [0.05, 0.2, 0.3, 0.5, 1.0])
@pytest.mark.parametrize("offset", [0.0, -66.0, 300.0, 20000.0])
@pytest.mark.parametrize("seed", [1, 2])
def test_intervals_are_the_predicates(qs, dx, offset, seed):
    rng, dx, _, o, ss, az, S, g, _, _ = _sample(dx, offset, seed)
    e = (az[:, None] - (o + (np.arange(g, dtype=F) * dx).astype(F)).astype(F)[None, :]).astype(F)
    pred = (S[:, None] + (e * e).astype(F)).astype(F) < ss[:, None]
    root = _root((ss - S).astype(F), rng)
    lo, hi, sure = (np.zeros(len(az), np.int32) for _ in range(3))
    assert qs.lib().qs_rule_interval(len(az), ctypes.c_float(o), g, ctypes.c_float(dx), _ptr(az), _ptr(ss), _ptr(S), _ptr(root),
                                     _ptr(lo), _ptr(hi), _ptr(sure)) == 0
    z = np.arange(g)[None, :]
    inside = (z >= lo[:, None]) & (z <= hi[:, None])
    sure = sure != 0
    assert np.array_equal(pred[sure], inside[sure])
    if abs(offset) < 1000 and dx >= 0.2:
        assert sure.mean() > 0.5  # (the sample is full of ends on grid points)


@pytest.mark.parametrize("dx", [0.05, 0.2, 0.5, 1.0])
@pytest.mark.parametrize("offset", [0.0, 300.0, 20000.0])
def test_rows_hold_every_reached_row(qs, dx, offset):
    rng, dx, _, o, ss, ay, X, g, rad, _ = _sample(dx, offset, 3)
    e = (ay[:, None] - (o + (np.arange(g, dtype=F) * dx).astype(F)).astype(F)[None, :]).astype(F)
    reached = (X[:, None] + (e * e).astype(F)).astype(F) < ss[:, None]
    root, rad = _root((ss - X).astype(F), rng), np.ascontiguousarray(rad, F)
    lo, hi = np.zeros(len(ay), np.int32), np.zeros(len(ay), np.int32)
    assert qs.lib().qs_rule_rows(len(ay), ctypes.c_float(o), g, ctypes.c_float(dx), _ptr(ay), _ptr(rad), _ptr(root), _ptr(lo),
                                 _ptr(hi)) == 0
    rows = np.arange(g)[None, :]
    assert not (reached & ~((rows >= lo[:, None]) & (rows <= hi[:, None]))).any()


def test_rules_refuse_bad_arguments(qs):
    out = (ctypes.c_int * 4)()
    for r, dx, keep in ((0, 0.5, 0), (3, 0.0, 0), (3, 0.5, 3), (3, 0.5, -1)):
        assert qs.lib().qs_rule_band(r, ctypes.c_float(dx), ctypes.c_float(64.0), keep, out) == -1
    assert qs.lib().qs_rule_rows(1, ctypes.c_float(0.0), 10, ctypes.c_float(0.5), None, None, None, None, None) == -1
