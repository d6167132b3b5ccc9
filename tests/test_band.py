"""The rule by which field pass 2 leaves voxels out (QsBand): every shell voxel that an edge with a
sign change touches is among the stored ones, and the signs of the voxels left out follow from their
window minimum.  Restated in numpy on the oracle's field."""
import math

import numpy as np
import pytest

PROBE = float(np.float32(1.4))


def _band(r, dx, coord_max):
    """klo, khi, lo, hi, edge, all: as build_offset_tables derives them."""
    delta = 16.0 * 2.0 ** -24 * (coord_max + 2.0 * r * dx)
    norms = range(3 * r * r + 1)
    klo = max([n for n in norms if dx * math.sqrt(n) + delta < PROBE], default=-1)
    khi = max([n for n in norms if dx * math.sqrt(n) - delta <= PROBE], default=-1)
    if klo < 0 or khi > r * r:
        return 0, 255, False, True
    lo = max([n for n in range(klo + 1) if math.sqrt(n) + 1.0 <= math.sqrt(klo) + 1e-9], default=-1)
    hi = min(int(math.floor((math.sqrt(khi) + 1.0) ** 2 + 1e-9)) + 1, 255)
    return lo, hi, khi == r * r, False


def _window_norm(out, r):
    n = np.where(out, 0, 10000).astype(np.int32)
    for axis in range(3):
        best = n.copy()
        size = n.shape[axis]
        for s in range(1, min(r, size - 1) + 1):
            for a, b in ((0, s), (s, 0)):
                i = [slice(None)] * 3
                j = [slice(None)] * 3
                i[axis], j[axis] = slice(a, a + size - s), slice(b, b + size - s)
                best[tuple(i)] = np.minimum(best[tuple(i)], n[tuple(j)] + s * s)
        n = best
    return n


def _shifted(mask, axis, s):
    out = np.zeros_like(mask)
    size = mask.shape[axis]
    if abs(s) >= size:
        return out
    i = [slice(None)] * 3
    j = [slice(None)] * 3
    i[axis], j[axis] = (slice(s, size), slice(0, size - s)) if s > 0 else (slice(0, size + s), slice(-s, size))
    out[tuple(i)] = mask[tuple(j)]
    return out


@pytest.mark.parametrize("reso,n", [(0.175, 40), (0.2, 60), (0.28, 120), (0.3, 150), (0.35, 200), (0.4, 250), (0.47, 300), (0.5, 400),
                                    (0.7, 500), (0.75, 500), (1.0, 700), (1.4, 900), (1.6, 900)])
@pytest.mark.parametrize("offset", [0.0, 900.0, 30000.0])
def test_read_voxels_are_stored(qs, orc, reso, n, offset):
    pos, rad = qs.synth_ball(77, n)
    pos = pos + np.float32(offset)
    G, _, _, _, _, lab, fld = orc.field(pos, rad, reso)
    g, r = G.g, G.r
    lab, fld = lab.reshape(g, g, g), fld.reshape(g, g, g)
    cmax = 1.0
    while cmax < max(np.abs(G.origin).max(), np.abs(G.origin + g * G.dx).max(), g * float(G.dx)):
        cmax *= 2.0
    lo, hi, edge, everything = _band(r, float(np.float32(reso)), cmax)
    out, shell = lab == 0, lab == 1
    norm = _window_norm(out, r)
    far = norm >= hi
    stored = shell & (norm > lo) & ~far
    if edge:
        stored |= shell & far & np.logical_or.reduce([_shifted(out, a, s) for a in range(3) for s in (-(r + 1), r + 1)])
    if everything:
        stored = shell
    neg = fld < 0
    left = shell & ~stored
    assert np.array_equal(neg[left], norm[left] > lo)
    read = np.zeros_like(neg)
    for a in range(3):
        cut = neg.take(range(g - 1), a) != neg.take(range(1, g), a)
        i, j = [slice(None)] * 3, [slice(None)] * 3
        i[a], j[a] = slice(0, g - 1), slice(1, g)
        read[tuple(i)] |= cut
        read[tuple(j)] |= cut
    assert not (read & left).any()
