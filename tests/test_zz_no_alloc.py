"""qs_compute_device_noalloc, through the C ABI: the same mesh as qs_compute_device, bit for bit,
on two calls in a row (the second with a smaller molecule, in the region the first one used);
too small an output capacity and too large a molecule are errors that write nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _reference(qs, hipmem, dp, dr, n, reso, smooth):
    nv, ni, pv, pt, pa = qs.compute_device(dp.ptr, dr.ptr, n, reso, smooth)
    return (hipmem.download(pv, (nv, 3), np.float32), hipmem.download(pt, (ni // 3, 3), np.int32),
            hipmem.download(pa, (nv,), np.int32))


def _noalloc(qs, hipmem, dp, dr, n, reso, smooth, vcap, tcap):
    dv, dt, da = hipmem.alloc(max(vcap, 1) * 12), hipmem.alloc(max(tcap, 1) * 12), hipmem.alloc(max(vcap, 1) * 4)
    try:
        nv, ni = qs.compute_device_noalloc(dp.ptr, dr.ptr, n, reso, smooth, dv, vcap, dt, tcap, da)
        return (hipmem.download(dv, (nv, 3), np.float32), hipmem.download(dt, (ni // 3, 3), np.int32),
                hipmem.download(da, (nv,), np.int32))
    finally:
        for p in (dv, dt, da):
            hipmem.free(p)


def _same(a, b):
    assert a[0].shape == b[0].shape and a[1].shape == b[1].shape
    assert np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32))
    assert np.array_equal(a[1], b[1])
    assert np.array_equal(a[2], b[2])


def test_noalloc_equals_device_entry_twice(qs):
    from quickses_amd import hipmem

    cases = [(401, 20000, 0.5, 1), (402, 2000, 0.4, 2)]  # the second call smaller than the first
    for seed, n, reso, smooth in cases:
        pos, rad = qs.synth_ball(seed, n)
        dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(rad)
        try:
            print("case noalloc seed=%d n=%d reso=%.1f" % (seed, n, reso), flush=True)
            ref = _reference(qs, hipmem, dp, dr, n, reso, smooth)
            got = _noalloc(qs, hipmem, dp, dr, n, reso, smooth, len(ref[0]) + 100, len(ref[1]) + 100)
        finally:
            dp.free()
            dr.free()
        assert len(ref[1]) > 0
        _same(got, ref)


def test_noalloc_errors(qs):
    from quickses_amd import hipmem

    pos, rad = qs.synth_ball(403, 1500)
    dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(rad)
    try:
        ref = _reference(qs, hipmem, dp, dr, len(rad), 0.5, 1)
        print("case noalloc capacity too small", flush=True)
        with pytest.raises(qs.QuickSESError, match="capacity"):
            _noalloc(qs, hipmem, dp, dr, len(rad), 0.5, 1, len(ref[0]) - 1, len(ref[1]))
        with pytest.raises(qs.QuickSESError, match="capacity"):
            _noalloc(qs, hipmem, dp, dr, len(rad), 0.5, 1, len(ref[0]), len(ref[1]) - 1)
        # exactly enough room
        _same(_noalloc(qs, hipmem, dp, dr, len(rad), 0.5, 1, len(ref[0]), len(ref[1])), ref)
    finally:
        dp.free()
        dr.free()
    # a grid beyond the fixed region: 20,000 atoms at 0.2 A (about 130 M grid points)
    big, brad = qs.synth_ball(404, 20000)
    dp, dr = hipmem.DeviceArray(big), hipmem.DeviceArray(brad)
    try:
        print("case noalloc molecule too large", flush=True)
        with pytest.raises(qs.QuickSESError, match="scratch region"):
            _noalloc(qs, hipmem, dp, dr, len(brad), 0.2, 1, 1 << 20, 1 << 21)
    finally:
        dp.free()
        dr.free()
    # the region is usable again after a rejected call
    pos, rad = qs.synth_ball(405, 800)
    dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(rad)
    try:
        ref = _reference(qs, hipmem, dp, dr, len(rad), 0.5, 1)
        _same(_noalloc(qs, hipmem, dp, dr, len(rad), 0.5, 1, len(ref[0]), len(ref[1])), ref)
    finally:
        dp.free()
        dr.free()


@pytest.mark.parametrize("kind", ["pageable", "pinned", "mixed"])
def test_noalloc_outputs_in_host_memory(qs, kind):
    """Output arrays that no kernel of the device may write are reached by copies."""
    import ctypes

    from quickses_amd import hipmem

    pos, rad = qs.synth_ball(406, 700)
    dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(rad)
    ref = _reference(qs, hipmem, dp, dr, len(rad), 0.5, 1)
    outs = [np.full(a.size, -7, a.dtype) for a in ref]
    pinned, pv = [], ctypes.c_void_p()
    ptrs = [o.ctypes.data for o in outs]
    if kind == "pinned":
        for o in outs:
            assert hipmem.hip().hipHostMalloc(ctypes.byref(pv), o.nbytes, 0) == 0
            pinned.append(pv.value)
        ptrs = pinned
    dev = hipmem.DeviceArray(outs[0]) if kind == "mixed" else None
    if dev:
        ptrs[0] = dev.ptr
    print("case noalloc into host memory: %s" % kind, flush=True)
    try:
        nv, ni = qs.compute_device_noalloc(dp.ptr, dr.ptr, len(rad), 0.5, 1, ptrs[0], len(ref[0]), ptrs[1], len(ref[1]), ptrs[2])
        assert (nv, ni) == (len(ref[0]), 3 * len(ref[1]))
        for k, p in enumerate(pinned):
            ctypes.memmove(outs[k].ctypes.data, p, outs[k].nbytes)
        if dev:
            outs[0] = hipmem.download(dev.ptr, outs[0].shape, outs[0].dtype)
    finally:
        for p in pinned:
            hipmem.hip().hipHostFree(ctypes.c_void_p(p))
    _same([o.reshape(a.shape) for o, a in zip(outs, ref)], ref)


@pytest.mark.parametrize("n,reso,smooth", [(1164000, 2.0, 1), (328600, 1.0, 1), (75300, 0.5, 1)])
def test_noalloc_region_holds_what_it_held(qs, n, reso, smooth):
    """Molecules that fill the region: their working buffers fit (the mesh then does not fit arrays of
    no entries), so no buffer beside them is larger than it has to be."""
    from quickses_amd import hipmem

    pos = (np.random.default_rng(5).random((n, 3)) * (n / 0.08) ** (1 / 3)).astype(np.float32)
    dp, dr = hipmem.DeviceArray(pos), hipmem.DeviceArray(np.full(n, 1.7, np.float32))
    print("case noalloc full region: n=%d reso=%.1f" % (n, reso), flush=True)
    try:
        with pytest.raises(qs.QuickSESError, match="capacity"):
            qs.compute_device_noalloc(dp.ptr, dr.ptr, n, reso, smooth, 0, 0, 0, 0, 0)
    finally:
        dp.free()
        dr.free()
