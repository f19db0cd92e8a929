"""sdv_pack_contiguous rejects bad arguments on the host (no GPU)."""
import ctypes

from specdec_amd import _native

P = ctypes.c_void_p(0x1000)


def test_host_validation():
    lib = _native.load()

    def f(k=P, v=P, s=P, b=1, kv=2, t=64, d=128, kp=P, vp=P, sp=P, bt=P):
        return lib.sdv_pack_contiguous(k, v, s, b, kv, t, d, kp, vp, sp, bt, None)
    for name in ("k", "v", "s", "kp", "vp", "sp", "bt"):
        assert f(**{name: None}) == _native.SDV_ERR_NULL
    for kw in (dict(b=0), dict(kv=0), dict(t=0), dict(t=-5), dict(t=2**31 - 1), dict(b=2**20, t=2**20)):
        assert f(**kw) == _native.SDV_ERR_SHAPE, kw
    assert f(d=96) == _native.SDV_ERR_UNSUPPORTED
    assert f(k=ctypes.c_void_p(0x1008)) == _native.SDV_ERR_ALIGN
    assert f(kp=ctypes.c_void_p(0x1008)) == _native.SDV_ERR_ALIGN
    assert f(v=ctypes.c_void_p(0x1002)) == _native.SDV_ERR_ALIGN


def test_varlen_slots_host_validation():
    lib = _native.load()

    def f(bt=P, mb=4, lens=(5, 64), slots=P, tiles=P, n=None):
        arr = (ctypes.c_int32 * max(1, len(lens)))(*lens) if lens is not None else None
        return lib.sdv_varlen_slots(bt, mb, arr, len(lens) if n is None else n, slots, tiles, None)
    assert f(bt=None) == _native.SDV_ERR_NULL and f(slots=None) == _native.SDV_ERR_NULL
    assert f(lens=None, n=2) == _native.SDV_ERR_NULL
    assert f(lens=(5, 65)) == _native.SDV_ERR_SHAPE and f(lens=(-1,)) == _native.SDV_ERR_SHAPE
    assert f(n=0) == _native.SDV_ERR_SHAPE and f(mb=0) == _native.SDV_ERR_SHAPE
    assert f(tiles=ctypes.c_void_p(0x1002)) == _native.SDV_ERR_ALIGN
    assert f(lens=(0, 0)) == _native.SDV_OK      # no rows: nothing to do, no launch
