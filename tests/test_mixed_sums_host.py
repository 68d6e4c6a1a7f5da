"""The launch that prepares attention and a selective scan from their projection's splits (csrc/window.hip) refuses what the launches of their own refuse, before anything is launched."""
import ctypes as C

import pytest

from chatts_amd import _lib


class SplitSums(C.Structure):
    _fields_ = [("slabs", C.c_void_p), ("scale", C.c_void_p), ("bias", C.c_void_p), ("plane", C.c_size_t), ("sk", C.c_int), ("n", C.c_int), ("most", C.c_int)]


AT = 0x40000000      # (no rows: nothing is read)
WINDOW = dict(proj=AT, ld_proj=1024, off_q=0, off_k=256, off_v=384, off_gate=0, heads=4, kv_heads=2, dim=64, vdim=64, dim_p=64, vdim_p=64, scale=0.1, eps=1e-5, kcache=AT, vcache=AT, table=AT, rows=AT,
              log_block=6, n_splits=1, **{})
SCAN = dict(proj=AT, ld_proj=1024, off_x=512, off_z=768, inner=256, state=16, taps=4, conv_ch=256, conv_w=AT, conv_b=AT, ring=AT, rows=AT)


def call(window={}, scan={}, u=AT, sk=4):
    w, c = _lib.WindowArgs(**{**WINDOW, **window}), _lib.SelectArgs(**{**SCAN, **scan})
    w.q.hi, w.q.lo, w.q.ld = AT, AT, 256
    c.u.f32, c.u.ld = u, 256
    lib = _lib.load()
    prep = getattr(lib, "_ZN6chatts18window_select_prepEPK16ChattsWindowArgsPK16ChattsSelectArgsRKNS_9SplitSumsEPfP12ihipStream_t")
    prep.argtypes, prep.restype = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p], C.c_int
    sums = SplitSums(slabs=AT, plane=1024, sk=sk, n=1024, most=8)
    apart = lib.chatts_window_prep(C.byref(w), None) or lib.chatts_select_conv(C.byref(c), None)
    return prep(C.addressof(w), C.addressof(c), C.addressof(sums), AT, None), apart


def test_what_both_take():
    assert call() == (0, 0)
    for taps in (1, 2, 3, 4):
        assert call(scan=dict(taps=taps)) == (0, 0)
    assert call(sk=8) == (0, 0) and call(sk=9)[0] != 0 and call(sk=0)[0] != 0


@pytest.mark.parametrize("kw", [dict(scan=dict(taps=0)), dict(scan=dict(taps=-1)), dict(scan=dict(inner=0)), dict(scan=dict(inner=-4)), dict(scan=dict(state=0)), dict(scan=dict(state=257)),
                                dict(scan=dict(off_z=-4)), dict(scan=dict(off_z=772)), dict(scan=dict(off_z=769)), dict(scan=dict(off_x=772)), dict(scan=dict(conv_ch=252)), dict(scan=dict(ring=None)),
                                dict(scan=dict(conv_w=AT + 4)), dict(scan=dict(rows=None)), dict(scan=dict(proj=None)), dict(scan=dict(proj=AT + 8)), dict(u=None), dict(u=AT + 4),
                                dict(window=dict(rows=None)), dict(window=dict(heads=3)), dict(window=dict(off_v=900)), dict(window=dict(log_block=5)), dict(window=dict(kcache=AT + 8))])
def test_what_both_refuse(kw):
    joint, apart = call(**kw)
    assert apart != 0 and joint == apart
