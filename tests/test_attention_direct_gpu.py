"""The forward on V itself (transposing LDS reads) against the forward on V_t:
the same operands in the same order, so bit-identical, at the edges of its key
blocks and rows, with non-finite values in the last rows of V (rows past the
end of the keys must add nothing)."""
import ctypes

import pytest
import torch

import moonmath_attention as ma
from moonmath_attention import _lib
from test_calls import _python_path

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(name, q, k, v, B, H, Sq, Skv, layout, mode, force):
    lib, p, st = _lib.lib, _lib.ptr, _lib.stream_ptr(DEV)
    out = torch.full_like(q, float("nan"))
    ws = torch.empty(lib.tail_workspace_bytes_rtne(), dtype=torch.uint8, device=DEV) if force else None
    src = v
    if name == "moonmath_attention_forward_ex":
        src = torch.empty(lib.moonmath_attention_vt_bytes(B, H, Skv) // 2, dtype=torch.bfloat16, device=DEV)
        assert lib.launch_v_transpose_rtne(p(v), p(src), B * H * Skv, Skv, H, layout, st) == 0
    assert getattr(lib, name)(p(q), p(k), p(src), p(out), B, H, Sq, Skv, 128, layout, mode, p(ws), force, st) == 0
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("B,H,Sq,Skv,force", [
    (1, 2, 256, 256, 0), (2, 3, 300, 1, 0), (1, 2, 33, 61, 0), (1, 3, 200, 65, 0), (1, 2, 257, 125, 0),
    (1, 2, 100, 193, 0), (2, 2, 520, 3000, 0), (1, 1, 64, 8191, 0),
    (1, 3, 21800, 77, 0), (2, 24, 4097, 1, 0), (2, 24, 4097, 128, 0),   # persistent short-KV kernel
    (1, 4, 1100, 1409, 3)])                                              # split parts
def test_direct_equals_vt(B, H, Sq, Skv, force, layout):
    g = torch.Generator(device=DEV).manual_seed(Sq + Skv)
    shape = (lambda s: (B, s, H, 128)) if layout else (lambda s: (B, H, s, 128))
    q, k, v = (torch.randn(shape(s), generator=g, device=DEV).bfloat16() for s in (Sq, Skv, Skv))
    last = (v.transpose(1, 2) if layout else v)[0, 0, Skv - 1]
    last[3], last[7], last[11] = float("inf"), float("nan"), float("-inf")
    for mode in range(3):
        a = _run("moonmath_attention_forward_ex", q, k, v, B, H, Sq, Skv, layout, mode, force)
        b = _run("moonmath_attention_forward_direct", q, k, v, B, H, Sq, Skv, layout, mode, force)
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), mode


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("B,H,Sq,Skv", [(1, 2, 300, 1000), (2, 3, 700, 8190), (1, 2, 256, 64), (1, 1, 50, 3)])
def test_lite_direct_equals_vt(B, H, Sq, Skv, layout):
    """Three steps from the full list on keys of growing norm (blocks drop out):
    outputs and written lists."""
    lib, p, st = _lib.lib, _lib.ptr, _lib.stream_ptr(DEV)
    g = torch.Generator(device=DEV).manual_seed(Sq + Skv)
    shape = (lambda s: (B, s, H, 128)) if layout else (lambda s: (B, H, s, 128))
    q, k, v = (torch.randn(shape(s), generator=g, device=DEV) for s in (Sq, Skv, Skv))
    ramp = torch.linspace(0.2, 3.0, Skv, device=DEV)
    k = k * (ramp.view(1, Skv, 1, 1) if layout else ramp.view(1, 1, Skv, 1))
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    nqb, nkb = -(-Sq // 256), -(-Skv // 64)
    vt = torch.empty(lib.moonmath_attention_vt_bytes(B, H, Skv) // 2, dtype=torch.bfloat16, device=DEV)
    assert lib.launch_v_transpose_rtne(p(v), p(vt), B * H * Skv, Skv, H, layout, st) == 0
    for mode, name in enumerate(("rtne", "rtna", "rtz")):
        got = []
        for direct in (False, True):
            pair = torch.zeros(2, B, H, nqb, nkb + 2, dtype=torch.int16, device=DEV)
            pair[0, ..., :3] = torch.tensor([2, nkb - 1, -1], dtype=torch.int16)
            for step in range(3):
                out = torch.full_like(q, float("nan"))
                ws = torch.empty(lib.lite_workspace_bytes_rtne(B, H, Sq), dtype=torch.uint8, device=DEV)
                head = (p(q), p(k), p(v if direct else vt), p(out), B, H, Sq, Skv, 128, p(pair[step & 1]),
                        p(pair[1 - (step & 1)]), None, -3.0, 1 - (step & 1), layout)
                rc = (lib.moonmath_attention_forward_lite_direct(*head, mode, p(ws), st) if direct else
                      getattr(lib, f"launch_attention_forward_lite_{name}")(*head, p(ws), st))
                assert rc == 0
                torch.cuda.synchronize()
                got.append((out.clone(), pair.clone()))
        for (a, x), (b, y) in zip(got[:3], got[3:], strict=True):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16)) and torch.equal(x, y)


@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("B,H,Sq,Skv", [
    (1, 1, 1, 1), (1, 2, 127, 64), (1, 2, 128, 65), (2, 3, 129, 128), (1, 3, 250, 700),   # one half CTA per CU
    (2, 12, 3000, 300), (2, 24, 2048, 2048),                                             # two per CU
    (1, 2, 100, 500), (1, 8, 128, 2000), (1, 1, 129, 4033), (1, 2, 1999, 2000)])         # split parts
def test_half_ctas(B, H, Sq, Skv, layout):
    """Calls that the launcher gives to half CTAs (with a workspace: split where
    it pays) against the 256-row CTAs of the V_t forward. Unsplit they are the
    same computation, bit for bit. Split, bf16 weights times powers of two add up
    in another order: Skv fp32 additions of terms within max |v| err by at most
    Skv 2^-24 max |v| on each side of the quotient, and one bf16 rounding then moves
    the results by a unit in the last place, 2^-7 of the larger at most. A part's
    max moves the last fp32 bit of the exponents, so a weight at a rounding boundary
    may be the next bf16: 2^-7 of its share, of two of the row's largest here."""
    g = torch.Generator(device=DEV).manual_seed(Sq + Skv)
    shape = (lambda s: (B, s, H, 128)) if layout else (lambda s: (B, H, s, 128))
    q, k, v = (torch.randn(shape(s), generator=g, device=DEV).bfloat16() for s in (Sq, Skv, Skv))
    lib, p, st = _lib.lib, _lib.ptr, _lib.stream_ptr(DEV)
    nbytes = lib.moonmath_attention_direct_workspace(B, H, Sq, Skv)
    qf, kf = (t.transpose(1, 2) if layout else t for t in (q.float(), k.float()))
    share = torch.softmax(qf @ kf.transpose(2, 3).contiguous() * 128 ** -0.5, -1).amax(-1, keepdim=True)
    if layout:
        share = share.transpose(1, 2)
    for mode in range(3):
        want = _run("moonmath_attention_forward_ex", q, k, v, B, H, Sq, Skv, layout, mode, 0)
        for ws in (None, torch.empty(max(1, nbytes), dtype=torch.uint8, device=DEV)):
            if ws is not None and nbytes == 0:
                continue
            out = torch.full_like(q, float("nan"))
            assert lib.moonmath_attention_forward_direct(p(q), p(k), p(v), p(out), B, H, Sq, Skv, 128, layout, mode,
                                                         p(ws), 0, st) == 0
            torch.cuda.synchronize()
            if ws is None:
                assert torch.equal(out.view(torch.int16), want.view(torch.int16)), mode
            else:
                a, b = out.float(), want.float()
                top = v.abs().max().float()
                bound = 2.0 ** -7 * (torch.maximum(a.abs(), b.abs()) + 2 * share * top) + 2 * Skv * 2.0 ** -24 * top
                assert ((a - b).abs() <= bound).all(), mode


def test_direct_argument_codes():
    nul = ctypes.c_void_p(0)
    f = _lib.lib.moonmath_attention_forward_direct
    assert f(nul, nul, nul, nul, 0, 1, 1, 1, 128, 0, 0, nul, 0, nul) == 1
    assert f(nul, nul, nul, nul, 1, 1, 1, 1, 128, 0, 0, nul, 0, nul) == 8
    assert f(nul, nul, nul, nul, 1, 1, 1, 1, 128, 0, 9, nul, 0, nul) == 10


def _ramp_lists(B, H, Sq, Skv):
    """A full read list and an empty list to write."""
    nqb, nkb = -(-Sq // 256), -(-Skv // 64)
    pair = torch.zeros(2, B, H, nqb, nkb + 2, dtype=torch.int16, device=DEV)
    pair[0, ..., :3] = torch.tensor([2, nkb - 1, -1], dtype=torch.int16)
    return pair


def _vt_result(monkeypatch, fn):
    """`fn` by the Python path with a V_t pass."""
    with monkeypatch.context() as m:
        _python_path(m)
        m.setattr(_lib.lib, "moonmath_attention_prefers_direct", lambda *a: 0)
        out = fn()
        torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("B,H,S,shift", [(1, 2, 256, 0), (1, 3, 1000, 0), (2, 8, 2048, 0), (2, 24, 1531, 0),
                                         (1, 3, 1000, 128), (2, 4, 1100, -256), (1, 2, 300, 128 * 599)])
def test_out_may_overlap_v(B, H, S, shift, layout, native, monkeypatch):
    """``out`` on V's own memory, or `shift` elements from it: V is read before
    any of it is overwritten, in both forwards."""
    g = torch.Generator(device=DEV).manual_seed(S)
    shape = (B, H, S, 128) if layout == "bhsd" else (B, S, H, 128)
    q, k, v0 = (torch.randn(shape, generator=g, device=DEV).bfloat16() for _ in range(3))
    n = v0.numel()
    for lite in (False, True):
        def call(v, out, pair):
            if lite:
                return ma.forward_lite(q, k, v, pair[0], pair[1], threshold=-3.0, phase=1, out=out, layout=layout)
            return ma.forward(q, k, v, out=out, layout=layout)

        want_pair, pair = _ramp_lists(B, H, S, S), _ramp_lists(B, H, S, S)
        want = _vt_result(monkeypatch, lambda: call(v0, None, want_pair))
        buf = torch.empty(n + abs(shift), dtype=torch.bfloat16, device=DEV)
        v, out = (buf[max(0, -s):][:n].view(shape) for s in (shift, -shift))
        v.copy_(v0)
        with monkeypatch.context() as m:
            if not native:
                _python_path(m)
            assert call(v, out, pair) is out
            torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        assert torch.equal(pair, want_pair)


@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
def test_out_may_be_q(layout):
    """Every CTA reads its query rows before it stores them, in both forwards."""
    for B, H, S in ((1, 2, 256), (2, 24, 1531), (1, 3, 4097)):
        g = torch.Generator(device=DEV).manual_seed(S)
        shape = (B, H, S, 128) if layout == "bhsd" else (B, S, H, 128)
        q, k, v = (torch.randn(shape, generator=g, device=DEV).bfloat16() for _ in range(3))
        want = ma.forward(q, k, v, layout=layout)
        q2 = q.clone()
        assert torch.equal(ma.forward(q2, k, v, out=q2, layout=layout).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("offset", [1, 4])
def test_v_off_a_16_byte_boundary(offset, native, monkeypatch):
    """V as a view that starts `offset` elements into its buffer: read by plain
    loads (the V_t pass), not by 16-byte gathers; the bits are those of an
    aligned copy."""
    B, H, S = 2, 3, 700
    g = torch.Generator(device=DEV).manual_seed(offset)
    q, k, v0 = (torch.randn(B, H, S, 128, generator=g, device=DEV).bfloat16() for _ in range(3))
    v = torch.empty(v0.numel() + offset, dtype=torch.bfloat16, device=DEV)[offset:].view(v0.shape)
    v.copy_(v0)
    for lite in (False, True):
        def call(v, pair):
            if lite:
                return ma.forward_lite(q, k, v, pair[0], pair[1], threshold=-3.0, phase=1)
            return ma.forward(q, k, v)

        want_pair, pair = _ramp_lists(B, H, S, S), _ramp_lists(B, H, S, S)
        want = _vt_result(monkeypatch, lambda: call(v0, want_pair))
        passes = []
        with monkeypatch.context() as m:
            if not native:
                _python_path(m)
                real = _lib.lib.launch_v_transpose_rtna
                m.setattr(_lib.lib, "launch_v_transpose_rtna", lambda *a: passes.append(1) or real(*a))
            got = call(v, pair)
            torch.cuda.synchronize()
        assert native or passes
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(pair, want_pair)
