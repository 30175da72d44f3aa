"""The native call path (csrc/calls.cpp): it takes plain GPU calls and nothing
else, and gives what the Python path gives."""
import sys
import threading
import types

import pytest
import torch

import moonmath_attention as ma
from moonmath_attention import _lib
from mla_inputs import KV_SCALE, QK, SCALE_192, paged_pool, rand_kv_rows, rand_q

DEV = "cuda:0"


class _Sub(torch.Tensor):
    pass


def test_leaves_everything_else_to_python():
    """CPU tensors, other types, subclasses, wrong counts of arguments: None, with
    nothing done, so that the wrapper's checks decide."""
    q = torch.zeros(1, 2, 8, 128, dtype=torch.bfloat16)
    c = _lib.calls
    for args in ((q, q, q, None, "rtna", "bhsd"), (q.float(), q, q, None, "rtna", "bhsd"),
                 (q.as_subclass(_Sub), q, q, None, "rtna", "bhsd"), (1, q, q, None, "rtna", "bhsd"),
                 (q, q, q, None, "xyz", "bhsd"), (q, q, q, None, 3, "bhsd"), (q, q)):
        assert c.forward(*args) is None
    assert c.forward_lite(q, q, q, q, q, -6.0, 1, None, "rtna", "bhsd") is None
    assert c.mla_slab(q, q, q, q, 1.0, 1.0, 1.0, False) is None
    assert c.mla_paged(q, q, q, q, q, None, q, q, 1, 1.0, 1.0, 1.0, True) is None
    assert c.mla_blocks(q, q, q, q, q, q, 1, 1.0, 1.0, 1.0, None) is None
    assert c.kv_quantize(q, q, q, q, 1.0, False) is None


def test_binds_every_launcher_it_uses():
    assert all(hasattr(_lib.lib, name) for name in _lib.calls.bound_names())


@pytest.mark.parametrize("why", ["missing", "other torch"])
def test_without_the_native_path(why, monkeypatch):
    """No module, or one of another torch: a warning, and the Python path alone."""
    if why == "missing":
        monkeypatch.setitem(sys.modules, "moonmath_attention._calls", None)
    else:
        monkeypatch.setattr(torch, "__version__", "1.2.3+other")
    with pytest.warns(RuntimeWarning, match="_calls module is not usable"):
        calls = _lib.load_calls()
    assert calls.forward(1, 2) is None and calls.kv_quantize() is None


def test_native_path_is_loaded():
    assert isinstance(_lib.calls, types.ModuleType)


def _python_path(monkeypatch):
    """The wrappers without the native path."""

    class Off:
        def __getattr__(self, name):
            return lambda *a: None

    monkeypatch.setattr(_lib, "calls", Off())


def _both(monkeypatch, fn):
    got = fn()
    torch.cuda.synchronize()
    with monkeypatch.context() as m:
        _python_path(m)
        want = fn()
        torch.cuda.synchronize()
    for a, b in zip(got, want, strict=True):
        assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device
        assert torch.equal(a.view(torch.int8), b.view(torch.int8))


def _qkv(layout, Sq=300, Skv=200, B=2, H=3):
    g = torch.Generator(device=DEV).manual_seed(3)
    shape = (lambda s: (B, H, s, 128)) if layout == "bhsd" else (lambda s: (B, s, H, 128))
    return [torch.randn(shape(s), generator=g, device=DEV).bfloat16() for s in (Sq, Skv, Skv)]


@pytest.mark.gpu
def test_plain_gpu_calls_are_taken(monkeypatch):
    """Each native function does a plain call itself, and its result is that of the
    Python path."""
    c = _lib.calls
    q, k, v = _qkv("bhsd")
    B, H, Sq, Skv = q.shape[0], q.shape[1], q.shape[2], k.shape[2]
    lists = [torch.zeros(2, B, H, -(-Sq // 256), -(-Skv // 64) + 2, dtype=torch.int16, device=DEV) for _ in range(2)]
    for pair in lists:
        pair[0, ..., :3] = torch.tensor([2, -(-Skv // 64) - 1, -1], dtype=torch.int16)
    lens = [700, 64, 1300]
    pool, idx, indptr = (t.to(DEV) for t in paged_pool(lens, 5))
    q4, p4 = (t.to(DEV) for t in rand_q(3, 3, 16, 5))
    q3, p3 = q4[:, 0].contiguous(), p4[:, 0].contiguous()
    n = torch.tensor(lens, dtype=torch.int32, device=DEV)
    slab = rand_kv_rows(3 * 500, 7).view(3, 500, QK).to(DEV)
    table = torch.arange(15, dtype=torch.int32, device=DEV).view(3, 5)
    blocks = pool.view(-1, 64, QK)
    ckv, kpe = (torch.randn(50, w, device=DEV).bfloat16() for w in (512, 64))
    slots = torch.arange(50, dtype=torch.int32, device=DEV)
    s, ks = SCALE_192, KV_SCALE

    got = [c.forward(q, k, v, None, "rtna", "bhsd"),
           c.forward_lite(q, k, v, lists[0][0], lists[0][1], -3.0, 1, None, "rtna", "bhsd"), lists[0]]
    outs = [torch.zeros_like(q3), torch.zeros_like(q4), torch.zeros_like(q3), torch.zeros_like(q4), torch.zeros_like(q3)]
    cache = [torch.zeros(60, QK, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn) for _ in range(2)]
    taken = [c.mla_slab(q3, p3, slab, outs[0], s, ks, 1.0, False), c.mla_slab(q4, p4, slab, outs[1], s, ks, 1.0, True),
             c.mla_paged(q3, p3, pool, outs[2], n, None, idx, indptr, 4, s, ks, 1.0, False),
             c.mla_paged(q4, p4, pool, outs[3], n, None, idx, indptr, 4, s, ks, 1.0, True),
             c.mla_blocks(q3, p3, blocks, outs[4], n, table, 4, s, ks, 1.0, None),
             c.kv_quantize(ckv, kpe, cache[0], slots, 0.03125, False)]
    assert all(t is not None for t in got) and all(t is True for t in taken)
    got += outs + [cache[0]]
    with monkeypatch.context() as m:
        _python_path(m)
        want = [ma.forward(q, k, v),
                ma.forward_lite(q, k, v, lists[1][0], lists[1][1], threshold=-3.0, phase=1), lists[1]]
        o = [torch.zeros_like(t) for t in outs]
        ma.mla_decode_a16w8(q3, p3, slab, o[0], s, ks)
        ma.mla_decode_a16w8_multiq(q4, p4, slab, o[1], s, ks)
        ma.mla_decode_a16w8_paged_dev(q3, p3, pool, o[2], n, None, idx, indptr, 4, s, ks)
        ma.mla_decode_a16w8_multiq_paged_dev(q4, p4, pool, o[3], n, None, idx, indptr, 4, s, ks)
        ma.mla_decode_a16w8_paged_blocks(q3, p3, blocks, o[4], n, table, 4, s, ks)
        ma.mla_kv_quantize(ckv, kpe, cache[1], slots, 0.03125)
        want += o + [cache[1]]
    torch.cuda.synchronize()
    for a, b in zip(got, want, strict=True):
        assert torch.equal(a.view(torch.int8), b.view(torch.int8))


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["bhsd", "bshd"])
@pytest.mark.parametrize("mode", ["rtna", "rtne", "rtz"])
def test_attention_equals_the_python_path(layout, mode, monkeypatch):
    q, k, v = _qkv(layout)
    _both(monkeypatch, lambda: [ma.forward(q, k, v, round_mode=mode, layout=layout)])
    out = torch.empty_like(q)
    assert ma.forward(q, k, v, out=out, round_mode=mode, layout=layout) is out
    _both(monkeypatch, lambda: [ma.forward(q, k, v, out=out, round_mode=mode, layout=layout).clone()])

    def lite():
        la = ma.LiteAttention(threshold=-3.0, round_mode=mode, layout=layout)
        outs = [la(q, k, v) for _ in range(3)]
        return outs + [la.read_list.clone(), la.write_list.clone()]

    _both(monkeypatch, lite)


@pytest.mark.gpu
@pytest.mark.parametrize("q_len", [1, 3])
def test_mla_equals_the_python_path(q_len, monkeypatch):
    B, H, lens = 3, 16, [700, 64, 1300]
    pool, idx, indptr = paged_pool(lens, 5)
    q_lat, q_pe = (t.to(DEV) for t in rand_q(B, q_len, H, 5))
    if q_len == 1:
        q_lat, q_pe = q_lat[:, 0].contiguous(), q_pe[:, 0].contiguous()
    pool, idx, indptr = pool.to(DEV), idx.to(DEV), indptr.to(DEV)
    n = torch.tensor(lens, dtype=torch.int32, device=DEV)
    rows = torch.tensor([2, 0, 1], dtype=torch.int32, device=DEV)
    slab = rand_kv_rows(B * 500, 7).view(B, 500, QK).to(DEV)
    table = torch.arange(3 * 5, dtype=torch.int32, device=DEV).view(3, 5)
    multi = q_len > 1

    def run():
        outs = [torch.full_like(q_lat, 7.0) for _ in range(4)]
        (ma.mla_decode_a16w8_multiq if multi else ma.mla_decode_a16w8)(q_lat, q_pe, slab, outs[0], SCALE_192, KV_SCALE)
        op = ma.mla_decode_a16w8_multiq_paged_dev if multi else ma.mla_decode_a16w8_paged_dev
        op(q_lat, q_pe, pool, outs[1], n, None, idx, indptr, 4, SCALE_192, KV_SCALE)
        op(q_lat, q_pe, pool, outs[2], n, rows, idx, indptr, 1, SCALE_192, KV_SCALE)
        ma.mla_decode_a16w8_paged_blocks(q_lat, q_pe, pool.view(-1, 64, QK), outs[3], n, table, 4, SCALE_192, KV_SCALE)
        return outs

    _both(monkeypatch, run)


@pytest.mark.gpu
def test_kv_quantize_equals_the_python_path(monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(9)
    c, r = (torch.randn(50, w, generator=g, device=DEV).bfloat16() * 20 for w in (512, 64))
    slots = torch.randperm(60, generator=g, device=DEV)[:50].int()

    def run():
        outs = []
        for sat in (False, True):
            pool = torch.zeros(60, QK, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn)
            ma.mla_kv_quantize(c, r, pool, slots, 0.03125, sat)
            outs.append(pool)
        return outs

    _both(monkeypatch, run)


@pytest.mark.gpu
def test_refusals_stay_refused_on_gpu():
    q, k, v = _qkv("bhsd")
    with pytest.raises(TypeError, match="must be torch.bfloat16"):
        ma.forward(q.float(), k, v)
    with pytest.raises(ValueError, match="must be contiguous"):
        ma.forward(q.transpose(1, 2), k, v, layout="bshd")
    with pytest.raises(ValueError, match="k shape mismatch"):
        ma.forward(q, k[:1].contiguous(), v)
    with pytest.raises(ValueError, match="out shape must match"):
        ma.forward(q, k, v, out=k)
    with pytest.raises(ValueError, match="round_mode must be"):
        ma.forward(q, k, v, round_mode="up")
    sub = ma.forward(q.as_subclass(_Sub), k, v)  # taken, by the Python path
    assert torch.equal(sub.as_subclass(torch.Tensor), ma.forward(q, k, v))


@pytest.mark.gpu
@pytest.mark.parametrize("bad,error", [("much", ValueError), (object(), TypeError), (None, TypeError)])
def test_scale_p_must_be_a_number(bad, error):
    """The single-query ops use scale_p nowhere and refuse what is no number; what
    converts to one is taken."""
    q_lat, q_pe = (t[:, 0].contiguous().to(DEV) for t in rand_q(1, 1, 16, 5))
    rows = rand_kv_rows(128, 7).to(DEV)
    n, idx, indptr, table = (torch.tensor(t, dtype=torch.int32, device=DEV)
                             for t in ([128], list(range(128)), [0, 128], [[0, 1]]))
    o = torch.zeros_like(q_lat)
    for scale_p in (bad, 1, "2.5"):
        for call in (lambda s: ma.mla_decode_a16w8(q_lat, q_pe, rows.view(1, 128, QK), o, SCALE_192, KV_SCALE, s),
                     lambda s: ma.mla_decode_a16w8_paged_dev(q_lat, q_pe, rows, o, n, None, idx, indptr, 1, SCALE_192,
                                                             KV_SCALE, s),
                     lambda s: ma.mla_decode_a16w8_paged_blocks(q_lat, q_pe, rows.view(2, 64, QK), o, n, table, 1,
                                                                SCALE_192, KV_SCALE, s)):
            if scale_p is bad:
                with pytest.raises(error):
                    call(scale_p)
            else:
                call(scale_p)
    torch.cuda.synchronize()


@pytest.mark.gpu
def test_streams_and_threads():
    """Calls from several threads, each on a stream of its own, on inputs of
    their own: every result is that of the call alone."""
    sets = [_qkv("bhsd", Sq=256 + 64 * i, Skv=1000) for i in range(4)]
    want = [ma.forward(*s) for s in sets]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            outs = [ma.forward(*sets[i]) for _ in range(20)]
        st.synchronize()
        bad.extend(i for o in outs if not torch.equal(o, want[i]))

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
