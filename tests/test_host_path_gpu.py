"""The wrappers' native fast path (csrc/host.cpp): every call it takes gives
what the checked Python path gives, and every call that path refuses it leaves
alone, so that the error is the same."""

import threading

import numpy as np
import pytest
import torch

import _kvdec as K
import dense_kernel
import kivi_stream
import paged_kernel
import quant_kernel
import sparse_kernel

pytestmark = pytest.mark.gpu

ENTRIES = ("sparse", "dense", "paged", "kivi", "step_attend", "quantize", "build")


class Recorder:
    """Stands in for K.host; `skip` answers None to everything."""

    def __init__(self, skip):
        self.taken = []
        for name in ENTRIES:
            setattr(self, name, self._entry(name, skip))

    def _entry(self, name, skip):
        real = getattr(K.host, name)

        def call(*args):
            out = None if skip else real(*args)
            self.taken.append(out is not None)
            return out
        return call


def _flat(x):
    if isinstance(x, dict):
        return [t for n in sorted(x) for t in _flat(x[n])]
    return [x] if isinstance(x, torch.Tensor) else [t for y in x for t in _flat(y)]


def _both(monkeypatch, call, taken=True):
    got = []
    for skip in (False, True):
        with monkeypatch.context() as m:
            rec = Recorder(skip)
            m.setattr(K, "host", rec)
            got.append(_flat(call()))
            if not skip:
                assert all(t == taken for t in rec.taken) and rec.taken
    for a, b in zip(*got):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        assert torch.equal(a.view(torch.uint8) if a.numel() else a, b.view(torch.uint8) if b.numel() else b)
    assert len(got[0]) == len(got[1])


def _randn(*shape, dtype=torch.float16):
    return torch.randn(*shape, device="cuda", dtype=torch.float32).to(dtype)


def _lens(*n):
    return torch.tensor(n, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_rows_same_as_checked_path(monkeypatch, dtype):
    q, k, v = _randn(2, 16, 128, dtype=dtype), _randn(2, 2, 68, 128, dtype=dtype), _randn(2, 2, 68, 128, dtype=dtype)
    for n in (40, 100000, _lens(1, 500)):
        for layout in ("linear", "ring"):
            _both(monkeypatch, lambda: sparse_kernel.sparse_decode_attention(q, k, v, n, 64, layout=layout))
    _both(monkeypatch, lambda: dense_kernel.dense_decode_attention(q, k, v, 68, sm_scale=0.1))
    if dtype == torch.float16:
        _both(monkeypatch, lambda: dense_kernel.dense_decode_attention(q, k, v, _lens(3, 68)))
        kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v))
        _both(monkeypatch, lambda: dense_kernel.dense_decode_attention(q, kt, vt, 68))
        for hnd in (False, True):
            shape = (9, 2, 16, 128) if hnd else (9, 16, 2, 128)
            kp, vp = _randn(*shape), _randn(*shape)
            table = torch.arange(8, dtype=torch.int32, device="cuda").view(2, 4)
            _both(monkeypatch, lambda: paged_kernel.paged_decode_attention(
                q, kp, vp, table, _lens(5, 61), max_seq_len=64, kv_layout="HND" if hnd else "NHD"))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_quantized_same_as_checked_path(monkeypatch, dtype):
    k, v = _randn(2, 2, 4 + 192, 128, dtype=dtype), _randn(2, 2, 4 + 192, 128, dtype=dtype)
    q = _randn(2, 16, 128, dtype=dtype)
    for bits, group in ((2, 32), (4, 32), (3, 64), (8, 32)):
        _both(monkeypatch, lambda: quant_kernel.quantize_k_cache(k[:, :, :192].contiguous(), group, bits))
        _both(monkeypatch, lambda: quant_kernel.quantize_v_cache(v, group, bits))
    for rd in (None, torch.float16):
        _both(monkeypatch, lambda: quant_kernel.build_quantized_kv_cache(k, v, residual_dtype=rd))
    _both(monkeypatch, lambda: quant_kernel.build_quantized_kv_cache(k[:, :, :37].contiguous(),
                                                                     v[:, :, :37].contiguous()))
    t = quant_kernel.build_quantized_kv_cache(k, v)
    parts = [t["k_residual"], t["v_residual"], *[t[n] for n in quant_kernel._KIVI_ORDER]]
    for n in (100, 163840, _lens(7, 900)):
        _both(monkeypatch, lambda: quant_kernel.sparse_decode_attention_quantized(q, *parts, n, 192))


def test_stream_step_same_as_checked_path(monkeypatch):
    k, v, q = _randn(2, 2, 300, 128), _randn(2, 2, 300, 128), _randn(2, 16, 128)
    kn, vn = _randn(2, 2, 128), _randn(2, 2, 128)
    for active in (None, _lens(1, 0)):
        def steps():
            c = kivi_stream.KiviStreamBatch.from_prefill(k, v, window=192)
            outs = [c.step_attend(q, kn * (i + 1), vn, active=active) for i in range(34)]
            return [outs, c.t, c.appended, c.ring]
        _both(monkeypatch, steps)


def test_stream_step_while_entries_are_replaced():
    """The step holds the cache's tensors: another thread may put copies of the
    parts it only reads in their place."""
    k, v, q = _randn(2, 2, 300, 128), _randn(2, 2, 300, 128), _randn(2, 16, 128)
    kn, vn = _randn(2, 2, 128), _randn(2, 2, 128)

    def steps(replace):
        c = kivi_stream.KiviStreamBatch.from_prefill(k, v, window=192)
        stop = threading.Event()

        def work():
            while not stop.is_set():
                for n in list(c.t):
                    if "_sink_" in n:
                        c.t[n] = c.t[n].clone()
        t = threading.Thread(target=work)
        if replace:
            t.start()
        try:
            return torch.stack([c.step_attend(q, kn * (i + 1), vn) for i in range(200)])
        finally:
            stop.set()
            if replace:
                t.join()
    assert torch.equal(steps(False), steps(True))


def test_calls_left_to_the_checks(monkeypatch):
    """Other argument types and views go through the wrapper's own path."""
    q, k, v = _randn(1, 16, 128), _randn(1, 2, 68, 128), _randn(1, 2, 68, 128)
    sparse = sparse_kernel.sparse_decode_attention
    _both(monkeypatch, lambda: sparse(q, k, v, np.int64(100), 64), taken=False)
    _both(monkeypatch, lambda: sparse(q, k, v, 100, 64.0), taken=False)
    _both(monkeypatch, lambda: sparse(q, k, v, 100, 64, sm_scale=1), taken=False)
    _both(monkeypatch, lambda: quant_kernel.quantize_v_cache(k.transpose(1, 2)), taken=False)

    class Sub(torch.Tensor):
        pass
    assert K.host.sparse(q.as_subclass(Sub), k, v, 100, 64, 4, 0, 0.1) is None
    with torch.overrides.TorchFunctionMode():
        assert K.host.sparse(q, k, v, 100, 64, 4, 0, 0.1) is None


def _same_error(monkeypatch, call):
    errors = []
    for skip in (False, True):
        with monkeypatch.context() as m:
            m.setattr(K, "host", Recorder(skip))
            with pytest.raises(Exception) as e:
                call()
            errors.append((e.type, str(e.value)))
    assert errors[0] == errors[1] and errors[0][0] is not NameError


@pytest.mark.parametrize("change", [
    dict(q=lambda q: q.cpu()), dict(q=lambda q: q.double()), dict(q=lambda q: q[0]), dict(k=lambda k: k.bfloat16()),
    dict(k=lambda k: k[:, :, :67].contiguous()), dict(k=lambda k: k.transpose(1, 2).contiguous().transpose(1, 2)),
    dict(v=lambda v: v[:, :1].contiguous()), dict(window=-1), dict(sink=-2), dict(layout="none"),
    dict(seq_len=lambda n: torch.ones(3, dtype=torch.int32, device="cuda")),
    dict(seq_len=lambda n: torch.ones(1, dtype=torch.int64, device="cuda"))])
def test_refused_as_before(monkeypatch, change):
    a = dict(q=_randn(1, 16, 128), k=_randn(1, 2, 68, 128), v=_randn(1, 2, 68, 128), seq_len=99, window=64, sink=4,
             layout="linear")
    for n, x in change.items():
        a[n] = x(a[n]) if callable(x) else x

    def call():
        return sparse_kernel.sparse_decode_attention(a["q"], a["k"], a["v"], a["seq_len"], a["window"], a["sink"],
                                                     layout=a["layout"])
    _same_error(monkeypatch, call)


def _ones(n, dtype=torch.int32):
    return torch.ones(n, dtype=dtype, device="cuda")


def _refused(fn, args, changes):
    """One case per change of a good call's arguments, all of them refused."""
    return [pytest.param(fn, args, c, id=f"{fn}-{i}") for i, c in enumerate(changes)]


_ROWS = dict(q=lambda: _randn(1, 16, 128), k=lambda: _randn(1, 2, 68, 128), v=lambda: _randn(1, 2, 68, 128))
_STRIDED = dict(k=lambda k: k.transpose(1, 2).contiguous().transpose(1, 2))


@pytest.mark.parametrize("fn,args,change", [
    *_refused("dense", dict(_ROWS, seq_len=68), [
        dict(q=lambda q: q.cpu()), dict(q=lambda q: q.double()), dict(q=lambda q: q[0]),
        dict(q=lambda q: q[:, :15].contiguous()), dict(k=lambda k: k.bfloat16()), dict(v=lambda v: v[:, :1].contiguous()),
        dict(k=lambda k: k[:, :, :67].contiguous()), dict(seq_len=67), dict(seq_len=0),
        dict(seq_len=lambda n: _ones(3)), dict(seq_len=lambda n: _ones(1, torch.int64)), _STRIDED,
        dict(q=lambda q: q.float(), k=lambda k: k.float(), v=lambda v: v.float(), seq_len=lambda n: _ones(1))]),
    *_refused("paged", dict(q=lambda: _randn(2, 16, 128), k_pages=lambda: _randn(9, 16, 2, 128),
                            v_pages=lambda: _randn(9, 16, 2, 128), block_table=lambda: _ones(8).view(2, 4),
                            seq_lens=lambda: _lens(5, 61), max_seq_len=64), [
        dict(q=lambda q: q.bfloat16()), dict(k_pages=lambda k: k.float()), dict(v_pages=lambda v: v[:, :8].contiguous()),
        dict(k_pages=lambda k: _randn(9, 12, 2, 128), v_pages=lambda v: _randn(9, 12, 2, 128)),
        dict(block_table=lambda t: t.long()), dict(block_table=lambda t: t[:1]), dict(block_table=lambda t: t.t()),
        dict(seq_lens=lambda n: n.long()), dict(seq_lens=lambda n: n[:1]), dict(max_seq_len=65), dict(kv_layout="DHN")]),
    *_refused("kivi", dict(q=lambda: _randn(1, 16, 128), seq_len=900, window=192), [
        dict(q=lambda q: q.cpu()), dict(q=lambda q: q.double()), dict(q=lambda q: q[:, :15].contiguous()),
        dict(window=193), dict(window=0), dict(seq_len=0), dict(sink=0), dict(sink=40), dict(residual_size=0),
        dict(residual_size=96), dict(bits=9), dict(bits=3), dict(bits=4), dict(group_size=64), dict(group_size=33),
        dict(seq_len=lambda n: _ones(2)), dict(seq_len=lambda n: _ones(1, torch.int64)),
        dict(k_cache=lambda k: k[:, :, 1:].contiguous()), dict(v_cache=lambda v: v.float()),
        dict(k_sink_scale=lambda x: x.float()), dict(v_win_packed=lambda x: x[:, :, ::2]),
        dict(k_win_zero=lambda x: x[:, :1].contiguous())]),
    *_refused("quantize_k", dict(x=lambda: _randn(1, 2, 64, 128)), [
        dict(x=lambda x: x[:, :, :63].contiguous()), dict(x=lambda x: x.cpu()), dict(x=lambda x: x.double()),
        dict(x=lambda x: x[0]), dict(bits=0), dict(bits=9), dict(group_size=0), dict(group_size=-32), dict(group_size=24),
        dict(group_size=2)]),
    *_refused("quantize_v", dict(x=lambda: _randn(1, 2, 64, 128)), [
        dict(x=lambda x: x[..., :120].contiguous()), dict(x=lambda x: x.cpu()), dict(x=lambda x: x.double()),
        dict(x=lambda x: x[0]), dict(bits=0), dict(bits=9), dict(group_size=0), dict(group_size=24), dict(group_size=2)]),
    *_refused("build", dict(k=lambda: _randn(1, 2, 196, 128), v=lambda: _randn(1, 2, 196, 128)), [
        dict(k=lambda k: k[:, :, :195].contiguous(), v=lambda v: v[:, :, :195].contiguous()),
        dict(k=lambda k: k.cpu()), dict(k=lambda k: k.bfloat16()), dict(v=lambda v: v[:, :1].contiguous()),
        dict(k=lambda k: k.double(), v=lambda v: v.double()), dict(k=lambda k: k[0]), dict(sink=0), dict(sink=33),
        dict(residual_size=0), dict(residual_size=100), dict(k=lambda k: k[:, :, :4].contiguous(),
                                                             v=lambda v: v[:, :, :4].contiguous()),
        dict(residual_dtype=torch.bfloat16)]),
    *_refused("step_attend", dict(q=lambda: _randn(2, 16, 128), k_new=lambda: _randn(2, 2, 128),
                                  v_new=lambda: _randn(2, 2, 128)), [
        dict(q=lambda q: q.cpu()), dict(q=lambda q: q.bfloat16()), dict(q=lambda q: q[:1]),
        dict(q=lambda q: q[:, :15].contiguous()), dict(k_new=lambda k: k[:1]), dict(k_new=lambda k: k.float()),
        dict(v_new=lambda v: v.cpu()), dict(active=lambda a: _ones(3))]),
])
def test_other_entries_refuse_as_before(monkeypatch, fn, args, change):
    a = {n: x() if callable(x) else x for n, x in args.items()}
    if fn == "kivi":
        t = quant_kernel.build_quantized_kv_cache(_randn(1, 2, 196, 128), _randn(1, 2, 196, 128))
        a.update(k_cache=t["k_residual"], v_cache=t["v_residual"], **{n: t[n] for n in quant_kernel._KIVI_ORDER})
    if fn == "step_attend":
        a["self"] = kivi_stream.KiviStreamBatch.from_prefill(_randn(2, 2, 300, 128), _randn(2, 2, 300, 128), window=192)
    for n, x in change.items():
        a[n] = x(a.get(n)) if callable(x) else x
    entry = {"dense": dense_kernel.dense_decode_attention, "paged": paged_kernel.paged_decode_attention,
             "kivi": quant_kernel.sparse_decode_attention_quantized, "build": quant_kernel.build_quantized_kv_cache,
             "quantize_k": lambda x, **kw: quant_kernel.quantize_k_cache(x, **kw),
             "quantize_v": lambda x, **kw: quant_kernel.quantize_v_cache(x, **kw),
             "step_attend": kivi_stream.KiviStreamBatch.step_attend}[fn]
    if fn == "build":
        a["k_compacted"], a["v_compacted"] = a.pop("k"), a.pop("v")
    _same_error(monkeypatch, lambda: entry(**a))
