"""Passes and operators whose host side is native code (csrc/host.cpp) against the operators in Python, bit for bit (the same launches), and the calls
that are left to those."""
import ctypes

import numpy as np
import pytest
import torch

import test_gpu_kuvonex as tk
import test_gpu_sitirax as ts
from helpers import KUVONEX_MIXED, SITIRAX_MIXED, make_awq, make_x
from test_gpu_q4nx import make
from test_gpu_stream_order import bits, dev

pytestmark = pytest.mark.gpu


def _leftovers(cache):
    return list(cache.rows.values()) if hasattr(cache, "rows") else [t for l in cache.layers for t in l.values()]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mod,config,entry", [(tk, KUVONEX_MIXED, "latent_rows"), (tk, tk.TALL, "latent_rows"), (tk, tk.WIDE, "latent_rows"), (tk, tk.ONE_LAYER, "latent_rows"),
                                              (ts, SITIRAX_MIXED, "mixed_rows"), (ts, ts.TALL, "mixed_rows"), (ts, ts.WIDE, "mixed_rows"),
                                              (ts, ts.ONE_PARALLEL, "mixed_rows")])
def test_passes(monkeypatch, mod, config, entry, dtype):
    from air_hip import _lib
    print("native pass", entry, dtype, flush=True)
    m, _ = mod._model(config, 5, dtype)
    host, ran = _lib.host_dense(), []
    run = getattr(host, entry)
    monkeypatch.setattr(host, entry, lambda *a: ran.append(run(*a)) or ran[-1])
    caches = [m.new_cache(242), m.new_cache(242)]
    for t in [t for c in caches for t in _leftovers(c)]:
        t.zero_()   # (rows behind the sequence are compared too)
    pos = 0
    for n in (2, 17, 1, 65, 130, 1):   # a few tokens, a portion's last one, edges of the forms' ranges, behind what is there
        ids = torch.tensor(mod._tokens(n, config["vocab"], seed=n), dtype=torch.int32, device="cuda")
        got, want = m._rows(caches[0], ids, pos), m._rows(caches[1], ids, pos, trace=[])
        assert len(ran) == 1 and (ran.pop() is None) == (n == 1 and mod is ts)   # (one token of a mixed model is the operators')
        assert torch.equal(got, want), n
        assert all(torch.equal(a, b) for a, b in zip(*map(_leftovers, caches))), n
        pos += n
    c = m.config
    logits, best = host.tail(m.tail_intake, got[-1], m.final_norm, m.head, c.eps, c.width, m.vocab, torch.cuda.current_stream().cuda_stream)
    logits2, best2 = m._tail(m._pending(want[-1].contiguous()))
    assert torch.equal(logits[:m.vocab], logits2) and torch.equal(best, best2)


def test_passes_left_to_the_operators():
    """Tensors of another type or shape: nothing is launched, and the operators say what is wrong."""
    m, _ = tk._model(KUVONEX_MIXED, 6, torch.float32)
    ids = torch.zeros(3, dtype=torch.int32, device="cuda")
    with pytest.raises(ValueError, match="do not fit a cache"):
        m._rows(m.new_cache(2), ids, 0)
    with pytest.raises(TypeError):
        m._rows(m.new_cache(8), ids.long(), 0)
    m.layers[0].norm1 = m.layers[0].norm1.double()
    with pytest.raises(TypeError, match="float32"):
        m._rows(m.new_cache(8), ids, 0)


@pytest.mark.parametrize("q4", [False, True])
def test_linear_forms(monkeypatch, q4):
    from air_hip import _lib, ops
    from oracle import awq as oawq
    K, N = 256, 128
    if q4:
        q, s, mins = make(N, K, seed=1)
        w = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(mins.T))
    else:
        w = ops.repack_stream(*map(dev, make_awq(K, N, seed=1)))
    gemv, gemm = (ops.q4nx_gemv_stream, ops.q4nx_gemm_stream) if q4 else (ops.w4a16_gemv_stream, ops.w4a16_gemm_stream)
    host, ran = _lib.host_w4a16(), []
    run = host.linear
    monkeypatch.setattr(host, "linear", lambda *a: ran.append(run(*a)) or ran[-1])
    for M in (1, 2, 16, 17, 70, 130):
        x = dev(make_x((M, K), seed=M))
        got = gemm(x, w)
        assert ran.pop() is not None and got.shape == (M, N)
        out = torch.empty_like(got)
        assert gemm(x, w, out=out).data_ptr() == out.data_ptr() and not ran   # a result of the caller's
        assert np.array_equal(bits(got), bits(out)), M
        assert np.array_equal(bits(gemm(x.view(torch.int16), w)), bits(out)) and ran.pop() is None   # 16-bit patterns
    row = dev(make_x((1, K), seed=1))
    for y in (gemm(row[0], w), gemv(row, w), gemv(row[0], w)):
        assert ran.pop() is not None and y.shape == (N,)
        assert np.array_equal(bits(y), bits(gemv(row, w, out=torch.empty(N, dtype=torch.bfloat16, device="cuda"))))
    for bad, error in ((row[0, 1:], ValueError), (row[0].float(), TypeError), (row.repeat(4, 2)[:, ::2], ValueError), (row.cpu(), RuntimeError)):
        for op in (gemv, gemm):
            with pytest.raises(error):
                op(bad, w)


def test_other_threads_run_while_a_call_launches():
    """Entry points are called without Python's lock: PyGILState_Check in their place, which returns 0 then, and 1, an error's code, where it is held.
    (Nothing is launched.)"""
    from air_hip import _lib, ops
    held = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    asked = ("_slices", "_splits", "gemm_parts", "_tile_rows", "_max_tiles", "gemv_keys", "_supported", "_bytes")   # (these launch nothing)
    stream = torch.cuda.current_stream().cuda_stream
    models = [mod._model(config, 5, torch.bfloat16)[0] for mod, config in ((tk, KUVONEX_MIXED), (ts, SITIRAX_MIXED))]
    w = ops.repack_stream(*map(dev, make_awq(256, 128, seed=1)))
    for bind, lib, names in ((_lib.host_dense().bind_dense, _lib.load_dense_library(), _lib.host_dense().dense_entries()),
                             (_lib.host_w4a16().bind_w4a16, _lib.load_library(), _lib.host_w4a16().w4a16_entries())):
        real = _lib._addresses(lib, names)
        bind({n: at if n.endswith(asked) else held for n, at in real.items()})
        try:
            if lib is _lib.load_library():
                for M in (1, 2, 17, 130):
                    assert _lib.host_w4a16().linear(dev(make_x((M, 256), seed=M)), w.buf, 256, 128, False, False, stream) is not None
                continue
            for m in models:
                for n in (2, 70):
                    assert m._rows(m.new_cache(80), torch.zeros(n, dtype=torch.int32, device="cuda"), 0).shape == (n, m.embed.shape[1])
                c = m.config
                assert _lib.host_dense().tail(m.tail_intake, torch.zeros(m.embed.shape[1], device="cuda"), m.final_norm, m.head, c.eps, c.width, m.vocab, stream) is not None
        finally:
            bind(real)


def test_errors_of_a_call():
    """What an entry point refuses is the same error as from Python."""
    from air_hip import _lib, ops
    w = ops.repack_stream(*map(dev, make_awq(256, 128, seed=1)))
    with pytest.raises(_lib.W4A16Error):
        _lib.host_w4a16().linear(dev(make_x((1, 192), seed=1)), w.buf, 192, 128, False, True, torch.cuda.current_stream().cuda_stream)   # no whole groups
