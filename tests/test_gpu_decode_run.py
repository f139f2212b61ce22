"""The decode steps launched from one native call against the same steps op by op: ids, logits and caches bit for bit (the same launches)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(codec, n_layers, n_heads, n_kv, hd, hidden, vocab, seed):
    from air_hip import decode, weights
    g = torch.Generator(device="cuda").manual_seed(seed)
    E = n_heads * hd
    cfg = weights.LlamaConfig(n_layers=n_layers, emb_dim=E, n_heads=n_heads, head_dim=hd, n_kv_heads=n_kv, hidden_dim=hidden, vocab_size=vocab)
    randn = lambda *shape: torch.randn(shape, device="cuda", generator=g)
    words = lambda *shape: torch.randint(-2 ** 31, 2 ** 31 - 1, shape, dtype=torch.int32, device="cuda", generator=g)

    def matrix(K, N):
        gs = 128 if codec == "awq" else 32
        scales = ((0.5 + randn(K // gs, N).abs()) * (K ** -0.5 / 8)).bfloat16()
        return (words(K, N // 8), words(K // gs, N // 8), scales) if codec == "awq" else (words(K, N // 8), scales, (scales.float() * -7.5).bfloat16())

    norm = lambda: (1 + 0.1 * randn(E)).bfloat16()
    layers = [decode.DecodeLayer(norm(), norm(), matrix(E, (n_heads + 2 * n_kv) * hd), matrix(E, E), matrix(E, hidden), matrix(E, hidden), matrix(hidden, E),
                                 codec=codec).with_stream() for _ in range(n_layers)]
    return cfg, layers, randn(vocab, E).bfloat16(), norm(), randn(vocab, E).bfloat16(), decode.generate_rope_lut(cfg, 200)


@pytest.mark.parametrize("codec,n_layers,n_heads,n_kv,hd,hidden,vocab,start,n", [("awq", 1, 4, 2, 64, 384, 40, 0, 5), ("awq", 3, 8, 1, 128, 640, 1003, 126, 4),
                                                                                 ("q4nx", 2, 4, 4, 64, 512, 200, 63, 3), ("awq", 2, 32, 8, 64, 8192, 512, 197, 3)])
def test_native_decode_steps(monkeypatch, codec, n_layers, n_heads, n_kv, hd, hidden, vocab, start, n):
    from air_hip import decode, ops
    print("decode run", codec, n_layers, n_heads, n_kv, hd, hidden, vocab, start, n, flush=True)
    cfg, layers, embed, final, head, lut = _model(codec, n_layers, n_heads, n_kv, hd, hidden, vocab, 3 * vocab + n)
    caches = decode.new_kv_cache(cfg, 200)
    for k, v in caches:
        k.normal_(), v.normal_()
    copies = [(k.clone(), v.clone()) for k, v in caches]
    first = torch.tensor([vocab - 1], dtype=torch.int32, device="cuda")
    ran = []
    run = ops.decode_run
    monkeypatch.setattr(ops, "decode_run", lambda *a: ran.append(run(*a)) or ran[-1])
    got = decode.decode_greedy(first, n, layers, embed, final, head, cfg, caches, start, lut)
    logits, best = decode.decode_token(int(first), layers, embed, final, head, cfg, caches, start, lut, return_argmax=True)
    assert len(ran) == 2 and all(r is not None for r in ran)
    assert run(embed[0], layers, embed, final, head, lut, cfg, caches, 200 - n + 1, n, got) is None   # past the cache: the ops' own errors
    monkeypatch.setattr(ops, "decode_run", lambda *a: None)
    want = decode.decode_greedy(first, n, layers, embed, final, head, cfg, copies, start, lut)
    logits2, best2 = decode.decode_token(int(first), layers, embed, final, head, cfg, copies, start, lut, return_argmax=True)
    assert torch.equal(got, want) and torch.equal(best, best2) and torch.equal(logits, logits2)
    assert all(torch.equal(a, b) and torch.equal(c, d) for (a, c), (b, d) in zip(caches, copies))


@pytest.mark.parametrize("n_heads,n_kv,hd,max_seq,positions", [(8, 2, 64, 3000, [2048, 2976, 2999]), (4, 4, 64, 2200, [2100]), (16, 2, 64, 2600, [64, 2500])])
def test_decode_attention_past_a_trip(n_heads, n_kv, hd, max_seq, positions):
    """More than 32 chunks of 64: several trips of a workgroup, and workgroups without a position."""
    import test_gpu_decode
    from air_hip import ops
    test_gpu_decode.test_decode_attention(ops, n_heads, n_kv, hd, max_seq, positions)


@pytest.mark.parametrize("n_heads,n_kv,hd", [(8, 2, 64), (4, 4, 128), (16, 2, 128)])
def test_decode_attention_with_infinities(n_heads, n_kv, hd):
    """Keys that no head looks at (scores of minus infinity: one, a wave's positions, a whole chunk), an infinite value, a NaN key, and NaN
    behind the last position; against float64 with the same rows."""
    from air_hip import ops
    print("attention infinities", n_heads, n_kv, hd, flush=True)
    g = torch.Generator(device="cuda").manual_seed(hd + n_heads)
    randn = lambda *shape: torch.randn(shape, device="cuda", generator=g).bfloat16()
    inf, pos, max_seq = float("inf"), 299, 320
    lut = torch.cat([torch.ones(hd // 2), torch.zeros(hd // 2)]).bfloat16().cuda()   # no rotation
    for rows, value, nan in ([77], None, None), (list(range(8)) + list(range(64, 136)), None, None), ([298], (150, -inf), None), ([0], (299, inf), 1):
        qkv, k, v = randn((n_heads + 2 * n_kv) * hd), randn(n_kv, max_seq, hd), randn(n_kv, max_seq, hd)
        q, k_new, v_new = (t.view(-1, hd) for t in qkv.split([n_heads * hd, n_kv * hd, n_kv * hd]))
        q[:, 5] = q[:, 5].abs() + 1.0
        k[:, rows, 5] = -inf
        k[:, pos + 1:], v[:, pos + 1:] = float("nan"), float("nan")
        if value:
            (v_new if value[0] == pos else v[:, value[0]])[:, 3] = value[1]
        if nan is not None:
            k[0, nan, 9] = float("nan")
        keys, values = k[:, :pos + 1].double(), v[:, :pos + 1].double()
        keys[:, pos], values[:, pos] = k_new.double(), v_new.double()
        out = ops.decode_attention(qkv, lut, k, v, pos, n_heads).view(n_heads, hd)
        for h in range(n_heads):
            kv = h // (n_heads // n_kv)
            w = torch.softmax((keys[kv] * q[h].double()).sum(-1) * hd ** -0.5, 0)
            want = (w[:, None] * values[kv]).sum(0)
            assert torch.equal(out[h].isnan(), want.isnan()) and torch.equal(out[h].isinf(), want.isinf()), (h, rows, value, nan)
            at = want.isfinite()
            assert torch.equal(out[h][want.isinf()].double(), want[want.isinf()])
            # as the other attention tests: 1 bf16 ulp (2^-7 of the value) and 2e-3
            assert bool(((out[h].double() - want)[at].abs() <= 2.0 ** -7 * want[at].abs() + 2e-3).all())
