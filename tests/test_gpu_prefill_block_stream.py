"""GPU parity of the two prompt-pass blocks on stream-order weights (RMSNorm + Q|K|V GEMM + RoPE; O projection +
residual + RMSNorm + SwiGLU FFN + residual), which run the tiled stream-order GEMM with fused epilogues.

Two kinds of check per stage.  Against the library's own plain product (w4a16_gemm_stream through the same tiled
kernel): the epilogues work on the bf16 product, so residual adds and rotations must come out bit for bit.  Against the
oracle: each stage on the kernel's own input to it within the roundings of that stage, and the whole block against the
restated CPU reference under the reference's gate.
"""
import numpy as np
import pytest
import torch

from helpers import bf16_ulp, dense_f64, make_awq, make_x
from oracle import awq as oawq, reference as oref
from oracle.bf16 import bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu


def dev(a):
    a = np.ascontiguousarray(a)
    if a.dtype == np.uint16:
        return torch.from_numpy(a.view(np.int16)).cuda().view(torch.bfloat16)
    return torch.from_numpy(a).cuda()


def bits(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


@pytest.fixture(scope="module")
def ops():
    from air_hip import ops
    return ops


@pytest.fixture
def tiled_gemm(ops):
    """w4a16_gemm_stream runs the tiled kernel from M = 17 on (by itself it does from M = 97 on), so that its output
    is the product inside the fused calls bit for bit."""
    ops.tune("prefill_min_m", 17)
    yield
    ops.tune("prefill_min_m", 0)


def _scaled(K, N, seed, scale):
    qw, qz, s = make_awq(K, N, seed=seed)
    return qw, qz, f32_to_bf16_bits(bf16_bits_to_f32(s) * np.float32(scale))


def _weights(E, H, seed, scale=1.0):
    return [_scaled(K, N, seed + i, scale) for i, (K, N) in enumerate(((E, E), (E, H), (E, H), (H, E)))]


def _sw(ops, w):
    return ops.repack_stream(*map(dev, w))


def _norm_w(E, seed):
    rng = np.random.default_rng(seed)
    return f32_to_bf16_bits((rng.standard_normal(E) * 0.1 + 1.0).astype(np.float32))


def _add_rounded(prod, add):
    return (prod.float() + add.float()).to(torch.bfloat16)


def _close_sum(got_bits, prod64, add32, what):
    want = prod64 + add32
    err = np.abs(bf16_bits_to_f32(got_bits).astype(np.float64) - want)
    tol = bf16_ulp(want) + bf16_ulp(prod64) + 2e-3
    assert np.all(err <= tol), f"{what}: worst {np.max(err - tol):.4g} over tolerance at {np.unravel_index(np.argmax(err - tol), err.shape)}"


@pytest.mark.parametrize("M,E,H", [(40, 256, 512), (300, 512, 1280), (17, 256, 256), (260, 1024, 2048)])
def test_prefill_block_stream_stage_by_stage(ops, tiled_gemm, M, E, H):
    print(f"prefill block (stream order) M={M} E={E} H={H}", flush=True)
    wo, wg, wu, wd = _weights(E, H, seed=M + E, scale=0.25)
    so, sg, su, sd = (_sw(ops, w) for w in (wo, wg, wu, wd))
    attn, xres, nw = make_x((M, E), seed=M), make_x((M, E), seed=M + 1), _norm_w(E, M + 2)
    y, res1, h = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), so, sg, su, sd, return_intermediates=True)
    y2 = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), so, sg, su, sd)
    torch.cuda.synchronize()
    y_b, res1_b, h_b = bits(y), bits(res1), bits(h)
    assert np.array_equal(bits(y2), y_b), "intermediates kept in the workspace give another result"
    f = lambda b: bf16_bits_to_f32(b).astype(np.float64)
    # 1. O projection + residual: the epilogue on the plain product, and the float64 product
    assert torch.equal(res1.view(torch.int16), _add_rounded(ops.w4a16_gemm_stream(dev(attn), so), dev(xres)).view(torch.int16))
    _close_sum(res1_b, f(attn) @ dense_f64(*wo, rounded=True), f(xres), "res1")
    # 2. row-wise RMSNorm of the kernel's res1
    normed = ops.rms_norm_rows(res1, dev(nw))
    n_gpu = bits(normed)
    n_ref = oref.rms_norm_rows_bf16(res1_b, nw)
    nd = np.abs(f(n_gpu) - f(n_ref))
    assert np.all(nd <= bf16_ulp(f(n_ref))) and np.mean(n_gpu != n_ref) < 0.01, (nd.max(), np.mean(n_gpu != n_ref))
    # 3. gate / up + SwiGLU: on the library's own bf16 products within one rounding (+ the exponential's last bits),
    #    and on float64 products of the kernel's normalised rows
    gb, ub = f(bits(ops.w4a16_gemm_stream(normed, sg))), f(bits(ops.w4a16_gemm_stream(normed, su)))
    h_exact = gb / (1.0 + np.exp(-gb)) * ub
    assert np.all(np.abs(f(h_b) - h_exact) <= 0.51 * bf16_ulp(h_exact) + 1e-6 * np.abs(h_exact) + 1e-30), \
        np.max(np.abs(f(h_b) - h_exact) / bf16_ulp(h_exact))
    G, U = f(n_gpu) @ dense_f64(*wg, rounded=True), f(n_gpu) @ dense_f64(*wu, rounded=True)
    g64, u64 = f(f32_to_bf16_bits(G.astype(np.float32))), f(f32_to_bf16_bits(U.astype(np.float32)))
    h_want = g64 / (1.0 + np.exp(-g64)) * u64
    h_tol = 4 * bf16_ulp(h_want) + 1.2 * bf16_ulp(g64) * np.abs(u64) + bf16_ulp(u64) * np.abs(g64) + 1e-3
    assert np.all(np.abs(f(h_b) - h_want) <= h_tol), np.max(np.abs(f(h_b) - h_want) - h_tol)
    # 4. down projection + residual on the kernel's h and res1
    assert torch.equal(y.view(torch.int16), _add_rounded(ops.w4a16_gemm_stream(h, sd), res1).view(torch.int16))
    _close_sum(y_b, f(h_b) @ dense_f64(*wd, rounded=True), f(res1_b), "y")
    # the whole block against the restated CPU reference, under the reference's gate and a tighter one
    l1 = [oawq.repack_hf_awq_linear(*w, 128) for w in (wo, wg, wu, wd)]
    want, _, _ = oref.o_ffn_int4_prefill_reference(*l1, attn, xres, nw)
    got_f, want_f = bf16_bits_to_f32(y_b), bf16_bits_to_f32(want)
    assert oref.check_outputs(got_f, want_f, rtol=0.5, atol=10.0, max_mismatch_percentage=0.5, min_correlation=0.99)
    assert np.max(np.abs(got_f - want_f)) <= 8 * 2.0**-8 * np.max(np.abs(want_f)), np.max(np.abs(got_f - want_f))


def test_prefill_block_stream_zero_projections_are_exact(ops):
    """q == z makes a projection exactly zero: res1 is the residual and y is res1, bit for bit."""
    M, E, H = 200, 256, 512
    wo, wg, wu, wd = _weights(E, H, seed=90)
    zero = lambda w: (w[1].repeat(128, axis=0), w[1], w[2])      # every q row equals its group's z row
    attn, xres, nw = make_x((M, E), seed=91), make_x((M, E), seed=92), _norm_w(E, 93)
    print("prefill block (stream order), zero O and down projections", flush=True)
    y, res1, h = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), _sw(ops, zero(wo)), _sw(ops, wg), _sw(ops, wu),
                                          _sw(ops, zero(wd)), return_intermediates=True)
    torch.cuda.synchronize()
    assert np.array_equal(bits(res1), xres) and np.array_equal(bits(y), xres)
    _, _, h0 = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), _sw(ops, wo), _sw(ops, zero(wg)), _sw(ops, wu),
                                        _sw(ops, wd), return_intermediates=True)
    assert np.all((bits(h0) & 0x7FFF) == 0)


@pytest.mark.parametrize("M,E,H,tile", [(300, 512, 1280, 0), (300, 512, 1024, 1), (130, 256, 768, 3), (2048, 2048, 8192, 0),
                                        (300, 512, 1280, 5), (260, 256, 1792, 5)])
def test_prefill_block_stream_paired_gate_up_launch_equals_two_launches(ops, M, E, H, tile):
    """Gate and up in one launch (a tile holds the same columns of both products) against the gate launch followed by
    the up launch with the SwiGLU epilogue: the same bits in h and y, at the tile width chosen by shape and forced."""
    ws = _weights(E, H, seed=70 + tile, scale=0.25)
    sws = [_sw(ops, w) for w in ws]
    attn, xres, nw = make_x((M, E), seed=71), make_x((M, E), seed=72), _norm_w(E, 73)
    print(f"prefill block (stream order), one launch for gate and up against two, M={M} E={E} H={H} tile={tile}", flush=True)
    ops.tune("prefill_tile", tile)
    try:
        y1, _, h1 = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), *sws, return_intermediates=True)
        ops.tune("prefill_swiglu_split", 1)
        y2, _, h2 = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), *sws, return_intermediates=True)
        torch.cuda.synchronize()
    finally:
        ops.tune("prefill_swiglu_split", 0)
        ops.tune("prefill_tile", 0)
    assert torch.equal(h1.view(torch.int16), h2.view(torch.int16)) and torch.equal(y1.view(torch.int16), y2.view(torch.int16))
    assert float(h1.float().abs().max()) > 0


def test_prefill_block_stream_agrees_with_the_checkpoint_layout_block(ops):
    """The same block on the checkpoint tensors (another kernel, another summation order inside a product): the
    outputs differ by roundings only."""
    M, E, H = 300, 512, 1024
    ws = _weights(E, H, seed=60, scale=0.25)
    attn, xres, nw = make_x((M, E), seed=61), make_x((M, E), seed=62), _norm_w(E, 63)
    print("prefill block, stream order against checkpoint layout", flush=True)
    a = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), *(_sw(ops, w) for w in ws))
    b = ops.prefill_o_ffn(dev(attn), dev(xres), dev(nw), *(tuple(map(dev, w)) for w in ws))
    err = (a.double() - b.double()).abs()
    assert float(err.max()) <= 4 * 2.0**-8 * float(b.double().abs().max()), float(err.max())


@pytest.mark.parametrize("M,E,H", [(2048, 2048, 8192), (512, 4096, 14336)])
def test_prefill_block_stream_model_sizes(ops, M, E, H):
    """Llama-3.2-1B's dimensions at the reference example's sequence length, and Llama-3-8B's at 512 tokens: the
    epilogues against the library's own products bit for bit, the products against float64 on the GPU."""
    print(f"prefill block (stream order) M={M} E={E} H={H}", flush=True)
    wo, wg, wu, wd = _weights(E, H, seed=7, scale=0.1)
    so, sg, su, sd = (_sw(ops, w) for w in (wo, wg, wu, wd))
    attn, xres, nw = make_x((M, E), seed=8), make_x((M, E), seed=9), _norm_w(E, 10)
    y, res1, h = ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), so, sg, su, sd, return_intermediates=True)
    torch.cuda.synchronize()
    assert torch.equal(res1.view(torch.int16), _add_rounded(ops.w4a16_gemm_stream(dev(attn), so), dev(xres)).view(torch.int16))
    assert torch.equal(y.view(torch.int16), _add_rounded(ops.w4a16_gemm_stream(h, sd), res1).view(torch.int16))
    d64 = lambda w: torch.from_numpy(dense_f64(*w, rounded=True)).cuda()
    rnd = lambda t: t.to(torch.bfloat16).double()
    res1_t = rnd(rnd(dev(attn).double() @ d64(wo)) + dev(xres).double())
    err = (res1.double() - res1_t).abs()
    assert float(err.max()) <= 2.0**-7 * float(res1_t.abs().max()) and float((err > 0).double().mean()) < 0.02
    n_t = rnd(torch.nn.functional.rms_norm(res1.double(), (E,), dev(nw).double(), eps=1e-5))
    g_t, u_t = rnd(n_t @ d64(wg)), rnd(n_t @ d64(wu))
    h_t = rnd(torch.nn.functional.silu(g_t) * u_t)
    herr = (h.double() - h_t).abs()
    assert float(herr.max()) <= 8 * 2.0**-8 * float(h_t.abs().max()) and float((herr > 0).double().mean()) < 0.1
    y_t = rnd(rnd(h.double() @ d64(wd)) + res1.double())
    yerr = (y.double() - y_t).abs()
    assert float(yerr.max()) <= 2.0**-7 * float(y_t.abs().max()) and float((yerr > 0).double().mean()) < 0.02


def test_prefill_block_stream_rejects_bad_arguments(ops):
    from air_hip import _lib
    lib = _lib.load_library()
    ws = lib.w4a16_prefill_block_workspace_bytes(32, 256, 256)
    wsq = lib.w4a16_prefill_qkv_workspace_bytes(32, 256)
    zeros = torch.zeros(1 << 18, dtype=torch.int32, device="cuda")
    out = torch.zeros(1 << 18, dtype=torch.int32, device="cuda")
    scratch = torch.zeros(max(ws, wsq), dtype=torch.uint8, device="cuda")
    P, Y, W = zeros.data_ptr(), out.data_ptr(), scratch.data_ptr()
    args = [P, P, P, 1e-5] + [P] * 4 + [Y, None, None, 32, 256, 256, 128, W, ws, None]
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*args) == 0
    torch.cuda.synchronize()
    bad = list(args); bad[16] = ws - 1
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*bad) == _lib.ERR_WORKSPACE
    bad = list(args); bad[12] = 128            # E must be a multiple of 256
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(args); bad[13] = 320            # and so must H
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(args); bad[14] = 64
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*bad) == _lib.ERR_GROUP
    bad = list(args); bad[5] = None
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*bad) == _lib.ERR_NULL
    bad = list(args); bad[0] = P + 2
    assert lib.w4a16_prefill_o_ffn_stream_bf16(*bad) == _lib.ERR_ALIGN
    qargs = [P, P, 1e-5, P, P, 64, 0, Y, 32, 256, 2, 1, 64, 128, W, wsq, None]
    assert lib.w4a16_prefill_rms_qkv_rope_stream_bf16(*qargs) == 0
    torch.cuda.synchronize()
    bad = list(qargs); bad[6] = 33             # positions 33 .. 64 of a 64-row table
    assert lib.w4a16_prefill_rms_qkv_rope_stream_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(qargs); bad[12] = 32            # head_dim
    assert lib.w4a16_prefill_rms_qkv_rope_stream_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(qargs); bad[15] = wsq - 1
    assert lib.w4a16_prefill_rms_qkv_rope_stream_bf16(*bad) == _lib.ERR_WORKSPACE
    bad = list(qargs); bad[3] = None
    assert lib.w4a16_prefill_rms_qkv_rope_stream_bf16(*bad) == _lib.ERR_NULL


def _qkv_weights(E, nh, nkv, hd, seed, scale=0.25):
    parts = [_scaled(E, N, seed + i, scale) for i, N in enumerate((nh * hd, nkv * hd, nkv * hd))]
    fused = tuple(np.concatenate([p[j] for p in parts], axis=1) for j in range(3))
    return parts, fused


# head widths 64 and 128 through every tile width that holds whole heads (tile 0: the width chosen by shape, which for
# these small matrices is 64 or 128 columns; 1: 256, 2: 192, 3: 128, 4: 64, 5: 256 mixed with 128), ragged M, one row
# tile and two
@pytest.mark.parametrize("M,E,nh,nkv,hd,pos0,tile", [(40, 256, 4, 2, 64, 0, 0), (300, 512, 8, 8, 64, 7, 0), (130, 256, 2, 1, 128, 100, 0),
                                                      (17, 256, 3, 1, 64, 1, 0), (270, 512, 1, 1, 128, 3, 0), (300, 256, 4, 2, 64, 5, 1),
                                                      (100, 256, 4, 1, 64, 2, 2), (260, 512, 2, 1, 128, 9, 1), (64, 256, 4, 2, 64, 0, 3),
                                                      (33, 256, 2, 1, 64, 11, 4), (270, 256, 4, 1, 128, 6, 5), (100, 512, 3, 2, 128, 0, 5)])
def test_prefill_rms_qkv_rope_stream(ops, tiled_gemm, M, E, nh, nkv, hd, pos0, tile):
    from oracle import decode as odec
    print(f"prefill qkv rope (stream order) M={M} E={E} heads {nh}/{nkv} hd={hd} pos0={pos0} tile={tile}", flush=True)
    parts, fused = _qkv_weights(E, nh, nkv, hd, seed=M + E)
    x, nw = make_x((M, E), seed=M + 3), _norm_w(E, M + 4)
    lut = odec.generate_rope_lut(hd, 500000.0, pos0 + M + 5)
    sw = _sw(ops, fused)
    ops.tune("prefill_tile", tile)
    try:
        out = ops.prefill_rms_qkv_rope_stream(dev(x), dev(nw), sw, dev(lut), pos0, nh, nkv, hd)
        torch.cuda.synchronize()
    finally:
        ops.tune("prefill_tile", 0)
    normed = ops.rms_norm_rows(dev(x), dev(nw))
    plain = ops.w4a16_gemm_stream(normed, sw)
    torch.cuda.synchronize()
    got = bits(out)
    f = lambda b: bf16_bits_to_f32(b).astype(np.float64)
    nq, nk = nh * hd, nkv * hd
    # V columns are the plain product, bit for bit the GEMM entry point's
    assert np.array_equal(got[:, nq + nk:], bits(plain)[:, nq + nk:])
    # Q and K: the rotation of the kernel's own bf16 product is reproduced exactly by the oracle's rotation
    rows = lut[pos0:pos0 + M]
    for lo, n in ((0, nh), (nq, nkv)):
        prod = bits(plain)[:, lo:lo + n * hd].reshape(M * n, hd)
        want = odec.rope_rows(prod, np.repeat(rows, n, axis=0)).reshape(M, n * hd)
        assert np.array_equal(got[:, lo:lo + n * hd], want)
    # and the whole call against the restated CPU reference (float32 BLAS products, one-ulp flips upstream)
    l1 = [oawq.repack_hf_awq_linear(*w, 128) for w in parts]
    ref_out = odec.prefill_rms_qkv_rope_reference(x, nw, *l1, lut, pos0, nh, nkv, hd)
    err = np.abs(f(got) - f(ref_out))
    assert np.max(err) <= 4 * 2.0**-8 * np.max(np.abs(f(ref_out))), err.max()
    ref_r = odec.prefill_rms_qkv_rope_reference(x, nw, *l1, lut, pos0, nh, nkv, hd, round_weights=True)
    assert np.mean(got != ref_r) < 0.1, np.mean(got != ref_r)


@pytest.mark.parametrize("M", [1, 17, 40, 100, 300])
def test_prefill_blocks_stream_in_the_least_workspace(ops, M):
    """2 M E bytes for the projections, the block's rows and split parts for the rest: what callers had to bring before few rows ran in slices, and nothing behind it is written.
    Slices only change the order of the fp32 sums: a bf16 step here and there, which the FFN carries on (2^-7 of a row's norm)."""
    from air_hip import _lib
    from oracle import decode as odec
    lib = _lib.load_library()
    E, H, nh, nkv, hd = 1024, 2048, 8, 4, 128
    _, fused = _qkv_weights(E, nh, nkv, hd, seed=M)
    ws = [_sw(ops, w) for w in _weights(E, H, seed=M)]
    sw, lut = _sw(ops, fused), dev(odec.generate_rope_lut(hd, 500000.0, M))
    x, attn, nw = dev(make_x((M, E), seed=M)), dev(make_x((M, E), seed=M + 1)), dev(_norm_w(E, 3))
    guard = 4096
    def least(n):
        buf = torch.full((n + guard,), 77, dtype=torch.uint8, device="cuda")
        return buf, buf[:n]
    print("prompt blocks, least workspace", M, flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    b1, w1 = least(lib.w4a16_prefill_qkv_workspace_bytes(M, E))
    assert w1.numel() == -(-2 * M * E // 256) * 256
    q1 = torch.empty((M, (nh + 2 * nkv) * hd), dtype=torch.bfloat16, device="cuda")
    _lib.check(lib.w4a16_prefill_rms_qkv_rope_stream_bf16(x.data_ptr(), nw.data_ptr(), 1e-5, sw.buf.data_ptr(), lut.data_ptr(), M, 0, q1.data_ptr(), M, E, nh, nkv, hd, 128,
                                                          w1.data_ptr(), w1.numel(), stream))
    b2, w2 = least(lib.w4a16_prefill_block_workspace_bytes(M, E, H))
    y1 = torch.empty((M, E), dtype=torch.bfloat16, device="cuda")
    _lib.check(lib.w4a16_prefill_o_ffn_stream_bf16(attn.data_ptr(), x.data_ptr(), nw.data_ptr(), 1e-5, *(w.buf.data_ptr() for w in ws), y1.data_ptr(), None, None, M, E, H, 128,
                                                   w2.data_ptr(), w2.numel(), stream))
    q2 = ops.prefill_rms_qkv_rope_stream(x, nw, sw, lut, 0, nh, nkv, hd)
    y2 = ops.prefill_o_ffn_stream(attn, x, nw, *ws)
    torch.cuda.synchronize()
    assert bool((b1[w1.numel():] == 77).all()) and bool((b2[w2.numel():] == 77).all())
    for got, want in ((q1, q2), (y1, y2)):
        got, want = got.double(), want.double()
        assert bool(((got - want).norm(dim=1) <= 2.0 ** -7 * want.norm(dim=1)).all())


@pytest.mark.parametrize("M", [33, 100])
def test_prefill_blocks_stream_after_those_on_the_checkpoint_layout(ops, monkeypatch, M):
    """The same sizes in both layouts in one process: the stream blocks run in as many slices, and so with the same bits, as where they come first."""
    from oracle import decode as odec
    E, H, nh, nkv, hd = 2048, 4096, 24, 4, 64
    parts, fused = _qkv_weights(E, nh, nkv, hd, seed=M)
    layer = _weights(E, H, seed=M)
    sw, ws = _sw(ops, fused), [_sw(ops, w) for w in layer]
    lut = dev(odec.generate_rope_lut(hd, 500000.0, M))
    x, attn, nw = dev(make_x((M, E), seed=M)), dev(make_x((M, E), seed=M + 1)), dev(_norm_w(E, 3))
    on_gpu = lambda w: tuple(map(dev, w))
    print("prompt blocks of both layouts", M, flush=True)

    def stream():
        return ops.prefill_rms_qkv_rope_stream(x, nw, sw, lut, 0, nh, nkv, hd), ops.prefill_o_ffn_stream(attn, x, nw, *ws)

    monkeypatch.setattr(ops, "_attn_ws", {})
    first = stream()
    monkeypatch.setattr(ops, "_attn_ws", {})
    ops.prefill_rms_qkv_rope(x, nw, on_gpu(fused), lut, 0, nh, nkv, hd)
    ops.prefill_o_ffn(attn, x, nw, *map(on_gpu, layer))
    for got, want in zip(stream(), first):
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_prompt_lengths_share_their_workspaces(ops, monkeypatch):
    """64 lengths take the memory of one, and each runs what it runs in a workspace of its own: the same bits after a shorter, after a longer one and alone."""
    from oracle import decode as odec
    E, H, nh, nkv, hd = 2048, 1024, 24, 4, 64
    sw, ws = _sw(ops, _qkv_weights(E, nh, nkv, hd, seed=1)[1]), [_sw(ops, w) for w in _weights(E, H, seed=1)]
    lut, nw = dev(odec.generate_rope_lut(hd, 500000.0, 200)), dev(_norm_w(E, 3))
    x, attn = dev(make_x((200, E), seed=1)), dev(make_x((200, E), seed=2))
    monkeypatch.setattr(ops, "_attn_ws", {})

    def run(M):
        print("prompt lengths", M, flush=True)
        return ops.prefill_rms_qkv_rope_stream(x[:M].contiguous(), nw, sw, lut, 0, nh, nkv, hd), ops.prefill_o_ffn_stream(attn[:M].contiguous(), x[:M].contiguous(), nw, *ws)

    lengths = (65, 128, 66, 100, 127)
    shared = [run(M) for M in lengths]
    kept = sum(t.numel() for t in ops._attn_ws.values())
    assert kept <= max(sum(int(f(M, *w)) for f, w in ((ops._lib.load_library().w4a16_prefill_qkv_workspace_most, (E,)),
                                                      (ops._lib.load_library().w4a16_prefill_block_workspace_most, (E, H)))) for M in range(65, 129)) * 1.1
    for M, outs in zip(lengths, shared):
        monkeypatch.setattr(ops, "_attn_ws", {})
        for got, want in zip(outs, run(M)):
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), M


def test_graphs_of_two_lengths_have_workspaces_of_their_own(ops, monkeypatch):
    """Lengths that share a workspace otherwise, captured on one stream and replayed on two at a time: each replay has the eager bits."""
    from oracle import decode as odec
    E, H, nh, nkv, hd = 2048, 1024, 24, 4, 64
    sw, ws = _sw(ops, _qkv_weights(E, nh, nkv, hd, seed=1)[1]), [_sw(ops, w) for w in _weights(E, H, seed=1)]
    lut, nw = dev(odec.generate_rope_lut(hd, 500000.0, 200)), dev(_norm_w(E, 3))
    monkeypatch.setattr(ops, "_attn_ws", {})
    runs = []
    for M in (70, 100):
        x, attn = dev(make_x((M, E), seed=M)), dev(make_x((M, E), seed=M + 1))
        run = lambda x=x, attn=attn: [t for _ in range(4) for t in (ops.prefill_rms_qkv_rope_stream(x, nw, sw, lut, 0, nh, nkv, hd), ops.prefill_o_ffn_stream(attn, x, nw, *ws))]
        want = run()
        torch.cuda.synchronize()
        kept = set(ops._attn_ws)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = run()
        assert set(ops._attn_ws) == kept
        runs.append((graph, outs, want, torch.cuda.Stream(), x, attn))
    for turn in range(3):
        print("two lengths on two streams", turn, flush=True)
        for _, outs, *_ in runs:
            for t in outs:
                t.zero_()
        torch.cuda.synchronize()
        for graph, _, _, stream, *_ in runs:
            with torch.cuda.stream(stream):
                graph.replay()
        torch.cuda.synchronize()
        for _, outs, want, *_ in runs:
            for got, w in zip(outs, want):
                assert torch.equal(got.view(torch.int16), w.view(torch.int16))


# 192-column tiles of heads of 128 (a head and half of one) and of gate and up: one of them, several, beside wide ones, ragged rows
@pytest.mark.parametrize("M,E,nh,nkv,pos0,tile", [(100, 256, 1, 1, 4, 2), (270, 512, 4, 1, 0, 2), (2048, 256, 9, 3, 9, 0), (1000, 256, 32, 8, 2, 0)])
def test_prefill_rms_qkv_rope_stream_in_192_columns(ops, tiled_gemm, M, E, nh, nkv, pos0, tile):
    test_prefill_rms_qkv_rope_stream(ops, tiled_gemm, M, E, nh, nkv, 128, pos0, tile)


@pytest.mark.parametrize("M,E,H,tile", [(130, 256, 768, 2), (300, 512, 1536, 2), (2048, 256, 14336, 0), (700, 256, 9728, 0)])
def test_prefill_block_stream_gate_up_in_192_columns(ops, M, E, H, tile):
    test_prefill_block_stream_paired_gate_up_launch_equals_two_launches(ops, M, E, H, tile)


def test_prefill_rms_qkv_rope_stream_position_zero_is_the_identity(ops, tiled_gemm):
    """Every row at position 0 (a one-row table, cos = 1, sin = 0) leaves Q and K unrotated: the fused call equals
    RMSNorm + plain GEMM bit for bit; and shifting pos0 equals shifting the table."""
    from oracle import decode as odec
    E, nh, nkv, hd = 256, 4, 2, 64
    _, fused = _qkv_weights(E, nh, nkv, hd, seed=5)
    sw = _sw(ops, fused)
    nw = _norm_w(E, 6)
    lut = odec.generate_rope_lut(hd, 500000.0, 64)
    x = make_x((40, E), seed=7)
    print("prefill qkv rope (stream order), position 0 and shifted tables", flush=True)
    plain = ops.w4a16_gemm_stream(ops.rms_norm_rows(dev(x), dev(nw)), sw)
    for m in (0, 17, 39):
        one = ops.prefill_rms_qkv_rope_stream(dev(x[m:m + 1]), dev(nw), sw, dev(lut[:1]), 0, nh, nkv, hd)
        assert torch.equal(one.view(torch.int16), plain[m:m + 1].view(torch.int16))
    a = ops.prefill_rms_qkv_rope_stream(dev(x), dev(nw), sw, dev(lut), 9, nh, nkv, hd)
    b = ops.prefill_rms_qkv_rope_stream(dev(x), dev(nw), sw, dev(lut[9:]), 0, nh, nkv, hd)
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M,E,nh,nkv,hd", [(2048, 2048, 32, 8, 64), (1024, 4096, 32, 8, 128)])
def test_prefill_rms_qkv_rope_stream_model_sizes(ops, M, E, nh, nkv, hd):
    """Llama-3.2-1B's and Llama-3-8B's projections (tiles of 256 and 192 columns for the first, 256 only for the
    second, whose heads are 128 wide)."""
    from oracle import decode as odec
    print(f"prefill qkv rope (stream order) M={M} E={E} {nh}/{nkv} heads of {hd}", flush=True)
    _, fused = _qkv_weights(E, nh, nkv, hd, seed=15, scale=0.1)
    sw = _sw(ops, fused)
    x, nw = make_x((M, E), seed=16), _norm_w(E, 17)
    lut = odec.generate_rope_lut(hd, 500000.0, M)
    out = ops.prefill_rms_qkv_rope_stream(dev(x), dev(nw), sw, dev(lut), 0, nh, nkv, hd)
    plain = ops.w4a16_gemm_stream(ops.rms_norm_rows(dev(x), dev(nw)), sw)
    torch.cuda.synchronize()
    got, prod = bits(out), bits(plain)
    nq, nk = nh * hd, nkv * hd
    want_q = odec.rope_rows(prod[:, :nq].reshape(M * nh, hd), np.repeat(lut, nh, axis=0)).reshape(M, nq)
    assert np.array_equal(got[:, :nq], want_q)
    want_k = odec.rope_rows(prod[:, nq:nq + nk].reshape(M * nkv, hd), np.repeat(lut, nkv, axis=0)).reshape(M, nk)
    assert np.array_equal(got[:, nq:nq + nk], want_k)
    assert np.array_equal(got[:, nq + nk:], prod[:, nq + nk:])
    # rotations preserve the norm of every (i, i + head_dim / 2) pair up to the bf16 roundings
    g = bf16_bits_to_f32(got[:, :nq]).reshape(M, nh, 2, hd // 2).astype(np.float64)
    p = bf16_bits_to_f32(prod[:, :nq]).reshape(M, nh, 2, hd // 2).astype(np.float64)
    n_g, n_p = np.sqrt((g**2).sum(axis=2)), np.sqrt((p**2).sum(axis=2))
    assert np.max(np.abs(n_g - n_p)) <= 2.0**-6 * np.max(n_p)


def test_prompt_layer_on_stream_order_weights_replays_from_a_hip_graph(ops):
    """RMSNorm + Q|K|V + RoPE, causal attention and the O + FFN block (the tiled kernel raises its LDS limit by a
    function attribute at every launch) captured in one HIP graph: every replay, with eager work and
    synchronisations in between, equals the eager results bit for bit."""
    from oracle import decode as odec
    M, E, H, nh, nkv, hd = 300, 512, 1280, 8, 2, 64
    print(f"prompt layer graph M={M} E={E} H={H}", flush=True)
    _, fused = _qkv_weights(E, nh, nkv, hd, seed=2100)
    wqkv = _sw(ops, fused)
    wo, wg, wu, wd = (_sw(ops, w) for w in _weights(E, H, seed=2110, scale=0.5))
    nw_a, nw_f = dev(_norm_w(E, 2120)), dev(_norm_w(E, 2121))
    lut = dev(odec.generate_rope_lut(hd, 500000.0, M))
    xs = [dev(make_x((M, E), seed=2130 + j)) for j in range(3)]
    cur = xs[0].clone()

    def layer(x):
        qkv = ops.prefill_rms_qkv_rope_stream(x, nw_a, wqkv, lut, 0, nh, nkv, hd)
        attn = ops.prefill_attention(qkv, nh, nkv, hd)
        return qkv, attn, ops.prefill_o_ffn_stream(attn, x, nw_f, wo, wg, wu, wd)

    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        layer(cur)   # warm-up: workspaces and function attributes outside the graph
        st.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=st):
            outs = layer(cur)
        for j in range(3):
            cur.copy_(xs[j])
            g.replay()
            st.synchronize()
            want = layer(xs[j])
            st.synchronize()
            for name, a, b in zip(("qkv", "attention", "block"), outs, want):
                assert torch.isfinite(a.float()).all(), (name, j)
                assert torch.equal(a.view(torch.int16), b.view(torch.int16)), (name, j)


@pytest.mark.parametrize("codec", ["awq", "q4nx"])
@pytest.mark.parametrize("M,E,H,nh,nkv,hd", [(1, 2048, 4096, 4, 2, 64), (16, 2048, 1024, 5, 1, 128), (33, 4096, 2048, 3, 1, 64), (130, 2048, 2304, 2, 1, 128), (512, 2048, 256, 2, 2, 64)])
def test_prompt_blocks_of_few_rows(ops, codec, M, E, H, nh, nkv, hd):
    """Products of few rows behind which RoPE, SwiGLU and the residual are launches of their own.  On whole K they have the tiled kernel's bits.  In slices the fp32 sum meets in another order: a
    product differs by its rounding (half an ulp and what the order moves, less than 2^-16 of the sum's magnitude, together less than an ulp), which each stage passes on."""
    from oracle import decode as odec
    print(f"prompt blocks of few rows {codec} M={M} E={E} H={H} heads {nh}/{nkv} of {hd}", flush=True)
    N = (nh + 2 * nkv) * hd

    def weight(K, n, seed):
        if codec == "awq":
            return _sw(ops, _scaled(K, n, seed, 0.1))
        from test_gpu_q4nx import make
        q, s, m = make(n, K, seed=seed)
        return ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T))

    wqkv, wo, wg, wu, wd = (weight(*a) for a in ((E, N, 1), (E, E, 2), (E, H, 3), (E, H, 4), (H, E, 5)))
    attn, xres, nw = make_x((M, E), seed=6), make_x((M, E), seed=7), _norm_w(E, 8)
    lut = odec.generate_rope_lut(hd, 500000.0, M + 3)

    def blocks(wsm, slices):
        ops.tune("prefill_wsm", wsm)
        ops.tune("gemm_wsm_slices", slices)
        try:
            qkv = ops.prefill_rms_qkv_rope_stream(dev(xres), dev(nw), wqkv, dev(lut), 3, nh, nkv, hd, codec=codec)
            return [qkv, *ops.prefill_o_ffn_stream(dev(attn), dev(xres), dev(nw), wo, wg, wu, wd, return_intermediates=True, codec=codec)]
        finally:
            ops.tune("prefill_wsm", 0)
            ops.tune("gemm_wsm_slices", 0)

    tiled = blocks(2, 0)
    for got, want in zip(blocks(1, 1), tiled):
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for slices in (2, 0):
        qkv, y, res1, h = blocks(1, slices)
        for got, want in ((qkv, tiled[0]), (res1, tiled[2])):
            # pairs of columns half a head apart share their products; res1: the residual's ulp besides
            bound = 2.0**-7 * want.float().abs().amax(1, keepdim=True)
            assert bool(((got.float() - want.float()).abs() <= bound).all())
            assert float((got != want).float().mean()) < 0.02
        # behind the norm of other roundings: from the kernel's own intermediates, on whole K
        normed = ops.rms_norm_rows(res1, dev(nw))
        f = lambda t: t.double().cpu().numpy()
        plain = ops.q4nx_gemm_stream if codec == "q4nx" else ops.w4a16_gemm_stream
        ops.tune("prefill_min_m", 17)
        ops.tune("prefill_wsm", 2)
        try:
            pad = lambda t: torch.cat([t, torch.zeros((max(0, 17 - M), t.shape[1]), dtype=t.dtype, device="cuda")])   # (fewer rows have another kernel)
            g, u, d = (plain(pad(t), w)[:M] for t, w in ((normed, wg), (normed, wu), (h, wd)))
        finally:
            ops.tune("prefill_min_m", 0)
            ops.tune("prefill_wsm", 0)
        g, u = f(g), f(u)
        want = g / (1.0 + np.exp(-g)) * u
        assert np.all(np.abs(f(h) - want) <= 2 * bf16_ulp(want) + 1.2 * bf16_ulp(g) * np.abs(u) + bf16_ulp(u) * np.abs(g) + 1e-3)
        want = f(d) + f(res1)
        assert np.all(np.abs(f(y) - want) <= bf16_ulp(want) + bf16_ulp(f(d)) + 2e-3)


@pytest.mark.parametrize("codec", ["awq", "q4nx"])
@pytest.mark.parametrize("M,E,H,nh,nkv,hd,slices", [(17, 1024, 14336, 8, 4, 128, 12), (33, 1024, 12288, 4, 2, 64, 8), (1, 1024, 6144, 1, 1, 128, 6), (33, 6144, 256, 3, 1, 128, 6),
                                                    (17, 8192, 256, 2, 1, 64, 8)])
def test_prompt_blocks_in_many_slices(ops, monkeypatch, codec, M, E, H, nh, nkv, hd, slices):
    """Six parts and more, of which some are asked for beside others and some alone: the projections with RoPE, O and down with the residual, gate and up with SwiGLU, where K holds so
    many (eight groups each).  Bounds as for few rows."""
    from oracle import decode as odec
    print(f"prompt blocks in many slices {codec} M={M} E={E} H={H} heads {nh}/{nkv} of {hd}, {slices}", flush=True)
    N = (nh + 2 * nkv) * hd

    def weight(K, n, seed):
        if codec == "awq":
            return _sw(ops, _scaled(K, n, seed, 0.1))
        from test_gpu_q4nx import make
        q, s, m = make(n, K, seed=seed)
        return ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T))

    monkeypatch.setattr(ops, "_attn_ws", {})
    many = E // 128 >= 8 * slices   # else down alone
    wg, wu, wd = weight(E, H, 3), weight(E, H, 4), weight(H, E, 5)
    wo = weight(E, E, 2)
    attn, xres, nw, lut = dev(make_x((M, E), seed=6)), dev(make_x((M, E), seed=7)), dev(_norm_w(E, 8)), dev(odec.generate_rope_lut(hd, 500000.0, M + 3))
    wqkv = weight(E, N, 1) if many else None

    def blocks(wsm, slices):
        ops.tune("prefill_wsm", wsm)
        ops.tune("gemm_wsm_slices", slices)
        try:
            qkv = ops.prefill_rms_qkv_rope_stream(xres, nw, wqkv, lut, 3, nh, nkv, hd, codec=codec) if many else None
            return [qkv, *ops.prefill_o_ffn_stream(attn, xres, nw, wo, wg, wu, wd, return_intermediates=True, codec=codec)]
        finally:
            ops.tune("prefill_wsm", 0)
            ops.tune("gemm_wsm_slices", 0)

    tiled = blocks(2, 0)
    for ws in ops._attn_ws.values():
        ws.fill_(0xFF)
    cut = blocks(1, slices)
    # so many parts were written behind the rows of each workspace
    round256 = lambda n: (n + 255) // 256 * 256
    rows = {"prefill_qkv_stream": round256(2 * M * E), "prefill_block_stream": 2 * round256(2 * M * E) + 2 * round256(2 * M * H)}
    parts = {"prefill_qkv_stream": slices * M * N, "prefill_block_stream": slices * M * (max(E, 2 * H) if many else E)}
    for key, ws in ops._attn_ws.items():
        behind = ws[rows[key[2]]:].view(torch.int32) != -1
        assert bool(behind[:parts[key[2]]].all()) and not bool(behind[parts[key[2]]:].any()), key
    for got, want in [(cut[0], tiled[0]), (cut[2], tiled[2])] if many else []:
        bound = 2.0**-7 * want.float().abs().amax(1, keepdim=True)
        assert bool(((got.float() - want.float()).abs() <= bound).all())
    _, y, res1, h = cut
    normed = ops.rms_norm_rows(res1, nw)
    plain = ops.q4nx_gemm_stream if codec == "q4nx" else ops.w4a16_gemm_stream
    f = lambda t: t.double().cpu().numpy()
    ops.tune("prefill_min_m", 17)
    ops.tune("prefill_wsm", 2)
    try:
        pad = lambda t: torch.cat([t, torch.zeros((max(0, 17 - M), t.shape[1]), dtype=t.dtype, device="cuda")])   # (fewer rows have another kernel)
        g, u, d = (plain(pad(t), w)[:M] for t, w in ((normed, wg), (normed, wu), (h, wd)))
    finally:
        ops.tune("prefill_min_m", 0)
        ops.tune("prefill_wsm", 0)
    g, u = f(g), f(u)
    want = g / (1.0 + np.exp(-g)) * u
    assert np.all(np.abs(f(h) - want) <= 2 * bf16_ulp(want) + 1.2 * bf16_ulp(g) * np.abs(u) + bf16_ulp(u) * np.abs(g) + 1e-3)
    want = f(d) + f(res1)
    assert np.all(np.abs(f(y) - want) <= bf16_ulp(want) + bf16_ulp(f(d)) + 2e-3)


@pytest.mark.parametrize("codec", ["awq", "q4nx"])
@pytest.mark.parametrize("wsm,slices", [(1, 1), (1, 2), (2, 0)])
def test_rows_that_are_not_finite_stay_alone(ops, codec, wsm, slices):
    """Infinities and NaN in one row of x or of the attention's output, through the sums, RoPE, the residual and SwiGLU: the other rows keep their bits, and nothing finite comes of these."""
    from oracle import decode as odec
    M, E, H, nh, nkv, hd = 40, 2048, 2048, 4, 2, 64
    print("rows that are not finite", codec, wsm, slices, flush=True)

    def weight(K, n, seed):
        if codec == "awq":
            return _sw(ops, _scaled(K, n, seed, 0.1))
        from test_gpu_q4nx import make
        q, s, m = make(n, K, seed=seed)
        return ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T))

    wqkv, wo, wg, wu, wd = (weight(*a) for a in ((E, (nh + 2 * nkv) * hd, 1), (E, E, 2), (E, H, 3), (E, H, 4), (H, E, 5)))
    x, attn, nw, lut = make_x((M, E), seed=6), make_x((M, E), seed=7), dev(_norm_w(E, 8)), dev(odec.generate_rope_lut(hd, 500000.0, M))

    def run(x, attn):
        ops.tune("prefill_wsm", wsm)
        ops.tune("gemm_wsm_slices", slices)
        try:
            return [ops.prefill_rms_qkv_rope_stream(dev(x), nw, wqkv, lut, 0, nh, nkv, hd, codec=codec),
                    *ops.prefill_o_ffn_stream(dev(attn), dev(make_x((M, E), seed=9)), nw, wo, wg, wu, wd, return_intermediates=True, codec=codec)]
        finally:
            ops.tune("prefill_wsm", 0)
            ops.tune("gemm_wsm_slices", 0)

    plain = run(x, attn)
    rows = {2: 0x7F80, 17: 0xFF80, 39: 0x7FC0}
    for row, value in rows.items():
        x[row, 100 + row] = attn[row, 1500 + row] = value
    others = torch.tensor([m for m in range(M) if m not in rows], device="cuda")
    for name, got, want in zip(("qkv", "y", "res1", "h"), run(x, attn), plain):
        assert bool(want.isfinite().all()), name
        assert torch.equal(got[others].view(torch.int16), want[others].view(torch.int16)), name
        assert not bool(got[list(rows)].isfinite().any()), name
