"""Host logic of the product package (no GPU): layout tools against the oracle, the runner's
comparator, backend argument checks, and the C ABI's symbols and error paths."""
import ctypes
import importlib.util
import os
import re
import warnings

import numpy as np
import pytest

from air_hip import _lib, awq, bf16
from air_hip.backend import AirBackendError, HIPBackend, HIPRunner, HipModule
from air_hip.examples import dequant_awq, matmul_int4_packed, matvec_int4_packed, matvec_int4_swiglu_rms, o_gemv_ffn_int4
from oracle import awq as oawq, reference as oref
from oracle.bf16 import f32_to_bf16_bits

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_bf16_helpers_match_oracle():
    rng = np.random.default_rng(0)
    a = np.concatenate([rng.standard_normal(50000).astype(np.float32) * 3, np.array([3.0234375, 0.0, -0.0, np.inf], np.float32)])
    assert np.array_equal(np.asarray(bf16.from_f32(a)), f32_to_bf16_bits(a))
    assert np.array_equal(bf16.to_f32(bf16.from_f32(a)), oawq.bf16_bits_to_f32(f32_to_bf16_bits(a)))
    assert bf16.is_bf16(bf16.from_f32(a)) and not bf16.is_bf16(a)


def test_pack_unpack_and_layout_converters_match_oracle():
    rng = np.random.default_rng(1)
    nib = rng.integers(0, 16, size=(256, 64), dtype=np.uint8)
    assert np.array_equal(awq.pack_int4(nib), oawq.pack_awq_int32(nib))
    assert np.array_equal(awq.unpack_int4(awq.pack_int4(nib)), nib)
    z = rng.integers(0, 16, size=(2, 64), dtype=np.uint8)
    s = f32_to_bf16_bits(rng.uniform(0.005, 0.02, size=(2, 64)).astype(np.float32))
    qw, qz = awq.pack_int4(nib), awq.pack_int4(z)
    a_q, a_s, a_z = awq.l1_from_awq(qw, qz, s)
    o_q, o_s, o_z = oawq.repack_hf_awq_linear(qw, qz, s, 128)
    assert np.array_equal(a_q, o_q) and np.array_equal(np.asarray(a_s), o_s) and np.array_equal(a_z, o_z)
    qw2, qz2, s2 = awq.awq_from_l1(a_q, a_s, a_z)
    assert np.array_equal(qw2, qw) and np.array_equal(qz2, qz) and np.array_equal(np.asarray(s2), s)
    with pytest.raises(ValueError):
        awq.pack_int4(nib[:, :60])


def test_packed_buffer_round_trip_and_alignment():
    rng = np.random.default_rng(2)
    K, N = 256, 96
    qw = awq.pack_int4(rng.integers(0, 16, size=(K, N), dtype=np.uint8))
    qz = awq.pack_int4(rng.integers(0, 16, size=(K // 128, N), dtype=np.uint8))
    s = f32_to_bf16_bits(rng.uniform(0.005, 0.02, size=(K // 128, N)).astype(np.float32))
    buf = awq.pack_buffer(qw, qz, s)
    lay = awq.packed_layout(K, N)
    assert buf.size == lay["total"] and lay["z_off"] % 256 == 0 and lay["s_off"] % 256 == 0
    q2, z2, s2 = awq.unpack_buffer(buf, K, N)
    assert np.array_equal(q2, qw) and np.array_equal(z2, qz) and np.array_equal(np.asarray(s2), s)
    with pytest.raises(ValueError):
        awq.unpack_buffer(buf[:-1], K, N)


def test_interleave_round_trip_matches_oracle():
    rng = np.random.default_rng(3)
    def l1(rows):
        q = rng.integers(0, 256, size=(rows, 64), dtype=np.uint8)
        return q, bf16.from_bits(rng.integers(0, 2**15, size=(1, rows)).astype(np.uint16)), rng.integers(0, 16, size=(1, rows), dtype=np.uint8)
    g, u = l1(8), l1(8)
    a_q, a_s, a_z = awq.interleave_rows(g, u)
    o_q, o_s, o_z = oref.interleave_gate_up((g[0], np.asarray(g[1]), g[2]), (u[0], np.asarray(u[1]), u[2]))
    assert np.array_equal(a_q, o_q) and np.array_equal(np.asarray(a_s), o_s) and np.array_equal(a_z, o_z)
    g2, u2 = awq.deinterleave_rows(a_q, a_s, a_z)
    assert np.array_equal(g2[0], g[0]) and np.array_equal(np.asarray(u2[1]), np.asarray(u[1])) and np.array_equal(u2[2], u[2])


def test_examples_draw_order_and_packing():
    a = matvec_int4_packed.parse_args(["--m", "64", "--k", "256"])
    A_q, A_s, A_z, B = matvec_int4_packed.draw_inputs(a)
    f = np.load(os.path.join(ROOT, "tests", "golden", "gemv_m64_k256_seed42.npz"))
    assert np.array_equal(A_q, f["A_q"]) and np.array_equal(np.asarray(A_s), f["A_s"]) and np.array_equal(A_z, f["A_z"])
    assert np.array_equal(np.asarray(B), f["B"])
    buf = matvec_int4_packed.pack_inputs(A_q, A_s, A_z, 64, 256, 128)
    qw, qz, s = awq.unpack_buffer(buf, 256, 64)
    assert np.array_equal(qw, f["qweight"]) and np.array_equal(qz, f["qzeros"])
    assert str(matvec_int4_packed.build_module(64, 256)) == "hip.module @matvec_int4 {M = 1, K = 256, N = 64, gs = 128}"
    assert matmul_int4_packed.build_module(32, 256, 64, 128, 16, 128, 128, 16, 2, 4) == HipModule("matmul_int4", K=256, N=64, M=32)
    assert matvec_int4_swiglu_rms.build_module(128, 256).N == 64
    d = dequant_awq.parse_args([])
    q, sc, z = dequant_awq.draw_inputs(d)
    g = np.load(os.path.join(ROOT, "tests", "golden", "dequant1d_n1024_seed0.npz"))
    assert np.array_equal(q, g["int4_vals"]) and np.array_equal(np.asarray(sc), g["scales"]) and np.array_equal(z, g["zeros"])
    # the fused RMSNorm example hands RMS_in (x row, weight row) to the kernel unchanged
    assert matvec_int4_swiglu_rms.build_module(128, 256).op == "matvec_int4_swiglu_rms"
    args = matvec_int4_swiglu_rms.parse_args(["--m", "32", "--k", "256"])
    *_, RMS_in = matvec_int4_swiglu_rms.draw_inputs(args)
    assert bf16.bits_of(RMS_in).shape == (2, 256)
    # block example: reference argument names, weight generator seeds and shapes
    a = o_gemv_ffn_int4.parse_args(["--emb-dim", "256", "--hidden-dim", "512"])
    wo, gu, wd, attn_out, x_residual, ffn_norm_w = o_gemv_ffn_int4.draw_inputs(a)
    assert wo[0].shape == (256, 128) and gu[0].shape == (1024, 128) and wd[0].shape == (256, 256)
    assert wd[1].shape == (4, 256) and set(np.unique(wo[2])) <= {7, 8}
    assert o_gemv_ffn_int4.build_module(256, 512) == HipModule("o_gemv_ffn_int4", K=256, N=512)
    rng = np.random.default_rng(100)
    q = rng.integers(0, 16, size=(256, 256), dtype=np.uint8)
    assert np.array_equal(wo[0], q[:, 0::2] | (q[:, 1::2] << 4))


def test_example_scripts_cli_without_a_gpu(tmp_path, capsys):
    """The stand-alone entry points: -p prints the module, compile-only validates it, a run without --expected or with
    a file written for other arguments returns 2 before anything touches the GPU."""
    import json
    import sys
    from air_hip.examples import _common
    assert matvec_int4_packed.main(["-p", "--m", "256", "--k", "512"]) == 0
    assert "hip.module @matvec_int4 {M = 1, K = 512, N = 256, gs = 128}" in capsys.readouterr().out
    assert matmul_int4_packed.main(["--compile-mode", "compile-only", "--output-format", "xclbin"]) == 0
    with pytest.raises(AirBackendError):
        matvec_int4_packed.main(["--compile-mode", "compile-only", "--k", "100"])
    assert o_gemv_ffn_int4.main([]) == 2
    assert "--expected" in capsys.readouterr().err
    args = dequant_awq.parse_args(["--n", "256"])
    path = str(tmp_path / "e.npz")
    _common.save_expected(path, args, np.zeros(256, np.uint16))
    with np.load(path) as f:
        assert json.loads(str(f["params"])) == {"group_size": 128, "herd_n": 4, "n": 256}
    assert dequant_awq.main(["--n", "512", "--expected", path]) == 2
    assert "was computed for" in capsys.readouterr().err
    sys.path.insert(0, os.path.join(os.path.dirname(__file__), "golden"))
    try:
        import make_expected
    finally:
        sys.path.pop(0)
    path = make_expected.write_expected("matvec_int4_packed", ["--m", "64", "--k", "256"], str(tmp_path / "m.npz"))
    a_q, a_s, a_z, b = matvec_int4_packed.draw_inputs(matvec_int4_packed.parse_args(["--m", "64", "--k", "256"]))
    with np.load(path) as f:
        assert np.array_equal(f["expected"], oref.matvec_cpu_reference_loop(a_q, bf16.bits_of(a_s), a_z, bf16.bits_of(b)))


def test_runner_comparator_semantics_match_reference_restatement(capsys):
    r = HIPRunner()
    e = np.linspace(1, 2, 1000)
    a = e.copy()
    a[:5] += 1.0
    for kw in (dict(rtol=0.1, atol=0.05), dict(rtol=0.1, atol=0.05, max_mismatch_percentage=0.5),
               dict(rtol=0.1, atol=0.05, max_mismatch_percentage=0.49), dict(rtol=0.1, atol=0.05, min_correlation=0.999)):
        assert r._check_outputs([a], [e], **kw) == oref.check_outputs(a, e, **kw), kw
    assert not r._check_outputs([np.ones(10)], [np.ones(10)], rtol=1, atol=1, min_correlation=0.5)   # NaN correlation
    # bf16 outputs are compared as floats, integers exactly
    eb = bf16.from_f32(np.array([1.0, 2.0, 3.0], np.float32))
    ab = bf16.from_f32(np.array([1.0, 2.0, 3.02], np.float32))
    assert r._check_outputs([ab], [eb], rtol=0.1, atol=0.05)
    assert not r._check_outputs([np.array([1, 2, 3])], [np.array([1, 2, 4])])
    capsys.readouterr()


def test_backend_compile_rejects_bad_modules_and_load_needs_gpu():
    b = HIPBackend()
    for bad in (HipModule("matvec_int4", K=100, N=64), HipModule("matvec_int4", K=128, N=40),
                HipModule("matvec_int4", K=128, N=64, gs=64), HipModule("nope", K=128, N=64),
                HipModule("matmul_int4", K=128, N=64, M=0)):
        with pytest.raises(AirBackendError):
            b.compile(bad)
    with pytest.raises(AirBackendError):
        b.compile("not a module")
    art = b.compile(HipModule("dequant_awq", K=128, N=40))
    import torch
    if not torch.cuda.is_available():
        with pytest.raises(AirBackendError):
            b.load(art)


def _declared_functions():
    text = open(os.path.join(ROOT, "include", "w4a16.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(?:int|size_t|const char \*)\s*\*?(\w+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load_library()
    names = _declared_functions()
    assert "w4a16_gemv_bf16" in names and "awq_dequant_bf16" in names and len(names) >= 12
    for n in names:
        assert hasattr(lib, n), f"{n} is declared in include/w4a16.h but not exported"
        assert n in _lib.SYMBOLS, f"{n} has no ctypes prototype"
    assert lib.w4a16_abi_version() == 1
    assert lib.w4a16_strerror(0) == b"ok" and b"128" in lib.w4a16_strerror(_lib.ERR_GROUP)


@pytest.mark.parametrize("E,H", [(256, 512), (2048, 8192), (4096, 14336)])
def test_prompt_workspaces_ask_for_no_more_than_is_used(E, H):
    """Parts of K slices, at most 12 MB, up to 512 rows; nothing for them past that."""
    lib = _lib.load_library()
    for M in (1, 40, 300, 512, 513, 600, 700, 3600, 8192):
        for least, most in ((lib.w4a16_prefill_qkv_workspace_bytes(M, E), lib.w4a16_prefill_qkv_workspace_most(M, E)),
                            (lib.w4a16_prefill_block_workspace_bytes(M, E, H), lib.w4a16_prefill_block_workspace_most(M, E, H))):
            assert least <= most <= least + ((12 << 20) if M <= 512 else 0), (M, E, H)


@pytest.mark.parametrize("E,H", [(64, 128), (1096, 2056), (2048, 8192), (4096, 14336), (8192, 28672)])
def test_prompt_workspaces_of_64_lengths_are_the_last_ones(E, H):
    """The longest of 64 lengths takes the most of them: its workspace is enough for all."""
    lib = _lib.load_library()
    for last in range(64, 513, 64):
        for f, widths in ((lib.w4a16_prefill_qkv_workspace_most, (E,)), (lib.w4a16_prefill_block_workspace_most, (E, H))):
            assert max(f(M, *widths) for M in range(last - 63, last + 1)) == f(last, *widths) > 0, (last, widths)


def test_c_abi_rejects_bad_arguments_before_touching_the_gpu():
    lib = _lib.load_library()
    P = 0x10000   # fake, aligned, never dereferenced: validation fails first
    assert lib.awq_dequant_bf16(None, P, P, P, 128, 8, 128, None) == _lib.ERR_NULL
    assert lib.awq_dequant_bf16(P, P, P, None, 128, 8, 128, None) == _lib.ERR_NULL
    assert lib.awq_dequant_bf16(P, P, P, P, 100, 8, 128, None) == _lib.ERR_SHAPE
    assert lib.awq_dequant_bf16(P, P, P, P, 128, 12, 128, None) == _lib.ERR_SHAPE
    assert lib.awq_dequant_bf16(P, P, P, P, 128, 8, 64, None) == _lib.ERR_GROUP
    assert lib.awq_dequant_bf16(P + 4, P, P, P, 128, 8, 128, None) == _lib.ERR_ALIGN
    ws = lib.w4a16_gemm_workspace_bytes(1, 128, 32)
    assert ws > 0 and lib.w4a16_gemm_workspace_bytes(0, 128, 32) == 0
    assert lib.w4a16_gemv_bf16(P, P, P, P, P, 128, 8, 128, P, ws, None) == _lib.ERR_SHAPE      # GEMV needs N % 32 == 0
    assert lib.w4a16_gemv_bf16(P, P, P, P, P, 128, 32, 128, None, ws, None) == _lib.ERR_WORKSPACE
    assert lib.w4a16_gemv_bf16(P, P, P, P, P, 128, 32, 128, P, ws - 1, None) == _lib.ERR_WORKSPACE
    assert lib.w4a16_gemm_bf16(P, P, P, P, P, 0, 128, 32, 128, P, ws, None) == _lib.ERR_SHAPE
    assert lib.w4a16_gemm_bf16(None, P, P, P, P, 4, 128, 32, 128, P, ws, None) == _lib.ERR_NULL
    fws = lib.w4a16_ffn_workspace_bytes(128, 256)
    args = [P] * 10 + [P, None, 128, 256, 128, P, fws, None]
    bad = list(args)
    bad[13] = 200                                                                              # H not a multiple of 128
    assert lib.w4a16_ffn_swiglu_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(args)
    bad[16] = fws - 1
    assert lib.w4a16_ffn_swiglu_bf16(*bad) == _lib.ERR_WORKSPACE
    qws = lib.w4a16_prefill_qkv_workspace_bytes(64, 256)
    assert qws >= 64 * 256 * 2 and lib.w4a16_prefill_qkv_workspace_bytes(64, 8200) == 0
    qargs = [P, P, 1e-5, P, P, P, P, 128, 0, P, 64, 256, 4, 2, 64, 128, P, qws, None]
    bad = list(qargs); bad[14] = 96
    assert lib.w4a16_prefill_rms_qkv_rope_bf16(*bad) == _lib.ERR_SHAPE        # head_dim 64 or 128
    bad = list(qargs); bad[8] = 65
    assert lib.w4a16_prefill_rms_qkv_rope_bf16(*bad) == _lib.ERR_SHAPE        # pos0 + M beyond the table
    bad = list(qargs); bad[17] = qws - 1
    assert lib.w4a16_prefill_rms_qkv_rope_bf16(*bad) == _lib.ERR_WORKSPACE
    bad = list(qargs); bad[6] = None
    assert lib.w4a16_prefill_rms_qkv_rope_bf16(*bad) == _lib.ERR_NULL
    pws = lib.w4a16_prefill_block_workspace_bytes(64, 256, 512)
    assert pws >= 4 * 64 * (256 + 512)
    pargs = [P, P, P, 1e-5] + [P] * 12 + [P, None, None, 64, 256, 512, 128, P, pws, None]
    bad = list(pargs); bad[21] = 500
    assert lib.w4a16_prefill_o_ffn_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(pargs); bad[24] = pws - 1
    assert lib.w4a16_prefill_o_ffn_bf16(*bad) == _lib.ERR_WORKSPACE
    assert lib.rms_norm_rows_bf16(P, P, 1e-5, P, 4, 100, None) == _lib.ERR_SHAPE    # K % 8
    lws = lib.lm_head_workspace_bytes(100)
    assert lws >= 8 * 7 and lib.lm_head_workspace_bytes(0) == 0
    assert lib.lm_head_gemv_bf16(P, None, 0.0, P, None, None, 100, 512, P, lws, None) == _lib.ERR_NULL
    assert lib.lm_head_gemv_bf16(P, None, 0.0, P, P, None, 100, 8200, P, lws, None) == _lib.ERR_SHAPE   # E above 8192
    assert lib.lm_head_gemv_bf16(P, P, -1.0, P, P, None, 100, 512, P, lws, None) == _lib.ERR_SHAPE
    assert lib.lm_head_gemv_bf16(P, None, 0.0, P, P, P + 2, 100, 512, P, lws, None) == _lib.ERR_ALIGN
    assert lib.lm_head_gemv_bf16(P, None, 0.0, P, P, None, 100, 512, P, lws - 1, None) == _lib.ERR_WORKSPACE
    aws = lib.w4a16_attention_workspace_bytes(4, 64)
    bws = lib.w4a16_block_workspace_bytes(256, 512)
    fargs = [P, P, P, P, P, 3, 16, 4, 2, 64, P, aws, P, P, 1e-5] + [P] * 12 + [P, None, 256, 512, 128, P, bws, None]
    bad = list(fargs); bad[4] = None
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_NULL
    bad = list(fargs); bad[29] = 512                                        # E != n_heads * head_dim
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(fargs); bad[5] = 16                                          # pos == max_seq
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_SHAPE
    bad = list(fargs); bad[11] = aws - 1
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_WORKSPACE
    bad = list(fargs); bad[33] = bws - 1
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_WORKSPACE
    bad = list(fargs); bad[12] = None                                       # x_residual
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_NULL
    bad = list(fargs); bad[28] = P + 4                                      # y_sumsq misaligned
    assert lib.w4a16_decode_attn_o_gemv_ffn_bf16(*bad) == _lib.ERR_ALIGN
    gws = lib.w4a16_gemm_workspace_bytes(1, 256, 64)
    assert lib.w4a16_rms_gemv_sumsq_bf16(P, None, 1, P, 1e-5, P, P, P, P, 256, 64, 128, P, gws, None) == _lib.ERR_NULL
    assert lib.w4a16_rms_gemv_sumsq_bf16(P, P, 65, P, 1e-5, P, P, P, P, 256, 64, 128, P, gws, None) == _lib.ERR_SHAPE
    assert lib.w4a16_rms_gemv_sumsq_bf16(P, P, 1, P, 1e-5, P, P, P, P, 256, 64, 128, P, gws - 1, None) == _lib.ERR_WORKSPACE
    assert lib.rope_halfsplit_bf16(P, P, None, 8, 64, None) == _lib.ERR_NULL
    assert lib.rope_halfsplit_bf16(P, P, P, 8, 24, None) == _lib.ERR_SHAPE        # dim % 16
    assert lib.rope_halfsplit_bf16(P, P, P, 0, 64, None) == _lib.ERR_SHAPE
    assert lib.rope_halfsplit_bf16(P, P + 8, P, 8, 64, None) == _lib.ERR_ALIGN
    assert lib.w4a16_workspace_init(None, 1024, None) == _lib.ERR_NULL
    assert lib.w4a16_workspace_init(P, 16, None) == _lib.ERR_WORKSPACE
    assert lib.w4a16_tune(b"no_such_key", 1) == _lib.ERR_TUNE and lib.w4a16_tune(b"gemv_waves", 0) == 0
    # the batched GEMM with caller scratch: scratch only where the split along K is the faster way (long K, enough rows, not
    # the widest matrices), and every argument checked before a launch
    need = lib.w4a16_gemm_stream_scratch_bytes(64, 14336, 4096)
    assert need == 14 * 64 * 4096 * 4
    assert lib.w4a16_gemm_stream_scratch_bytes(64, 4096, 14336) == 0 and lib.w4a16_gemm_stream_scratch_bytes(64, 2048, 4096) == 0
    assert lib.w4a16_gemm_stream_scratch_bytes(16, 14336, 4096) == 0 and lib.w4a16_gemm_stream_scratch_bytes(129, 14336, 4096) == 0
    assert lib.w4a16_gemm_stream_scratch_bytes(64, 14336, 4100) == 0
    big = (P, P, P, 64, 14336, 4096, 128)
    assert lib.w4a16_gemm_stream_scratch_bf16(*big, None, 0, None) == _lib.ERR_WORKSPACE
    assert lib.w4a16_gemm_stream_scratch_bf16(*big, P, need - 1, None) == _lib.ERR_WORKSPACE
    assert lib.w4a16_gemm_stream_scratch_bf16(*big, P + 8, need, None) == _lib.ERR_ALIGN
    assert lib.w4a16_gemm_stream_scratch_bf16(None, P, P, 64, 14336, 4096, 128, P, need, None) == _lib.ERR_NULL
    assert lib.w4a16_gemm_stream_scratch_bf16(P, P, P, 64, 14336, 4096, 64, P, need, None) == _lib.ERR_GROUP
    assert lib.w4a16_gemm_stream_scratch_bf16(P, P, P, 64, 14336, 4100, 128, P, need, None) == _lib.ERR_SHAPE
    assert lib.w4a16_gemm_stream_scratch_bf16(P, P, None, 64, 4096, 14336, 128, None, 0, None) == _lib.ERR_NULL   # (whole-K route)
    assert lib.w4a16_tune(b"gemm_splitk", 3) == _lib.ERR_TUNE and lib.w4a16_tune(b"gemm_splitk", 0) == 0
    # Q4NX order: blocks -> stream order, and the prompt-pass entry points
    assert lib.w4a16_q4nx_blocks_to_stream(None, P, 32, 256, 0, None) == _lib.ERR_NULL
    assert lib.w4a16_q4nx_blocks_to_stream(P, P, 48, 256, 0, None) == _lib.ERR_SHAPE      # whole blocks of 32 rows
    assert lib.w4a16_q4nx_blocks_to_stream(P, P, 32, 128, 0, None) == _lib.ERR_SHAPE      # and of 256 columns
    assert lib.w4a16_q4nx_blocks_to_stream(P, P, 32, 256, 3, None) == _lib.ERR_SHAPE
    assert lib.w4a16_q4nx_blocks_to_stream(P, P + 4, 32, 256, 0, None) == _lib.ERR_ALIGN
    wsq = lib.w4a16_prefill_qkv_workspace_bytes(64, 256)
    assert lib.w4a16_q4nx_prefill_rms_qkv_rope_stream_bf16(P, P, 1e-5, None, P, 80, 0, P, 64, 256, 4, 2, 64, P, wsq, None) == _lib.ERR_NULL
    assert lib.w4a16_q4nx_prefill_rms_qkv_rope_stream_bf16(P, P, 1e-5, P, P, 80, 20, P, 64, 256, 4, 2, 64, P, wsq, None) == _lib.ERR_SHAPE
    assert lib.w4a16_q4nx_prefill_rms_qkv_rope_stream_bf16(P, P, 1e-5, P, P, 80, 0, P, 64, 256, 4, 2, 64, P, wsq - 1, None) == _lib.ERR_WORKSPACE
    wsb = lib.w4a16_prefill_block_workspace_bytes(64, 256, 512)
    blk = [P, P, P, 1e-5, P, P, P, P, P, None, None, 64, 256, 512]
    assert lib.w4a16_q4nx_prefill_o_ffn_stream_bf16(*blk, None, wsb, None) == _lib.ERR_WORKSPACE
    assert lib.w4a16_q4nx_prefill_o_ffn_stream_bf16(*(blk[:4] + [None] + blk[5:]), P, wsb, None) == _lib.ERR_NULL
    assert lib.w4a16_q4nx_prefill_o_ffn_stream_bf16(*(blk[:13] + [500]), P, wsb, None) == _lib.ERR_SHAPE
    with pytest.raises(_lib.W4A16Error):
        _lib.check(_lib.ERR_ALIGN)


def test_kernel_cache_host_contract(tmp_path):
    """What KernelCache decides before it touches the device: module shape rules, registration, the manifest,
    unknown kernels, the shared_alias checks (the reference makes these before any XRT call,
    shared/infra/cache.py:569-603) and the profiler's bookkeeping."""
    from air_hip import cache as kc

    with pytest.raises(AssertionError):
        kc.build_rms_qkv_int4_rope_module(emb_dim=2048, kv_dim=512, n_heads=16, n_kv_heads=8, head_dim=64)
    with pytest.raises(AssertionError):
        kc.build_rms_qkv_int4_rope_module(emb_dim=1024, kv_dim=256, n_heads=16, n_kv_heads=4, head_dim=64)   # k_chunk != emb
    with pytest.raises(AssertionError):
        kc.build_o_gemv_ffn_int4_module(emb_dim=2048, hidden_dim=3072)
    with pytest.raises(AssertionError):
        kc.build_o_gemv_ffn_int4_module(emb_dim=4096, hidden_dim=8192)
    c = kc.KernelCache(cache_dir=tmp_path, profiler=kc.Profiler(enabled=True))
    with pytest.raises(AirBackendError):
        c.compile_and_cache("x", "not a module", {})
    with pytest.raises(AirBackendError):
        c.compile_and_cache("x", kc.DecodeModule("o_gemv_ffn_int4", emb_dim=2048, hidden_dim=8192, gs=64), {})
    c.compile_and_cache("rms_qkv_int4_rope", kc.build_rms_qkv_int4_rope_module(), {"verbose": False})
    c.compile_and_cache("o_gemv_ffn_int4", kc.build_o_gemv_ffn_int4_module(), {})
    c.compile_and_cache("lm_head_gemv", kc.build_lm_head_gemv_module(2048), {})
    assert set(c.profiler.compile_times) == {"rms_qkv_int4_rope", "o_gemv_ffn_int4", "lm_head_gemv"}
    c._save_manifest()
    c2 = kc.KernelCache(cache_dir=tmp_path)
    assert c2.load_manifest() and c2.artifacts == c.artifacts
    assert not kc.KernelCache().load_manifest()

    with pytest.raises(RuntimeError, match="not found in cache"):
        c.load_and_run("attn_gemms", {}, np.zeros(4, np.uint16))
    z = bf16.from_f32(np.zeros(2048))
    args = [z] * 15
    with pytest.raises(ValueError, match="is static"):
        c.load_and_run("o_gemv_ffn_int4", {}, *args, static_input_indices={0, 6}, shared_alias={6: "res"})
    with pytest.raises(ValueError, match="does not exist"):
        c.load_and_run("o_gemv_ffn_int4", {}, *args, shared_alias={15: "res"})
    with pytest.raises(ValueError, match="no pool name"):
        c.load_and_run("o_gemv_ffn_int4", {}, *args, shared_alias={14: ""})
    with pytest.raises(AirBackendError, match="takes 15 arguments"):
        c.load_and_run("o_gemv_ffn_int4", {}, *args[:14])

    prof = kc.Profiler(enabled=True)
    with prof.time_cpu("decode_attention_cpu"):
        pass
    for layer in range(4):
        prof.end_layer(layer % 2, prof.start_layer())
    prof.record_kernel("k", 0.5)
    prof.record_breakdown("k", 1.0, 2.0, 3.0, 4, 5, 6)
    assert len(prof.cpu_times["decode_attention_cpu"]) == 1 and len(prof.per_token_walls_ms(2)) == 2
    assert prof.per_token_walls_ms(3) == [] and prof.kernel_breakdowns["k"][0]["bytes_written"] == 5
    off = kc.Profiler()
    off.record_kernel("k", 1.0)
    assert off.start_layer() is None and off.kernel_times == {} and off.per_token_walls_ms(1) == []


def test_fake_quantize_matches_the_oracle_loop():
    """The vectorised host quantiser against the oracle's scalar restatement, bit for bit, on groups with outliers,
    constant groups and one-sided groups; accepts bf16 bits or floats."""
    rng = np.random.default_rng(9)
    w = (rng.standard_normal((12, 512)) * 10.0 ** rng.uniform(-3, 1, (12, 1))).astype(np.float32)
    w[3, 128:256] = 0.25
    w[4, :128] = np.abs(w[4, :128]) + 1.0
    w[5, 17] = 40.0
    wb = bf16.from_f32(w)
    got = awq.fake_quantize_awq_int4(wb, 128)
    want = oawq.fake_quantize_awq_int4_loop(bf16.to_f32(bf16.bits_of(wb)), 128)
    assert np.array_equal(got[0], want[0]) and np.array_equal(bf16.bits_of(got[1]), want[1]) and np.array_equal(got[2], want[2])
    got_f = awq.fake_quantize_awq_int4(bf16.to_f32(bf16.bits_of(wb)), 128)
    assert all(np.array_equal(np.asarray(a), np.asarray(b)) for a, b in zip(got, got_f))
    assert got[0].shape == (12, 256) and got[1].shape == (4, 12) and got[2].dtype == np.uint8
    with pytest.raises(ValueError):
        awq.fake_quantize_awq_int4(w[:, :100], 128)


def test_decode_token_takes_its_layers_once(monkeypatch):
    """Layers and caches that can be walked only once: looking whether the native steps take them leaves them to the steps op by op."""
    import types

    import torch
    from air_hip import decode, ops

    ran = []
    monkeypatch.setattr(decode, "run_decode_block", lambda x, layer, *a, **k: (ran.append(layer), (x, None))[1])
    monkeypatch.setattr(ops, "lm_head", lambda x, head, **k: (x, torch.zeros(1)))
    layers = [types.SimpleNamespace(stream=None, name=i) for i in range(3)]
    decode.decode_token(0, iter(layers), torch.zeros((2, 8)), None, None, types.SimpleNamespace(rms_eps=1e-5), iter([(0, 0)] * 3), 0, None)
    assert ran == layers
    decode.decode_greedy(torch.zeros(1), 1, iter(layers), torch.zeros((2, 8)), None, None, types.SimpleNamespace(rms_eps=1e-5), iter([(0, 0)] * 3), 0, None)
    assert ran == layers + layers


def test_decode_run_leaves_a_model_without_a_final_norm_to_the_ops():
    import types

    import torch
    from air_hip import ops

    buf = types.SimpleNamespace(is_cuda=True, is_contiguous=lambda: True, data_ptr=lambda: 256)
    matrix = lambda K, N: types.SimpleNamespace(order="awq", K=K, N=N, buf=buf)
    E, H, V = 256, 512, 8
    layer = types.SimpleNamespace(codec="awq", attn_norm=torch.ones(E), ffn_norm=torch.ones(E),
                                  stream={"wqkv": matrix(E, 3 * E), "wo": matrix(E, E), "w_gate": matrix(E, H), "w_up": matrix(E, H), "w_down": matrix(H, E)})
    cache = (torch.zeros((4, 16, 64)), torch.zeros((4, 16, 64)))
    on_gpu = lambda *shape: types.SimpleNamespace(shape=shape, is_cuda=True, dtype=torch.bfloat16, is_contiguous=lambda: True, data_ptr=lambda: 256,
                                                  dim=lambda: len(shape), numel=lambda: shape[-1])
    args = (on_gpu(E), [layer], on_gpu(V, E))
    rest = (torch.zeros((V, E)), torch.zeros((16, 64)), types.SimpleNamespace(n_heads=4, rms_eps=1e-5), [cache], 0, 1, torch.zeros(1, dtype=torch.int32))
    assert ops.decode_run(*args, torch.ones(E), *rest) is None   # (a norm that is not on the GPU)
    assert ops.decode_run(*args, None, *rest) is None


def test_experts_with_few_rows_get_their_own_tiles():
    """64 rows an expert on average or less: plans of 128-row tiles, two workgroups to a CU."""
    lib = _lib.load_dense_library()
    assert [lib.dlm_gemm_tile_rows(0, rows, 2048, 64) for rows in (0, 1, 16, 64, 65, 256, 4096)] == [128, 128, 128, 128, 384, 384, 384]
    assert [lib.dlm_gemm_tile_rows(1, rows, 2048, 64) for rows in (16, 48, 49, 256)] == [32, 32, 128, 128]   # fp32


def test_slices_that_a_launch_adds_up_are_charged_for_it():
    """fp32 products whose parts nobody takes: a router's narrow one runs whole; one whose caller takes the parts is cut."""
    lib = _lib.load_dense_library()
    assert [lib.dlm_gemm_slices(0, M, 64, 2048, 1) for M in (2048, 4096, 8192)] == [1] * 3
    assert lib.dlm_gemm_parts(0, 2048, 2048, 8192) > 1 and lib.dlm_gemm_parts(0, 64, 2048, 8192) > 1
    assert lib.dlm_gemm_parts(0, 2048, 64, 2048) > 1 and lib.dlm_gemm_parts(0, 16384, 32, 512) == 1   # a router's: very many tokens' choices wait for parts
    assert lib.dlm_gemm_slices(0, 64, 2048, 8192, 1) > 1                                     # worth its launch
    assert lib.dlm_gemm_parts(1, 64, 2048, 8192) == 1 and lib.dlm_gemm_parts(0, 0, 64, 64) == 0   # fp32 weights, no rows


def test_int4_slices_are_ranked_by_time_and_advised_past_what_their_launch_costs():
    """Products under the 12.5 us that two launches and a buffer take a host: among sliced plans the fastest, not the first; and none where
    the call without scratch is done by then."""
    lib = _lib.load_library()
    slices = lambda M, K, N: lib.w4a16_q4nx_gemm_stream_best_scratch_bytes(M, K, N, 0) / (4 * M * N)
    assert slices(64, 4096, 1024) > 4 and slices(20, 5120, 1280) > 4 and slices(33, 128 * 19, 272) == 0   # (four were the first below 12 us)
    assert lib.w4a16_gemm_stream_best_scratch_bytes(30, 3328, 1472) == 0 and lib.w4a16_gemm_stream_best_scratch_bytes(20, 5120, 1280) == 0
    assert lib.w4a16_gemm_stream_best_scratch_bytes(64, 14336, 4096) >= lib.w4a16_gemm_stream_scratch_bytes(64, 14336, 4096)


@pytest.mark.parametrize("broken", [False, True])
def test_without_the_host_module_the_operators_run_in_python(monkeypatch, tmp_path, broken):
    """A missing module, or one that does not load (built against another torch, say), leaves every call to Python, and says so once a library."""
    path = tmp_path / "air_host.so"
    if broken:
        path.write_bytes(b"not a library")
    monkeypatch.setattr(_lib, "_HOST_PATH", str(path))
    for name in ("_host", "_host_w4a16", "_host_dense"):
        monkeypatch.setattr(_lib, name, None)
    for get in (_lib.host_w4a16, _lib.host_dense):
        with pytest.warns(RuntimeWarning, match="air_host"):
            host = get()
        with warnings.catch_warnings():
            warnings.simplefilter("error")
            assert get() is host
    assert all(f(1, 2, 3) is None for f in (host.linear, host.latent_rows, host.mixed_rows, host.tail))


def test_build_links_the_libraries_where_the_host_module_cannot_be_built(monkeypatch, tmp_path, capsys):
    """Without g++ or torch's headers: an error behind the link, and a library that is asked for alone is built without one."""
    spec = importlib.util.spec_from_file_location("build_under_test", os.path.join(ROOT, "mlir-air_amd", "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    for name in ("LIB_DIR", "OBJ_DIR"):
        monkeypatch.setattr(build, name, str(tmp_path / name))

    def no_host():
        raise RuntimeError("no compiler for the host module")

    monkeypatch.setattr(build, "_build_host", no_host)
    monkeypatch.setattr(build, "_compile", lambda src, extra: (src, ""))
    monkeypatch.setattr(build.subprocess, "check_call", lambda cmd: open(cmd[cmd.index("-o") + 1], "w").close())
    with pytest.raises(RuntimeError, match="no compiler"):
        build.build()
    for name in build.LIBRARIES:
        assert os.path.exists(build.lib_path(name))
        os.remove(build.lib_path(name))
        assert build.ensure(name) == build.lib_path(name) and os.path.exists(build.lib_path(name))
        assert "no compiler" in capsys.readouterr().err


def test_a_host_module_built_against_other_headers_is_not_used(monkeypatch):
    """Versions and struct sizes are those of the ctypes side, and one that differs leaves the calls to Python."""
    module = _lib.load_host()
    compiled = module.compiled_for()
    assert compiled["w4a16"] == _lib.load_library().w4a16_abi_version() and compiled["dense_lm"] == _lib.load_dense_library().dlm_abi_version()
    text = open(os.path.join(ROOT, "mlir-air_amd", "csrc", "host.cpp")).read()
    handed_over = set(re.findall(r"\bdlm_(\w+) \w+{", text)) | {"latent_shape", "head_shape"}
    assert {n.title().replace("_", "") for n in handed_over} <= set(compiled)   # every struct that it fills in
    assert _lib._host_misfits(module) == "" and "no record" in _lib._host_misfits(object())
    for name in ("GemmArgs", "HeadRows"):
        class Longer(getattr(_lib, name)):
            _fields_ = [("more", ctypes.c_int64)]
        with monkeypatch.context() as m:
            m.setattr(_lib, name, Longer)
            for cached in ("_host", "_host_dense"):
                m.setattr(_lib, cached, None)
            with pytest.raises(_lib.LibraryNotBuiltError, match=name):
                _lib.load_host()
            with pytest.warns(RuntimeWarning, match="other headers"):
                assert _lib.host_dense().latent_rows(1) is None


def test_a_model_with_a_tail_of_its_own():
    """A further dense-weight model gives its passes and the tail's two steps; a prompt goes by those unless the class names the native tail's form."""
    import torch
    from air_hip import dense
    from air_hip.dense_model import DenseModel, SequenceCache
    from air_hip.kuvonex import KuvonexModel
    from air_hip.sitirax import SitiraxModel

    class Own(DenseModel):
        device, vocab = torch.device("cpu"), 9

        def _rows(self, cache, tokens, pos, trace=None):
            return tokens.float()[:, None].expand(-1, 4)

        def _pending(self, row):
            return row + 1

        def _tail(self, pending):
            return pending, pending.argmax().reshape(1)

    model = Own()
    cache = SequenceCache(model, 8)
    for tokens in ([3, 5], torch.tensor([1, 5], dtype=torch.int32)):
        row, _ = model.prefill(cache, tokens)
        assert row.tolist() == [6.0] * 4

    class Scaled(KuvonexModel):
        def _head(self, r, keys=None):
            return super()._head(r, keys)

    class Kept(SitiraxModel):
        def _tail(self, pending):
            return super()._tail(pending)

    class Longer(SitiraxModel):
        max_portion = 64

    assert Kept.tail_intake is None and Scaled.tail_intake is None and KuvonexModel.tail_intake == dense.FINAL
    assert Longer.tail_intake == SitiraxModel.tail_intake == dense.NORMED


def test_splits_of_the_keys():
    """One rule for passes in Python and in native code: what the operators have always launched."""
    lib = _lib.load_dense_library()
    lengths = [1, 2, 17, 31, 32, 33, 64, 100, 300, 511, 513, 1000, 2048, 4097, 10000, 32768, 65537, 1 << 20]
    for heads in (1, 2, 3, 4, 8, 12, 16, 24, 32, 64, 128, 255):
        for M in (1, 2, 3, 5, 8, 16, 17, 33, 64, 1000):
            rows = M * heads
            for total in lengths:
                blocks = (total + 31) // 32
                assert lib.dlm_latent_splits(heads, M, total) == max(1, min(256, 512 // ((rows + 15) // 16), blocks, round((512 * blocks / rows) ** 0.5))), (heads, M, total)
            for kv_heads in {1, heads, max(1, heads // 4)}:
                if heads % kv_heads:
                    continue
                tiles = kv_heads * ((M * (heads // kv_heads) + 15) // 16)
                for window in (1, 64, 1000, 1 << 30):
                    for total in lengths:
                        assert lib.dlm_head_splits(heads, kv_heads, window, M, total) == max(1, min(256, 512 // tiles, (min(total, window + M - 1) + 31) // 32 + 1))
    assert lib.dlm_latent_splits(0, 1, 5) == lib.dlm_head_splits(4, 0, 5, 1, 5) == 1
