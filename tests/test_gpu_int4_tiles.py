"""Int4 products of 17 rows and more at the edges of their row blocks, column sets, steps and slices, both codecs: exact weights against the
float64 product (one bf16 rounding of an fp32 sum: 1 ulp and 2e-3, as for the other exact products); rounded weights against the tiled kernel,
bit for bit.  What the rule picks and two slices at a range of shapes, then every kernel that there is, set by hand, with slices of uneven length;
the scratch says how many there were."""
import numpy as np
import pytest
import torch

from helpers import assert_bf16_close, dense_f64, make_awq, make_x
from oracle import awq as oawq
from oracle.bf16 import bf16_bits_to_f32, f32_to_bf16_bits
from test_gpu_q4nx import make
from test_gpu_stream_order import bits, dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [(17, 128, 16), (32, 384, 48), (33, 128 * 19, 272), (64, 4096, 64), (65, 1024, 528), (96, 512, 128), (112, 2176, 144),
                                   (113, 512, 1040), (129, 640, 320), (129, 256, 64), (257, 1024, 192), (300, 2048, 1088)])
@pytest.mark.parametrize("q4", [False, True])
def test_int4_tiles(q4, M, K, N):
    from air_hip import _lib, ops
    print("int4 tiles", "q4nx" if q4 else "awq", M, K, N, flush=True)
    lib, stream = _lib.load_library(), torch.cuda.current_stream().cuda_stream
    x = make_x((M, K), seed=M + K)
    res = make_x((M, N), seed=N) if q4 else None
    if q4:
        q, s, m = make(N, K, seed=M + N)   # [N, K] and [N, K / 32]
        w = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T))
        dense = (q.astype(np.float64).reshape(N, K // 32, 32) * bf16_bits_to_f32(s).astype(np.float64)[:, :, None]
                 + bf16_bits_to_f32(m).astype(np.float64)[:, :, None]).reshape(N, K).T
    else:
        tri = make_awq(K, N, seed=M + N)
        w, dense = ops.repack_stream(*map(dev, tri)), dense_f64(*tri)
    want = bf16_bits_to_f32(x).astype(np.float64) @ dense
    xd, rd = dev(x), dev(res) if q4 else None
    scratch = torch.full((1 << 26,), 0xFF, dtype=torch.uint8, device="cuda")

    def call(nbytes, residual):
        y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
        at = scratch.data_ptr() if nbytes else None
        if q4:
            _lib.check(lib.w4a16_q4nx_gemm_stream_scratch_bf16(xd.data_ptr(), w.buf.data_ptr(), residual, y.data_ptr(), M, K, N, at, nbytes, stream))
        elif nbytes:
            _lib.check(lib.w4a16_gemm_stream_scratch_bf16(xd.data_ptr(), w.buf.data_ptr(), y.data_ptr(), M, K, N, 128, at, nbytes, stream))
        else:
            _lib.check(lib.w4a16_gemm_stream_bf16(xd.data_ptr(), w.buf.data_ptr(), y.data_ptr(), M, K, N, 128, stream))
        return bits(y)

    rounded = M >= (65 if q4 else 129) and K % 256 == 0 and N % 64 == 0
    ops.tune("gemm_splitk", 1)
    ops.tune("prefill_wsm", 1)
    try:
        for nbytes in (0, 1 << 26):
            got = call(nbytes, None)
            if rounded:
                ops.tune("prefill_tile", 4)
                assert np.array_equal(got, call(0, None))
                ops.tune("prefill_tile", 0)
            else:
                assert_bf16_close(got, want, ulps=1.0, atol=2e-3, what=f"int4 tiles, {nbytes} bytes of scratch")
            if q4:
                assert_bf16_close(call(nbytes, rd.data_ptr()), want + bf16_bits_to_f32(res).astype(np.float64), ulps=1.0, atol=2e-3,
                                  what=f"int4 tiles with a residual, {nbytes} bytes of scratch")
    finally:
        ops.tune("gemm_splitk", 0)
        ops.tune("prefill_wsm", 0)
        ops.tune("prefill_tile", 0)


@pytest.mark.parametrize("rt", [2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("mode", ["awq", "q4nx", "awq rounded", "q4nx rounded"])
def test_every_int4_tile(mode, rt):
    """Two blocks of rows or more, the last one ragged; two sets of columns and a ragged third; an odd number of groups in one slice, two and three."""
    from air_hip import _lib, ops
    q4, rounded = mode.startswith("q4nx"), mode.endswith("rounded")
    lib, stream = _lib.load_library(), torch.cuda.current_stream().cuda_stream
    M = 16 * rt * (max(129 // (16 * rt), 1) + 1) - 5
    K = 256 * 3 if rounded else 128 * 11
    for nt in (1, 2, 3) if rounded and 3 <= rt <= 5 else (1, 2):
        N = 64 * nt * 2 + (64 if rounded else 48)
        if rounded and nt == 1:
            N = 128
        print("int4 tile", mode, rt, nt, M, K, N, flush=True)
        x = make_x((M, K), seed=M)
        if q4:
            q, s, m = make(N, K, seed=rt)
            w = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T))
            dense = (q.astype(np.float64).reshape(N, K // 32, 32) * bf16_bits_to_f32(s).astype(np.float64)[:, :, None]
                     + bf16_bits_to_f32(m).astype(np.float64)[:, :, None]).reshape(N, K).T
        else:
            tri = make_awq(K, N, seed=rt)
            w, dense = ops.repack_stream(*map(dev, tri)), dense_f64(*tri)
        want = bf16_bits_to_f32(x).astype(np.float64) @ dense
        xd = dev(x)
        fill = torch.full((1,), -1, dtype=torch.int32, device="cuda")

        def call(scratch):
            y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device="cuda")
            at, nbytes = (None, 0) if scratch is None else (scratch.data_ptr(), scratch.numel() * 4)
            if q4:
                _lib.check(lib.w4a16_q4nx_gemm_stream_scratch_bf16(xd.data_ptr(), w.buf.data_ptr(), None, y.data_ptr(), M, K, N, at, nbytes, stream))
            elif scratch is not None:
                _lib.check(lib.w4a16_gemm_stream_scratch_bf16(xd.data_ptr(), w.buf.data_ptr(), y.data_ptr(), M, K, N, 128, at, nbytes, stream))
            else:
                _lib.check(lib.w4a16_gemm_stream_bf16(xd.data_ptr(), w.buf.data_ptr(), y.data_ptr(), M, K, N, 128, stream))
            return bits(y)

        keys = {"gemm_splitk": 1, "prefill_wsm": 1, "prefill_min_m": M if rounded else M + 1, "gemm_wsm_rt": rt, "gemm_wsm_nt": nt}
        try:
            for key, value in keys.items():
                ops.tune(key, value)
            if rounded:
                got = call(None)
                ops.tune("prefill_tile", 4)
                assert np.array_equal(got, call(None)), (mode, rt, nt)
                dense_r = bf16_bits_to_f32(f32_to_bf16_bits(np.ascontiguousarray(dense.astype(np.float32)))).astype(np.float64)
                assert_bf16_close(got, bf16_bits_to_f32(x).astype(np.float64) @ dense_r, ulps=1.0, atol=2e-3, what=f"{mode} {rt} {nt}")
                continue
            for slices in (1, 2, 3):
                ops.tune("gemm_wsm_slices", slices)
                scratch = fill.repeat(4 * M * N)   # NaNs: a part is written whole, and nothing behind the parts
                assert_bf16_close(call(scratch), want, ulps=1.0, atol=2e-3, what=f"{mode} {rt} {nt}, {slices} slices")
                parts = slices * M * N if slices > 1 else 0
                assert bool((scratch[:parts] != -1).all()) and bool((scratch[parts:] == -1).all()), "parts in the scratch"
        finally:
            for key in [*keys, "gemm_wsm_slices", "prefill_tile"]:
                ops.tune(key, 0)


@pytest.mark.parametrize("M,K,N", [(17, 128, 48), (40, 640, 272), (64, 2048, 528), (100, 384, 1040)])
@pytest.mark.parametrize("residual", [False, True])
def test_q4nx_minima_of_any_size(residual, M, K, N):
    """Row m adds 32 rows of one scale block and takes away 32 of the next; a column has one q and one scale everywhere, so what is left is
    32 times the difference of two minima, from 2^-12 to 2^4 scales.  Exact products in fp32: three matrix instructions a block, each at most two
    roundings of 2^-24 of the sum of magnitudes, then a bf16 rounding.  Weights kept in 16 bits miss it by up to 2^-17 of that sum."""
    from air_hip import _lib, ops
    print("q4nx minima", residual, M, K, N, flush=True)
    rng = np.random.default_rng(M + K + N)
    B = K // 32
    q = np.repeat(rng.integers(1, 16, (N, 1), dtype=np.uint8), K, axis=1)
    s = np.repeat(f32_to_bf16_bits(rng.uniform(0.5, 2.0, (N, 1)).astype(np.float32)), B, axis=1)
    m = f32_to_bf16_bits((bf16_bits_to_f32(s) * 2.0 ** rng.uniform(-12, 4, (N, B)) * rng.choice([-1.0, 1.0], (N, B))).astype(np.float32))
    x = np.zeros((M, K), np.float32)
    for i in range(M):
        x[i, 32 * (i % B):32 * (i % B) + 32], x[i, 32 * ((i + 1) % B):32 * ((i + 1) % B) + 32] = 1.0, -1.0
    w = (q.astype(np.float64).reshape(N, B, 32) * bf16_bits_to_f32(s).astype(np.float64)[:, :, None] + bf16_bits_to_f32(m).astype(np.float64)[:, :, None]).reshape(N, K).T
    parts = (q.astype(np.float64).reshape(N, B, 32) * bf16_bits_to_f32(s).astype(np.float64)[:, :, None]
             + np.abs(bf16_bits_to_f32(m)).astype(np.float64)[:, :, None]).reshape(N, K).T
    res = make_x((M, N), seed=N) if residual else None
    want = x.astype(np.float64) @ w + (bf16_bits_to_f32(res) if residual else 0.0)
    sums = np.abs(x).astype(np.float64) @ parts
    stream = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(np.ascontiguousarray(s.T)), dev(np.ascontiguousarray(m.T)))
    lib = _lib.load_library()
    xd, y = dev(f32_to_bf16_bits(x)), torch.empty((M, N), dtype=torch.bfloat16, device="cuda")
    rd = dev(res) if residual else None
    ops.tune("gemm_splitk", 1)
    try:
        _lib.check(lib.w4a16_q4nx_gemm_stream_bf16(xd.data_ptr(), stream.buf.data_ptr(), rd.data_ptr() if residual else None, y.data_ptr(), M, K, N,
                                                   torch.cuda.current_stream().cuda_stream))
    finally:
        ops.tune("gemm_splitk", 0)
    got = bf16_bits_to_f32(bits(y)).astype(np.float64)
    bad = np.abs(got - want) > 2.0 ** -8 * np.abs(want) + 2.0 ** -24 * 12 * sums
    assert not bad.any(), (int(bad.sum()), bad.size, float((np.abs(got - want) / sums).max()))


@pytest.mark.parametrize("q4", [False, True])
def test_tiled_products_in_slices(q4):
    """Many rows of a long K with few columns: the tiled kernel in slices of K, alone and behind an FFN's down projection (bit for bit)."""
    from air_hip import _lib, ops
    M, K, N = 1030, 14336, 1024
    print("tiled slices", "q4nx" if q4 else "awq", M, K, N, flush=True)
    lib = _lib.load_library()
    x, aux = make_x((M, K), seed=3), make_x((M, N), seed=4)
    if q4:
        q, s, m = make(N, K, seed=5)
        w = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T))
        exact = (q.astype(np.float32).reshape(N, K // 32, 32) * bf16_bits_to_f32(s)[:, :, None] + bf16_bits_to_f32(m)[:, :, None]).reshape(N, K).T
        dense = bf16_bits_to_f32(f32_to_bf16_bits(np.ascontiguousarray(exact))).astype(np.float64)
    else:
        tri = make_awq(K, N, seed=5)
        w, dense = ops.repack_stream(*map(dev, tri)), dense_f64(*tri, rounded=True)
    need = lib.w4a16_q4nx_gemm_stream_best_scratch_bytes(M, K, N, 0) if q4 else lib.w4a16_gemm_stream_best_scratch_bytes(M, K, N)
    assert need >= 2 * M * N * 4
    y = (ops.q4nx_gemm_stream if q4 else ops.w4a16_gemm_stream)(dev(x), w)
    want = (torch.from_numpy(bf16_bits_to_f32(x)).double().cuda() @ torch.from_numpy(dense).cuda()).cpu().numpy()
    assert_bf16_close(bits(y), want, ulps=1.0, atol=2e-3, what="tiled slices")
    if not q4:
        H, E = K, N
        mats = [ops.repack_stream(*map(dev, make_awq(E, n, seed=6 + i))) for i, n in enumerate((E, H, H))]
        nw = dev(make_x((E,), seed=9))
        out, res1, h = ops.prefill_o_ffn_stream(dev(make_x((M, E), seed=10)), dev(aux), nw, *mats, w, return_intermediates=True)
        torch.cuda.synchronize()
        prod = ops.w4a16_gemm_stream(h, w)
        both = (prod.float() + res1.float()).bfloat16()
        assert torch.equal(out.view(torch.int16), both.view(torch.int16))


@pytest.mark.parametrize("nt,rt", [(1, 2), (2, 5), (3, 4)])
def test_every_weight_of_rounded_tiles(nt, rt):
    """One-hot rows of x return the rounded weights bit for bit: every pair of nibble and zero point, under scales of either sign, down to the
    smallest numbers and up to 2^116."""
    from air_hip import ops
    print("every weight", nt, rt, flush=True)
    K, N = 256, 256
    k, n = np.arange(K)[:, None], np.arange(N)[None, :]
    q = ((k + n // 16) % 16).astype(np.uint8)
    z = np.broadcast_to((n % 16).astype(np.uint8), (K // 128, N))
    values = np.array([1.0, -0.3711, 2.0**-120, 9.2e-41, -(2.0**-126), 2.0**116, -1.99 * 2.0**115, 0.0], np.float32)
    s = f32_to_bf16_bits(np.ascontiguousarray(values[(n // 16 + np.arange(K // 128)[:, None]) % len(values)]))
    tri = dev(oawq.pack_awq_int32(q)), dev(oawq.pack_awq_int32(np.ascontiguousarray(z))), dev(s)
    x, w = torch.eye(K, dtype=torch.bfloat16, device="cuda"), ops.repack_stream(*tri)
    want = bits(ops.awq_dequant(*tri))
    keys = ("prefill_wsm", "gemm_wsm_nt", "gemm_wsm_rt")
    try:
        for values in ((1, nt, rt), (2, 0, 0)):   # the tile; the tiled kernel
            for key, value in zip(keys, values):
                ops.tune(key, value)
            got = bits(ops.w4a16_gemm_stream(x, w))
            assert np.array_equal(np.where(got == 0x8000, 0, got), np.where(want == 0x8000, 0, want))   # (a sum's zero has no sign)
    finally:
        for key in keys:
            ops.tune(key, 0)


@pytest.mark.parametrize("M,K,N,forms", [(257, 512, 384, [(1, nt, rt, 0) for nt, rt in ((1, 2), (1, 7), (2, 4), (2, 6), (3, 3), (3, 5))] + [(2, 0, 0, tile) for tile in (1, 2, 3, 4)]),
                                         (1500, 14336, 4096, [(2, 0, 0, 0)])])   # (the last one in slices of K)
def test_scales_up_to_the_largest(M, K, N, forms):
    """Scales of 2^118 to 2^124, whose offsets are past fp32, in half of the columns: a power of two on scales and off x changes no bit of what is
    added up, here or in the other columns.  The kernels of fewer rows take any scale as it is."""
    from air_hip import ops
    print("largest scales", M, K, N, flush=True)
    rng = np.random.default_rng(M)
    q, z = rng.integers(0, 16, (K, N), dtype=np.uint8), rng.integers(0, 16, (K // 128, N), dtype=np.uint8)
    s = np.exp2(rng.uniform(8, 14, (K // 128, N))).astype(np.float32) * rng.choice([-1, 1], (K // 128, N))
    x = (rng.uniform(0.125, 4, (M, K)) * rng.choice([-1, 1], (M, K))).astype(np.float32)
    exact = lambda b, by: f32_to_bf16_bits(bf16_bits_to_f32(b) * by)
    s, x = (f32_to_bf16_bits(np.ascontiguousarray(t.astype(np.float32))) for t in (s, x))
    large = np.broadcast_to(np.arange(N) // 16 % 2 == 0, (K // 128, N))
    qz = dev(oawq.pack_awq_int32(q)), dev(oawq.pack_awq_int32(z))
    w, w_large = (ops.repack_stream(*qz, dev(t)) for t in (s, exact(s, np.where(large, 2.0**110, 1.0).astype(np.float32))))
    small_x = exact(x, np.float32(2.0**-110))
    keys = ("prefill_wsm", "gemm_wsm_nt", "gemm_wsm_rt", "prefill_tile")
    try:
        for values in forms:
            for key, value in zip(keys, values):
                ops.tune(key, value)
            want = bits(ops.w4a16_gemm_stream(dev(x), w))
            got = bits(ops.w4a16_gemm_stream(dev(small_x), w_large))
            assert np.array_equal(got, np.where(large[0], want, exact(want, np.float32(2.0**-110)))), values
    finally:
        for key in keys:
            ops.tune(key, 0)


@pytest.mark.parametrize("nt,rt", [(1, 2), (2, 6), (3, 5)])
def test_scales_up_to_the_largest_in_slices(nt, rt):
    """Scales of 2^118 to 2^124 in some groups of K, and so in some slices and not in others, which decide alone what they take again: the powers of two cancel against x, so every
    product and sum has the bits of moderate scales."""
    from air_hip import ops
    print("largest scales in slices", nt, rt, flush=True)
    M, K, N = 200, 4096, 256
    rng = np.random.default_rng(rt)
    q, z = rng.integers(0, 16, (K, N), dtype=np.uint8), rng.integers(0, 16, (K // 128, N), dtype=np.uint8)
    s = np.exp2(rng.uniform(8, 14, (K // 128, N))).astype(np.float32) * rng.choice([-1, 1], (K // 128, N))
    x = (rng.uniform(0.125, 4, (M, K)) * rng.choice([-1, 1], (M, K))).astype(np.float32)
    exact = lambda b, by: f32_to_bf16_bits(bf16_bits_to_f32(b) * by)
    s, x = (f32_to_bf16_bits(np.ascontiguousarray(t.astype(np.float32))) for t in (s, x))
    qz = dev(oawq.pack_awq_int32(q)), dev(oawq.pack_awq_int32(z))
    w = ops.repack_stream(*qz, dev(s))
    keys = ("prefill_wsm", "gemm_wsm_nt", "gemm_wsm_rt", "gemm_wsm_slices")
    lib, parts = ops._lib.load_library(), torch.empty(4 * M * N, dtype=torch.float32, device="cuda")

    def product(xb, w, slices):
        for key, value in zip(keys, (1, nt, rt, slices)):
            ops.tune(key, value)
        y, xd = torch.empty((M, N), dtype=torch.bfloat16, device="cuda"), dev(xb)
        parts.fill_(float("nan"))
        ops._lib.check(lib.w4a16_gemm_stream_scratch_bf16(xd.data_ptr(), w.buf.data_ptr(), y.data_ptr(), M, K, N, 128, parts.data_ptr(), parts.numel() * 4,
                                                          torch.cuda.current_stream().cuda_stream))
        assert int(parts.isfinite().sum()) == (slices * M * N if slices > 1 else 0), "parts in the scratch"
        return bits(y)

    try:
        for large in (np.arange(K // 128) < 8, np.arange(K // 128) == 20, np.arange(K // 128) % 16 == 15):
            by = np.where(large, 2.0**110, 1.0).astype(np.float32)
            w_large, small_x = ops.repack_stream(*qz, dev(exact(s, by[:, None]))), exact(x, np.repeat(1 / by, 128)[None, :])
            for slices in (1, 2, 4):
                assert np.array_equal(product(small_x, w_large, slices), product(x, w, slices)), (slices, np.flatnonzero(large))
    finally:
        for key in keys:
            ops.tune(key, 0)


@pytest.mark.parametrize("form", [(1, 1, 2, 0), (1, 3, 4, 0), (2, 0, 0, 1), (2, 0, 0, 3)])
def test_every_weight_under_the_largest_scales(form):
    """One-hot rows of x, small and largest scales in one column: the dequantised weights bit for bit."""
    from air_hip import ops
    print("every weight, largest scales", form, flush=True)
    K, N = 256, 256
    k, n = np.arange(K)[:, None], np.arange(N)[None, :]
    q = ((k + n // 16) % 16).astype(np.uint8)
    z = np.broadcast_to((n % 16).astype(np.uint8), (K // 128, N))
    values = np.array([1.0, 2.0**118, 2.0**-120, -1.99 * 2.0**117, 2.0**122, 2.0**117, -(2.0**124)], np.float32)
    s = f32_to_bf16_bits(np.ascontiguousarray(values[(n // 16 + 3 * np.arange(K // 128)[:, None]) % len(values)]))
    tri = dev(oawq.pack_awq_int32(q)), dev(oawq.pack_awq_int32(np.ascontiguousarray(z))), dev(s)
    x, w = torch.eye(K, dtype=torch.bfloat16, device="cuda"), ops.repack_stream(*tri)
    want = bits(ops.awq_dequant(*tri))
    keys = ("prefill_wsm", "gemm_wsm_nt", "gemm_wsm_rt", "prefill_tile")
    try:
        for key, value in zip(keys, form):
            ops.tune(key, value)
        got = bits(ops.w4a16_gemm_stream(x, w))
        assert np.array_equal(np.where(got == 0x8000, 0, got), np.where(want == 0x8000, 0, want))   # (a sum's zero has no sign)
    finally:
        for key in keys:
            ops.tune(key, 0)


@pytest.mark.parametrize("codec", ["awq", "q4nx"])
@pytest.mark.parametrize("rt,nt", [(2, 1), (4, 2), (5, 2), (8, 2), (10, 2), (3, 3), (6, 3), (7, 3)])
def test_rounded_tiles_of_every_ring(codec, rt, nt):
    """Forms with two and with one workgroup to a CU, rings of three and four stages, from fewer groups than stages on; a ragged last block of rows and set of columns:
    the tiled kernel's bits."""
    from air_hip import ops
    for K in (256, 512, 1280):
        for M in (16 * rt * max(2, 144 // (16 * rt)) - 7, 16 * rt * 9 + 1):
            N = 64 * nt + 64
            print("rounded ring", codec, rt, nt, M, K, N, flush=True)
            if codec == "awq":
                w, product = ops.repack_stream(*map(dev, make_awq(K, N, seed=rt))), ops.w4a16_gemm_stream
            else:
                q, s, m = make(N, K, seed=rt)
                w, product = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T)), ops.q4nx_gemm_stream
            x = dev(make_x((M, K), seed=K))
            keys = ("prefill_min_m", "prefill_wsm", "gemm_wsm_rt", "gemm_wsm_nt")
            try:
                results = []
                for values in ((17, 1, rt, nt), (17, 2, 0, 0)):
                    for key, value in zip(keys, values):
                        ops.tune(key, value)
                    results.append(product(x, w))
                assert torch.equal(*(r.view(torch.int16) for r in results)), (codec, rt, nt, M, K)
            finally:
                for key in keys:
                    ops.tune(key, 0)


@pytest.mark.parametrize("codec", ["awq", "q4nx"])
@pytest.mark.parametrize("rt,nt,two", [(2, 1, 1), (4, 1, 1), (5, 1, 1), (6, 1, 1), (6, 1, 2), (3, 2, 1), (4, 2, 1), (6, 2, 1), (7, 2, 1), (7, 2, 2), (5, 3, 1), (5, 3, 2)])
def test_rounded_tiles_of_one_and_two_workgroups_to_a_cu(codec, rt, nt, two):
    """Rings of two, three and four stages of half of LDS, from as many groups as stages on, whole and in slices: on whole K the tiled kernel's bits, a grid that leaves no CU
    with one workgroup included; in slices one more rounding of fp32 sums."""
    from air_hip import ops
    keys = ("prefill_min_m", "prefill_wsm", "gemm_wsm_rt", "gemm_wsm_nt", "gemm_wsm_two", "gemm_wsm_slices")
    for M, K, N in ((16 * rt * max(1, 80 // (16 * rt)) + 1, 256, 64 * nt + 64), (16 * rt * 2 - 7, 512, 64 * nt), (16 * rt * 4 - 1, 768, 64 * 3 * nt), (200, 2048 + 256, 1024),
                    (16 * rt * 24, 1024, 64 * nt * 24)):
        print("rounded tiles, workgroups to a CU", codec, rt, nt, two, M, K, N, flush=True)
        if codec == "awq":
            w, product = ops.repack_stream(*map(dev, make_awq(K, N, seed=rt))), ops.w4a16_gemm_stream
        else:
            q, s, m = make(N, K, seed=rt)
            w, product = ops.q4nx_repack_stream(dev(oawq.pack_awq_int32(q.T)), dev(s.T), dev(m.T)), ops.q4nx_gemm_stream
        x = dev(make_x((M, K), seed=K))
        try:
            results = []
            for values in ((17, 1, rt, nt, two, 1), (17, 2, 0, 0, 0, 0), (17, 1, rt, nt, two, 2)):
                for key, value in zip(keys, values):
                    ops.tune(key, value)
                results.append(product(x, w))
            assert torch.equal(*(r.view(torch.int16) for r in results[:2])), (codec, rt, nt, two, M, K)
            whole, cut = results[0].double(), results[2].double()
            assert bool(((whole - cut).abs() <= 2.0 ** -7 * whole.abs() + 2.0 ** -14 * whole.abs().amax()).all()), (codec, rt, nt, two, M, K)
        finally:
            for key in keys:
                ops.tune(key, 0)


@pytest.mark.parametrize("rt,nt", [(3, 1), (4, 1), (7, 1), (3, 2), (4, 2), (6, 2)])
def test_exact_tiles_of_few_groups(rt, nt):
    """Pipelined exact tiles with fewer groups than sets of waves, than stages, and one more than whole steps: one bf16 rounding of an fp32 sum; a row of infinities stays
    in its row."""
    from air_hip import ops
    keys = {"gemm_splitk": 1, "gemm_wsm_rt": rt, "gemm_wsm_nt": nt, "gemm_wsm_slices": 1}
    M, N = 16 * rt - 5, 64 * nt + 48
    for K in (128, 256, 384, 640, 896):
        print("exact tiles of few groups", rt, nt, M, K, N, flush=True)
        tri = make_awq(K, N, seed=K)
        x = make_x((M, K), seed=rt)
        want = bf16_bits_to_f32(x).astype(np.float64) @ dense_f64(*tri)
        x[3, 5] = 0x7F80
        w, xd = ops.repack_stream(*map(dev, tri)), dev(x)
        try:
            for key, value in keys.items():
                ops.tune(key, value)
            got = bits(ops.w4a16_gemm_stream(xd, w))
        finally:
            for key in keys:
                ops.tune(key, 0)
        rows = np.arange(M) != 3
        assert not np.isfinite(bf16_bits_to_f32(got[3])).any()
        assert_bf16_close(np.ascontiguousarray(got[rows]), want[rows], ulps=1.0, atol=2e-3, what=f"{rt} {nt} {K}")


@pytest.mark.parametrize("slices", [4, 5, 8, 9, 16])
def test_sums_of_many_slices(slices):
    """Parts asked for several at a time, with and without some left over, against the float64 product."""
    from air_hip import ops
    M, K, N = 33, 34 * 128, 80
    qw, qz, s = make_awq(K, N, seed=slices)
    x = make_x((M, K), seed=slices)
    try:
        for key, value in (("gemm_splitk", 1), ("gemm_wsm_slices", slices)):
            ops.tune(key, value)
        got = ops.w4a16_gemm_stream(dev(x), ops.repack_stream(dev(qw), dev(qz), dev(s)))
        assert_bf16_close(bits(got), bf16_bits_to_f32(x).astype(np.float64) @ dense_f64(qw, qz, s), ulps=1.0, atol=2e-3, what=f"{slices} slices")
    finally:
        for key in ("gemm_splitk", "gemm_wsm_slices"):
            ops.tune(key, 0)
