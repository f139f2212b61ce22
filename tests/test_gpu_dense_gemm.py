"""Products over many rows at the edges of their tiles and slices, each tile set by hand and as the rule picks them, against float64 products of the
same bf16 numbers.

fp32 results: sums of K products of 16 significant bits in fp32, any order, stay within K 2^-24 of the sum of magnitudes, which for
random signs is about K^1/2 times the result's rms; 2^-24 K^3/2 is 4e-5 at K = 8192, and what is seen is 30 times less.  bf16 results add
half an ulp of the value, 2^-8 with the rounding to either neighbour."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dense():
    from air_hip import dense as d
    return d


def rand(seed, *shape):
    return torch.randn(shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(seed))


def close(got, want, bf16, what):
    rms = want.square().mean().sqrt()
    bound = 4e-5 * rms + (2.0 ** -8 * want.abs() if bf16 else 0.0)
    bad = (got.double() - want).abs() > bound
    assert not bad.any(), (what, int(bad.sum()), bad.nonzero()[0].tolist())


def interleaved(g, u):
    n, K = g.shape
    return torch.stack([g.reshape(n // 16, 16, K), u.reshape(n // 16, 16, K)], 1).reshape(2 * n, K).contiguous()


SHAPES = [(1, 16, 64, 1), (17, 144, 192, 3), (31, 96, 1024, 8), (33, 272, 128, 2), (64, 400, 512, 4), (127, 256, 576, 5), (128, 528, 64, 1), (129, 784, 320, 2),
          (255, 240, 704, 4), (256, 512, 128, 2), (257, 1040, 448, 7), (300, 2048, 8192, 8), (513, 208, 640, 1), (700, 1104, 1216, 2), (1025, 3088, 192, 1)]


def products(dense, M, N, K, counts, tile=0):
    """Every epilogue in each number of slices, against float64; rows of A and out are longer than what is used of them."""
    from air_hip import _lib
    lib, stream = _lib.load_dense_library(), torch.cuda.current_stream().cuda_stream
    a, w = rand(M, M, K + 64).bfloat16()[:, 8:K + 8], (rand(N + 1, N, K) * K ** -0.5).bfloat16()
    want = a.double() @ w.double().t()
    pair = N // 32 * 32
    silu, gelu = torch.nn.functional.silu, lambda t: torch.nn.functional.gelu(t, approximate="tanh")
    for n in counts:
        for epilogue in (dense.OUT_F32, dense.OUT_ELEM, dense.OUT_SWIGLU, dense.OUT_GEGLU):
            cols, width = (N, N) if epilogue < 2 else (pair, pair // 2)
            if not cols:
                continue
            out = torch.full((M, width + 8), 7.0, device="cuda", dtype=torch.float32 if epilogue == dense.OUT_F32 else torch.bfloat16)
            parts = torch.full((n, M, cols), float("nan"), device="cuda")
            begin, end = (16, N // 32 * 16) if epilogue == dense.OUT_ELEM else (0, 0)
            g = _lib.GemmArgs(a=a.data_ptr(), w=w.data_ptr(), out=out.data_ptr(), lda=a.stride(0), ldo=width + 8, M=M, N=cols, K=K, epilogue=epilogue,
                              silu_begin=begin, silu_end=end, tile_rows=tile)
            _lib.check_dense(lib.dlm_gemm_sliced(0, ctypes.byref(g), n, parts.data_ptr(), stream))
            ref = want[:, :cols].clone()
            if epilogue >= 2:
                q = ref.reshape(M, -1, 2, 16)
                ref = ((silu if epilogue == dense.OUT_SWIGLU else gelu)(q[:, :, 0]) * q[:, :, 1]).reshape(M, width)
            elif begin < end:
                ref[:, begin:end] = silu(ref[:, begin:end])
            close(out[:, :width], ref, epilogue != dense.OUT_F32, (n, epilogue))
            assert (out[:, width:] == 7.0).all(), "columns past the width were written"
            assert bool(parts.isnan().all()) if n == 1 else bool(parts.isfinite().all()), "as many parts as slices"


@pytest.mark.parametrize("M,N,K,slices", SHAPES)
def test_sliced_products(dense, M, N, K, slices):
    """The tiles that the rule picks."""
    print("sliced", M, N, K, slices, flush=True)
    from air_hip import _lib
    products(dense, M, N, K, {1, slices, _lib.load_dense_library().dlm_gemm_slices(0, M, N, K, dense.OUT_F32)})


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("M,N,K", [(255, 208, 64), (257, 272, 128), (129, 144, 192), (513, 544, 256), (33, 400, 320)])
def test_every_tile(dense, tile, M, N, K):
    """Each of the six tiles at one row less and more than its blocks, one 16-column tile past its columns, one to five K-steps, in one slice and
    in uneven ones (three, of one or two K-steps)."""
    print("tile", tile, M, N, K, flush=True)
    products(dense, M, N, K, {1, min(3, K // 64)}, -tile)


@pytest.mark.parametrize("tile", [4, 5, 6])
@pytest.mark.parametrize("M,N,K", [(2100, 8208, 64), (1300, 12304, 320), (513, 33296, 128)])
def test_wide_tiles_one_after_the_other(dense, tile, M, N, K):
    """More tiles than CUs, whole ones and those at the edges in turn, one to five K-steps each."""
    print("wide tiles", tile, M, N, K, flush=True)
    products(dense, M, N, K, {1, 2} if K > 64 else {1}, -tile)


@pytest.mark.parametrize("M,N,K,slices", [(64, 4096, 64, 1), (260, 2048, 128, 2), (1040, 512, 64, 1)])
@pytest.mark.parametrize("gated", [False, True])
def test_silu_behind_a_product_is_an_fp32_one(dense, gated, M, N, K, slices):
    """Two products of bf16 numbers make the argument, exact in fp32 (multiples of 2^-16), from -80 to -47.  silu in fp32 is off by one unit of
    2^-24 on average at most, which changes one bf16 rounding (2^-8 apart at least) in 2^16; an exponent rounded after log2 e is off by
    2^-19 ln 2 on average."""
    from air_hip import _lib
    print("silu", gated, M, N, K, slices, flush=True)
    lib, stream = _lib.load_dense_library(), torch.cuda.current_stream().cuda_stream
    a, w = torch.zeros((M, K), device="cuda").bfloat16(), torch.zeros((N, K), device="cuda").bfloat16()
    g = torch.Generator(device="cuda").manual_seed(M)
    uniform = lambda n, lo, hi: (lo + (hi - lo) * torch.rand(n, device="cuda", generator=g)).bfloat16()
    a[:, 0], a[:, 1], a[:, 2] = -8.0, uniform(M, 0.5, 1.0), 1.0
    width = N // 2 if gated else N
    z = torch.stack([uniform(width, 6.0, 10.0), uniform(width, 0.5, 1.0)], 1)
    if gated:   # 16 gate rows, 16 rows that give 1
        v = w.view(N // 32, 2, 16, K)
        v[:, 0, :, :2], v[:, 1, :, 2] = z.view(-1, 16, 2), 1.0
    else:
        w[:, :2] = z
    out, parts = torch.empty((M, width), device="cuda", dtype=torch.bfloat16), torch.empty((slices, M, N), device="cuda")
    args = _lib.GemmArgs(a=a.data_ptr(), w=w.data_ptr(), out=out.data_ptr(), lda=K, ldo=width, M=M, N=N, K=K, silu_begin=0, silu_end=0 if gated else N,
                         epilogue=dense.OUT_SWIGLU if gated else dense.OUT_ELEM)
    _lib.check_dense(lib.dlm_gemm_sliced(0, ctypes.byref(args), slices, parts.data_ptr(), stream))
    want = torch.nn.functional.silu(a[:, :2].double() @ z.double().t())
    down = want.float().bfloat16().double()   # (fp32 first: a double rounding shows as rarely)
    wrong = int((out.double() != down).sum())
    assert wrong <= out.numel() * 2.0 ** -16 + 4 * (out.numel() * 2.0 ** -16) ** 0.5, (wrong, out.numel())
    if not gated:
        a[:3, 0] = torch.tensor([float("inf"), float("-inf"), float("nan")])   # inf, -inf / inf, NaN
        _lib.check_dense(lib.dlm_gemm_sliced(0, ctypes.byref(args), slices, parts.data_ptr(), stream))
        assert bool((out[0] == float("inf")).all()) and bool(out[1:3].isnan().all()) and bool(out[3:].isfinite().all())


@pytest.mark.parametrize("M,K", [(3, 64), (300, 2048)])
def test_parts_meet_in_the_row_kernels(dense, M, K):
    a, w = rand(1, M, 512).bfloat16(), (rand(2, K, 512) * 512 ** -0.5).bfloat16()
    res, nw = rand(3, M, K), 1.0 + 0.1 * rand(4, K)
    y = a.double() @ w.double().t()
    parts = torch.stack([dense.gemm(a[:, i:i + 64].contiguous(), w[:, i:i + 64].contiguous(), out_f32=True) for i in range(0, 512, 64)])
    norm = lambda v: v / torch.sqrt(v.square().mean(-1, keepdim=True) + 1e-5) * nw.double()
    for dtype in (torch.float32, torch.bfloat16):
        r = res.clone()
        h = dense.residual_norm_rows(r, parts, nw, 1e-5, K, dtype)
        close(r, res.double() + norm(y), False, "residual")
        close(h, res.double() + norm(y), dtype == torch.bfloat16, "residual, element type")
        r = res.clone()
        h = dense.add_norm_rows(r, parts, nw, 1e-5, K, dtype)
        close(r, res.double() + y, False, "sum")
        close(h, norm(res.double() + y), dtype == torch.bfloat16, "norm of the sum")
    assert dense.gemm(a, w, out_f32=True, parts=True).shape[1:] == (M, K)


@pytest.mark.parametrize("width", [64, 1024, 1088, 2048, 2112, 4096, 4160])
def test_row_kernels_of_every_form(dense, width):
    """Few rows (loads together, sums in registers) and many (loads in turn, sums by way of LDS) add up in the same order: the same bits."""
    many = 1100
    res, nw = rand(1, many, width), 1.0 + 0.1 * rand(2, width)
    norm = lambda v: v / torch.sqrt(v.square().mean(-1, keepdim=True) + 1e-5) * nw.double()
    for n in (1, 2, 3, 5, 9):
        y, ys, wt = rand(n, n, many, width), rand(n + 20, many, n, width).bfloat16(), rand(n + 40, many, n).abs()
        calls = {"residual": lambda r, m: dense.residual_norm_rows(r, y[:, :m].contiguous(), nw, 1e-5, width, torch.bfloat16),
                 "sum": lambda r, m: dense.add_norm_rows(r, y[:, :m].contiguous(), nw, 1e-5, width, torch.bfloat16),
                 "experts": lambda r, m: dense.residual_norm_rows(r, ys[:m].reshape(m * n, width), nw, 1e-5, width, torch.bfloat16, weights=wt[:m].contiguous())}
        wants = {"residual": res.double() + norm(y.double().sum(0)), "sum": res.double() + y.double().sum(0),
                 "experts": res.double() + norm((wt.double()[..., None] * ys.double()).sum(1))}
        for name, call in calls.items():
            all_r = res.clone()
            all_h = call(all_r, many)
            close(all_r, wants[name], False, (name, n))
            for m in (1, 512, 513):
                r = res[:m].clone()
                h = call(r, m)
                assert torch.equal(r, all_r[:m]) and torch.equal(h, all_h[:m]), (name, n, m)


COUNTS = [(0, 1, 15, 128, 129, 255, 256, 257), (512, 0, 0, 300, 64, 127, 383, 385), (16, 16, 16, 16, 16, 16, 16, 16), (0, 0, 0, 700, 0, 0, 0, 0), [384, 385, 320, 770, 192, 321]]


@pytest.mark.parametrize("tile_rows,launched", [(32, 32), (128, 128), (256, 256), (384, 384), (384, 128), (64, 384)])   # of the plan, of the launch
@pytest.mark.parametrize("counts", COUNTS)
def test_experts_with_tiles_of_every_fill(dense, counts, tile_rows, launched):
    print("experts", counts, tile_rows, launched, flush=True)
    from air_hip import _lib
    lib, stream = _lib.load_dense_library(), torch.cuda.current_stream().cuda_stream
    E, K, ff, N, top = len(counts), 192, 144, 272, 2
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    if len(ids) % top:
        ids = torch.cat([ids, ids[-1:]])
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(5))].to(torch.int32).cuda()
    entries = len(ids)
    h = rand(6, entries // top, K).bfloat16()
    gate, up = ((rand(7 + i, E, ff, K) * K ** -0.5).bfloat16() for i in range(2))
    w1, w2 = torch.stack([interleaved(g, u) for g, u in zip(gate, up)]), (rand(9, E, N, 192) * ff ** -0.5).bfloat16()
    order = torch.empty((entries,), dtype=torch.int32, device="cuda")
    n_tiles = lib.dlm_moe_max_tiles(entries, E, tile_rows)
    tiles = torch.empty((n_tiles + 1, 4), dtype=torch.int32, device="cuda")
    _lib.check_dense(lib.dlm_moe_plan(ids.data_ptr(), entries, E, tile_rows, order.data_ptr(), tiles.data_ptr(), stream))
    act = torch.zeros((entries, 192), dtype=torch.bfloat16, device="cuda")
    out = torch.full((entries, N), 7.0, dtype=torch.bfloat16, device="cuda")
    common = dict(tiles=tiles.data_ptr(), order=order.data_ptr(), M=entries, n_tiles=n_tiles, tile_rows=launched)
    g = _lib.GemmArgs(a=h.data_ptr(), w=w1.data_ptr(), out=act.data_ptr(), lda=K, ldo=192, w_stride=2 * ff * K, N=2 * ff, K=K, epilogue=dense.OUT_SWIGLU,
                      gather=top, **common)
    _lib.check_dense(lib.dlm_gemm(0, ctypes.byref(g), stream))
    g = _lib.GemmArgs(a=act.data_ptr(), w=w2.data_ptr(), out=out.data_ptr(), lda=192, ldo=N, w_stride=N * 192, N=N, K=192, epilogue=dense.OUT_ELEM, gather=0,
                      **common)
    _lib.check_dense(lib.dlm_gemm(0, ctypes.byref(g), stream))
    e, token = ids.long(), torch.arange(entries, device="cuda") // top
    for i in range(E):
        at = (e == i).nonzero()[:, 0]
        if not len(at):
            continue
        x = h[token[at]].double()
        a = torch.nn.functional.silu(x @ gate[i].double().t()) * (x @ up[i].double().t())
        place = torch.empty((entries,), dtype=torch.long, device="cuda")
        place[order.long()] = torch.arange(entries, device="cuda")
        got = act[place[at]]
        close(got[:, :ff], a, True, ("gate / up", i))
        close(out[at], got.double() @ w2[i].double().t(), True, ("down", i))


@pytest.mark.parametrize("tile_rows", [128, 384])
@pytest.mark.parametrize("past", [-1, 0, 1])
def test_experts_with_tiles_of_every_height(dense, tile_rows, past):
    test_experts_with_tiles_of_every_fill(dense, [32 * r + past for r in range(1, 1 + tile_rows // 32)], tile_rows, tile_rows)


@pytest.mark.parametrize("gather,lda", [(1, 1 << 30), (2, 1 << 29), (0, 6 << 20)])   # 3 tokens' rows past 2^32 bytes, below them, a tile's past them
def test_experts_with_rows_far_apart(dense, gather, lda):
    print("experts with rows of", lda, "gathered", gather, flush=True)
    from air_hip import _lib
    lib, stream = _lib.load_dense_library(), torch.cuda.current_stream().cuda_stream
    E, K, N, tokens = 3, 128, 144, 3
    entries = tokens * max(gather, 1)
    ids = torch.tensor([2, 0, 2, 0, 0, 2][:entries], dtype=torch.int32, device="cuda")
    a = torch.empty(((tokens if gather else entries) - 1) * lda + K, dtype=torch.bfloat16, device="cuda").as_strided((tokens if gather else entries, K), (lda, 1))
    a.copy_(rand(1, *a.shape))
    w = (rand(2, E, N, K) * K ** -0.5).bfloat16()
    order = torch.empty((entries,), dtype=torch.int32, device="cuda")
    n_tiles = lib.dlm_moe_max_tiles(entries, E, 128)
    tiles = torch.empty((n_tiles + 1, 4), dtype=torch.int32, device="cuda")
    _lib.check_dense(lib.dlm_moe_plan(ids.data_ptr(), entries, E, 128, order.data_ptr(), tiles.data_ptr(), stream))
    out = torch.full((entries, N), 7.0, dtype=torch.bfloat16, device="cuda")
    g = _lib.GemmArgs(a=a.data_ptr(), w=w.data_ptr(), out=out.data_ptr(), lda=lda, ldo=N, w_stride=N * K, N=N, K=K, gather=gather, tiles=tiles.data_ptr(),
                      epilogue=dense.OUT_ELEM, order=order.data_ptr(), M=entries, n_tiles=n_tiles, tile_rows=128)
    _lib.check_dense(lib.dlm_gemm(0, ctypes.byref(g), stream))
    at = order.long()
    rows = a[at // gather] if gather else a
    want = torch.stack([w[e].double() @ r.double() for e, r in zip(ids[at].tolist(), rows)])
    close(out if gather else out[at], want, True, (gather, lda))


@pytest.mark.parametrize("dtype,tile_rows", [(torch.bfloat16, 32), (torch.bfloat16, 128), (torch.bfloat16, 384), (torch.float32, 32), (torch.float32, 128)])
@pytest.mark.parametrize("pair", [False, True])
def test_grouped_products_with_rows_in_either_order(dense, dtype, tile_rows, pair):
    """Both sides of `gather` with both epilogues: rows of A by entry and results at sorted places, or the other way round."""
    print("grouped rows", dtype, tile_rows, pair, flush=True)
    from air_hip import _lib
    lib, stream, dt = _lib.load_dense_library(), torch.cuda.current_stream().cuda_stream, int(dtype == torch.float32)
    counts, K, N, top = (1, 130, 0, 400, 65), 128, 160, 4
    E, entries, width = len(counts), sum(counts), 80 if pair else 160
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(entries, generator=torch.Generator().manual_seed(1))].to(torch.int32).cuda()
    order = torch.empty((entries,), dtype=torch.int32, device="cuda")
    n_tiles = lib.dlm_moe_max_tiles(entries, E, tile_rows)
    tiles = torch.empty((n_tiles + 1, 4), dtype=torch.int32, device="cuda")
    _lib.check_dense(lib.dlm_moe_plan(ids.data_ptr(), entries, E, tile_rows, order.data_ptr(), tiles.data_ptr(), stream))
    a, w = rand(2, entries, K).bfloat16().to(dtype), (rand(3, E, N, K) * K ** -0.5).bfloat16().to(dtype)
    w1 = torch.stack([interleaved(m[:N // 2], m[N // 2:]) for m in w]) if pair else w
    e, at = ids.long(), order.long()
    for gather in (0, top):
        out = torch.full((entries, width), 7.0, dtype=dtype, device="cuda")
        g = _lib.GemmArgs(a=a.data_ptr(), w=w1.data_ptr(), out=out.data_ptr(), lda=K, ldo=width, w_stride=N * K, N=N, K=K, gather=gather, tiles=tiles.data_ptr(),
                          epilogue=dense.OUT_SWIGLU if pair else dense.OUT_ELEM, order=order.data_ptr(), M=entries, n_tiles=n_tiles, tile_rows=tile_rows)
        _lib.check_dense(lib.dlm_gemm(dt, ctypes.byref(g), stream))
        rows = a[at // top] if gather else a                      # by sorted place
        y = torch.bmm(w[e[at]].float(), rows.float()[:, :, None]).squeeze(2).double()   # (fp32 products of 128 bf16 numbers: 2^-24 of their sum)
        y = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:] if pair else y
        close(out if gather else out[at], y, not dt, (gather, pair))


@pytest.mark.parametrize("entries,experts", [(1, 1), (1000, 7), (16384, 64), (16385, 1024), (50000, 3)])
def test_expert_plan(dense, entries, experts):
    print("plan", entries, experts, flush=True)
    from air_hip import _lib
    lib, stream = _lib.load_dense_library(), torch.cuda.current_stream().cuda_stream
    ids = torch.randint(0, experts, (entries,), dtype=torch.int32, device="cuda", generator=torch.Generator(device="cuda").manual_seed(entries))
    for bm in (32, 384):
        most = lib.dlm_moe_max_tiles(entries, experts, bm)
        order, tiles = torch.full((entries,), -1, dtype=torch.int32, device="cuda"), torch.empty((most + 1, 4), dtype=torch.int32, device="cuda")
        _lib.check_dense(lib.dlm_moe_plan(ids.data_ptr(), entries, experts, bm, order.data_ptr(), tiles.data_ptr(), stream))
        n = int(tiles[most, 0])
        assert torch.equal(order.sort()[0], torch.arange(entries, dtype=torch.int32, device="cuda"))
        assert torch.equal(ids[order.long()], ids.sort()[0])
        rows = tiles[:n].long()
        assert n <= most and bool(((rows[:, 2] > 0) & (rows[:, 2] <= bm)).all())
        # the tiles follow each other and stay within their expert
        ends = rows[:, 2].cumsum(0)
        assert torch.equal(rows[:, 1], ends - rows[:, 2]) and int(ends[-1]) == entries
        assert torch.equal(ids[order.long()].long(), torch.repeat_interleave(rows[:, 0], rows[:, 2]))
