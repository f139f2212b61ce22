// Products of 17 rows and more on stream-order weights (wstream.h), both codecs, any K % 128 == 0 and N % 16 == 0:
// y[M, N] = bf16(x[M, K] . W (+ residual)) with the exact weights, fp32 accumulation.
//
// A wave alone goes through a group of 128 k (4 x 2 tiles, exact) in about 1900 cycles, of which the matrix pipe works a third: LDS reads, 145 vector and 60
// scalar instructions and the barrier are a chain.  So a workgroup puts KW waves on every SIMD, each set of four on a group of its own
// (their sums meet in LDS at the end), and K is cut into slices besides where there are few columns; and two waves make a K-step's operands beside the products
// of the one before (AWQ).  64 rows, K = 14336, N = 4096: 18.4 us, the launches of 64 whole-K rows that ran before there was this kernel 27.3 us (split along K) and 54.9 us;
// Q4NX, 2000 rows of the ragged K = 2176, N = 5744 151 us (16 rows a launch: 949 us).
//
//   workgroup  = 16 RT rows x 64 NT columns; wave (part kq < KW of K, wq < 4): row tiles all, stream tiles NT wq .. of the column set
//   step       = KW groups; x goes global -> LDS once per workgroup (global_load_lds_dwordx4) and so do a wave's cells and scale words
//                (a cell is the B operand of four K-steps), R - 1 steps ahead, in a ring of R.  (Cells in registers instead: the
//                compiler waits for every request in flight once per turn of a loop that carries loads from one turn to the next.)
//   AWQ        : operands are (128 + q) exactly, flushed per group: y += s (sum (128 + q) x - (128 + z) sum x); the sums of x are taken by one wave per row
//                tile with an MFMA against ones and handed round through LDS (by every wave for itself with four waves a SIMD and R = 2).  Two waves a SIMD, one group
//                after the other / pipelined, us: 64 rows of 4096 x 14336 in 4 x 2 tiles 25.8 / 22.8, 4 x 1 20.6 / 19.1; 128 of 4096 x 11008 26.2 / 23.3; 3 x 2 of 64 of 14336 x 4096 24.4 / 22.2
//   Q4NX       : a scale and a minimum per K-step would make that flush four times as dear: s q, which has 12 significant bits, is cut
//                into two bf16, and the minimum is an operand of its own: three MFMAs per K-step with every product exact, as s sum q x +
//                min sum x has them.  (s q + min in two operands keeps 16 bits of it, which loses minima small against the scale.)
//   rounded    : bf16 weights as the tiled kernel of gemm_ws.hip multiplies them, on whole K in its order of sums: the same bits, and a residual is
//                added to the rounded product as its epilogue does.  KW = 1, and an accumulator's products follow each other, so what hides a wave's LDS reads and
//                dequantisation are its own products: those of a K-step run beside the reads and the dequantisation of the next one (sm_interleave), across
//                groups too.  What bounds it then is issue, 4 cycles an instruction: a group of 5 x 3 tiles has 240 vector, 60 matrix and 110 other ones.  Tall and wide
//                forms (up to 10 x 2 and 7 x 3 tiles, one workgroup to a CU, rings of 160 KB) need the fewest; two workgroups to a CU, each with half of LDS, hide each
//                other's latencies and fill the chip with twice as many tiles.  Reading a group ahead takes a stage of the ring: with four it is asked for two groups
//                before it is needed, with three one group, with two it could not be.  So with fewer than four all of a group's x is read in its first half (kEarly: 8 RT more
//                registers) and its own stage is filled again: three stages are two groups, two stages one.
//                Weights from memory, us, K-steps one after the other / read ahead without kEarly, where two stages leave one workgroup to a CU / now: 349 rows of 4352 x 13760
//                54.9 / 64.5 / 52.5, 386 of 6656 x 12800 82.2 / 95.4 / 82.9, 652 of 1280 x 8896 22.6 / 27.8 / 22.2, 170 of 2048 x 5120 11.5 / 12.4 / 11.5, 1519 of 1536 x 5568 31.6 /
//                40.2 / 32.6, 300 of 4096 x 11008 43.0 / 39.1 / 38.4, Q4NX 486 of 2560 x 12480 45.1 / 60.0 / 42.3, 282 of 10240 x 6336 69.4 / 77.3 / 67.5.  400 random products of 129 to
//                2000 rows against the loop of K-steps one after the other: 1.14 times as fast (from memory 0.88 at worst, seven below 0.95: 1000 to 1300 rows of wide short matrices,
//                where the tiled kernel and the tallest forms are close, and eight to ten groups of K; from the last-level cache 0.95, one); 17 to 128 rows, exact ones mostly, 1.06 and
//                1.07 (0.94 and 0.96 at worst).  (Every instruction in its place by
//                volatile asm, none behind one that it depends on, 300 of 4096 x 11008 36.4 -> 38.3: not taken.)
//   slices > 1 : fp32 sums to plain scratch, added in slice order by a second launch (deterministic)
#include <algorithm>
#include <utility>

#include "common.h"
#include "kernels.h"
#include "wsdequant.h"
#include "wstream.h"

namespace w4a16 {

namespace {

constexpr int kSmLds = 160 * 1024;
enum : int { kSmAwq, kSmQ4, kSmAwqRounded, kSmQ4Rounded };

struct SmArgs {
    const uint16_t *x;
    const char *w, *w2;            // w2: a second matrix of the same shape, whose product goes to y2 (rounded weights)
    float *partial;                // [slices][matrices][M][N]
    uint16_t *y, *y2;
    const uint16_t *residual;
    int M, K, N, G, NB;
    int sets, slices, blocks;      // column sets of all matrices, slices of K, blocks of rows
    int own_sets;                  // column sets of one matrix
};

// A step in LDS: the x tiles of its groups, then per wave its cells and its scale words ([64]: tile lane / 16, column lane % 16; Q4NX:
// [NT][64], K-step lane / 16)
constexpr int sm_wave_bytes(int nt, bool q4) { return nt * (int)kWsCellBytes + (q4 ? nt : 1) * 256; }
constexpr int sm_stage(int rt, int nt, int kw, bool q4) { return kw * (16 * rt * 256 + 4 * sm_wave_bytes(nt, q4)); }
constexpr int sm_sums(int rt, int kw, bool q4) { return q4 ? 0 : 2 * kw * 16 * rt * 4; }   // bytes of the sums of x of two steps
constexpr int sm_ring(int rt, int nt, int kw, bool q4, bool two) {
    const int n = ((two ? kSmLds / 2 : kSmLds) - sm_sums(rt, kw, q4)) / sm_stage(rt, nt, kw, q4);
    return n < 4 ? n : 4;
}

// The compiler's schedule of P products: behind each its share of VALU vector instructions; the READS LDS reads behind the first half, so that they are there when the
// next K-step begins; the COPIES requests, which may not pass them, behind the other.  (Reads behind all of the products, copies first: 300 x 4096 x 11008 38 us, 36.4 so.)
template <int P, int VALU, int READS, int COPIES, int... I>
__device__ __forceinline__ void sm_interleave(std::integer_sequence<int, I...>) {
    auto one = [](auto n) __attribute__((always_inline)) {
        constexpr int i = decltype(n)::value;
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        constexpr int E = P / 2;
        constexpr int r = (i + 1 < E ? (i + 1) * READS / E : READS) - (i < E ? i * READS / E : READS);
        constexpr int c = (i < E ? 0 : (i + 1 - E) * COPIES / (P - E)) - (i <= E ? 0 : (i - E) * COPIES / (P - E)), v = (i + 1) * VALU / P - i * VALU / P;
        if constexpr (r > 0) __builtin_amdgcn_sched_group_barrier(0x100, r, 0);
        if constexpr (v > 0) __builtin_amdgcn_sched_group_barrier(0x2, v, 0);
        if constexpr (c > 0) __builtin_amdgcn_sched_group_barrier(0x20, c, 0);
    };
    (one(std::integral_constant<int, I>()), ...);
}

__device__ __forceinline__ floatx4 widen4(uint2 v) {
    return floatx4{bf16_bits_to_float(v.x & 0xFFFFu), bf16_bits_to_float(v.x >> 16), bf16_bits_to_float(v.y & 0xFFFFu), bf16_bits_to_float(v.y >> 16)};
}
__device__ __forceinline__ uint2 narrow4(floatx4 v) { return uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])}; }
__device__ __forceinline__ floatx4 rounded4(floatx4 v) { return widen4(narrow4(v)); }

template <int RT, int NT, int KW, int MODE, bool TWO>
__global__ void __launch_bounds__(256 * KW, KW == 1 ? 2 : KW) gemm_wsm_kernel(const SmArgs p) {
    constexpr bool Q4 = MODE == kSmQ4 || MODE == kSmQ4Rounded, kExact = MODE == kSmAwq;
    constexpr int ROWS = 16 * RT, XT = ROWS * 256;                     // rows and bytes of an x tile (a group: 128 bf16 a row)
    constexpr int MC = Q4 ? NT : 1;                                    // copies (256 bytes) of a wave's scale words
    constexpr int V = RT + NT + MC;                                    // requests of a wave and step: x, cells, scale words
    constexpr int kWave = sm_wave_bytes(NT, Q4), kStage = sm_stage(RT, NT, KW, Q4), R = sm_ring(RT, NT, KW, Q4, TWO);
    // Exact AWQ by two waves a SIMD: pipelined.  (Four waves hide each other's latencies, and there are few registers: 2 x 2 tiles 16.0 us without, 17.0 with, 64 rows of 4096 x 14336.)
    constexpr bool kAhead = kExact && KW == 2 && RT * NT <= 12;
    constexpr bool kSums = kExact && !kAhead && R > 2 && RT <= 4;      // sums of x handed round, taken a step ahead; else a wave takes its own
    constexpr int CW = 64 * NT, kThreads = 256 * KW;
    static_assert(R >= 2, "two steps fit LDS");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    float *xs_lds = reinterpret_cast<float *>(lds + R * kStage);       // [2][KW][ROWS]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kq = wave >> 2, wq = wave & 3;
    const int lg = lane >> 4, ln = lane & 15;

    // An XCD takes a contiguous range of (slice, column set, row block), row blocks first: those that run together on it share the
    // weights of a set and the x of a slice in its L2.
    const int total = p.sets * p.slices * p.blocks, per_xcd = (total + 7) / 8;
    const int id = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || id >= total) return;
    const int block = id % p.blocks, set_of_all = id / p.blocks % p.sets, slice = id / (p.blocks * p.sets);
    const bool second = MODE >= kSmAwqRounded && set_of_all >= p.own_sets;
    const int set = second ? set_of_all - p.own_sets : set_of_all;
    const char *const w = second ? p.w2 : p.w;
    const int g_lo = (int)((long)p.G * slice / p.slices), g_hi = (int)((long)p.G * (slice + 1) / p.slices);
    const int m0 = block * ROWS, rows = min(ROWS, p.M - m0);

    // tiles past the matrix (ragged last set) read the last tile and are not stored
    const int ntiles = p.N / kWsTileCols;
    constexpr int kMd = Q4 ? kWsQ4MdKiB : 1;   // KiB of scale words in front of a block's cells
    const size_t tile_bytes = (size_t)(kMd * p.NB + p.G) * kWsCellBytes;
    const int first = min((set * 4 + wq) * NT, ntiles - 1);
    gptr tb[NT];
#pragma unroll
    for (int c = 0; c < NT; ++c) tb[c] = scalar_ptr(w + (size_t)min(first + c, ntiles - 1) * tile_bytes);
    // this lane's cell and scale words: 32-bit offsets from a tile's start (from the first tile's for the AWQ words, one copy of which
    // serves all the wave's tiles)
    const uint32_t lane16 = 16 * lane;
    const uint32_t word_off = 16 * ln + (Q4 ? lg * (uint32_t)kWsCellBytes : (uint32_t)(min(first + lg % NT, ntiles - 1) - first) * (uint32_t)tile_bytes);

    // copy j of the wave: rows 4 q .. + 3 of its group's x, q = 4 j + wq; lane l fetches chunk (l % 16) ^ row % 16 of row l / 16
    const gptr xbase = scalar_ptr(p.x + (size_t)m0 * p.K);
    uint32_t xoff[RT];   // (at most 127 rows: the host keeps K below 2^24; 2^23 with more)
#pragma unroll
    for (int j = 0; j < RT; ++j) {
        const int row = 4 * (4 * j + wq) + lg;
        xoff[j] = (uint32_t)min(row, rows - 1) * (uint32_t)(p.K * 2) + 16 * (ln ^ (row & 15));
    }
    const int x_lds = kq * XT, wave_lds = KW * XT + wave * kWave;
    auto copy16 = [&](gptr src, int dst) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src, (__attribute__((address_space(3))) void *)(lds + dst), 16, 0, 0);
    };
    auto copy4 = [&](gptr src, int dst) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src, (__attribute__((address_space(3))) void *)(lds + dst), 4, 0, 0);
    };
    auto request_x = [&](int g, int stage, int j0, int j1) {
        const gptr xs = xbase + (size_t)g * 256;
#pragma unroll
        for (int j = 0; j < RT; ++j)
            if (j >= j0 && j < j1) copy16(xs + xoff[j], stage + x_lds + 1024 * (4 * j + wq));
    };
    auto request_w = [&](int g, int stage) {
        const uint32_t blk = (uint32_t)(g >> 4) * (uint32_t)((kWsBlockGroups + kMd) * kWsCellBytes);
        uint32_t cell = lane16 + (blk + (uint32_t)(kMd + (g & 15)) * (uint32_t)kWsCellBytes), word = word_off + (blk + 64 * (g & 12) + 4 * (g & 3));
        asm volatile("" : "+v"(cell), "+v"(word));   // (a 32-bit sum: folds into the copies as their offset)
#pragma unroll
        for (int c = 0; c < NT; ++c) copy16(tb[c] + cell, stage + wave_lds + c * (int)kWsCellBytes);
#pragma unroll
        for (int c = 0; c < MC; ++c) copy4(tb[c] + word, stage + wave_lds + NT * (int)kWsCellBytes + 256 * c);
    };
    auto request = [&](int g, int stage) {
        request_x(g, stage, 0, RT);
        request_w(g, stage);
    };
    auto cell_at = [&](int stage, int c) { return *reinterpret_cast<const u32x4 *>(lds + stage + wave_lds + c * (int)kWsCellBytes + 16 * lane); };
    auto word_at = [&](int stage, int c, int t) {   // (AWQ: t = 0)
        return *reinterpret_cast<const uint32_t *>(lds + stage + wave_lds + NT * (int)kWsCellBytes + (Q4 ? 256 * c + 64 * t : 64 * c) + 4 * ln);
    };

    uint32_t nib_mask = kLowNibbles, high_mask = kHighNibbles, magic = kExact ? 0x43004300u : kHalf1024;
    asm volatile("" : "+s"(nib_mask));
    asm volatile("" : "+v"(magic));
    if constexpr (MODE == kSmAwqRounded) asm volatile("" : "+s"(high_mask));
    auto exact_operand = [&](uint32_t w) {   // rows (2 v, 2 v + 1) as bf16 (128 + q)
        u32x4 b;
#pragma unroll
        for (int v = 0; v < 4; ++v) b[v] = ((w >> (4 * v)) & nib_mask) | magic;
        return __builtin_bit_cast(bf16x8, b);
    };
    // eight products s q as the sum of two bf16: 8 + 4 bits, exact (the cuts do not round, so nothing carries into the first one)
    auto two_operands = [&](uint32_t w, float s, bf16x8 &high, bf16x8 &rest) {
        uint32_t e = w & 0x0F0F0F0Fu, o = (w >> 4) & 0x0F0F0F0Fu;   // rows 0, 4, 1, 5 and 2, 6, 3, 7
        asm volatile("" : "+v"(e), "+v"(o));
        const uint32_t src[4] = {e, o, e, o};
        u32x4 h, l;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint32_t n = src[v] >> (v < 2 ? 0 : 8);
            const float w0 = static_cast<float>(n & 0xFFu) * s, w1 = static_cast<float>((n >> 16) & 0xFFu) * s;
            const uint32_t b0 = __builtin_bit_cast(uint32_t, w0), b1 = __builtin_bit_cast(uint32_t, w1);
            const float r0 = w0 - __builtin_bit_cast(float, b0 & 0xFFFF0000u), r1 = w1 - __builtin_bit_cast(float, b1 & 0xFFFF0000u);
            h[v] = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
            l[v] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, r1), __builtin_bit_cast(uint32_t, r0), 0x07060302u);
        }
        high = __builtin_bit_cast(bf16x8, h);
        rest = __builtin_bit_cast(bf16x8, l);
    };
    auto operand_a = [&](int stage, int t, int rt) {
        return *reinterpret_cast<const bf16x8 *>(lds + stage + x_lds + (16 * rt + ln) * 256 + (((4 * t + lg) ^ ln) << 4));
    };
    // the sums of x of row tile `wave` of a stage, left for its flush
    auto sum_rows = [&](const bf16x8 (&a)[4], int half) {
        const uint32_t one = 0x3F803F80u;
        const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{one, one, one, one});
        floatx4 s = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; ++t) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], ones, s, 0, 0, 0);
        if (ln == 0) *reinterpret_cast<floatx4 *>(xs_lds + (half * KW + kq) * ROWS + 16 * wq + 4 * lg) = s;
    };
    auto read_sum_operands = [&](int stage, bf16x8 (&a)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) a[t] = operand_a(stage, t, wq);
    };
    const bool sums = kSums && wq < RT;

    floatx4 Y[RT][NT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int c = 0; c < NT; ++c) Y[rt][c] = floatx4{0.f, 0.f, 0.f, 0.f};

    // The first steps are requested; past the slice's end its last group once more (into a stage that nobody reads again).
    const int g_wave = g_lo + kq, g_last = g_hi - 1;
    constexpr bool kEarly = MODE >= kSmAwqRounded && R < 4 && TWO;   // (2 x 1 and 3 x 1 tiles have four stages: 1 to 4 % slower with it)
    constexpr int kFirst = kAhead || kEarly ? R : R - 1;
#pragma unroll
    for (int i = 0; i < kFirst; ++i) request(min(g_wave + i * KW, g_last), i * kStage);
    // VALU instructions, LDS reads and copies of a K-step
    auto interleave = [&](auto products, auto valu, auto reads, auto copies) {
        constexpr int P = decltype(products)::value;
        sm_interleave<P, decltype(valu)::value, decltype(reads)::value, decltype(copies)::value>(std::make_integer_sequence<int, P>());
    };

    int stage = 0;
    if constexpr (kAhead) {
        // Products of K-step t from one side of a and b, while the other one is made.  A group's accumulators are flushed beside the first products of the next, and
        // its sums of x are taken by four waves, row tiles wq and wq + 4 each.  Between K-steps 2 and 3 the next group has landed for everybody, and nobody
        // reads this one any more: its stage is filled from there on.
        constexpr int ST = (RT + 3) / 4, P = RT * NT;
        const uint32_t one = 0x3F803F80u;
        const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{one, one, one, one});
        const floatx4 zero = floatx4{0.f, 0.f, 0.f, 0.f};
        floatx4 acc[RT][NT], xs[RT];
        bf16x8 a[2][RT], b[2][NT], as[ST][4];
        u32x4 cell[NT];
        uint32_t word[NT];
        float sc[NT], nz[NT];
        int half = 0;
        auto read_a = [&](int at, int t, int side) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) a[side][rt] = operand_a(at, t, rt);
        };
        auto read_next = [&](int at) {   // cells, words and what the sums are taken of
#pragma unroll
            for (int c = 0; c < NT; ++c) cell[c] = cell_at(at, c), word[c] = word_at(at, c, 0);
#pragma unroll
            for (int i = 0; i < ST; ++i)
#pragma unroll
                for (int t = 0; t < 4; ++t) as[i][t] = operand_a(at, t, min(wq + 4 * i, RT - 1));
        };
        auto dequant = [&](int t, int side) {
#pragma unroll
            for (int c = 0; c < NT; ++c) b[side][c] = exact_operand(cell[c][t]);
        };
        auto products = [&](int t) {
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t & 1][rt], b[t & 1][c], t ? acc[rt][c] : zero, 0, 0, 0);
        };
        auto sums_at = [&](int rt) { return reinterpret_cast<floatx4 *>(xs_lds + (half * KW + kq) * ROWS + 16 * rt + 4 * lg); };   // register i of lane group lg is row 16 rt + 4 lg + i
        auto sum_rows = [&]() {
#pragma unroll
            for (int i = 0; i < ST; ++i) {
                floatx4 s = zero;
#pragma unroll
                for (int t = 0; t < 4; ++t) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as[i][t], ones, s, 0, 0, 0);
                *sums_at(min(wq + 4 * i, RT - 1)) = s;   // (the same from every column, and from every wave that takes the tile)
            }
        };
        auto flush = [&](const floatx4 (&x)[RT]) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int c = 0; c < NT; ++c)
#pragma unroll
                    for (int i = 0; i < 4; ++i) Y[rt][c][i] = fmaf(sc[c], fmaf(nz[c], x[rt][i], acc[rt][c][i]), Y[rt][c][i]);
        };
        auto scales = [&]() {
#pragma unroll
            for (int c = 0; c < NT; ++c) sc[c] = __builtin_bit_cast(float, word[c] << 16), nz[c] = __builtin_bit_cast(float, word[c] & 0xFFFF0000u);
        };
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            xs[rt] = zero;
#pragma unroll
            for (int c = 0; c < NT; ++c) acc[rt][c] = zero;
        }
#pragma unroll
        for (int c = 0; c < NT; ++c) sc[c] = nz[c] = 0.f;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * V) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read_next(0);
        read_a(0, 0, 0);
        dequant(0, 0);
        const int whole = (g_hi - g_lo) / KW;   // steps in which every set of four waves has a group
        for (int step = 0; step < whole; ++step) {
            const int next = stage == (R - 1) * kStage ? 0 : stage + kStage, gn = min(g_wave + (step + R) * KW, g_last);
#pragma unroll
            for (int j = 0; j < RT; ++j) asm volatile("" : "+v"(xoff[j]));
            __builtin_amdgcn_sched_barrier(0);
            flush(xs);
            read_a(stage, 1, 1);
            dequant(1, 1);
            products(0);
            sum_rows();
            interleave(std::integral_constant<int, P + 4 * ST>(), std::integral_constant<int, 7 * NT + 8 * P>(), std::integral_constant<int, RT>(), std::integral_constant<int, 0>());
            __builtin_amdgcn_sched_barrier(0);
            read_a(stage, 2, 0);
            dequant(2, 0);
            products(1);
            interleave(std::integral_constant<int, P>(), std::integral_constant<int, 7 * NT>(), std::integral_constant<int, RT>(), std::integral_constant<int, 0>());
            __builtin_amdgcn_sched_barrier(0);
            read_a(stage, 3, 1);
            dequant(3, 1);
            products(2);
            interleave(std::integral_constant<int, P>(), std::integral_constant<int, 7 * NT>(), std::integral_constant<int, RT>(), std::integral_constant<int, 0>());
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((R - 2) * V) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            scales();
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) xs[rt] = *sums_at(rt);
            read_next(next);
            read_a(next, 0, 0);
            dequant(0, 0);
            products(3);
            request(gn, stage);
            interleave(std::integral_constant<int, P>(), std::integral_constant<int, 9 * NT>(), std::integral_constant<int, 2 * RT + 2 * NT + 4 * ST>(), std::integral_constant<int, V>());
            __builtin_amdgcn_sched_barrier(0);
            stage = next;
            half ^= 1;
        }
        flush(xs);
        // the groups that are not a whole step: a set's own sums of x
        if (g_wave + whole * KW < g_hi) {
            floatx4 own[RT];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) own[rt] = zero;
            scales();
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t > 0) {
                    read_a(stage, t, t & 1);
                    dequant(t, t & 1);
                }
                products(t);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) own[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t & 1][rt], ones, own[rt], 0, 0, 0);
            }
            flush(own);
        }
    } else if constexpr (MODE >= kSmAwqRounded) {
        static_assert(kEarly || R >= 3, "a group lands while another is multiplied");
        // Products of K-step t from one side of a and b, while the other one is made.  Between K-steps 1 and 2 the next group has landed for everybody, and nobody
        // reads the one before this any more (kEarly: this one), whose stage is filled from there on.
        bf16x8 a[kEarly ? 4 : 2][RT], b[2][NT];
        u32x4 cell[NT];
        uint32_t word[NT][Q4 ? 4 : 1];
        AwqScale d[NT];
        auto read_a = [&](int at, int t, int side) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) a[side][rt] = operand_a(at, t, rt);
        };
        auto read_w = [&](int at) {
#pragma unroll
            for (int c = 0; c < NT; ++c) cell[c] = cell_at(at, c);
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int t = 0; t < (Q4 ? 4 : 1); ++t) word[c][t] = word_at(at, c, t);
        };
        auto scales = [&]() {
            if constexpr (!Q4) {
#pragma unroll
                for (int c = 0; c < NT; ++c) d[c] = awq_scale(word[c][0]);
            }
        };
        uint32_t last[NT], last_word[NT];   // of K-step 3, while the next group's are read
        auto keep_last = [&]() {
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                last[c] = cell[c][3];
                asm volatile("" : "+v"(last[c]));
                if constexpr (Q4) {
                    last_word[c] = word[c][Q4 ? 3 : 0];
                    asm volatile("" : "+v"(last_word[c]));
                }
            }
        };
        auto dequant = [&](int t, int side) {
#pragma unroll
            for (int c = 0; c < NT; ++c) {
                const uint32_t v = t == 3 ? last[c] : cell[c][t];
                if constexpr (Q4) {
                    float s, low;
                    decode_md_q4(t == 3 ? last_word[c] : word[c][t], s, low);
                    b[side][c] = dequant_operand(v, s, low);
                } else {
                    b[side][c] = dequant_operand_awq(v, d[c], nib_mask, high_mask, magic);
                }
            }
        };
        auto products = [&](int t) {
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) Y[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kEarly ? t : t & 1][rt], b[t & 1][c], Y[rt][c], 0, 0, 0);
        };
        constexpr int kDq = NT * (Q4 ? 25 : 17);
        constexpr std::integral_constant<int, RT * NT> P;
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kFirst - 1) * V) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        read_w(0);
        read_a(0, 0, 0);
        scales();
        dequant(0, 0);
        for (int g = g_lo; g < g_hi; ++g) {
#pragma unroll
            for (int j = 0; j < RT; ++j) asm volatile("" : "+v"(xoff[j]));
            const int fill = kEarly ? stage : stage == 0 ? (R - 1) * kStage : stage - kStage, next = stage == (R - 1) * kStage ? 0 : stage + kStage;
            const int gn = min(g + kFirst, g_last);
            __builtin_amdgcn_sched_barrier(0);
            read_a(stage, 1, 1);
            if constexpr (kEarly) read_a(stage, 2, 2);
            dequant(1, 1);
            products(0);
            interleave(P, std::integral_constant<int, kDq>(), std::integral_constant<int, kEarly ? 2 * RT : RT>(), std::integral_constant<int, 0>());
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (kEarly) read_a(stage, 3, 3);
            else read_a(stage, 2, 0);
            dequant(2, 0);
            keep_last();
            products(1);
            interleave(P, std::integral_constant<int, kDq>(), std::integral_constant<int, RT>(), std::integral_constant<int, 0>());
            __builtin_amdgcn_sched_barrier(0);
            // the next group has landed for everybody, and nobody reads the stage to fill any more
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((kFirst - 2) * V) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if constexpr (!kEarly) read_a(stage, 3, 1);
            read_w(next);
            dequant(3, 1);
            products(2);
            request_x(gn, fill, 0, RT);
            interleave(P, std::integral_constant<int, kDq>(), std::integral_constant<int, (kEarly ? 0 : RT) + NT * (Q4 ? 5 : 2)>(), std::integral_constant<int, RT>());
            __builtin_amdgcn_sched_barrier(0);
            read_a(next, 0, 0);
            scales();
            dequant(0, 0);
            products(3);
            request_w(gn, fill);
            interleave(P, std::integral_constant<int, kDq + (Q4 ? 0 : 4 * NT)>(), std::integral_constant<int, RT>(), std::integral_constant<int, NT + MC>());
            __builtin_amdgcn_sched_barrier(0);
            stage = next;
        }
    } else {
        int half = 0;
        // One group.  A wave's LDS reads are in flight long before their products: everything at the head of the group where there are
        // registers for it (four row tiles or less), else the operands of a K-step while the one before it multiplies.
        constexpr int AHEAD = RT <= 4 ? 4 : 2;
        auto multiply = [&](int half, int stage, int next) {
            u32x4 cell[NT];
            uint32_t word[NT][Q4 ? 4 : 1];
            bf16x8 a[AHEAD][RT], as[4];
#pragma unroll
            for (int c = 0; c < NT; ++c) cell[c] = cell_at(stage, c);
#pragma unroll
            for (int t = 0; t < (AHEAD == 4 ? 4 : 1); ++t)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) a[t][rt] = operand_a(stage, t, rt);
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int t = 0; t < (Q4 ? 4 : 1); ++t) word[c][t] = word_at(stage, c, t);
            __builtin_amdgcn_sched_barrier(0);
            floatx4 acc[RT][NT], own[RT];
            if constexpr (kExact && !kSums) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) own[rt] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
            if constexpr (MODE == kSmAwq) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int c = 0; c < NT; ++c) acc[rt][c] = floatx4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if constexpr (AHEAD == 2) {
                    if (t < 3) {
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) a[(t + 1) & 1][rt] = operand_a(stage, t + 1, rt);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                if (t == 2 && sums) read_sum_operands(next, as);
                if constexpr (kExact && !kSums) {
                    const uint32_t one = 0x3F803F80u;
                    const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{one, one, one, one});
#pragma unroll
                    for (int rt = 0; rt < RT; ++rt) own[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t % AHEAD][rt], ones, own[rt], 0, 0, 0);
                }
#pragma unroll
                for (int c = 0; c < NT; ++c) {
                    const bf16x8(&at)[RT] = a[t % AHEAD];
                    if constexpr (MODE == kSmAwq) {
                        const bf16x8 b = exact_operand(cell[c][t]);
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) acc[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[rt], b, acc[rt][c], 0, 0, 0);
                    } else {
                        bf16x8 high, rest;
                        two_operands(cell[c][t], __builtin_bit_cast(float, word[c][t] << 16), high, rest);
                        const uint32_t min2 = __builtin_amdgcn_perm(word[c][t], word[c][t], 0x03020302u);
                        const bf16x8 low8 = __builtin_bit_cast(bf16x8, u32x4{min2, min2, min2, min2});
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) Y[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[rt], high, Y[rt][c], 0, 0, 0);
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) Y[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[rt], rest, Y[rt][c], 0, 0, 0);
#pragma unroll
                        for (int rt = 0; rt < RT; ++rt) Y[rt][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(at[rt], low8, Y[rt][c], 0, 0, 0);
                    }
                }
                if (AHEAD == 2) __builtin_amdgcn_sched_barrier(0);
            }
            if (sums) sum_rows(as, half ^ 1);
            if constexpr (MODE == kSmAwq) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {   // register i of lane group lg is row 16 rt + 4 lg + i
                    const floatx4 xs = kSums ? *reinterpret_cast<const floatx4 *>(xs_lds + (half * KW + kq) * ROWS + 16 * rt + 4 * lg) : own[rt];
#pragma unroll
                    for (int c = 0; c < NT; ++c) {
                        const float sc = __builtin_bit_cast(float, word[c][0] << 16), nz = __builtin_bit_cast(float, word[c][0] & 0xFFFF0000u);
#pragma unroll
                        for (int i = 0; i < 4; ++i) Y[rt][c][i] = fmaf(sc, fmaf(nz, xs[i], acc[rt][c][i]), Y[rt][c][i]);
                    }
                }
            }
        };

        if (kSums) {
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((R - 1) * V - RT) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            bf16x8 as[4];
            if (sums) {
                read_sum_operands(0, as);
                sum_rows(as, 0);
            }
        }

        for (int g0 = g_lo; g0 < g_hi; g0 += KW) {
            // This step's requests and, for the sums, the next step's x have landed (younger ones: R - 2 steps, less that x); this wave is done
            // with the step before, and behind the barrier so is everybody.
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kSums ? (R - 2) * V - RT : (R - 2) * V) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int j = 0; j < RT; ++j) asm volatile("" : "+v"(xoff[j]));
            const int fill = stage == 0 ? (R - 1) * kStage : stage - kStage, next = stage == (R - 1) * kStage ? 0 : stage + kStage;
            request(min(g0 + kq + (R - 1) * KW, g_last), fill);
            __builtin_amdgcn_sched_barrier(0);
            if (KW == 1 || g0 + kq < g_hi) multiply(half, stage, next);
            stage = next;
            half ^= 1;
        }
    }

    // Scales from 2^117 on (wsdequant.h): the wave's columns once more, a tile at a time in the same order, operand by operand from memory, in place of what it stores.  (21 forms and
    // 5 sizes against the kernel without: 0.96 to 1.05, 1.002 on average; with two tiles side by side in registers, behind the loop, 6 x 2 and 7 x 2 tiles 1.04 to 1.10.)
    bool over = false;
    auto again = [&](int rt, int c) {
        typedef const __attribute__((address_space(1))) uint32_t *Word;
        const gptr tile = (gptr)(w + (size_t)min(first + c, ntiles - 1) * tile_bytes);
        const uint16_t *x = p.x + (size_t)(m0 + min(16 * rt + ln, rows - 1)) * p.K + 8 * lg;
        floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int k = 4 * g_lo; k < 4 * g_hi; ++k) {   // K-steps
            const int g = k >> 2;
            const uint32_t blk = (uint32_t)(g >> 4) * (uint32_t)((kWsBlockGroups + kMd) * kWsCellBytes);
            const uint32_t cell = lane16 + blk + (uint32_t)(kMd + (g & 15)) * (uint32_t)kWsCellBytes + 4 * (k & 3), word = 16 * ln + blk + 64 * (g & 12) + 4 * (g & 3);
            float s, low;
            decode_md(*reinterpret_cast<Word>(tile + word), s, low);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8 *>(x + 32 * k), dequant_operand(*reinterpret_cast<Word>(tile + cell), s, low), acc, 0, 0, 0);
        }
        return acc;
    };
    if constexpr (MODE == kSmAwqRounded) {
        static_assert(KW == 1, "a wave has all of K");
#pragma unroll
        for (int c = 0; c < NT; ++c) over |= awq_overflowed(Y[0][c][0], Y[RT - 1][c][0]);
    }

    // The parts of K meet, then the sums leave through LDS, so that a store is whole rows of the workgroup's columns.  (No copy of
    // any wave may still be on its way into it.)
    constexpr int LDP = CW + 4;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if constexpr (KW > 1) {
        floatx4 *parts = reinterpret_cast<floatx4 *>(lds);
        if (kq > 0) {
#pragma unroll
            for (int i = 0; i < RT * NT; ++i) parts[((wave - 4) * RT * NT + i) * 64 + lane] = Y[i / NT][i % NT];
        }
        __syncthreads();
        if (kq == 0) {
#pragma unroll
            for (int k = 1; k < KW; ++k)
#pragma unroll
                for (int i = 0; i < RT * NT; ++i) Y[i / NT][i % NT] += parts[((4 * (k - 1) + wq) * RT * NT + i) * 64 + lane];
        }
        __syncthreads();
    }
    float *yt = reinterpret_cast<float *>(lds);
    if (kq == 0) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int c = 0; c < NT; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) yt[(16 * rt + 4 * lg + i) * LDP + (NT * wq + c) * kWsTileCols + ln] = Y[rt][c][i];
    }
    if constexpr (MODE == kSmAwqRounded) {
        if (__ballot(over)) {
#pragma unroll 1
            for (int n = 0; n < RT * NT; ++n) {
                const int rt = n / NT, c = n % NT;
                const floatx4 acc = again(rt, c);
#pragma unroll
                for (int i = 0; i < 4; ++i) yt[(16 * rt + 4 * lg + i) * LDP + (NT * wq + c) * kWsTileCols + ln] = acc[i];
            }
        }
    }
    __syncthreads();
    const int col0 = set * CW, ncols = min(CW, p.N - col0);   // a multiple of 16
    for (int i = tid; i < rows * (CW / 4); i += kThreads) {
        const int row = i / (CW / 4), col = i % (CW / 4) * 4;
        if (col >= ncols) continue;
        floatx4 v = *reinterpret_cast<const floatx4 *>(yt + row * LDP + col);
        const size_t at = (size_t)(m0 + row) * p.N + col0 + col;
        if (p.slices > 1) {
            const int part = MODE >= kSmAwqRounded ? (p.w2 ? 2 * slice + second : slice) : slice;
            *reinterpret_cast<floatx4 *>(p.partial + (size_t)part * p.M * p.N + at) = v;
            continue;
        }
        if (p.residual) {
            const uint2 q = *reinterpret_cast<const uint2 *>(p.residual + at);
            if constexpr (MODE >= kSmAwqRounded) {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = bf16_bits_to_float(float_to_bf16_bits(v[i]));
            }
            v[0] += bf16_bits_to_float(q.x & 0xFFFFu), v[1] += bf16_bits_to_float(q.x >> 16);
            v[2] += bf16_bits_to_float(q.y & 0xFFFFu), v[3] += bf16_bits_to_float(q.y >> 16);
        }
        *reinterpret_cast<uint2 *>((second ? p.y2 : p.y) + at) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    }
}

// y = bf16(sum over the slices, in slice order (+ residual)); four columns per thread.  With their loads in flight together, not in turn, the whole of 64 x 14336 x 4096 in 4 slices
// takes 18.6 us instead of 19.5, in 8 18.8 instead of 19.6, and 100 x 8192 x 2048 in 8 15.8 instead of 16.7.  ROUNDED: the residual is added to the rounded sum.
template <int AT, bool ROUNDED>
__global__ void __launch_bounds__(256) gemm_wsm_sum_kernel(const float *__restrict__ partial, const uint16_t *__restrict__ residual,
                                                           uint16_t *__restrict__ y, size_t mn, int slices) {
    const size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (at >= mn) return;
    uint2 r = uint2{0u, 0u};
    if (residual) r = *reinterpret_cast<const uint2 *>(residual + at);
    floatx4 s = sum_parts<AT>(partial + at, mn, slices);
    if (residual) {
        if constexpr (ROUNDED) s = rounded4(s);
        s += widen4(r);
    }
    *reinterpret_cast<uint2 *>(y + at) = narrow4(s);
}

// What the tiled prompt kernel does to a bf16 product where it stores it, as launches of their own (2 to 5 us): its tiles of 256 rows leave few rows most of the chip idle, and these kernels'
// narrower ones, cut along K besides, have no columns' partners at hand.  A layer of 4096 x 14336, 40 rows, projections / O / gate and up / down: 56 / 16 / 61 / 75 us in the tiled
// kernel, 16 / 14 / 32 / 19 with these launches (under the profiler); four such layers and the head 835 -> 393 us, of 3 rows 1369 -> 328, 100 rows 916 -> 536, 300 rows 1195 -> 979.
// Half-split RoPE on the heads of the first `rope_cols` columns; a thread has four columns of a head's lower half and the four they pair with.  AT = 0: in place.
template <int AT>
__global__ void __launch_bounds__(256) gemm_wsm_rope_kernel(const float *__restrict__ partial, int slices, const uint16_t *__restrict__ lut, uint16_t *y, int M, int N, int cols,
                                                            int rope_cols, int hd, int pos0) {
    const int half = hd >> 1, quads = half >> 2, per_row = cols / hd * quads;
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int m = (int)(t / per_row), q = (int)(t % per_row), i = q % quads * 4, col = q / quads * hd + i;
    if (m >= M) return;
    const size_t at = (size_t)m * N + col;
    const uint16_t *angles = lut + (size_t)(pos0 + m) * hd + i;
    const floatx4 cs = widen4(*reinterpret_cast<const uint2 *>(angles)), sn = widen4(*reinterpret_cast<const uint2 *>(angles + half));
    floatx4 lo, hi;
    if constexpr (AT > 0) {
        lo = rounded4(sum_parts<AT>(partial + at, (size_t)M * N, slices));
        hi = rounded4(sum_parts<AT>(partial + at + half, (size_t)M * N, slices));
    } else {
        lo = widen4(*reinterpret_cast<const uint2 *>(y + at));
        hi = widen4(*reinterpret_cast<const uint2 *>(y + at + half));
    }
    if (col < rope_cols) {
        const floatx4 x = lo, z = hi;
#pragma unroll
        for (int e = 0; e < 4; ++e) lo[e] = x[e] * cs[e] - z[e] * sn[e], hi[e] = z[e] * cs[e] + x[e] * sn[e];
    }
    *reinterpret_cast<uint2 *>(y + at) = narrow4(lo);
    *reinterpret_cast<uint2 *>(y + at + half) = narrow4(hi);
}

// h = bf16(silu(bf16 gate) * bf16 up) from both products' parts, or (AT = 0) from the products, `gate` and what is in h
template <int AT>
__global__ void __launch_bounds__(256) gemm_wsm_swiglu_kernel(const float *__restrict__ partial, int slices, const uint16_t *__restrict__ gate, uint16_t *h, size_t mn) {
    const size_t at = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (at >= mn) return;
    floatx4 g, u;
    if constexpr (AT > 0) {
        g = rounded4(sum_parts<AT>(partial + at, 2 * mn, slices));
        u = rounded4(sum_parts<AT>(partial + mn + at, 2 * mn, slices));
    } else {
        g = widen4(*reinterpret_cast<const uint2 *>(gate + at));
        u = widen4(*reinterpret_cast<const uint2 *>(h + at));
    }
    floatx4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = gated_f32(g[e], g[e]) * u[e];
    *reinterpret_cast<uint2 *>(h + at) = narrow4(v);
}

// f(parts asked for at a time)
template <class F>
void parts_at_a_time(int slices, F f) {
    if (slices <= 2) f(std::integral_constant<int, 2>());
    else if (slices <= 4) f(std::integral_constant<int, 4>());
    else f(std::integral_constant<int, 8>());
}

template <int RT, int NT, int KW, int MODE, bool TWO>
hipError_t launch_wsm(const SmArgs &p, hipStream_t stream) {
    constexpr bool Q4 = MODE == kSmQ4 || MODE == kSmQ4Rounded;
    constexpr size_t ring = (size_t)sm_ring(RT, NT, KW, Q4, TWO) * sm_stage(RT, NT, KW, Q4) + sm_sums(RT, KW, Q4);
    constexpr size_t out = (size_t)16 * RT * (64 * NT + 4) * sizeof(float), parts = (size_t)(KW - 1) * 4 * RT * NT * 1024;
    constexpr size_t lds = ring > out ? (ring > parts ? ring : parts) : out > parts ? out : parts;
    static_assert(lds <= kSmLds, "fits LDS");
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_wsm_kernel<RT, NT, KW, MODE, TWO>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    if ((p.blocks - 1) * 16 * RT >= p.M || p.blocks * 16 * RT < p.M) return hipErrorInvalidValue;   // every block has rows, every row a block
    const int total = p.sets * p.slices * p.blocks;
    hipLaunchKernelGGL((gemm_wsm_kernel<RT, NT, KW, MODE, TWO>), dim3((total + 7) / 8 * 8), dim3(256 * KW), lds, stream, p);
    return hipGetLastError();
}

// Four groups to a step for the smallest row tiles, whose waves have least to do in one.
template <int NT, int MODE>
hipError_t launch_wsm_exact(int rt, const SmArgs &p, hipStream_t stream) {
    switch (rt) {
        case 2: return launch_wsm<2, NT, 4, MODE, false>(p, stream);
        case 3: return launch_wsm<3, NT, 2, MODE, false>(p, stream);
        case 4: return launch_wsm<4, NT, 2, MODE, false>(p, stream);
        case 5: return launch_wsm<5, NT, 2, MODE, false>(p, stream);
        case 6: return launch_wsm<6, NT, 2, MODE, false>(p, stream);
        case 7: return launch_wsm<7, NT, 2, MODE, false>(p, stream);
        default: return hipErrorInvalidValue;
    }
}

// Forms of products of rounded weights (KW = 1: the sums in one order).  `two`: two workgroups to a CU.  For AWQ and Q4NX the microseconds that a workgroup takes besides its groups,
// that a group takes one that is alone, what is added with every CU full, and with just more workgroups than CUs.  Fitted to 1200 products in a graph with every form (17 .. 1600
// rows, K and N 1024 .. 14336; half of them on weights from memory, which takes the forms of few tiles up to a tenth longer): rms error 4 to 5 %, the form it picks takes 0.2 to 0.7 % more
// than the best of them on average.  (3 x 3 tiles, and 4 x 3 by two workgroups, are never more than 1 % faster than all others.)
struct SmForm {
    int rt, nt;
    bool two;
    float each[2], alone[2], more[2], half[2];
};
constexpr SmForm kSmForms[] = {{4, 3, false, {3.93f, 3.87f}, {0.856f, 0.974f}, {0.079f, 0.067f}}, {5, 3, false, {4.49f, 4.59f}, {0.880f, 1.031f}, {0.106f, 0.082f}},
                               {6, 1, false, {2.47f, 2.32f}, {0.497f, 0.542f}, {0.049f, 0.050f}}, {7, 1, false, {2.81f, 2.62f}, {0.521f, 0.563f}, {0.072f, 0.065f}},
                               {5, 2, false, {3.26f, 3.36f}, {0.682f, 0.777f}, {0.077f, 0.065f}}, {6, 2, false, {3.87f, 3.78f}, {0.703f, 0.810f}, {0.090f, 0.074f}},
                               {7, 2, false, {4.22f, 4.21f}, {0.748f, 0.956f}, {0.109f, 0.078f}}, {8, 2, false, {3.72f, 3.38f}, {0.936f, 1.112f}, {0.084f, 0.024f}},
                               {10, 2, false, {4.61f, 4.49f}, {1.019f, 1.163f}, {0.128f, 0.103f}}, {6, 3, false, {4.97f, 4.98f}, {0.916f, 1.125f}, {0.149f, 0.100f}},
                               {7, 3, false, {4.98f, 4.73f}, {1.028f, 1.275f}, {0.154f, 0.077f}}, {2, 1, true, {1.18f, 1.11f}, {0.415f, 0.441f}, {0.021f, 0.034f}, {0.157f, 0.196f}},
                               {3, 1, true, {1.72f, 1.44f}, {0.407f, 0.456f}, {0.200f, 0.206f}, {0.193f, 0.223f}}, {4, 1, true, {1.96f, 1.79f}, {0.437f, 0.484f}, {0.265f, 0.263f}, {0.239f, 0.254f}},
                               {5, 1, true, {2.28f, 2.19f}, {0.479f, 0.500f}, {0.333f, 0.338f}, {0.294f, 0.308f}}, {6, 1, true, {1.93f, 1.36f}, {0.686f, 0.727f}, {0.260f, 0.245f}, {0.180f, 0.224f}},
                               {3, 2, true, {2.46f, 2.44f}, {0.592f, 0.690f}, {0.360f, 0.351f}, {0.355f, 0.406f}}, {4, 2, true, {2.97f, 3.05f}, {0.645f, 0.737f}, {0.414f, 0.445f}, {0.394f, 0.463f}},
                               {6, 2, true, {2.96f, 2.69f}, {0.816f, 0.935f}, {0.499f, 0.504f}, {0.455f, 0.512f}}, {7, 2, true, {3.29f, 3.21f}, {0.876f, 1.017f}, {0.560f, 0.534f}, {0.521f, 0.559f}},
                               {5, 3, true, {3.81f, 3.59f}, {0.942f, 1.191f}, {0.679f, 0.564f}, {0.646f, 0.686f}}};

template <int MODE, size_t... I>
hipError_t launch_wsm_rounded(const WsmPlan &plan, const SmArgs &p, hipStream_t stream, std::index_sequence<I...>) {
    hipError_t e = hipErrorInvalidValue;
    auto one = [&](auto i) {
        constexpr SmForm f = kSmForms[decltype(i)::value];
        if (plan.rt == f.rt && plan.nt == f.nt && plan.two == f.two) e = launch_wsm<f.rt, f.nt, 1, MODE, f.two>(p, stream);
    };
    (one(std::integral_constant<size_t, I>()), ...);
    return e;
}

template <int MODE>
hipError_t launch_wsm_mode(const WsmPlan &plan, const SmArgs &p, hipStream_t stream) {
    if constexpr (MODE >= kSmAwqRounded) return launch_wsm_rounded<MODE>(plan, p, stream, std::make_index_sequence<sizeof(kSmForms) / sizeof(SmForm)>());
    else return plan.nt == 1 ? launch_wsm_exact<1, MODE>(plan.rt, p, stream) : launch_wsm_exact<2, MODE>(plan.rt, p, stream);
}

// The time of a launch on the GPU in microseconds.
// Exact Q4NX: fitted to 1900 timings in a graph (11 matrices from 2432 x 272 to 13056 x 5744, 17 .. 700 rows, every tile, 1 .. 16 slices; rms error 5 %).  Start, a
// workgroup, a step alone on the chip (a1 rt + a2 nt + a3 rt nt), plus (b0 + b1 rt + b2 nt) with every CU busy; a step of four groups costs 1 + four of one of
// two.  The launch that adds up: sum, and per slice `part` and its bytes.
struct SmCost {
    double start, group, a1, a2, a3, b0, b1, b2, four, sum, part, tb_s;
};
constexpr SmCost kSmCostQ4 = {3.79, 1.28, 0.018, 0.422, 0.165, 0.138, 0.019, 0.089, 0.83, 0.60, 0.21, 5.6};
// Exact AWQ: a step's time for each form, fitted to 3000 timings (14 matrices from 1024 x 4096 to 10240 x 8192, 17 .. 128 rows, every form and number of slices;
// rms error 4 %; the plan it picks takes 0.5 % more than the best of them on average, 5 % at worst).  Of 64 rows of 14336 x 4096 in 4 slices start and end are 5.5 us, seven steps 10, the
// parts and their sum 3.6.
struct SmExactForm {
    float alone, more;
};
constexpr SmExactForm kSmExact[2][6] = {{{0.874f, 0.172f}, {0.690f, 0.044f}, {0.827f, 0.023f}, {1.013f, 0.067f}, {1.072f, 0.082f}, {1.256f, 0.116f}},
                                        {{1.208f, 0.206f}, {0.866f, 0.057f}, {1.077f, 0.066f}, {1.336f, 0.085f}, {1.620f, 0.102f}, {2.023f, 0.f}}};   // [nt - 1][rt - 2]
double wsm_rounded_us(const SmForm &f, int blocks, int K, int N, bool q4) {
    const int chip = f.two ? 512 : 256, groups = K / kGroup;
    const long wgs = (long)((N + 64 * f.nt - 1) / (64 * f.nt)) * blocks, full = wgs / chip;
    const double rest = (double)(wgs % chip) / chip;
    double us = (q4 ? 2.01 : 1.80) + full * (f.each[q4] + groups * (f.alone[q4] + f.more[q4]));
    // (two to a CU: from half a round on some CUs have both)
    const double more = !f.two ? f.more[q4] * rest : rest <= 0.5 ? 0.37 * f.more[q4] * rest : f.half[q4] + (q4 ? 0.72 : 0.79) * f.more[q4] * (rest - 0.5);
    if (rest > 0) us += f.each[q4] + groups * (f.alone[q4] + more);
    return us;
}

double wsm_us(const WsmPlan &p, int M, int K, int N, bool q4) {
    const bool four = p.rt <= 2;   // groups to a step
    const int kw = four ? 4 : 2, chip = 256;
    const int groups = (K / kGroup + p.slices - 1) / p.slices, steps = (groups + kw - 1) / kw;
    const long wgs = (long)((N + 64 * p.nt - 1) / (64 * p.nt)) * p.blocks * p.slices, full = wgs / chip;
    const double rest = (double)(wgs % chip) / chip, mb = (double)M * N * 8e-6;   // a part written and read
    if (!q4) {
        const SmExactForm &f = kSmExact[p.nt - 1][p.rt - 2];
        double us = 3.26 + full * (2.24 + steps * (f.alone + f.more));
        if (rest > 0) us += 2.24 + steps * (f.alone + f.more * rest);
        if (p.slices > 1) us += 0.98 + 0.21 * ((p.slices + 7) / 8) + p.slices * mb / 3.52;
        return us;
    }
    const SmCost &c = kSmCostQ4;
    const double alone = c.a1 * p.rt + c.a2 * p.nt + c.a3 * p.rt * p.nt, more = c.b0 + c.b1 * p.rt + c.b2 * p.nt, step = steps * (four ? 1 + c.four : 1.0);
    double us = c.start + full * (c.group + step * (alone + more));
    if (rest > 0) us += c.group + step * (alone + more * rest);
    if (p.slices > 1) us += c.sum + p.slices * (c.part + mb / c.tb_s);
    return us;
}

}  // namespace

size_t gemm_wsm_scratch_bytes(const WsmPlan &p, int M, int N) { return p.slices > 1 ? (size_t)p.slices * M * N * sizeof(float) : 0; }

// Parts of products of rounded weights: within 12 MB, as they are where there are fewer workgroups than the chip takes (512 of 64 x 64 results are 8 MB)
size_t gemm_wsm_parts_bytes(int M, int N) { return M > kWsmSliceRows ? 0 : std::min((size_t)16 * M * N * sizeof(float), (size_t)12 << 20); }

// Slices where few rows leave the chip idle: at least eight groups each, and no more parts than the workspace of a prompt pass has at most (gemm_wsm_parts_bytes); of one
// matrix, from the rows on from which its plain product has rounded weights, only where whole K would take longer than two launches take the host.  So a plain product and the same
// one inside such a pass run the same slices, if the pass has that workspace (with less of it fewer).  Whole K / slices: 297 x 8704 x 1280 36.8 / 19.5 us, 369 x 13568 x 1088 53.7 / 23.5, Q4NX 108 x 8448 x 1664 38.8 / 14.0.
WsmPlan plan_wsm_rounded(int M, int K, int N, int matrices, bool q4, size_t scratch_bytes) {
    const auto &tune = g_gemv_ws_tune;
    const int tiles = (M + 15) / 16;
    WsmPlan best, whole;
    best.us = whole.us = -1;
    double best_rank = 0;   // slices have to be 2 % faster: a second launch and its scratch for nothing
    // a tune key's form, or the tallest of its width where there is none so tall
    int only_rt = tune.wsm_rt, only_nt = tune.wsm_nt;
    if (only_rt || only_nt) {
        int tallest = 0, fits = 0;
        for (const SmForm &f : kSmForms) {
            if (f.nt != (only_nt ? only_nt : f.nt)) continue;
            tallest = std::max(tallest, f.rt);
            if (f.rt >= only_rt && (!fits || f.rt < fits)) fits = f.rt;
        }
        if (only_rt) only_rt = fits ? fits : tallest;
    }
    for (const SmForm &f : kSmForms) {
        if ((only_rt && f.rt != only_rt) || (only_nt && f.nt != only_nt) || (f.rt > 8 && K >= 1 << 23)) continue;   // (the copies' 32-bit offsets)
        if (tune.wsm_two && f.two != (tune.wsm_two == 1) && std::any_of(std::begin(kSmForms), std::end(kSmForms), [&](const SmForm &o) { return o.rt == f.rt && o.nt == f.nt && o.two != f.two; })) continue;
        WsmPlan p;
        p.rt = f.rt, p.nt = f.nt, p.two = f.two, p.blocks = (tiles + f.rt - 1) / f.rt;
        auto fits = [&](int slices) {
            p.slices = slices;
            return slices <= 1 || (K / kGroup / slices >= 8 && M <= kWsmSliceRows &&
                                   gemm_wsm_scratch_bytes(p, M, N * matrices) <= std::min(scratch_bytes, gemm_wsm_parts_bytes(M, N * matrices)));
        };
        const int only = tune.wsm_slices && fits(tune.wsm_slices) ? tune.wsm_slices : 0;
        for (int slices : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (only) slices = only;
            if (!fits(slices)) break;
            p.us = wsm_rounded_us(f, p.blocks * slices * matrices, (K / kGroup + slices - 1) / slices * kGroup, N, q4);
            if (slices > 1) p.us += 0.98 + 0.21 * ((slices + 7) / 8) + slices * matrices * ((double)M * N * 8e-6 / 3.52);
            const double rank = slices > 1 ? 1.02 * p.us : p.us;
            if (best.us < 0 || rank < best_rank) best = p, best_rank = rank;
            if (slices == 1 && (whole.us < 0 || p.us < whole.us)) whole = p;
            if (only) break;
        }
    }
    if (matrices == 1 && M >= gemm_rounded_rows(q4) && best.slices > 1 && whole.us >= 0 && 0.98 * whole.us <= std::max(best.us, kTwoLaunchesUs)) return whole;
    return best;
}

WsmPlan plan_gemm_wsm(int M, int K, int N, bool q4, bool rounded, size_t scratch_bytes) {
    if (rounded) return plan_wsm_rounded(M, K, N, 1, q4, scratch_bytes);
    const auto &tune = g_gemv_ws_tune;
    const int tiles = (M + 15) / 16, G = K / kGroup, most = 7, least = 2, few = (tiles + most - 1) / most;
    const int only_nt = tune.wsm_nt <= 2 ? tune.wsm_nt : 0, only_slices = std::min(tune.wsm_slices ? tune.wsm_slices : tune.splitk == 1 ? 2 : 0, G);
    WsmPlan best;
    best.us = -1;
    double best_rank = 0;   // slices have to be 2 % faster: a second launch and its scratch for nothing
    for (int nt = 1; nt <= 2; ++nt) {
        if (only_nt && nt != only_nt) continue;
        const int options[3] = {few, few + 1, (tiles + 3) / 4};   // blocks of rows
        for (int blocks : options) {
            WsmPlan p;
            p.nt = nt;
            p.rt = std::max((tiles + blocks - 1) / blocks, least);
            if (tune.wsm_rt) p.rt = std::min(std::max(tune.wsm_rt, least), most);
            p.blocks = (tiles + p.rt - 1) / p.rt;
            auto try_slices = [&](int slices) {   // false: no room for so many
                p.slices = slices;
                if (slices > 1 && gemm_wsm_scratch_bytes(p, M, N) > scratch_bytes) return false;
                p.us = wsm_us(p, M, K, N, q4);
                const double rank = slices > 1 ? 1.02 * p.us : p.us;
                if (best.us < 0 || rank < best_rank) best = p, best_rank = rank;
                return true;
            };
            if (only_slices > 1 && try_slices(only_slices)) continue;
            for (int slices : {1, 2, 3, 4, 6, 8, 12, 16})
                if ((slices > 1 && (only_slices || G / slices < 2)) || !try_slices(slices)) break;
        }
    }
    return best;
}

bool gemm_wsm_supported(int M, int K, int N) { return M > 16 && K > 0 && K % kGroup == 0 && K < 1 << 24 && N > 0 && N % kWsTileCols == 0; }

// (a second matrix: rounded weights; both products' parts, or each to its own y)
static hipError_t launch_wsm_products(const WsmPlan &plan, const uint16_t *x, const void *w, const void *w2, uint16_t *y, uint16_t *y2, const uint16_t *residual, float *scratch, int M,
                                      int K, int N, bool q4, bool rounded, hipStream_t stream) {
    SmArgs p;
    p.x = x;
    p.w = static_cast<const char *>(w), p.w2 = static_cast<const char *>(w2);
    p.partial = scratch;
    p.y = y, p.y2 = y2;
    p.residual = residual;
    p.M = M, p.K = K, p.N = N, p.G = K / kGroup, p.NB = ws_blocks(K);
    if (M < 1 || !gemm_wsm_supported(std::max(M, 17), K, N) || (w2 && !rounded)) return hipErrorInvalidValue;   // (the smallest products have other kernels, not other limits)
    p.own_sets = (N + 64 * plan.nt - 1) / (64 * plan.nt);
    p.sets = w2 ? 2 * p.own_sets : p.own_sets;
    p.slices = plan.slices, p.blocks = plan.blocks;
    if (plan.slices > 1 && !scratch) return hipErrorInvalidValue;
    return q4 ? (rounded ? launch_wsm_mode<kSmQ4Rounded>(plan, p, stream) : launch_wsm_mode<kSmQ4>(plan, p, stream))
              : (rounded ? launch_wsm_mode<kSmAwqRounded>(plan, p, stream) : launch_wsm_mode<kSmAwq>(plan, p, stream));
}

hipError_t launch_gemm_wsm(const WsmPlan &plan, const uint16_t *x, const void *w, uint16_t *y, const uint16_t *residual, float *scratch, int M, int K, int N,
                           bool q4, bool rounded, hipStream_t stream) {
    const hipError_t e = launch_wsm_products(plan, x, w, nullptr, y, nullptr, residual, scratch, M, K, N, q4, rounded, stream);
    if (e != hipSuccess || plan.slices == 1) return e;
    const size_t mn = (size_t)M * N;   // N % 16 == 0: whole groups of four columns
    parts_at_a_time(plan.slices, [&](auto at) {
        constexpr int AT = decltype(at)::value;
        hipLaunchKernelGGL((rounded ? &gemm_wsm_sum_kernel<AT, true> : &gemm_wsm_sum_kernel<AT, false>), dim3((unsigned)((mn / 4 + 255) / 256)), dim3(256), 0, stream, scratch, residual, y, mn,
                           plan.slices);
    });
    return hipGetLastError();
}

hipError_t launch_gemm_wsm_rope(const WsmPlan &plan, const uint16_t *x, const void *w, uint16_t *y, const uint16_t *lut, const GemmRope &rope, float *scratch, int M, int K, int N,
                                bool q4, hipStream_t stream) {
    if (rope.head_dim % 8 || rope.head_dim <= 0 || rope.cols % rope.head_dim || N % rope.head_dim) return hipErrorInvalidValue;
    const hipError_t e = launch_wsm_products(plan, x, w, nullptr, y, nullptr, nullptr, scratch, M, K, N, q4, true, stream);
    if (e != hipSuccess) return e;
    const int cols = plan.slices > 1 ? N : rope.cols;
    const unsigned grid = (unsigned)(((size_t)M * (cols / 8) + 255) / 256);
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, stream, scratch, plan.slices, lut, y, M, N, cols, rope.cols, rope.head_dim, rope.pos0); };
    if (plan.slices == 1) run(&gemm_wsm_rope_kernel<0>);
    else parts_at_a_time(plan.slices, [&](auto at) { run(&gemm_wsm_rope_kernel<decltype(at)::value>); });
    return hipGetLastError();
}

hipError_t launch_gemm_wsm_swiglu(const WsmPlan &plan, const uint16_t *x, const void *w_gate, const void *w_up, uint16_t *gate, uint16_t *h, float *scratch, int M, int K, int H, bool q4,
                                  hipStream_t stream) {
    const hipError_t e = launch_wsm_products(plan, x, w_gate, w_up, gate, h, nullptr, scratch, M, K, H, q4, true, stream);
    if (e != hipSuccess) return e;
    const size_t mn = (size_t)M * H;
    const unsigned grid = (unsigned)((mn / 4 + 255) / 256);
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, stream, scratch, plan.slices, gate, h, mn); };
    if (plan.slices == 1) run(&gemm_wsm_swiglu_kernel<0>);
    else parts_at_a_time(plan.slices, [&](auto at) { run(&gemm_wsm_swiglu_kernel<decltype(at)::value>); });
    return hipGetLastError();
}

}  // namespace w4a16
