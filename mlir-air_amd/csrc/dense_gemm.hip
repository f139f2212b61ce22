// Products over many rows with dense weights for gfx950: out[M, N] = A[M, K] W[N, K]^T, A and W row-major in the element
// type, fp32 accumulation; plain, or grouped over the experts of a mixture (row tiles from moe_plan_kernel).
//
// Both operands have k contiguous, so a tile of either is a set of rows of 128 bytes per K-step (64 bf16 or 32 floats) and
// goes global -> LDS without passing through registers (global_load_lds_dwordx4): one wave instruction fills 1 KiB, 8 rows, lane l
// writing 16-byte slot l % 8 of row l / 8 and fetching chunk slot ^ row % 8, so that the operand reads of 16 consecutive rows are
// spread over the banks without padding.  W is the first MFMA operand: a lane then holds four consecutive n of one row m.
//
//   dense_gemm_kernel        fp32, few rows, experts with few rows: a ring of STAGES buffers, STAGES - 1 K-steps ahead, one barrier
//                            per K-step, the compiler's own order of reads and products
//   dense_gemm_wide_kernel   bf16 from 128 rows on: one wave per SIMD with 128 x 128 results in AGPRs, every read and copy at its
//                            place between the products
//
// Products with too few tiles for the GPU run in slices along K (blockIdx.y) whose fp32 parts are added afterwards.
//
// Row gathers cost nothing here: every lane of a copy has its own source row.  The waves of a SIMD differ in their rows, so
// that a wave whose rows lie behind the end of an expert's run can leave the matrix pipe to the other.
//
// Requirements: K a multiple of 128 bytes of elements (the loader pads), N of 16.  Rows past M and N are read from the last
// row and never stored.
#include "dense.h"
#include "dense_kernels.h"
#include <type_traits>
#include <utility>

namespace w4a16 {

namespace {

constexpr int kRowBytes = 128;

template <class T>
struct GemmKernelArgs {
    const T *a, *w;
    void *out;
    int M, N, K;
    long lda, ldo;
    const int32_t *tiles, *order;
    int gather;
    long w_stride;
    int tiles_m, tiles_n;
    int silu_begin, silu_end;
    long slice_stride;   // elements between the parts of two slices along K (blockIdx.y); one slice: anything
};

// The K-steps of this workgroup's slice.
struct KSlice {
    int first, steps;
};
__device__ __forceinline__ KSlice k_slice(int steps) {
    const int first = (int)((long)steps * blockIdx.y / gridDim.y);
    return {first, (int)((long)steps * (blockIdx.y + 1) / gridDim.y) - first};
}

// silu on the columns of [silu_begin, silu_end), whole 16-column tiles: ahead of the stores, whose code then is in one piece where a wave has none of
// them.  (Between the stores, 64 jumps over 40 KiB of it: 2048 x 2752 x 2048 without any silu 28.8 us, 27.8 so; 2048 x 11264 x 2048 80.4 / 78.9.)
template <class T, int MT, int NT, int EPI, bool GROUPED>
__device__ __forceinline__ void silu_columns(const GemmKernelArgs<T> &p, floatx4 (&acc)[NT][MT], int n_first) {
    if constexpr (EPI == kOutElem && !GROUPED) {
        if (n_first >= p.silu_end || n_first + 16 * NT <= p.silu_begin) return;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const int n = n_first + 16 * j;
            if (n < p.silu_begin || n >= p.silu_end) continue;
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[j][i][r] = silu_of<T>(acc[j][i][r]);
        }
    }
}

// A wave's block of the result, NT x MT tiles of 16 x 16: a lane holds row ql of every tile and its columns 4 g .. + 3.
template <class T, int MT, int NT, int EPI, bool GROUPED>
__device__ __forceinline__ void store_tile(const GemmKernelArgs<T> &p, floatx4 (&acc)[NT][MT], int m_first, int m_end, int n_first) {
    const int lane = threadIdx.x & 63, ql = lane & 15, g = lane >> 4;
    silu_columns<T, MT, NT, EPI, GROUPED>(p, acc, n_first);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int m = m_first + 16 * i + ql;
        if (m >= m_end) continue;
        size_t row = m;
        if constexpr (GROUPED)
            if (p.gather == 0) row = p.order[m];
        if constexpr (EPI == kOutSwiglu || EPI == kOutGeglu) {
#pragma unroll
            for (int j = 0; j < NT; j += 2) {
                const int n = n_first + 16 * j;
                if (n >= p.N) continue;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = (EPI == kOutGeglu ? gelu_tanh_of<T>(acc[j][i][r]) : silu_of<T>(acc[j][i][r])) * acc[j + 1][i][r];
                store4(static_cast<T *>(p.out) + row * p.ldo + n / 2 + 4 * g, v[0], v[1], v[2], v[3]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int n = n_first + 16 * j + 4 * g;
                if (n >= p.N) continue;
                if constexpr (EPI == kOutF32)
                    store4(static_cast<float *>(p.out) + blockIdx.y * p.slice_stride + row * p.ldo + n, acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]);
                else
                    store4(static_cast<T *>(p.out) + row * p.ldo + n, acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]);
            }
        }
    }
}

// BM x BN tile, WM x WN waves (m x n); GROUPED: expert row tiles
template <class T, int BM, int BN, int WM, int WN, int STAGES, int EPI, bool GROUPED>
__global__ void __launch_bounds__(64 * WM * WN) dense_gemm_kernel(const GemmKernelArgs<T> p) {
    constexpr int NW = WM * WN, KE = kRowBytes / sizeof(T), KS = KE / 32;
    constexpr int MT = BM / WM / 16, NT = BN / WN / 16;
    constexpr int COPIES = (BM + BN) / 8 / NW;
    static_assert((BM + BN) % (8 * NW) == 0, "whole copies per wave");
    constexpr int kStage = (BM + BN) * kRowBytes;
    extern __shared__ __attribute__((aligned(16))) char gemm_lds[];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int ql = lane & 15, g = lane >> 4;

    // An XCD (blockIdx % 8) takes a contiguous range of tiles; in a band of four row panels the columns go by first, so
    // that the workgroups running together on one XCD share both operands in its L2.
    // (Experts: the launch covers the most tiles that there can be, the table's last row says how many there are.)
    const int tiles_m = GROUPED ? p.tiles[4 * p.tiles_m] : p.tiles_m;
    const int total = tiles_m * p.tiles_n, per_xcd = (total + 7) / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= total) return;
    const int band = tile / (4 * p.tiles_n), in_band = tile % (4 * p.tiles_n);
    const int rows_in_band = tiles_m - 4 * band < 4 ? tiles_m - 4 * band : 4;
    const int tm = 4 * band + in_band % rows_in_band, tn = in_band / rows_in_band;

    const T *w = p.w;
    int m0 = tm * BM, m_end = p.M;
    if constexpr (GROUPED) {
        const int32_t *t = p.tiles + 4 * tm;
        w += (size_t)t[0] * p.w_stride;
        m0 = t[1];
        m_end = m0 + t[2];
    }
    const int n0 = tn * BN;

    // copy sources of this lane: row (lane / 8) of the eight rows of copy i, chunk (lane % 8) ^ row % 8
    const char *src[COPIES];
#pragma unroll
    for (int i = 0; i < COPIES; ++i) {
        const int row = 8 * (i * NW + wave) + (lane >> 3);   // row of the stage: A rows, then W rows
        const T *base;
        if (row < BM) {
            int m = m0 + row < m_end ? m0 + row : m_end - 1;
            if constexpr (GROUPED)
                if (p.gather > 0) m = p.order[m] / p.gather;
            base = p.a + (size_t)m * p.lda;
        } else {
            const int n = n0 + row - BM < p.N ? n0 + row - BM : p.N - 1;
            base = w + (size_t)n * p.K;
        }
        src[i] = reinterpret_cast<const char *>(base) + 16 * ((lane & 7) ^ (row & 7));
    }
    auto copy = [&](int buf, int kt) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src[i] + (size_t)kt * kRowBytes),
                                             (__attribute__((address_space(3))) void *)(gemm_lds + buf * kStage + 1024 * (i * NW + wave)), 16, 0, 0);
    };
    auto operand = [&](const char *stage, int row, int ks) -> Vec8<T> {   // 8 consecutive k of a stage row
        const char *r = stage + row * kRowBytes;
        if constexpr (sizeof(T) == 2) {
            return load8(reinterpret_cast<const T *>(r + 16 * ((4 * ks + g) ^ (row & 7))));
        } else {
            Vec8<T> v;
            v.lo = *reinterpret_cast<const floatx4 *>(r + 16 * ((2 * g) ^ (row & 7)));
            v.hi = *reinterpret_cast<const floatx4 *>(r + 16 * ((2 * g + 1) ^ (row & 7)));
            return v;
        }
    };

    floatx4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};

    const KSlice slice = k_slice(p.K / KE);
    const int steps = slice.steps;
#pragma unroll
    for (int i = 0; i < COPIES; ++i) src[i] += (size_t)slice.first * kRowBytes;
    const bool idle = GROUPED && m0 + wm * (BM / WM) >= m_end;
#pragma unroll
    for (int i = 0; i < STAGES - 1; ++i)
        if (i < steps) copy(i, i);
    int buf = 0;
    for (int kt = 0; kt < steps; ++kt) {
        // The copies write LDS behind the compiler's back: step kt's have landed once at most those of the STAGES - 2 steps
        // after it are outstanding; this wave's reads of the step before have returned.  Then, behind the barrier, so have
        // everybody's, and the buffer of the step before can be filled again.
        if (STAGES > 2 && kt + STAGES - 2 < steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * COPIES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int next = buf == 0 ? STAGES - 1 : buf - 1;   // the buffer of the step before = of the step STAGES - 1 ahead
        if (kt + STAGES - 1 < steps) copy(next, kt + STAGES - 1);
        const char *stage = gemm_lds + buf * kStage;
        buf = buf + 1 == STAGES ? 0 : buf + 1;
        if (idle) continue;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            Vec8<T> b[MT], a[NT];
#pragma unroll
            for (int i = 0; i < MT; ++i) b[i] = operand(stage, wm * (BM / WM) + 16 * i + ql, ks);
#pragma unroll
            for (int j = 0; j < NT; ++j) a[j] = operand(stage, BM + wn * (BN / WN) + 16 * j + ql, ks);
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) acc[j][i] = mma32(a[j], b[i], acc[j][i]);
        }
    }

    store_tile<T, MT, NT, EPI, GROUPED>(p, acc, m0 + wm * (BM / WM), m_end, n0 + wn * (BN / WN));
}

// ---- wide tiles, bf16 ------------------------------------------------------------------------------------------------------
// 128 WM rows x 16 NT (4 / WM) columns, four waves WM x 4 / WM, a wave 128 rows x 16 NT columns.
//
// What bounds it: the matrix pipe at the clock that the power limit leaves (1.9 GHz), if nothing else holds the one wave of a SIMD
// up, which issues in order.  A K-step of 256 x 256 is 128 products of 16 cycles a wave, in four quarters: (columns 0 .. 63 | 64 .. 127 of the
// wave) x (k 0 .. 31 | 32 .. 63).  Each quarter's operands are read during the one before it, two products apart; the last quarter
// reads the next K-step's, so the one wait and barrier of a K-step stands in front of it, with the matrix pipe full and the operands of
// 32 products in registers.  Copies: A of K-step t + 2 in the last quarter of t and the first of t + 1, W of t + 3 (three buffers; A has two)
// in the middle ones, evenly: LDS is filled at 64 bytes a cycle, so the 64 KiB of a K-step take half of its 2048 cycles, and copies in
// bursts stopped the products (215 -> 197 us below).
// Two waves per SIMD with 128 x 64 each (the kernel before) read half as much again from LDS: 1536 + 512 cycles of reads and copies for
// 2048 of products.  2048 x 8192 x 8192 236 -> 197 us = 1.39 PFLOP/s, 4096^3 122 -> 100 us = 1.38, 2048 x 16384 x 2048 with gelu 135 -> 106.
// More tiles than CUs: a workgroup takes one after the other, and asks for a tile's first K-steps before it stores the one before (that waited for a workgroup's
// start, its addresses and HBM: 2048 x 16384 x 2048 with gelu, two tiles each, 110.7 -> 108.2 us, 2048 x 11264 x 2048 77.2 -> 75.4, 2048 x 28672 x 4096 with silu 383.7 -> 372.0).
constexpr int kWideThreads = 256, kWideStagesW = 3;
constexpr size_t wide_lds(int wm, int nt) { return (2 * (size_t)(128 * wm) + kWideStagesW * (size_t)(4 / wm * 16 * nt)) * kRowBytes; }

// acc += w a.  Volatile asm: the accumulators stay in their AGPRs and the order of the source is kept.
__device__ __forceinline__ void mfma_in_place(floatx4 &acc, const bf16x8 &w, const bf16x8 &a) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(a));
}
// COLS x 8 products, `behind(n)` issued behind the n-th of them
// (LAST: the last of them are the compiler's, so that what it puts behind the loop, a move of the accumulators say, waits for them)
template <int COLS, bool LAST = false, int W, class F>
__device__ __forceinline__ void quarter(floatx4 (*acc)[8], const bf16x8 (&w)[W], const bf16x8 (&a)[8], F behind) {
#pragma unroll
    for (int n = 0; n < 8 * COLS; ++n) {
        __builtin_amdgcn_sched_barrier(0);
        if (LAST && n >= 8 * COLS - 4) acc[n / 8][n % 8] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[n / 8], a[n % 8], acc[n / 8][n % 8], 0, 0, 0);
        else mfma_in_place(acc[n / 8][n % 8], w[n / 8], a[n % 8]);
        __builtin_amdgcn_sched_barrier(0);
        behind(n);
    }
}
// Which of `items` LDS reads goes behind product n of `products`: every second product has one, or every one where that would run
// into their last quarter.  Which of `items` copies: spread evenly, because the four waves' copies fill LDS at 64 bytes a cycle, 16
// cycles each, and one that finds the path taken holds up its wave's products.  -1: none.
__device__ constexpr int read_behind(int n, int products, int items) {
    const int stride = items * 8 <= products * 3 ? 2 : 1;
    return n % stride == 0 && n / stride < items ? n / stride : -1;
}
__device__ constexpr int copy_behind(int n, int products, int items) {
    const int stride = products / items;
    return n % stride == stride - 1 && n / stride < items ? n / stride : -1;
}
// A wave's NT x MT tiles by way of LDS, 16 rows at a time: what leaves is whole 16-byte pieces, as many rows' side by side as a wave
// has lanes for.  (store_tile's pieces are 8 bytes, 32 together: 2048 x 6656 x 2048 took 61 us with them, 56 with these.)
constexpr int kWideStore = 16 * (16 * 8 + 8) * (int)sizeof(float);   // of a wave: 16 rows and their padding
// SCATTER: rows of the result are entries; without a pair out_rows holds where the wave's rows go, 64 an element, a lane each.
template <int NT, int MT, int EPI, bool GROUPED, bool SCATTER>
__device__ __forceinline__ void store_rows(const GemmKernelArgs<bf16> &p, floatx4 (&acc)[NT][MT], char *lds, int m_first, int m_end, int n_first,
                                           const int (&out_rows)[3] = {0, 0, 0}) {
    typedef typename std::conditional<EPI == kOutF32, float, bf16>::type Out;
    constexpr bool kPair = EPI == kOutSwiglu || EPI == kOutGeglu;
    constexpr int kCols = 16 * NT / (kPair ? 2 : 1), kPiece = 16 / (int)sizeof(Out), kPitch = kCols + kPiece;
    constexpr int kPieces = 16 * kCols / kPiece;   // of 16 rows
    static_assert(16 * kPitch * sizeof(Out) <= kWideStore, "fits the wave's part");
    const int lane = threadIdx.x & 63, ql = lane & 15, g = lane >> 4;
    Out *rows = reinterpret_cast<Out *>(lds);
    const int n_out = kPair ? n_first / 2 : n_first, n_end = kPair ? p.N / 2 : p.N;
    silu_columns<bf16, MT, NT, EPI, GROUPED>(p, acc, n_first);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (m_first + 16 * i >= m_end) break;   // uniform
#pragma unroll
        for (int j = 0; j < NT; j += kPair ? 2 : 1) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = acc[j][i][r];
                if constexpr (kPair) v[r] = (EPI == kOutGeglu ? gelu_tanh_of<bf16>(v[r]) : silu_of<bf16>(v[r])) * acc[j + 1][i][r];
            }
            store4(rows + ql * kPitch + 16 * (kPair ? j / 2 : j) + 4 * g, v[0], v[1], v[2], v[3]);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int t = lane; t < kPieces; t += 64) {
            const int row = t / (kCols / kPiece), col = t % (kCols / kPiece) * kPiece, m = m_first + 16 * i + row;
            size_t to = m;
            if constexpr (SCATTER && !kPair) to = __shfl(out_rows[i / 4], 16 * (i % 4) + row);
            if (m >= m_end || n_out + col >= n_end) continue;
            if constexpr (SCATTER && kPair) to = p.order[m];   // (no product of the mixture)
            const long part = EPI == kOutF32 ? blockIdx.y * p.slice_stride : 0;
            *reinterpret_cast<u32x4 *>(static_cast<Out *>(p.out) + part + to * p.ldo + n_out + col) = *reinterpret_cast<const u32x4 *>(rows + row * kPitch + col);
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// (fp32 rows need more LDS for their stores than is free then; with 256 accumulators and silu on some columns there are no registers for both)
constexpr bool wide_loops(int nt, int epi) { return epi != kOutF32 && !(nt == 8 && epi == kOutElem); }

template <int WM, int NT, int EPI>
__device__ __forceinline__ void wide_tiles(const GemmKernelArgs<bf16> &p, char *lds, int tile, int tiles_end, int stride, KSlice slice) {
    constexpr int WN = 4 / WM, BM = 128 * WM, BN = 16 * NT * WN;
    constexpr int H0 = (NT + 1) / 2, H1 = NT - H0;        // column tiles of the two halves of a wave's columns
    static_assert(H1 >= 2, "room for a quarter's LDS reads");
    constexpr int CA = BM / 32, CW = BN / 32;             // copies of a wave and K-step
    constexpr int CA0 = CA / 2, CW0 = (CW + 1) / 2;
    constexpr int kSideA = BM * kRowBytes, kSideW = BN * kRowBytes;
    static_assert(!wide_loops(NT, EPI) || 4 * (kWideStore / 2) <= kSideW, "rows on their way out fit the buffer that no copy goes to");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int ql = lane & 15, g = lane >> 4;

    // Copy i of a wave fills KiB i of the wave's part of a stage: eight rows, lane's chunk (lane % 8) ^ row % 8.  Four copies share
    // their LDS base (M0) and differ in the instruction's offset, which the hardware adds to both addresses: the source takes it back.
    // (Offsets from the wave's first row, 64 rows at most.)
    uint32_t off_a[CA], off_w[CW];
    gptr base_a, base_w;
    int m0, n0;
    const int m_end = p.M;
    auto place = [&](int tile) {   // where a tile is, and the offsets of its copies; then the copies' bases
        const int band = tile / (4 * p.tiles_n), in_band = tile % (4 * p.tiles_n);
        const int rows_in_band = p.tiles_m - 4 * band < 4 ? p.tiles_m - 4 * band : 4;
        m0 = (4 * band + in_band % rows_in_band) * BM, n0 = in_band / rows_in_band * BN;
        const int m_wave = m0 + 8 * CA * wave < m_end ? m0 + 8 * CA * wave : m_end - 1, n_wave = n0 + 8 * CW * wave < p.N ? n0 + 8 * CW * wave : p.N - 1;
#pragma unroll
        for (int i = 0; i < CA; ++i) {
            const int row = 8 * (CA * wave + i) + (lane >> 3), m = m0 + row < m_end ? m0 + row : m_end - 1;
            off_a[i] = (uint32_t)(m - m_wave) * (uint32_t)(p.lda * sizeof(bf16)) + 16 * ((lane & 7) ^ (row & 7)) + 4096 - 1024 * (i & 3);
        }
#pragma unroll
        for (int i = 0; i < CW; ++i) {
            const int row = 8 * (CW * wave + i) + (lane >> 3), n = n0 + row < p.N ? n0 + row : p.N - 1;
            off_w[i] = (uint32_t)(n - n_wave) * (uint32_t)(p.K * sizeof(bf16)) + 16 * ((lane & 7) ^ (row & 7)) + 4096 - 1024 * (i & 3);
        }
        return int2{m_wave, n_wave};
    };
    auto begin = [&](int2 at) {
        const size_t from = (size_t)slice.first * kRowBytes;
        base_a = scalar_ptr(reinterpret_cast<const char *>(p.a + (size_t)at.x * p.lda) + from - 4096);
        base_w = scalar_ptr(reinterpret_cast<const char *>(p.w + (size_t)at.y * p.K) + from - 4096);
    };
    auto copy = [&](gptr from, int at, int i) {
        const auto *src = (const __attribute__((address_space(1))) void *)from;
        auto *dst = (__attribute__((address_space(3))) void *)(lds + at + 1024 * (i & ~3));
        switch (i & 3) {
            case 0: __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0); break;
            case 1: __builtin_amdgcn_global_load_lds(src, dst, 16, 1024, 0); break;
            case 2: __builtin_amdgcn_global_load_lds(src, dst, 16, 2048, 0); break;
            default: __builtin_amdgcn_global_load_lds(src, dst, 16, 3072, 0); break;
        }
    };
    auto copy_a = [&](int side, int i) { copy(base_a + off_a[i], side + 1024 * CA * wave, i); };
    auto copy_w = [&](int side, int i) { copy(base_w + off_w[i], 2 * kSideA + side + 1024 * CW * wave, i); };

    const int steps = slice.steps;
    auto read = [&](uint32_t at, int i) { return *reinterpret_cast<const bf16x8 *>(lds + at + i * 16 * kRowBytes); };

    // A of K-steps 0 and 1, W of 0, 1 and 2 are on their way when the loop begins (past the end: the last K-step's once more, into
    // a buffer that nobody reads)
    int next_a, next_w;   // K-steps that the sources stand at
    auto step_a = [&]() { return next_a + 1 < steps ? (++next_a, kRowBytes) : 0; };
    auto step_w = [&]() { return next_w + 1 < steps ? (++next_w, kRowBytes) : 0; };
    auto ask = [&] {
        next_a = next_w = 0;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < CW; ++i) copy_w(s * kSideW, i);
            base_w += step_w();
#pragma unroll
            for (int i = 0; i < (s == 0 ? CA : CA0); ++i) copy_a(s * kSideA, i);
            if (s == 0) base_a += step_a();
        }
    };
    begin(place(tile));
    ask();
    for (;;) {
        floatx4 acc[NT][8];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};

        // operand addresses of the two halves (32 k) of a K-step; tile i is the instruction's offset
        uint32_t at_a[2], at_w[2];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const uint32_t o = ql * kRowBytes + 16 * ((4 * ks + g) ^ (ql & 7));
            at_a[ks] = o + wm * 128 * kRowBytes;
            at_w[ks] = o + 2 * kSideA + wn * 16 * NT * kRowBytes;
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(CW + CA0) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");

        // (the zeros have been written when the first product, of which the compiler does not know, adds to them)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            asm volatile("s_nop 1" : "+a"(acc[j][0]), "+a"(acc[j][1]), "+a"(acc[j][2]), "+a"(acc[j][3]), "+a"(acc[j][4]), "+a"(acc[j][5]), "+a"(acc[j][6]), "+a"(acc[j][7]));
        bf16x8 a0[8], a1[8], w0[H0], w1[H0];
#pragma unroll
        for (int i = 0; i < 8; ++i) a0[i] = read(at_a[0], i);
#pragma unroll
        for (int j = 0; j < H0; ++j) w0[j] = read(at_w[0], j);

        int side_a = 0, side_w = 0, fill_w = 2 * kSideW;   // of the K-step that is multiplied; of the one that W is copied for
#pragma unroll 1
        for (int kt = 0; kt < steps; ++kt) {
            // (opaque in this block: the offsets' zero extension folds into the copies only if it is not taken out of the loop)
#pragma unroll
            for (int i = 0; i < CA; ++i) asm volatile("" : "+v"(off_a[i]));
#pragma unroll
            for (int i = 0; i < CW; ++i) asm volatile("" : "+v"(off_w[i]));
            // first columns, first half of the K-step; the other half of A's copies for the next K-step
            quarter<H0>(acc, w0, a0, [&](int n) {
                if (const int r = read_behind(n, 8 * H0, H0 + 8); r >= 0) {
                    if (r < H0) w1[r] = read(at_w[1], r);
                    else a1[r - H0] = read(at_a[1], r - H0);
                }
                if (const int i = copy_behind(n, 8 * H0, CA - CA0); i >= 0) copy_a(side_a ^ kSideA, CA0 + i);
            });
            base_a += step_a();
            // second half; W two K-steps on
            quarter<H0>(acc, w1, a1, [&](int n) {
                if (const int r = read_behind(n, 8 * H0, H1); r >= 0) w0[r] = read(at_w[0], H0 + r);
                if (const int i = copy_behind(n, 8 * H0, CW0); i >= 0) copy_w(fill_w, i);
            });
            // the other columns, first half
            quarter<H1>(acc + H0, w0, a0, [&](int n) {
                if (const int r = read_behind(n, 8 * H1, H1); r >= 0) w1[r] = read(at_w[1], H0 + r);
                if (const int i = copy_behind(n, 8 * H1, CW - CW0); i >= 0) copy_w(fill_w, CW0 + i);
            });
            base_w += step_w();
            __builtin_amdgcn_sched_barrier(0);
            // everything of the next K-step has landed (W of the one after it need not have), everybody has read all of this one
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(CW) : "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const int filled = side_a;
            side_a ^= kSideA;
            const int ahead = side_w == 2 * kSideW ? -2 * kSideW : kSideW;
            side_w += ahead;
            fill_w = fill_w == 2 * kSideW ? 0 : fill_w + kSideW;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                at_a[ks] ^= kSideA;
                at_w[ks] += ahead;
            }
            // second half; A two K-steps on
            quarter<H1, true>(acc + H0, w1, a1, [&](int n) {
                if (const int r = read_behind(n, 8 * H1, H0 + 8); r >= 0) {
                    if (r < H0) w0[r] = read(at_w[0], r);
                    else a0[r - H0] = read(at_a[0], r - H0);
                }
                if (const int i = copy_behind(n, 8 * H1, CA0); i >= 0) copy_a(filled, i);
            });
        }
        // no copy, of any wave, is on its way to LDS any more; the products have left the matrix pipe
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int j = 0; j < NT; ++j)
            asm volatile("" : "+a"(acc[j][0]), "+a"(acc[j][1]), "+a"(acc[j][2]), "+a"(acc[j][3]), "+a"(acc[j][4]), "+a"(acc[j][5]), "+a"(acc[j][6]), "+a"(acc[j][7]));
        const int m_store = m0 + wm * 128, n_store = n0 + wn * 16 * NT;
        tile += stride;
        const bool more = wide_loops(NT, EPI) && tile < tiles_end;
        if (more) {
            begin(place(tile));
            ask();
        }
        // (the third buffer of W, which nothing is on its way to; fp32 rows, of one tile only, need more)
        store_rows<NT, 8, EPI, false, false>(p, acc, lds + (wide_loops(NT, EPI) ? 2 * kSideA + 2 * kSideW + wave * (kWideStore / 2) : wave * kWideStore), m_store, m_end, n_store);
        if (!more) return;
        // the offsets once more, so that they need no registers beside the rows that are stored
        asm volatile("" : "+s"(tile));
        place(tile);
    }
}

template <int WM, int NT, int EPI>
__global__ void __launch_bounds__(kWideThreads, 1) dense_gemm_wide_kernel(const GemmKernelArgs<bf16> p) {
    extern __shared__ __attribute__((aligned(16))) char gemm_lds[];
    const int per_xcd = (p.tiles_m * p.tiles_n + 7) / 8, total = p.tiles_m * p.tiles_n;
    const int first = (blockIdx.x & 7) * per_xcd, end = first + per_xcd < total ? first + per_xcd : total, tile = first + (blockIdx.x >> 3);
    if (tile < end) wide_tiles<WM, NT, EPI>(p, gemm_lds, tile, end, gridDim.x / 8, k_slice(p.K / 64));
}


// ---- experts, bf16 -----------------------------------------------------------------------------------------------------------
// 32 R rows of an expert (R <= 12) x 128 columns, four waves two by two, a wave 16 R rows x 64 columns.
//
// What bounds it: an expert's W is read for its few hundred rows alone, so HBM (W once: 64 experts of 2048 x 2048 take 100 us) as well as the
// matrix pipe, and LDS beside it: a K-step of 256 rows reads 96 KiB and fills 48, 1152 cycles of LDS for 1024 of products.  A workgroup has all of an
// expert's rows where they are 384 or less (else even parts of them), so W leaves HBM once, in
// 128 columns, so that there are many workgroups of even work, and does whole 32-row steps' products only.  (Four waves one below the other, 64-row
// steps: the same reads from LDS at 256 rows, but 32 rows of padding an expert on average instead of 16, multiplied, copied and read.  64 experts
// of 2 x 1024 x 2048 and 1024 x 2048, 16384 entries 196 + 111 -> 191.5 + 108 us; 8 experts of 2 x 1408 x 1024, 600 entries 13.2 + 13.2 -> 12.1 + 11.8.)
// A K-step is two halves of 4 R products of 16 cycles; each half's operands are read during the one before it.  One wait and barrier
// stand between the halves: all of the next K-step has landed, everybody has read all of this one, and the copies of a K-step two or three
// on (buffers: W three, A three up to 256 rows, else two; more of them for few rows were no faster) go out behind the products after it.
// Few rows (plans of 128 to a tile): two workgroups to a CU, whose starts and stores then stand beside each other's products; 80 KiB of LDS and
// 192 registers each.  64 experts of 2 x 1024 x 2048 and 1024 x 2048, one / two to a CU, gate and up, then down: 16 tokens of 8 92 / 84 + 50 / 44 us,
// 128 tokens 100 / 97 + 57 / 53, 512 tokens 108 / 107 + 69 / 62 (32- and 128-row tiles before: 96 + 42, 118 + 54, 137 + 64); 768 tokens, 96 rows an
// expert on average and up to 188, 117 / 138 + 77 / 80, which is where the second reading of W costs more: up to 64 on average.
constexpr int kExpertCols = 128, kExpertRows = 384, kFewRows = 128, kFewMean = 64;
constexpr int kExpertStagesW = 3;
constexpr int expert_stages_a(int r, bool few) { return r <= (few ? 2 : 8) ? 3 : 2; }
constexpr size_t expert_lds(int r, bool few) { return (size_t)(expert_stages_a(r, few) * 32 * r + kExpertStagesW * kExpertCols) * kRowBytes; }
// f(0) .. f(N - 1), the number known to the compiler (which leaves long loops around loops as they are)
template <class F, int... N>
__device__ __forceinline__ void each_of(F &&f, std::integer_sequence<int, N...>) { (f(std::integral_constant<int, N>()), ...); }
template <int N, class F>
__device__ __forceinline__ void each(F &&f) { each_of(f, std::make_integer_sequence<int, N>()); }
// of `items` that are to be spread over the products [0, upto): the first one that goes behind product n or later
__device__ constexpr int items_before(int n, int upto, int items) { return n >= upto ? items : n * items / upto; }

// (LONG: rows of A further apart than 32-bit offsets reach; a 64-bit address a copy, added up in two steps, holds the products up.  4096 tokens of 8
// experts, 64 of 2 x 1024 x 2048 and 1024 x 2048: 308 + 173 us with them, 294 + 166 without.)
template <int R, int EPI, bool SCATTER, bool FEW, bool LONG>
__device__ __forceinline__ void expert_tile(const GemmKernelArgs<bf16> &p, char *lds, const bf16 *w, int m0, int m_end, int n0, int first) {
    constexpr int kSideA = 32 * R * kRowBytes, kSideW = kExpertCols * kRowBytes, RA = expert_stages_a(R, FEW), RW = kExpertStagesW;
    constexpr int kBehind = RA == RW ? (RA - 2) * (R + 4) : 4;   // copies that may be on their way at the wait
    constexpr int CA = R, CW = 4, V = CA + CW, kEarly = V / 2;   // copies of a wave and K-step; those right behind the barrier
    constexpr int kProducts = 4 * R, kReads = 4 + R, kReadsUpto = kProducts * 3 / 4;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / 2, wn = wave % 2;
    const int ql = lane & 15, g = lane >> 4;

    // copies as in wide_tile: KiB i of the wave's part of a stage, eight rows, lane's chunk (lane % 8) ^ row % 8
    uint32_t off_a[CA], off_w[CW];
    size_t far_a[LONG ? CA : 1];
    const int m_wave = p.gather > 0 ? 0 : m0 + 8 * CA * wave < m_end ? m0 + 8 * CA * wave : m_end - 1;
    const int n_wave = n0 + 8 * CW * wave < p.N ? n0 + 8 * CW * wave : p.N - 1;
#pragma unroll
    for (int i = 0; i < CA; ++i) {
        const int row = 8 * (CA * wave + i) + (lane >> 3);
        int m = m0 + row < m_end ? m0 + row : m_end - 1;
        if (p.gather > 0) m = p.order[m] / p.gather;
        const uint32_t chunk = 16 * ((lane & 7) ^ (row & 7)) + 4096 - 1024 * (i & 3);
        if constexpr (LONG) far_a[i] = (size_t)(m - m_wave) * (p.lda * sizeof(bf16)) + chunk;
        else off_a[i] = (uint32_t)(m - m_wave) * (uint32_t)(p.lda * sizeof(bf16)) + chunk;
    }
#pragma unroll
    for (int i = 0; i < CW; ++i) {
        const int row = 8 * (CW * wave + i) + (lane >> 3);
        const int n = n0 + row < p.N ? n0 + row : p.N - 1;
        off_w[i] = (uint32_t)(n - n_wave) * (uint32_t)(p.K * sizeof(bf16)) + 16 * ((lane & 7) ^ (row & 7)) + 4096 - 1024 * (i & 3);
    }
    const int steps = p.K / 64;
    const ptrdiff_t from = (ptrdiff_t)first * kRowBytes - 4096;
    gptr base_a = scalar_ptr(reinterpret_cast<const char *>(p.a + (size_t)m_wave * p.lda) + from);
    gptr base_w = scalar_ptr(reinterpret_cast<const char *>(w + (size_t)n_wave * p.K) + from);
    auto copy = [&](gptr from, int at, int i) {
        const auto *src = (const __attribute__((address_space(1))) void *)from;
        auto *dst = (__attribute__((address_space(3))) void *)(lds + at + 1024 * (i & ~3));
        switch (i & 3) {
            case 0: __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0); break;
            case 1: __builtin_amdgcn_global_load_lds(src, dst, 16, 1024, 0); break;
            case 2: __builtin_amdgcn_global_load_lds(src, dst, 16, 2048, 0); break;
            default: __builtin_amdgcn_global_load_lds(src, dst, 16, 3072, 0); break;
        }
    };
    int fill_a = 0, fill_w = 0;   // stages that the next K-step's copies go to
    // copy i of a K-step, A's first; behind the last one of each the source moves on, from the last K-step to the first, but not past all of
    // them (what is copied then, into buffers that nobody reads, comes from L2)
    int next_a = first, next_w = first, left_a = steps - 1, left_w = steps - 1;
    auto step_copy = [&](int i) {
        if (i < CA) {
            if constexpr (LONG) copy((gptr)(base_a + far_a[i < CA ? i : 0]), fill_a + 1024 * CA * wave, i);
            else copy(base_a + off_a[i < CA ? i : 0], fill_a + 1024 * CA * wave, i);
            if (i == CA - 1) {
                const bool more = left_a-- > 0, wrap = next_a + 1 == steps;
                next_a = wrap ? 0 : next_a + 1;
                base_a += !more ? 0 : wrap ? kRowBytes - steps * kRowBytes : kRowBytes;
                fill_a = fill_a == (RA - 1) * kSideA ? 0 : fill_a + kSideA;
            }
        } else {
            copy(base_w + off_w[i < CA ? 0 : i - CA], RA * kSideA + fill_w + 1024 * CW * wave, i - CA);
            if (i == V - 1) {
                const bool more = left_w-- > 0, wrap = next_w + 1 == steps;
                next_w = wrap ? 0 : next_w + 1;
                base_w += !more ? 0 : wrap ? kRowBytes - steps * kRowBytes : kRowBytes;
                fill_w = fill_w == (RW - 1) * kSideW ? 0 : fill_w + kSideW;
            }
        }
    };

    // operand addresses of the two halves (32 k) of a K-step; tile i is the instruction's offset
    uint32_t at_a[2], at_w[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const uint32_t o = ql * kRowBytes + 16 * ((4 * ks + g) ^ (ql & 7));
        at_a[ks] = o + wm * 16 * R * kRowBytes;
        at_w[ks] = o + RA * kSideA + wn * 64 * kRowBytes;
    }
    auto read = [&](uint32_t at, int i) { return *reinterpret_cast<const bf16x8 *>(lds + at + i * 16 * kRowBytes); };

    // where the second product's rows go: asked for here, because a store that has to ask waits once per 16 rows (down of 64 experts of
    // 1024 x 2048, 16384 entries: 109 -> 101 us, with nothing read past the last K-step)
    int out_rows[3] = {0, 0, 0};
    if constexpr (SCATTER && EPI == kOutElem) {
#pragma unroll
        for (int i = 0; i < (R + 3) / 4; ++i) {
            const int own = m0 + wm * 16 * R + 64 * i + lane;
            out_rows[i] = p.order[own < m_end ? own : m_end - 1];
        }
    }

    floatx4 acc[4][R];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < R; ++i) acc[j][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    bf16x8 a0[R], a1[R], w0[4], w1[4];
    // 4 R products with the reads of the next half and copies [c0, c1) of a K-step behind them
    auto half = [&](const bf16x8 (&wh)[4], const bf16x8 (&ah)[R], bf16x8 (&wx)[4], bf16x8 (&ax)[R], uint32_t from_wx, uint32_t from_ax, auto c0, auto c1) {
        each<kProducts>([&](auto product) __attribute__((always_inline)) {
            constexpr int n = decltype(product)::value;
            constexpr int r0 = items_before(n, kReadsUpto, kReads), r1 = items_before(n + 1, kReadsUpto, kReads);
            constexpr int k0 = decltype(c0)::value + items_before(n, kProducts, decltype(c1)::value - decltype(c0)::value);
            constexpr int k1 = decltype(c0)::value + items_before(n + 1, kProducts, decltype(c1)::value - decltype(c0)::value);
            __builtin_amdgcn_sched_barrier(0);
            // (the last ones are the compiler's: what it puts behind the loop, a move of the accumulators say, it then makes wait for them)
            if constexpr (n < kProducts - 4) mfma_in_place(acc[n % 4][n / 4], wh[n % 4], ah[n / 4]);
            else acc[n % 4][n / 4] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wh[n % 4], ah[n / 4], acc[n % 4][n / 4], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = r0; r < r1; ++r) {
                if (r < 4) wx[r < 4 ? r : 0] = read(from_wx, r);
                else ax[r < 4 ? 0 : r - 4] = read(from_ax, r - 4);
            }
#pragma unroll
            for (int c = k0; c < k1; ++c) step_copy(c);
        });
    };

    // All buffers but one each, and the first copies of the next K-step (with two buffers for A and three for W, A of K-step t + 2 goes with
    // W of t + 3)
#pragma unroll
    for (int s = 0; s < RW - 1; ++s)
#pragma unroll
        for (int i = s == 1 && RA == 2 ? CA : 0; i < V; ++i) step_copy(i);
#pragma unroll
    for (int i = 0; i < kEarly; ++i) step_copy(i);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kBehind + kEarly) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 4; ++j) w0[j] = read(at_w[0], j);
#pragma unroll
    for (int i = 0; i < R; ++i) a0[i] = read(at_a[0], i);

    int side_a = 0, side_w = 0;   // of the K-step that is multiplied
#pragma unroll 1
    for (int kt = 0; kt < steps; ++kt) {
#pragma unroll
        for (int i = 0; i < CA; ++i)
            if constexpr (!LONG) asm volatile("" : "+v"(off_a[i]));
#pragma unroll
        for (int i = 0; i < CW; ++i) asm volatile("" : "+v"(off_w[i]));
        half(w0, a0, w1, a1, at_w[1], at_a[1], std::integral_constant<int, kEarly>(), std::integral_constant<int, V>());
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kBehind) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int by_a = side_a == (RA - 1) * kSideA ? -side_a : kSideA, by_w = side_w == (RW - 1) * kSideW ? -side_w : kSideW;
        side_a += by_a;
        side_w += by_w;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) at_a[ks] += by_a, at_w[ks] += by_w;
        half(w1, a1, w0, a0, at_w[0], at_a[0], std::integral_constant<int, 0>(), std::integral_constant<int, kEarly>());
    }
    // no copy, of any wave, is on its way to LDS any more
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    store_rows<4, R, EPI, true, SCATTER>(p, acc, lds + wave * kWideStore, m0 + wm * 16 * R, m_end, n0 + wn * 64, out_rows);
}

// (SCATTER is gather == 0: asked at run time it cost gate and up 1.7 %)
template <int EPI, bool SCATTER, bool FEW, bool LONG>
__global__ void __launch_bounds__(kWideThreads, FEW ? 2 : 1) dense_gemm_expert_kernel(const GemmKernelArgs<bf16> p) {
    extern __shared__ __attribute__((aligned(16))) char gemm_lds[];
    const int tiles_m = p.tiles[4 * p.tiles_m];
    const int total = tiles_m * p.tiles_n, per_xcd = (total + 7) / 8;
    const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per_xcd || tile >= total) return;
    const int32_t *t = p.tiles + 4 * (tile / p.tiles_n);   // columns first: an XCD's workgroups share the rows of two experts or so in its L2
    const int n0 = tile % p.tiles_n * kExpertCols, m0 = t[1], m_end = m0 + t[2];
    const bf16 *w = p.w + (size_t)t[0] * p.w_stride;
    const int first = (5 * t[0] + 3 * (tile % p.tiles_n)) % (p.K / 64);
    if constexpr (FEW) {
        for (int m = m0; m < m_end; m += kFewRows) {   // (once, for a plan of the tile_rows that the launch was given)
            if (m > m0) __syncthreads();
            const int end = m_end - m < kFewRows ? m_end : m + kFewRows;
            switch ((end - m + 31) / 32) {
                case 1: expert_tile<1, EPI, SCATTER, true, false>(p, gemm_lds, w, m, end, n0, first); break;
                case 2: expert_tile<2, EPI, SCATTER, true, false>(p, gemm_lds, w, m, end, n0, first); break;
                case 3: expert_tile<3, EPI, SCATTER, true, false>(p, gemm_lds, w, m, end, n0, first); break;
                default: expert_tile<4, EPI, SCATTER, true, false>(p, gemm_lds, w, m, end, n0, first); break;
            }
        }
    } else if constexpr (LONG) {
        expert_tile<12, EPI, SCATTER, false, true>(p, gemm_lds, w, m0, m_end, n0, first);
    } else {
        switch ((t[2] + 31) / 32) {
            case 1: return expert_tile<1, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 2: return expert_tile<2, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 3: return expert_tile<3, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 4: return expert_tile<4, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 5: return expert_tile<5, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 6: return expert_tile<6, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 7: return expert_tile<7, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 8: return expert_tile<8, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 9: return expert_tile<9, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 10: return expert_tile<10, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            case 11: return expert_tile<11, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
            default: return expert_tile<12, EPI, SCATTER, false, false>(p, gemm_lds, w, m0, m_end, n0, first);
        }
    }
}

template <class T>
GemmKernelArgs<T> kernel_args(const GemmArgs &g, int bm, int bn) {
    GemmKernelArgs<T> p;
    p.a = static_cast<const T *>(g.a);
    p.w = static_cast<const T *>(g.w);
    p.out = g.out;
    p.M = g.M;
    p.N = g.N;
    p.K = g.K;
    p.lda = g.lda;
    p.ldo = g.ldo;
    p.tiles = g.tiles;
    p.order = g.order;
    p.gather = g.gather;
    p.w_stride = g.w_stride;
    p.silu_begin = g.silu_begin;
    p.silu_end = g.silu_end;
    p.slice_stride = (long)g.M * g.ldo;
    p.tiles_m = g.tiles ? g.n_tiles : (g.M + bm - 1) / bm;
    p.tiles_n = (g.N + bn - 1) / bn;
    return p;
}

template <class P>
hipError_t run_tiles(void (*kernel)(P), const P &p, int threads, size_t lds, int slices, hipStream_t stream, int most = 1 << 30) {
    if (lds > 48 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const int total = (p.tiles_m * p.tiles_n + 7) / 8 * 8;
    hipLaunchKernelGGL(kernel, dim3(total < most ? total : most, slices), dim3(threads), lds, stream, p);
    return hipGetLastError();
}

template <class T, int BM, int BN, int WM, int WN, int STAGES>
hipError_t launch_tile(const GemmArgs &g, int slices, hipStream_t stream) {
    const GemmKernelArgs<T> p = kernel_args<T>(g, BM, BN);
    constexpr size_t lds = STAGES * (size_t)(BM + BN) * kRowBytes;
    auto run = [&](auto kernel) { return run_tiles<GemmKernelArgs<T>>(kernel, p, 64 * WM * WN, lds, slices, stream); };
    if constexpr (std::is_same<T, float>::value)
        if (g.tiles)
            return g.epilogue == kOutSwiglu ? run(&dense_gemm_kernel<T, BM, BN, WM, WN, STAGES, kOutSwiglu, true>)
                                            : run(&dense_gemm_kernel<T, BM, BN, WM, WN, STAGES, kOutElem, true>);
    switch (g.epilogue) {
        case kOutF32: return run(&dense_gemm_kernel<T, BM, BN, WM, WN, STAGES, kOutF32, false>);
        case kOutSwiglu: return run(&dense_gemm_kernel<T, BM, BN, WM, WN, STAGES, kOutSwiglu, false>);
        case kOutGeglu: return run(&dense_gemm_kernel<T, BM, BN, WM, WN, STAGES, kOutGeglu, false>);
        default: return run(&dense_gemm_kernel<T, BM, BN, WM, WN, STAGES, kOutElem, false>);
    }
}

template <int WM, int NT>
hipError_t launch_wide(const GemmArgs &g, int slices, hipStream_t stream) {
    const GemmKernelArgs<bf16> p = kernel_args<bf16>(g, 128 * WM, 16 * NT * (4 / WM));
    auto run = [&](auto kernel) { return run_tiles<GemmKernelArgs<bf16>>(kernel, p, kWideThreads, wide_lds(WM, NT), slices, stream, wide_loops(NT, g.epilogue) ? 256 : 1 << 30); };
    switch (g.epilogue) {
        case kOutF32: return run(&dense_gemm_wide_kernel<WM, NT, kOutF32>);
        case kOutSwiglu: return run(&dense_gemm_wide_kernel<WM, NT, kOutSwiglu>);
        case kOutGeglu: return run(&dense_gemm_wide_kernel<WM, NT, kOutGeglu>);
        default: return run(&dense_gemm_wide_kernel<WM, NT, kOutElem>);
    }
}

template <bool FEW, bool LONG>
hipError_t launch_experts(const GemmArgs &g, hipStream_t stream) {
    const GemmKernelArgs<bf16> p = kernel_args<bf16>(g, kExpertRows, kExpertCols);
    constexpr size_t lds = FEW ? expert_lds(4, true) : expert_lds(12, false);
    static_assert(lds <= (FEW ? 80 : 160) * 1024 && 4 * kWideStore <= lds, "fits LDS, twice for few rows");
    static_assert(FEW ? expert_lds(2, true) <= lds : expert_lds(8, false) <= lds, "the heights with a buffer more too");
    auto run = [&](auto kernel) { return run_tiles<GemmKernelArgs<bf16>>(kernel, p, kWideThreads, lds, 1, stream); };
    if (g.epilogue == kOutSwiglu) return g.gather == 0 ? run(&dense_gemm_expert_kernel<kOutSwiglu, true, FEW, LONG>) : run(&dense_gemm_expert_kernel<kOutSwiglu, false, FEW, LONG>);
    return g.gather == 0 ? run(&dense_gemm_expert_kernel<kOutElem, true, FEW, LONG>) : run(&dense_gemm_expert_kernel<kOutElem, false, FEW, LONG>);
}

// out = the epilogue of the sum of `slices` parts [M][N]; a thread has four neighbouring columns of out
template <int EPI, int AT>
__global__ void __launch_bounds__(256) gemm_sum_kernel(const float *parts, int slices, int M, int N, void *out, long ldo, int silu_begin, int silu_end) {
    constexpr bool kPair = EPI == kOutSwiglu || EPI == kOutGeglu;
    const int quads = (kPair ? N / 2 : N) / 4;
    const long t = (long)blockIdx.x * 256 + threadIdx.x, size = (long)M * N;
    if (t >= (long)M * quads) return;
    const long m = t / quads;
    const int col = (int)(t % quads) * 4;
    const float *p = parts + m * N + (kPair ? col / 16 * 32 + col % 16 : col);
    floatx4 v = sum_parts<AT>(p, size, slices);
    if constexpr (kPair) {
        const floatx4 up = sum_parts<AT>(p + 16, size, slices);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (EPI == kOutGeglu ? gelu_tanh_of<bf16>(v[r]) : silu_of<bf16>(v[r])) * up[r];
    } else if (EPI == kOutElem && col >= silu_begin && col < silu_end) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = silu_of<bf16>(v[r]);
    }
    if constexpr (EPI == kOutF32) store4(static_cast<float *>(out) + m * ldo + col, v[0], v[1], v[2], v[3]);
    else store4(static_cast<bf16 *>(out) + m * ldo + col, v[0], v[1], v[2], v[3]);
}

// ---- choice of tile and slices ---------------------------------------------------------------------------------------------------
// A kernel's time: full rounds of its workgroups on 256 CUs (`together` of them to a CU), then a last one whose K-steps are the
// faster the emptier it is; in us.  Fitted to 18 products of 16 .. 2048 rows, K = 2048 .. 8192, in 1, 2, 4 and 8 slices, each alone
// on the GPU with cold weights (rms error of the time 4 to 10 %; the choice it leads to is within 8 % of the best kernel's time at 17 of
// the 18).  M x N x K with the parts added up, before there were slices / now: 64 x 2048 x 8192 130 / 16 us, 300 x 2048 x 8192 79 / 28,
// 2048 x 2048 x 8192 90 / 71; 64 x 16384 x 2048 with gelu 50 / 13 (64-row tiles).
// Narrow tiles read W from L2 once per 32 or 64 rows, which costs more in a model, where other kernels have been there, than alone:
// up to eight of them (2048 x 2048 x 2048 behind an attention: 32 us with 64-row tiles, 25 with wide ones alone).  128 x 128 tiles stay
// for what fills less than a round (808 x 1472 x 1664 with gelu: 23.6 us, 24.4 in wide tiles; 808 x 640 x 1664 5.7 / 7.6).
struct GemmKind {
    int rows, cols, together;
    float tile_us, step_us, step_full_us, store_tbs;   // per tile; per K-step alone and in a full round; fp32 results
};
enum : int { kTile32, kTile64, kTile128, kWide128, kWide192, kWide256, kKinds };
static_assert(kKinds == kGemmTiles, "");
constexpr GemmKind kGemmKinds[kKinds] = {
    {32, 128, 2, 1.0f, 0.215f, 0.43f, 6.8f}, {64, 128, 2, 0.f, 0.364f, 0.541f, 3.7f},  {128, 128, 2, 0.f, 0.547f, 0.866f, 4.4f},
    {128, 256, 1, 2.6f, 0.566f, 0.696f, 5.8f},
    {256, 192, 1, 5.8f, 0.728f, 0.947f, 10.3f}, {256, 256, 1, 7.5f, 0.953f, 1.201f, 11.f}};
float gemm_time(const GemmKind &k, int M, int N, int steps, int epilogue, int slices, bool kept) {
    const long tiles = (long)((M + k.rows - 1) / k.rows) * ((N + k.cols - 1) / k.cols) * slices, cap = 256 * k.together;
    const long full = tiles / cap, rest = tiles % cap;
    const int per = (steps + slices - 1) / slices;
    const float mb = 4e-6f * M * N;   // of one part
    float t = 4.f + full * (k.tile_us + per * k.step_full_us);
    if (rest) t += k.tile_us + per * (k.step_us + (k.step_full_us - k.step_us) * rest / cap);
    if (epilogue == kOutF32 || slices > 1) t += slices * mb / k.store_tbs;
    // whoever adds them up: the next kernel where the parts are kept, else a launch (3.5 us on the GPU, 6 with its allocation on the host, which
    // short prompts wait for)
    // (a router's parts: the choice of the experts waits for them, a wave to a token.  16384 x 32 x 512 13.1 us in one launch, 14.8 in two slices)
    if (slices > 1 && kept && N <= 128) t += 1.5e-4f * M;
    if (slices > 1) t += kept ? (slices - 1) * mb / 5.f : 6.f + (slices + 0.5f) * mb / 4.f;
    return t;
}

struct GemmChoice {
    int kind, slices;
};
// slices 0: any number; kept: the caller takes the parts.  Up to 128 columns are one tile's in any kind, so narrow tiles read nothing but their
// little W again: a router, 2048 x 64 x 2048, takes 13.7 us in one launch of 32-row tiles (its 32 K-steps on 64 CUs are all latency), 7.4 in eight
// slices of 64-row ones whose sum is left to the choice of the experts (5.0 -> 5.3 us), 17 in slices of 128-row ones and their sum.
GemmChoice choose_gemm(int M, int N, int K, int epilogue, int slices, bool kept) {
    GemmChoice best{kWide256, 1};
    float least = 1e30f;
    const int steps = K / 64, first = slices ? slices : 1, last = slices ? slices : steps >= 8 ? (steps / 4 < 8 ? steps / 4 : 8) : 1;
    for (int kind = N <= 128 ? kTile32 : M > 1024 ? kWide128 : M > 512 ? kTile128 : M > 256 ? kTile64 : kTile32; kind < kKinds; ++kind)
        for (int n = first; n <= last; n *= 2) {
            const float t = gemm_time(kGemmKinds[kind], M, N, steps, epilogue, n, kept);
            if (t < least) {
                least = t;
                best = {kind, n};
            }
        }
    return best;
}

// Rows as long as this do not fit the wide tiles' 32-bit offsets (64 rows of them).
bool long_rows(const GemmArgs &g) { return g.K >= 1 << 25 || (!g.tiles && g.lda >= 1 << 25); }

hipError_t launch_kind(const GemmArgs &g, int kind, int slices, hipStream_t stream) {
    if (long_rows(g) && kind > kTile64) kind = kTile64;
    switch (kind) {
        case kTile32: return launch_tile<bf16, 32, 128, 1, 4, 4>(g, slices, stream);
        case kTile64: return launch_tile<bf16, 64, 128, 1, 4, 3>(g, slices, stream);
        case kTile128: return launch_tile<bf16, 128, 128, 2, 2, 2>(g, slices, stream);
        case kWide128: return launch_wide<1, 4>(g, slices, stream);
        case kWide192: return launch_wide<2, 6>(g, slices, stream);
        default: return launch_wide<2, 8>(g, slices, stream);
    }
}

}  // namespace

// Rows of A per tile for a product of `rows` rows with each of `matrices` matrices.
int dense_gemm_tile_rows(int dtype, int rows, int N, int matrices) {
    if (dtype == kBf16 && matrices > 1) return rows <= kFewMean ? kFewRows : kExpertRows;
    if (rows <= 48 || N < 96) return 32;
    return dtype == kBf16 && rows > 128 ? 256 : 128;
}

hipError_t launch_dense_gemm(int dtype, const GemmArgs &g, int tile_rows, hipStream_t stream) {
    if (dtype == kF32) return tile_rows == 32 ? launch_tile<float, 32, 128, 1, 4, 4>(g, 1, stream) : launch_tile<float, 128, 128, 2, 2, 2>(g, 1, stream);
    if (g.tiles) {   // (any plan: its tiles are 384 rows or less)
        if (g.K >= 1 << 26) return hipErrorInvalidValue;
        // the copies' 32-bit offsets: from the first row of A where rows are gathered, else within a wave's part of a tile
        const long rows = g.gather > 0 ? (g.M + g.gather - 1) / g.gather : kExpertRows;
        if (rows * g.lda >= (1L << 31) - 4096) return launch_experts<false, true>(g, stream);
        return tile_rows <= kFewRows ? launch_experts<true, false>(g, stream) : launch_experts<false, false>(g, stream);
    }
    if (tile_rows == 32) return launch_tile<bf16, 32, 128, 1, 4, 4>(g, 1, stream);
    return launch_kind(g, tile_rows == 256 ? kWide256 : kWide128, 1, stream);
}

int dense_gemm_slices(int dtype, int M, int N, int K, int epilogue, bool kept) { return dtype == kBf16 ? choose_gemm(M, N, K, epilogue, 0, kept).slices : 1; }

hipError_t launch_dense_gemm_sliced(int dtype, const GemmArgs &g, int slices, float *parts, hipStream_t stream, int tile) {
    if (dtype != kBf16 || g.tiles) return launch_dense_gemm(dtype, g, dense_gemm_tile_rows(dtype, g.M, g.N, 1), stream);
    const int kind = tile >= 0 && tile < kKinds ? tile : choose_gemm(g.M, g.N, g.K, g.epilogue, slices, !g.out).kind;
    if (slices == 1) return launch_kind(g, kind, 1, stream);
    GemmArgs p = g;
    p.out = parts;
    p.ldo = g.N;
    p.epilogue = kOutF32;
    p.silu_begin = p.silu_end = 0;
    const hipError_t e = launch_kind(p, kind, slices, stream);
    if (e != hipSuccess || !g.out) return e;
    const bool pair = g.epilogue == kOutSwiglu || g.epilogue == kOutGeglu;
    const long threads = (long)g.M * (pair ? g.N / 2 : g.N) / 4;
    auto add = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, parts, slices, g.M, g.N, g.out, g.ldo, g.silu_begin, g.silu_end);
        return hipGetLastError();
    };
    auto pick = [&](auto epi) {
        constexpr int EPI = decltype(epi)::value;
        return slices <= 2 ? add(&gemm_sum_kernel<EPI, 2>) : slices <= 4 ? add(&gemm_sum_kernel<EPI, 4>) : add(&gemm_sum_kernel<EPI, 8>);
    };
    switch (g.epilogue) {
        case kOutF32: return pick(std::integral_constant<int, kOutF32>());
        case kOutSwiglu: return pick(std::integral_constant<int, kOutSwiglu>());
        case kOutGeglu: return pick(std::integral_constant<int, kOutGeglu>());
        default: return pick(std::integral_constant<int, kOutElem>());
    }
}

}  // namespace w4a16
