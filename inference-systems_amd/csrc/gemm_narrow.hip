// mfma_narrow: mfma_staged's form for grids of at most one round on the CUs, from a
// K that grows with the tile, C[M,N] = A[M,K] * W[N,K]^T (or B[K,N]) on tiles
// down to 32 x 32.  Such a grid is bound by the chain of K-tiles in each workgroup (copies, barrier,
// fragment reads, MFMAs; 0.27 us per 64 elements of K on 4 waves of 64 x 64,
// however deep the ring), so:
//   * tiles are as small as fills the CUs once: fewer bytes copied and read
//     per K-tile, and more CUs at work (200 x 1024 x 3584: 64 workgroups on 64
//     x 64 tiles, 224 on 32 x 32);
//   * a K-tile is 128 or 256 elements (KS sub-tiles of 64), so a barrier and
//     the latencies after it are paid half or a quarter as often; larger tiles
//     run on 8 waves, whose latencies hide under each other;
//   * every fragment read of the K-tile is issued before the copies that refill
//     the stage behind it, so the copies issue while the reads return.
// v_mfma_f32_16x16x32 sums K in the order of mfma_staged's 32x32x16, and copies
// past K are zeros, so every output has the bits of the larger tiles.
// bf16, us: 200 x 1024 x 3584 17.1 -> 8.9, 512 x 1024 x 3584 17.7 -> 11.1, 1024 x
// 1024 x 3584 18.4 -> 13.9, gate/up pairs of 47 x (2 x 2624) x 1024 9.4 -> 6.3.
#include "gemm_common.hpp"

namespace nvg {
namespace {

constexpr int kLdsPerCu = 160 * 1024;

__device__ u32x4_t g_narrow_zero = {0u, 0u, 0u, 0u};

// Column chunks of B[K,N] k-rows within a panel of 64 columns: the key of
// splitk_decode's B[K,N] lines (conflict-free for the transposing reads).
__device__ __forceinline__ int panel_swizzle(int r) { return 2 * (((r >> 1) & 1) | ((r >> 2) & 2)); }

// BM x BN tile (W rows, or columns of B), KS sub-tiles of 64 elements per
// K-tile, WGM x WGN waves, STAGES K-tiles in LDS.
template <int DT, int DT_OUT, int BM, int BN, int KS, int WGM, int WGN, int STAGES, int EPI, int RS, int KN>
__global__ __launch_bounds__(WGM * WGN * 64) void mfma_narrow_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, int64_t m, int64_t n, int64_t k, int64_t lda,
    int64_t ldb, void* __restrict__ c, int64_t ldc, int c_vec, const float* __restrict__ row_scale) {
    constexpr int NW = WGM * WGN, NT = NW * 64;
    constexpr int BK = 64 * KS;
    constexpr int BNO = EPI == EPI_SILU_MUL ? BN / 2 : BN;
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int MI = WM / 16, NI = WN / 16;
    constexpr int ROWS = BM + BN;
    constexpr int STAGE = KS * ROWS * 8;          // 16-byte chunks per stage
    constexpr int IPW = KS * ROWS / 8 / NW;       // copy instructions per wave and K-tile
    constexpr int AHEAD = STAGES - 1;
    static_assert(IPW * 8 * NW == KS * ROWS && WM % 16 == 0 && WN % 16 == 0, "tile shape");
    static_assert((AHEAD - 1) * IPW < 64, "vmcnt range");
    static_assert(EPI != EPI_SILU_MUL || (NI % 2 == 0 && !KN), "gate/up pairs per wave");
    static_assert(!KN || (BN % 64 == 0 && BM % 8 == 0), "B[K,N] panels of 64 columns");
    constexpr int OB = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    constexpr int PITCH = BNO * OB + 16;
    constexpr int RING = STAGES * STAGE * 16;
    constexpr int LDS = RING > BM * PITCH ? RING : BM * PITCH;
    static_assert(LDS <= kLdsPerCu, "LDS per CU");
    __shared__ u32x4_t ring[LDS / 16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int r16 = lane & 15, quad = lane >> 4;
    const int tiles_m = static_cast<int>((m + BM - 1) / BM);
    const int tiles_n = static_cast<int>((n + BNO - 1) / BNO);
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BNO;

    // Copy instruction j of a wave is number i = wave * IPW + j of the stage:
    // sub-tile i / (ROWS / 8), 8 LDS rows (or, in the B[K,N] part, 8 k-rows of
    // a 64-column panel); lane L fills row L / 8, position L % 8.
    const uint16_t* src[IPW];
    int kpos[IPW];
    bool krow[IPW];
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
        const int i = wave * IPW + j;
        const int sub = i / (ROWS / 8), r = 8 * (i % (ROWS / 8)) + (lane >> 3);
        krow[j] = false;
        if (KN && r >= BM) {
            const int q = r - BM, panel = q >> 6, kr = q & 63;
            const int64_t col = n0 + 64 * panel + 8 * ((lane & 7) ^ panel_swizzle(kr));
            src[j] = w + min_i64(col, n - 8) + int64_t(64 * sub + kr) * ldb;
            kpos[j] = 64 * sub + kr;
            krow[j] = true;
        } else {
            const int ch = (lane & 7) ^ ((r >> 1) & 7);
            kpos[j] = 64 * sub + 8 * ch;
            if (r < BM) {
                src[j] = a + min_i64(m0 + r, m - 1) * lda + kpos[j];
            } else {
                const int wr = r - BM;
                int64_t row;
                // 16 gate rows, then the 16 up rows of the same columns.
                if constexpr (EPI == EPI_SILU_MUL)
                    row = min_i64(n0 + 16 * (wr >> 5) + (wr & 15), n - 1) + ((wr & 16) ? n : 0);
                else
                    row = min_i64(n0 + wr, n - 1);
                src[j] = w + row * ldb + kpos[j];
            }
        }
    }
    const int kk = static_cast<int>(k);
    const int ktiles = (kk + BK - 1) / BK;
    const uint32_t lds0 = lds_address(ring);
    const void* zero = &g_narrow_zero;
    asm volatile("" : "+s"(zero));
    // Chunks past K (and K-tiles past the last) copy zeros, so every K-tile
    // issues the same number of copies.
    auto issue = [&](int t, int stage) {
        const int k0 = t * BK;
        const uint32_t dst = lds0 + uint32_t(stage * STAGE + 64 * wave * IPW) * 16u;
        if (k0 + BK <= kk) {
#pragma unroll
            for (int j = 0; j < IPW; ++j) dma16(src[j] + (KN && krow[j] ? int64_t(k0) * ldb : k0), dst + 1024u * j);
        } else {
#pragma unroll
            for (int j = 0; j < IPW; ++j) {
                const void* p = src[j] + (KN && krow[j] ? int64_t(k0) * ldb : k0);
                dma16(k0 + kpos[j] < kk ? p : zero, dst + 1024u * j);
            }
        }
    };

    f32x4_t acc[NI][MI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) acc[i][j] = f32x4_t{};

#pragma unroll
    for (int t = 0; t < AHEAD; ++t) issue(t, t);
    asm volatile("" :: "s"(c), "s"(ldc), "s"(c_vec), "s"(m), "s"(n), "s"(row_scale));

    const int swz = (r16 >> 1) & 7;
    auto read_step = [&](const u32x4_t* tile, int s, u32x4_t (&af)[MI], u32x4_t (&wf)[NI]) {
        const u32x4_t* sub = tile + (s >> 1) * ROWS * 8;
        const int ch = (4 * (s & 1) + quad) ^ swz;
#pragma unroll
        for (int i = 0; i < MI; ++i) af[i] = sub[(wm * WM + 16 * i + r16) * 8 + ch];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if constexpr (KN) {
                typedef short v4i16_t __attribute__((ext_vector_type(4)));
                typedef __attribute__((address_space(3))) v4i16_t* lds_v4;
                const int kr = 32 * (s & 1) + 8 * quad + (r16 >> 2);
                const int col = wn * WN + 16 * i;
                const int cc = (((col & 63) >> 3) + ((r16 & 3) >> 1)) ^ panel_swizzle(kr);
                const uint32_t a0 = lds_address(sub + (BM + 64 * (col >> 6)) * 8) + uint32_t(kr) * 128u +
                                    uint32_t(cc) * 16u + 8u * (r16 & 1);
                const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(uintptr_t)a0));
                const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(uintptr_t)(a0 + 512u)));
                wf[i] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
            } else {
                wf[i] = sub[(BM + wn * WN + 16 * i + r16) * 8 + ch];
            }
        }
    };

    int cur = 0;
    for (int t = 0; t < ktiles; ++t) {
        // K-tile t has landed in every wave's part, and every wave has read
        // K-tile t - 1, whose stage is refilled.
        wait_vmcnt<(AHEAD - 1) * IPW>();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const u32x4_t* tile = ring + cur * STAGE;
        u32x4_t af[2 * KS][MI], wf[2 * KS][NI];
#pragma unroll
        for (int s = 0; s < 2 * KS; ++s) read_step(tile, s, af[s], wf[s]);
        __builtin_amdgcn_sched_barrier(0);
        issue(t + AHEAD, cur == 0 ? STAGES - 1 : cur - 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2 * KS; ++s)
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < MI; ++j) acc[i][j] = mfma_16x16x32<DT>(wf[s][i], af[s][j], acc[i][j]);
        cur = cur + 1 == STAGES ? 0 : cur + 1;
    }
    wait_vmcnt<0>();   // copies of zeros past the last K-tile

    // Output through LDS, as in mfma_wide.
    constexpr int CPR = BNO * OB / 16, EPC = 16 / OB;
    constexpr int NJ = EPI == EPI_SILU_MUL ? NI / 2 : NI;
    char* ctile = reinterpret_cast<char*>(ring);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < MI; ++j) {
        const int row = wm * WM + 16 * j + r16;
        float rs = 1.0f;
        if constexpr (RS) rs = row_scale[min_i64(m0 + row, m - 1)];
#pragma unroll
        for (int i = 0; i < NJ; ++i) {
            f32x4_t x = acc[EPI == EPI_SILU_MUL ? 2 * i : i][j];
            if constexpr (RS) x *= rs;
            if constexpr (EPI == EPI_SILU_MUL) {
                f32x4_t u = acc[2 * i + 1][j];
                if constexpr (RS) u *= rs;
#pragma unroll
                for (int v = 0; v < 4; ++v) x[v] = silu_f32(x[v]) * u[v];
            }
            char* p = ctile + row * PITCH + (wn * 16 * NJ + 16 * i + 4 * quad) * OB;
            if constexpr (OB == 4) *reinterpret_cast<f32x4_t*>(p) = x;
            else *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack2<DT_OUT>(x[0], x[1]), pack2<DT_OUT>(x[2], x[3])};
        }
    }
    __syncthreads();
    if (!c_vec) {
        store_unaligned<OB, BM, BNO, NT>(ctile, PITCH, static_cast<char*>(c) + (m0 * ldc + n0) * OB, ldc, m - m0, n - n0,
                                         tid);
        return;
    }
#pragma unroll 2
    for (int e = tid; e < BM * CPR; e += NT) {
        const int r = e / CPR, chunk = e % CPR;
        const int64_t grow = m0 + r, gcol = n0 + chunk * EPC;
        if (grow >= m || gcol >= n) continue;
        const u32x4_t val = *reinterpret_cast<const u32x4_t*>(ctile + r * PITCH + chunk * 16);
        char* gdst = static_cast<char*>(c) + (grow * ldc + gcol) * OB;
        if (gcol + EPC <= n) {
            __builtin_nontemporal_store(val, reinterpret_cast<u32x4_t*>(gdst));
        } else {
            const int valid = int(min_i64(EPC, n - gcol));
            if constexpr (OB == 4) {
                for (int x = 0; x < valid; ++x) reinterpret_cast<uint32_t*>(gdst)[x] = val[x];
            } else {
                for (int x = 0; x < valid; ++x)
                    reinterpret_cast<uint16_t*>(gdst)[x] = uint16_t(val[x >> 1] >> (16 * (x & 1)));
            }
        }
    }
}

template <int DT, int DT_OUT, int BM, int BN, int KS, int WGM, int WGN, int STAGES, int EPI, int RS, int KN>
int launch_tile(const Problem& p, hipStream_t s) {
    constexpr int BNO = EPI == EPI_SILU_MUL ? BN / 2 : BN;
    const int64_t tiles = ((p.m + BM - 1) / BM) * ((p.n + BNO - 1) / BNO);
    if (tiles > INT32_MAX) return set_error(NANOVLLM_GEMM_EINVAL, "mfma_narrow: grid too large");
    const int out_bytes = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    const int c_vec = (reinterpret_cast<uintptr_t>(p.c) % 16 == 0) && ((p.ldc * out_bytes) % 16 == 0);
    hipLaunchKernelGGL((mfma_narrow_kernel<DT, DT_OUT, BM, BN, KS, WGM, WGN, STAGES, EPI, RS, KN>),
                       dim3(static_cast<uint32_t>(tiles)), dim3(WGM * WGN * 64), 0, s,
                       static_cast<const uint16_t*>(p.a), static_cast<const uint16_t*>(p.b), p.m, p.n, p.k, p.lda, p.ldb,
                       p.c, p.ldc, c_vec, p.row_scale);
    return check_launch("mfma_narrow", BM, BNO);
}

constexpr int64_t kCus = 256;

int64_t tiles(const Problem& p, int64_t rows, int64_t cols) {
    return ((p.m + rows - 1) / rows) * ((p.n + cols - 1) / cols);
}

// Plain GEMM: the smallest tile whose grid fits the CUs at one workgroup each
// (bf16, us, against mfma_staged's 64 x 64):
//   * 32 x 32 (4 waves), K-tiles of 256 from K = 1536 (200 x 1024 x 3584 8.9, on
//     K-tiles of 128 9.3, 32 x 64 10.4-10.7, 64 x 64 17.1) and of 128 below
//     (48 x 4096 x 1024 4.9 / 5.0 / 5.5 / 7.2, 130 x 576 x 256 3.4 against 3.7);
//   * 32 x 64 (8 waves): 512 x 1024 x 1024 5.8 (32 x 32 6.1, 64 x 64 6.5), 700 x
//     700 x 8000 21.0 (25.8, 36.3), 333 x 1024 x 2048 7.8 (8.5, 11.0);
//   * 64 x 64 (8 waves): 512 x 2048 x 1024 6.7 against 7.3, 256 x 4096 x 2048
//     9.5 / 11.5, 1024 x 1024 x 3584 13.9 / 18.4.  From 257 tiles, two of
//     mfma_staged's fit a CU and overlap (2048 x 1024 x 1024 8.7 against 11.3).
// B[K,N] has the last two (panels of 64 columns): 200 x 1024 x 3584 12.2 against
// 16.9, 100 x 512 x 512 4.5 / 4.8, 256 x 4096 x 2048 10.9 / 12.0.
template <int DT, int DT_OUT, int EPI, int RS, int KN>
int launch_plain(const Problem& p, hipStream_t s) {
    if constexpr (!KN) {
        if (tiles(p, 32, 32) <= kCus) {
            if (p.k >= 1536) return launch_tile<DT, DT_OUT, 32, 32, 4, 2, 2, 4, EPI, RS, 0>(p, s);
            return launch_tile<DT, DT_OUT, 32, 32, 2, 2, 2, 4, EPI, RS, 0>(p, s);
        }
    }
    if (tiles(p, 32, 64) <= kCus) return launch_tile<DT, DT_OUT, 32, 64, 2, 2, 4, 5, EPI, RS, KN>(p, s);
    return launch_tile<DT, DT_OUT, 64, 64, 2, 2, 4, 4, EPI, RS, KN>(p, s);
}

// SiLU pairs, in rows x output columns (bf16, us, K = 1024 unless given, against
// mfma_staged's 64 x 64): 32 x 32 (4 waves) while those fit the CUs at one
// each (47 x 2624 6.3 against 9.4, 64 x 3584 x K 2048 9.2 / 14.7), then 64 x 32 on
// 8 waves (100 x 3584 6.8 against 10.9 on 32 x 32 and 9.7), then 64 x 32 on 4
// waves, two workgroups to a CU (200 x 3584 8.9 / 9.8).
template <int DT, int DT_OUT, int RS>
int launch_silu(const Problem& p, hipStream_t s) {
    if (tiles(p, 32, 32) <= kCus) return launch_tile<DT, DT_OUT, 32, 64, 2, 2, 2, 4, EPI_SILU_MUL, RS, 0>(p, s);
    if (tiles(p, 64, 32) <= kCus) return launch_tile<DT, DT_OUT, 64, 64, 2, 4, 2, 4, EPI_SILU_MUL, RS, 0>(p, s);
    return launch_tile<DT, DT_OUT, 64, 64, 1, 2, 2, 4, EPI_SILU_MUL, RS, 0>(p, s);
}

// Which plain grids take these tiles, up to one round of 64 x 64.  A long
// K-tile fills and drains once per workgroup, so they need a K to spread that
// over; more of it where 8 waves share the tile, and where rows of A and B are
// not whole 128-byte lines, which adds a line to most copy instructions of
// every K-tile (mfma_staged's 64 x 64 against these, bf16 and f16, us):
//   * 32 x 32: 983 x 256 x 64 3.25 / 3.41, 795 x 128 x 96 3.43 / 3.29;
//   * 32 x 64: K = 320 544 x 832 4.15 / 4.32, 384 573 x 832 4.60 / 4.32, 512
//     312 x 1600 5.00 / 4.70; rows of other lengths: K = 552 2259 x 192 5.00 /
//     5.44, 584 245 x 1472 5.67 / 5.31, 608 517 x 576 5.48 / 5.17;
//   * 64 x 64: K = 448 264 x 2816 5.01 / 5.34, 512 67 x 5248 5.27 / 4.89, 1024 842
//     x 704 7.34 / 6.64; rows of other lengths: K = 816 395 x 2240 6.64 / 7.22, 1456
//     452 x 1856 9.25 / 9.82, 1848 1727 x 448 11.84 / 11.66, 2016 203 x 3264 11.56 /
//     10.88;
//   * B[K,N], 32 x 64: K = 320 78 x 832 4.12 / 4.31, 512 447 x 192 4.80 / 4.56;
//     rows of other lengths: K = 560 83 x 3912 5.95 / 6.23, 768 149 x 592 6.32 /
//     5.82; 64 x 64: K = 704 2619 x 384 6.30 / 6.60, 1024 1272 x 512 7.40 / 7.13,
//     1152 237 x 2112 7.83 / 7.20; rows of other lengths: K = 1160 132 x 3696 8.84
//     / 9.43, 2256 56 x 11520 18.0 / 17.1.
bool plain_pays(const Problem& p) {
    if (tiles(p, 64, 64) > kCus) return false;
    const bool lines = p.lda % 64 == 0 && p.ldb % 64 == 0;
    const bool rows32 = tiles(p, 32, 64) <= kCus;
    if (p.b_layout == NANOVLLM_GEMM_B_KN) return p.k >= (rows32 ? (lines ? 512 : 768) : (lines ? 1024 : 2048));
    if (tiles(p, 32, 32) <= kCus) return p.k > 64;
    return p.k >= (rows32 ? (lines ? 384 : 576) : (lines ? 512 : 1792));
}

// SiLU pairs: all grids of one round of 64 x 32 outputs; up to two rounds, where
// a workgroup of 64 x 32 copies as many rows of A as W rows, mfma_staged's 64 x 64
// outputs copy less and win where rows are not whole 128-byte lines (unless only
// its 128 x 128 tiles are left) and on a very long K (these / those, bf16, us:
// 729 x 1216 x 992 10.7 / 10.3, norm + 827 x 1024 x 616 12.7 / 11.9, norm + 59 x 9344
// x 3968 45.5 / 43.8; taken: 929 x 736 x 1024 9.1 / 10.0).
bool silu_pays(const Problem& p) {
    if (tiles(p, 64, 32) <= kCus) return true;
    if (tiles(p, 64, 32) > 2 * kCus || p.k > 3072) return false;
    const int64_t tiles128 = (p.m + 127) / 128 * ((2 * p.n + 127) / 128);
    return (p.lda % 64 == 0 && p.ldb % 64 == 0) || tiles128 > kCus / 2;
}

template <int DT, int DT_OUT>
int launch_typed(const Problem& p, hipStream_t s) {
    if (p.b_layout == NANOVLLM_GEMM_B_KN) return launch_plain<DT, DT_OUT, EPI_NONE, 0, 1>(p, s);
    if (p.row_scale != nullptr) {
        if (p.epi == EPI_SILU_MUL) return launch_silu<DT, DT_OUT, 1>(p, s);
        return launch_plain<DT, DT_OUT, EPI_NONE, 1, 0>(p, s);
    }
    if (p.epi == EPI_SILU_MUL) return launch_silu<DT, DT_OUT, 0>(p, s);
    return launch_plain<DT, DT_OUT, EPI_NONE, 0, 0>(p, s);
}

}  // namespace

// K-tiles are counted in 32 bits.
bool mfma_narrow_pays(const Problem& p) {
    if (p.k >= (int64_t(1) << 30)) return false;
    if (p.b_layout == NANOVLLM_GEMM_B_KN && (p.epi != EPI_NONE || p.row_scale != nullptr)) return false;
    if (p.epi == EPI_SILU_MUL) return silu_pays(p);
    return p.epi == EPI_NONE && plain_pays(p);
}

int launch_mfma_narrow(const Problem& p, hipStream_t s) {
    if (p.dtype_in == NANOVLLM_GEMM_BF16) {
        if (p.dtype_out == NANOVLLM_GEMM_BF16) return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_BF16>(p, s);
        return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_F32>(p, s);
    }
    if (p.dtype_out == NANOVLLM_GEMM_F16) return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F16>(p, s);
    return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F32>(p, s);
}

}  // namespace nvg
