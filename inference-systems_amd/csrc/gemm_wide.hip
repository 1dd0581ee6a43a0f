// mfma_wide: mfma_staged's form for large grids, C[M,N] = A[M,K] * W[N,K]^T
// on 256 x 256 tiles.  What bounds these grids is how evenly a CU's copies
// into LDS, its fragment reads and its matrix instructions overlap:
//   * 256 x 256 x 64 K-tiles copy 64 KiB per 2048 clocks of MFMAs, 32 B per
//     clock where global -> LDS copies sustain 45-57 (a 128 x 256 tile needs
//     47), and read 192 KiB of fragments (8 waves of 128 x 64), about half of
//     what LDS reads sustain;
//   * only two 64 KiB stages fit a CU, so a stage is refilled in two parts.
//     Region P (W, and the lower 64 rows of both wave tiles of A: 6 of a
//     wave's 8 copies) is free as soon as its second K-step has been read,
//     5/16 into a K-tile; region Q (the upper rows of A, 2 copies) at the end.
//     That lets the 8 copies be spread one per two groups of 4 MFMAs over
//     the whole K-tile, each with 10 groups (1280 clocks) or more to land.
//     Issued back to back in 8 groups instead, they ask for 64 B per clock:
//     4096^3 98 against 91.5 us, 8192^3 818 against 717 us;
//   * v_mfma_f32_16x16x32, whose products the chip runs at a higher clock
//     under its power limit than 32x32x16; both sum K in the same order, so
//     every output has the bits mfma_staged's tiles give it;
//   * within a group, the fragment of A the group has just used is reloaded
//     for the next K-step, so the reads too are spread over the MFMAs.
// Against the 128 x 256 and 128 x 128 tiles of mfma_staged (bf16, inputs
// rotated): 4096^3 116.5 -> 91.6 us (1500 TFLOP/s), 8192^3 915 -> 717, 4096 x
// 4096 x 1024 33.5 -> 28.4, 8192 x 8192 x 1024 129-139 -> 112, the fused
// gate/up projection of 8192 x (2 x 3584) x 1024 140 -> 125 us.
#include <type_traits>

#include "gemm_common.hpp"

namespace nvg {
namespace {

constexpr int kBM = 256, kBN = 256, kBK = 64;
constexpr int kChunks = kBK / 8;              // 16-byte chunks per LDS row
constexpr int kRows = kBM + kBN;              // LDS rows per stage: A, then W
constexpr int kStageChunks = kRows * kChunks; // 64 KiB
constexpr int kThreads = 512;                 // 8 waves, 2 x 4 over the tile
constexpr int kWM = 128, kWN = 64;            // wave tile
constexpr int kMI = kWM / 16, kNI = kWN / 16; // 16 x 16 blocks of a wave tile
constexpr int kCopies = kRows / 64;           // copy instructions per wave and K-tile (8 rows each)
constexpr int kLdsBytes = 160 * 1024;

__device__ u32x4_t g_wide_zero = {0u, 0u, 0u, 0u};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// dma16 from a scalar base and a 32-bit byte offset per lane.
__device__ __forceinline__ void dma16_at(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2"
                 :: "v"(off), "s"(lds), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

template <int DT, int DT_OUT, int EPI, int RS>
__global__ __launch_bounds__(kThreads) void mfma_wide_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, int64_t m, int64_t n, int64_t k, int64_t lda,
    int64_t ldb, void* __restrict__ c, int64_t ldc, int c_vec, const float* __restrict__ row_scale) {
    constexpr int BNO = EPI == EPI_SILU_MUL ? kBN / 2 : kBN;   // output columns per tile
    constexpr int OB = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    constexpr int PITCH = BNO * OB + 16;
    constexpr int EP_ROWS = kBM * PITCH <= kLdsBytes ? kBM : kWM;   // C-tile rows per epilogue pass
    constexpr int EPASS = kBM / EP_ROWS;
    constexpr int RING_BYTES = 2 * kStageChunks * 16;
    constexpr int LDS_BYTES = RING_BYTES > EP_ROWS * PITCH ? RING_BYTES : EP_ROWS * PITCH;
    static_assert(LDS_BYTES <= kLdsBytes, "LDS per CU");
    __shared__ u32x4_t ring[LDS_BYTES / 16];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int r16 = lane & 15, quad = lane >> 4;

    const int tiles_m = static_cast<int>((m + kBM - 1) / kBM);
    const int tiles_n = static_cast<int>((n + BNO - 1) / BNO);
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int64_t m0 = int64_t(tm) * kBM;
    const int64_t n0 = int64_t(tn) * BNO;

    // Copies: instruction j of a wave fills 8 LDS rows, lane L row L / 8,
    // position L % 8, which holds logical chunk (L % 8) ^ ((row >> 1) & 7).
    // j = 0..3: W rows; j = 4, 5: the lower 64 rows of both wave tiles of A
    // (with W, region P); j = 6, 7: the upper 64 rows (region Q).
    // EPI_SILU_MUL alternates 32 gate rows and the 32 up rows of the same
    // output columns, as mfma_staged does.
    auto copy_row = [&](int j) {   // first LDS row of instruction j
        if (j < 4) return kBM + 32 * wave + 8 * j;
        const int i = 2 * wave + (j & 1);
        return 128 * (i >> 3) + 8 * (i & 7) + (j < 6 ? 0 : 64);
    };
    const uint16_t* abase = a + m0 * lda;
    const uint16_t* wbase = w + n0 * ldb;
    uint32_t off[kCopies];
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
        const int row = copy_row(j) + (lane >> 3);
        const int chunk = (lane & 7) ^ ((row >> 1) & 7);
        int64_t src;
        if (j >= 4) {
            src = (min_i64(m0 + row, m - 1) - m0) * lda;
        } else {
            const int wr = row - kBM;
            if constexpr (EPI == EPI_SILU_MUL)
                src = (min_i64(n0 + 32 * (wr >> 6) + (wr & 31), n - 1) - n0 + ((wr & 32) ? n : 0)) * ldb;
            else
                src = (min_i64(n0 + wr, n - 1) - n0) * ldb;
        }
        off[j] = static_cast<uint32_t>((src + chunk * 8) * 2);
    }
    const int ktiles = static_cast<int>((k + kBK - 1) / kBK);
    const uint32_t lds0 = lds_address(ring);
    using Yes = std::true_type;
    using No = std::false_type;
    auto copy = [&](int t, int j, auto last_c) {
        const uint16_t* kb = (j < 4 ? wbase : abase) + int64_t(t) * kBK;
        const uint32_t dst = lds0 + uint32_t((t & 1) * kStageChunks) * 16u + uint32_t(copy_row(j)) * 128u;
        if (!decltype(last_c)::value || (t + 1) * kBK <= k) {
            dma16_at(kb, off[j], dst);
        } else {
            // The last K-tile of a K that is not a multiple of 64: chunks
            // past K copy zeros.
            const int chunk = (lane & 7) ^ (((copy_row(j) + (lane >> 3)) >> 1) & 7);
            const void* src = t * kBK + chunk * 8 < k ? reinterpret_cast<const char*>(kb) + off[j]
                                                      : reinterpret_cast<const char*>(&g_wide_zero);
            dma16(src, dst);
        }
    };

    f32x4_t acc[kNI][kMI];
#pragma unroll
    for (int i = 0; i < kNI; ++i)
#pragma unroll
        for (int j = 0; j < kMI; ++j) acc[i][j] = f32x4_t{};

    // Fragment of a 16-row block: lane l reads row l % 16, chunk 4 s + l / 16
    // of K-step s.
    const int swz = (r16 >> 1) & 7;
    const u32x4_t* a_base = ring + (wm * kWM + r16) * kChunks;
    const u32x4_t* w_base = ring + (kBM + wn * kWN + r16) * kChunks;
    u32x4_t af[kMI], wf0[kNI], wf1[kNI];
    auto read_a = [&](int stage, int s, int i) {
        return a_base[stage * kStageChunks + 16 * i * kChunks + ((4 * s + quad) ^ swz)];
    };
    auto read_w = [&](int stage, int s, int i) {
        return w_base[stage * kStageChunks + 16 * i * kChunks + ((4 * s + quad) ^ swz)];
    };
    auto barrier = [&] {
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

#pragma unroll
    for (int j = 0; j < kCopies; ++j) copy(0, j, Yes{});
    if (ktiles > 1) {
#pragma unroll
        for (int j = 0; j < 6; ++j) copy(1, j, Yes{});
        wait_vmcnt<6>();
    } else {
        wait_vmcnt<0>();
    }
    asm volatile("" :: "s"(c), "s"(ldc), "s"(c_vec), "s"(m), "s"(n), "s"(row_scale));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
#pragma unroll
    for (int i = 0; i < kNI; ++i) wf0[i] = read_w(0, 0, i);
#pragma unroll
    for (int i = 0; i < kMI; ++i) af[i] = read_a(0, 0, i);

    // last_c: K-tile t + 2 is the last.  The vmcnt waits count the copies
    // issued after the awaited ones: region P of t + 1 is followed by Q of
    // t + 1 (2) and the first two of t + 2, Q of t + 1 by four of t + 2.
    auto k_tile = [&](int t, auto next_c, auto copy_c, auto last_c) {
        constexpr bool NEXT = decltype(next_c)::value;    // K-tile t + 1 exists
        constexpr bool COPY = decltype(copy_c)::value;    // K-tile t + 2 exists
        constexpr std::integral_constant<bool, NEXT && !COPY> last1{};   // t + 1 is the last K-tile
        const int st = t & 1;
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
            if constexpr (COPY) {
                if (i == 5) {
                    // Every wave has read region P of K-tile t.
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_waitcnt lgkmcnt(1)" ::: "memory");
                    barrier();
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < kNI; ++j) acc[j][i] = mfma_16x16x32<DT>(wf0[j], af[i], acc[j][i]);
            if (i < kNI) wf1[i] = read_w(st, 1, i);
            af[i] = read_a(st, 1, i);
            if constexpr (NEXT) {
                if (i == 0) copy(t + 1, 6, last1);
                if (i == 2) copy(t + 1, 7, last1);
            }
            if constexpr (COPY) {
                if (i == 5) copy(t + 2, 0, last_c);
                if (i == 7) copy(t + 2, 1, last_c);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (NEXT) {
            // Region P of K-tile t + 1 has landed in every wave's part.
            if constexpr (COPY) wait_vmcnt<4>();
            else wait_vmcnt<2>();
            barrier();
        }
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < kNI; ++j) acc[j][i] = mfma_16x16x32<DT>(wf1[j], af[i], acc[j][i]);
            if constexpr (NEXT) {
                if (i == 4) {
                    // Region Q of K-tile t + 1 has landed, and every wave has
                    // read that of K-tile t.
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (COPY) wait_vmcnt<4>();
                    else wait_vmcnt<0>();
                    asm volatile("s_waitcnt lgkmcnt(8)" ::: "memory");
                    barrier();
                }
                if (i < kNI) wf0[i] = read_w(st ^ 1, 0, i);
                af[i] = read_a(st ^ 1, 0, i);
            }
            if constexpr (COPY) {
                if (i == 1) copy(t + 2, 2, last_c);
                if (i == 3) copy(t + 2, 3, last_c);
                if (i == 5) copy(t + 2, 4, last_c);
                if (i == 7) copy(t + 2, 5, last_c);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int t = 0;
    for (; t + 3 < ktiles; ++t) k_tile(t, Yes{}, Yes{}, No{});
    if (t + 2 < ktiles) k_tile(t++, Yes{}, Yes{}, Yes{});
    if (t + 1 < ktiles) k_tile(t++, Yes{}, No{}, Yes{});
    k_tile(t, No{}, No{}, No{});

    // Epilogue through LDS, as in mfma_staged: acc[j][i][v] is output row
    // 16 i + l % 16, column 16 j + 4 (l / 16) + v of the wave tile.
    constexpr int CPR = BNO * OB / 16;
    constexpr int EPC = 16 / OB;
    constexpr int ROWS_PER_PASS = kThreads / CPR;
    constexpr int NJ = EPI == EPI_SILU_MUL ? kNI / 2 : kNI;
    static_assert(EP_ROWS % ROWS_PER_PASS == 0, "copy passes");
    char* ctile = reinterpret_cast<char*>(ring);
    const int chunk = tid % CPR;
    // The row scales from a scalar base and 32-bit rows: 64-bit row numbers are
    // kept through the K loop, which has no register left for them.
    const float* scale = RS ? row_scale + m0 : nullptr;
    const int last_row = static_cast<int>(min_i64(kBM, m - m0)) - 1;
#pragma unroll 1
    for (int ep = 0; ep < EPASS; ++ep) {
        __syncthreads();
        if (EPASS == 1 || wm == ep) {
#pragma unroll
            for (int i = 0; i < kMI; ++i) {
                const int row = wm * kWM + 16 * i + r16;
                float rs = 1.0f;
                if constexpr (RS) rs = scale[row < last_row ? row : last_row];
                char* rowp = ctile + (row - ep * EP_ROWS) * PITCH;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    f32x4_t x = acc[j][i];
                    if constexpr (RS) x *= rs;
                    if constexpr (EPI == EPI_SILU_MUL) {
                        f32x4_t u = acc[j + NJ][i];
                        if constexpr (RS) u *= rs;
#pragma unroll
                        for (int v = 0; v < 4; ++v) x[v] = silu_f32(x[v]) * u[v];
                    }
                    char* dst = rowp + (wn * 16 * NJ + 16 * j + 4 * quad) * OB;
                    if constexpr (DT_OUT == NANOVLLM_GEMM_F32) *reinterpret_cast<f32x4_t*>(dst) = x;
                    else *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{pack2<DT_OUT>(x[0], x[1]), pack2<DT_OUT>(x[2], x[3])};
                }
            }
        }
        __syncthreads();
        const int64_t mp = m0 + int64_t(ep) * EP_ROWS;
        if (c_vec && mp + EP_ROWS <= m && n0 + BNO <= n) {
#pragma unroll
            for (int pass = 0; pass < EP_ROWS / ROWS_PER_PASS; ++pass) {
                const int r = tid / CPR + pass * ROWS_PER_PASS;
                const u32x4_t val = *reinterpret_cast<const u32x4_t*>(ctile + r * PITCH + chunk * 16);
                __builtin_nontemporal_store(
                    val, reinterpret_cast<u32x4_t*>(static_cast<char*>(c) + ((mp + r) * ldc + n0 + chunk * EPC) * OB));
            }
            continue;
        }
        if (!c_vec) {
            store_unaligned<OB, EP_ROWS, BNO, kThreads>(ctile, PITCH, static_cast<char*>(c) + (mp * ldc + n0) * OB, ldc,
                                                        m - mp, n - n0, tid);
            continue;
        }
        for (int r = tid / CPR; r < EP_ROWS; r += ROWS_PER_PASS) {
            const int64_t grow = mp + r;
            const int64_t gcol = n0 + chunk * EPC;
            if (grow >= m || gcol >= n) continue;
            const u32x4_t val = *reinterpret_cast<const u32x4_t*>(ctile + r * PITCH + chunk * 16);
            char* gdst = static_cast<char*>(c) + (grow * ldc + gcol) * OB;
            if (gcol + EPC <= n) {
                __builtin_nontemporal_store(val, reinterpret_cast<u32x4_t*>(gdst));
            } else {
                const int valid = int(min_i64(EPC, n - gcol));
                if constexpr (OB == 4) {
                    for (int e = 0; e < valid; ++e) reinterpret_cast<uint32_t*>(gdst)[e] = val[e];
                } else {
                    for (int e = 0; e < valid; ++e)
                        reinterpret_cast<uint16_t*>(gdst)[e] = uint16_t(val[e >> 1] >> (16 * (e & 1)));
                }
            }
        }
    }
}

template <int DT, int DT_OUT, int EPI, int RS>
int launch_tile(const Problem& p, hipStream_t s) {
    constexpr int BNO = EPI == EPI_SILU_MUL ? kBN / 2 : kBN;
    const int64_t tiles = ((p.m + kBM - 1) / kBM) * ((p.n + BNO - 1) / BNO);
    if (tiles > INT32_MAX) return set_error(NANOVLLM_GEMM_EINVAL, "mfma_wide: grid too large");
    const int out_bytes = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    // The copy-out writes 16-byte chunks: every row start must be 16-byte aligned.
    const int c_vec = (reinterpret_cast<uintptr_t>(p.c) % 16 == 0) && ((p.ldc * out_bytes) % 16 == 0);
    hipLaunchKernelGGL((mfma_wide_kernel<DT, DT_OUT, EPI, RS>), dim3(static_cast<uint32_t>(tiles)), dim3(kThreads), 0, s,
                       static_cast<const uint16_t*>(p.a), static_cast<const uint16_t*>(p.b), p.m, p.n, p.k, p.lda,
                       p.ldb, p.c, p.ldc, c_vec, p.row_scale);
    return check_launch("mfma_wide", kBM, BNO);
}

template <int DT, int DT_OUT>
int launch_typed(const Problem& p, hipStream_t s) {
    if (p.row_scale != nullptr) {
        if (p.epi == EPI_SILU_MUL) return launch_tile<DT, DT_OUT, EPI_SILU_MUL, 1>(p, s);
        return launch_tile<DT, DT_OUT, EPI_NONE, 1>(p, s);
    }
    if (p.epi == EPI_SILU_MUL) return launch_tile<DT, DT_OUT, EPI_SILU_MUL, 0>(p, s);
    return launch_tile<DT, DT_OUT, EPI_NONE, 0>(p, s);
}

}  // namespace

// Which grids take 256 x 256 tiles: those whose time on them, from a cost
// model in units of 10 ns fitted to bf16 timings over M 512-8192, N 1024-12288
// and K 256-4096 (kt K-tiles), is below that of the 128-row tiles:
//   * 256 x 256, one workgroup per CU: 8 + 1.25 kt us per full round of 256
//     tiles, 4.5 + 0.9 kt us for a partial one plus up to 3.5 + 0.28 kt us as
//     it fills (the chip clocks higher with CUs idle);
//   * 128 x 256 (gemm_mid.hip): 1.6 us, 4.8 + 0.73 kt us per full round, 2.2 +
//     0.48 kt us for a partial one plus up to 1.2 + 0.27 kt us as it fills; or 4 +
//     1.08 kt us on 128 x 128 tiles where those are at most 512, two to each CU.
// Both sides measured (us, 128-row tiles against 256 x 256), K = 1024: 272 tiles
// of 128 x 256 28.6 / 25.3, 320 28.5 / 25.7, 416 31.5 / 28.9, 896 (SiLU pairs) 66.0 /
// 59.4, 1579 x 4992 (260, and 507 of 128 x 128) 21.6 / 24.6 (not taken), 576 44.4 /
// 50.2 and 768 49.4 / 53.5 (not taken); K = 512: 416 20.4 / 19.2, 768 31.9 / 34.3
// (not taken); K = 3072: 272 68.2 / 59.7, 576 109 / 123 (not taken).  Up to 8
// K-tiles the model has to promise 7%: a partial round there costs more than it
// says (K = 256: 624 tiles of 128 x 256 (f16) 21.1 / 23.1, 750 21.6 / 23.8, 646 (SiLU
// pairs) 25.4 / 26.3; K = 480, 1050 (f16) 59.9 / 61.3; not taken).  fp16 inputs
// and fp32 outputs go by the same rule: over 550 random grids with all of them,
// K 256 to 1040, none was slower by more than 3% than on mfma_staged's tiles.
bool mfma_wide_pays(const Problem& p) {
    if (p.b_layout != NANOVLLM_GEMM_B_NK || p.k < 256 || p.k > (int64_t(1) << 30)) return false;
    if (p.epi != EPI_NONE && p.epi != EPI_SILU_MUL) return false;
    // 32-bit byte offsets from a tile's first rows.
    constexpr int64_t kRange = int64_t(1) << 31;
    const int64_t w_rows = p.epi == EPI_SILU_MUL ? p.n + kBN : kBN;
    if (p.lda >= kRange / (2 * kBM) || p.ldb >= kRange / (2 * w_rows)) return false;
    const int64_t cols = p.epi == EPI_SILU_MUL ? 2 * p.n : p.n;
    const int64_t tiles_n = (cols + kBN - 1) / kBN;
    const int64_t wide = (p.m + kBM - 1) / kBM * tiles_n;
    const int64_t narrow = (p.m + 127) / 128 * tiles_n;   // 128 x 256 tiles
    constexpr int64_t kCus = 256;
    if (narrow <= kCus) return false;
    const int64_t kt = (p.k + kBK - 1) / kBK;
    const int64_t rest = wide % kCus;
    const int64_t wide_cost =
        wide / kCus * (800 + 125 * kt) + (rest > 0 ? 450 + 90 * kt + rest * (350 + 28 * kt) / kCus : 0);
    const int64_t tiles128 = (p.m + 127) / 128 * ((cols + 127) / 128);
    const int64_t part = narrow % kCus;
    int64_t narrow_cost =
        160 + narrow / kCus * (480 + 73 * kt) + (part > 0 ? 220 + 48 * kt + part * (120 + 27 * kt) / kCus : 0);
    if (tiles128 <= 2 * kCus && 400 + 108 * kt < narrow_cost) narrow_cost = 400 + 108 * kt;
    return wide_cost * 100 < narrow_cost * (kt <= 8 ? 93 : 100);
}

int launch_mfma_wide(const Problem& p, hipStream_t s) {
    if (p.dtype_in == NANOVLLM_GEMM_BF16) {
        if (p.dtype_out == NANOVLLM_GEMM_BF16) return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_BF16>(p, s);
        return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_F32>(p, s);
    }
    if (p.dtype_out == NANOVLLM_GEMM_F16) return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F16>(p, s);
    return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F32>(p, s);
}

}  // namespace nvg
