// mfma_mid: mfma_staged's 128 x 256 and 128 x 128 tiles, C[M,N] = A[M,K] *
// W[N,K]^T, for grids of about one round on the CUs, where 256 x 256 tiles leave
// half of them idle.  A 128 x 256 tile copies 48 KiB per K-tile of 64, 48 bytes
// per clock of its MFMAs and about what copies into LDS sustain (128 x 128: 64),
// so copies, fragment reads and MFMAs have to overlap over the whole K-tile:
//   * fragments are reloaded in place as soon as their MFMAs have issued, a
//     K-step ahead;
//   * one barrier per K-tile, inside its second half: by then every fragment of
//     the K-tile has been read, so its stage of the 3-deep ring is refilled (one
//     copy per wave and group of MFMAs through the following K-tile), and the
//     next K-tile, whose copies are a K-tile old, is read;
//   * 8 waves: 4 of 128 x 64 read 96 KiB of fragments per K-tile against 128, but
//     start and store slower (2048 x 4096 x 1024 19.8 against 18.3 us, x 4096 56.0
//     / 54.1);
//   * v_mfma_f32_16x16x32, which the chip clocks higher than 32x32x16 and which
//     sums K in the same order: outputs keep the bits of the other tiles.
#include <type_traits>

#include "gemm_common.hpp"

namespace nvg {
namespace {

constexpr int kBM = 128, kBK = 64;
constexpr int kChunks = kBK / 8;
constexpr int kStages = 3;
constexpr int kThreads = 512;                   // 8 waves, 2 x 4 over the tile
constexpr int kWM = kBM / 2, kMI = kWM / 16;

__device__ u32x4_t g_mid_zero = {0u, 0u, 0u, 0u};

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// dma16 from a scalar base and a 32-bit byte offset per lane.
__device__ __forceinline__ void dma16_at(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %2"
                 :: "v"(off), "s"(lds), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop

// BN: 256 or 128 W rows per tile.
template <int DT, int DT_OUT, int EPI, int RS, int BN>
__global__ __launch_bounds__(kThreads) void mfma_mid_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, int64_t m, int64_t n, int64_t k, int64_t lda,
    int64_t ldb, void* __restrict__ c, int64_t ldc, int c_vec, const float* __restrict__ row_scale) {
    constexpr int kWN = BN / 4, kNI = kWN / 16;
    constexpr int kStageChunks = (kBM + BN) * kChunks;   // 48 or 32 KiB
    constexpr int kCopies = (kBM + BN) / 64;             // copy instructions per wave and K-tile
    constexpr int kWCopies = BN / 64;                    // of which W rows
    constexpr int kHalf = kCopies / 2;
    constexpr int kAt = kMI - kHalf;   // group of the second half that opens with the barrier
    static_assert(EPI != EPI_SILU_MUL || BN == 256, "gate/up pairs per wave");
    constexpr int BNO = EPI == EPI_SILU_MUL ? BN / 2 : BN;   // output columns per tile
    constexpr int OB = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    constexpr int PITCH = BNO * OB + 16;
    constexpr int RING_BYTES = kStages * kStageChunks * 16;
    static_assert(kBM * PITCH <= RING_BYTES, "the C tile takes the ring's place");
    __shared__ u32x4_t ring[RING_BYTES / 16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;
    const int r16 = lane & 15, quad = lane >> 4;
    const int tiles_m = static_cast<int>((m + kBM - 1) / kBM);
    const int tiles_n = static_cast<int>((n + BNO - 1) / BNO);
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int64_t m0 = int64_t(tm) * kBM, n0 = int64_t(tn) * BNO;

    // Copy instruction j of a wave fills 8 LDS rows, lane L row L / 8, position
    // L % 8, which holds logical chunk (L % 8) ^ ((row >> 1) & 7).  j <
    // kWCopies: W rows (EPI_SILU_MUL alternates 32 gate rows and the 32 up rows
    // of the same output columns); the others: A rows.
    auto copy_row = [&](int j) { return j < kWCopies ? kBM + 8 * (kWCopies * wave + j) : 8 * ((kCopies - kWCopies) * wave + j - kWCopies); };
    const uint16_t* abase = a + m0 * lda;
    const uint16_t* wbase = w + n0 * ldb;
    uint32_t off[kCopies];
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
        const int row = copy_row(j) + (lane >> 3);
        const int chunk = (lane & 7) ^ ((row >> 1) & 7);
        int64_t src;
        if (j >= kWCopies) {
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
    using No = std::false_type;
    // Copy j of K-tile t into `stage`; last_c: t may be the last K-tile.
    auto copy = [&](int t, int stage, int j, auto last_c) {
        const uint16_t* kb = (j < kWCopies ? wbase : abase) + int64_t(t) * kBK;
        const uint32_t dst = lds0 + uint32_t(stage * kStageChunks) * 16u + uint32_t(copy_row(j)) * 128u;
        if (!decltype(last_c)::value || (t + 1) * kBK <= k) {
            dma16_at(kb, off[j], dst);
        } else {
            // The last K-tile of a K that is not a multiple of 64: chunks
            // past K copy zeros.
            const int chunk = (lane & 7) ^ (((copy_row(j) + (lane >> 3)) >> 1) & 7);
            const void* src = t * kBK + chunk * 8 < k ? reinterpret_cast<const char*>(kb) + off[j]
                                                      : reinterpret_cast<const char*>(&g_mid_zero);
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

    // Prologue: K-tiles 0 and 1, and the first half of K-tile 2's copies (K >=
    // 256 is the launcher's rule, so K-tile 3 exists).
#pragma unroll
    for (int j = 0; j < kCopies; ++j) copy(0, 0, j, No{});
#pragma unroll
    for (int j = 0; j < kCopies; ++j) copy(1, 1, j, No{});
#pragma unroll
    for (int j = 0; j < kHalf; ++j) copy(2, 2, j, No{});
    asm volatile("" :: "s"(c), "s"(ldc), "s"(c_vec), "s"(m), "s"(n), "s"(row_scale));
    wait_vmcnt<kCopies + kHalf>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    barrier();
#pragma unroll
    for (int i = 0; i < kNI; ++i) wf0[i] = read_w(0, 0, i);
#pragma unroll
    for (int i = 0; i < kMI; ++i) af[i] = read_a(0, 0, i);

    int cur = 0;   // ring stage of K-tile t
    // LEFT: how many K-tiles follow t, capped at 4 (K-tile t + 3 is then not
    // the last).
    auto k_tile = [&](int t, auto left_c) {
        constexpr int LEFT = decltype(left_c)::value;
        const int next = cur + 1 == kStages ? 0 : cur + 1;
        const int after = next + 1 == kStages ? 0 : next + 1;
        constexpr std::integral_constant<bool, LEFT == 2> last2{};   // t + 2 is the last K-tile
        constexpr std::integral_constant<bool, LEFT == 3> last3{};   // t + 3 is
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < kNI; ++j) acc[j][i] = mfma_16x16x32<DT>(wf0[j], af[i], acc[j][i]);
            if (i < kNI) wf1[i] = read_w(cur, 1, i);
            af[i] = read_a(cur, 1, i);
            if constexpr (LEFT >= 2)
                if (i < kHalf) copy(t + 2, after, kHalf + i, last2);
        }
#pragma unroll
        for (int i = 0; i < kMI; ++i) {
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (LEFT >= 1) {
                if (i == kAt) {
                    // K-tile t + 1 has landed in every wave's part, and every
                    // wave has read all of K-tile t.
                    if constexpr (LEFT >= 2) wait_vmcnt<kCopies>();
                    else wait_vmcnt<0>();
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    barrier();
                }
            }
#pragma unroll
            for (int j = 0; j < kNI; ++j) acc[j][i] = mfma_16x16x32<DT>(wf1[j], af[i], acc[j][i]);
            if constexpr (LEFT >= 1) {
                if (i >= kAt) {
#pragma unroll
                    for (int j = (i - kAt) * kNI / kHalf; j < (i - kAt + 1) * kNI / kHalf; ++j) wf0[j] = read_w(next, 0, j);
                    if (i < 2 * kAt) af[i - kAt] = read_a(next, 0, i - kAt);
                    af[i] = read_a(next, 0, i);
                }
            }
            if constexpr (LEFT >= 3)
                if (i >= kAt) copy(t + 3, cur, i - kAt, last3);
        }
        __builtin_amdgcn_sched_barrier(0);
        cur = next;
    };
    static_assert(kAt >= 1 && 2 * kAt <= kMI, "one copy per group behind the barrier");
    int t = 0;
    for (; t + 4 < ktiles; ++t) k_tile(t, std::integral_constant<int, 4>{});
    k_tile(t++, std::integral_constant<int, 3>{});
    k_tile(t++, std::integral_constant<int, 2>{});
    k_tile(t++, std::integral_constant<int, 1>{});
    k_tile(t, std::integral_constant<int, 0>{});

    // Epilogue through LDS: acc[j][i][v] is output row 16 i + l % 16, column
    // 16 j + 4 (l / 16) + v of the wave tile.
    constexpr int CPR = BNO * OB / 16;
    constexpr int EPC = 16 / OB;
    constexpr int ROWS_PER_PASS = kThreads / CPR;
    constexpr int NJ = EPI == EPI_SILU_MUL ? kNI / 2 : kNI;
    static_assert(kThreads % CPR == 0 && kBM % ROWS_PER_PASS == 0, "copy passes");
    char* ctile = reinterpret_cast<char*>(ring);
    const int chunk = tid % CPR;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMI; ++i) {
        const int row = wm * kWM + 16 * i + r16;
        float rs = 1.0f;
        if constexpr (RS) rs = row_scale[min_i64(m0 + row, m - 1)];
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
            char* dst = ctile + row * PITCH + (wn * 16 * NJ + 16 * j + 4 * quad) * OB;
            if constexpr (OB == 4) *reinterpret_cast<f32x4_t*>(dst) = x;
            else *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{pack2<DT_OUT>(x[0], x[1]), pack2<DT_OUT>(x[2], x[3])};
        }
    }
    __syncthreads();
    if (c_vec && m0 + kBM <= m && n0 + BNO <= n) {
#pragma unroll
        for (int pass = 0; pass < kBM / ROWS_PER_PASS; ++pass) {
            const int r = tid / CPR + pass * ROWS_PER_PASS;
            const u32x4_t val = *reinterpret_cast<const u32x4_t*>(ctile + r * PITCH + chunk * 16);
            __builtin_nontemporal_store(
                val, reinterpret_cast<u32x4_t*>(static_cast<char*>(c) + ((m0 + r) * ldc + n0 + chunk * EPC) * OB));
        }
        return;
    }
    if (!c_vec) {
        store_unaligned<OB, kBM, BNO, kThreads>(ctile, PITCH, static_cast<char*>(c) + (m0 * ldc + n0) * OB, ldc, m - m0,
                                                n - n0, tid);
        return;
    }
    for (int r = tid / CPR; r < kBM; r += ROWS_PER_PASS) {
        const int64_t grow = m0 + r;
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

template <int DT, int DT_OUT, int EPI, int RS, int BN>
int launch_tile(const Problem& p, hipStream_t s) {
    constexpr int BNO = EPI == EPI_SILU_MUL ? BN / 2 : BN;
    const int64_t tiles = ((p.m + kBM - 1) / kBM) * ((p.n + BNO - 1) / BNO);
    if (tiles > INT32_MAX) return set_error(NANOVLLM_GEMM_EINVAL, "mfma_mid: grid too large");
    const int out_bytes = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    // The copy-out writes 16-byte chunks: every row start must be 16-byte aligned.
    const int c_vec = (reinterpret_cast<uintptr_t>(p.c) % 16 == 0) && ((p.ldc * out_bytes) % 16 == 0);
    hipLaunchKernelGGL((mfma_mid_kernel<DT, DT_OUT, EPI, RS, BN>), dim3(static_cast<uint32_t>(tiles)), dim3(kThreads), 0, s,
                       static_cast<const uint16_t*>(p.a), static_cast<const uint16_t*>(p.b), p.m, p.n, p.k, p.lda,
                       p.ldb, p.c, p.ldc, c_vec, p.row_scale);
    return check_launch("mfma_mid", kBM, BNO);
}

constexpr int64_t kCus = 256;

int64_t tiles(const Problem& p, int64_t w_rows) {
    const int64_t rows = p.epi == EPI_SILU_MUL ? 2 * p.n : p.n;
    return (p.m + kBM - 1) / kBM * ((rows + w_rows - 1) / w_rows);
}

template <int DT, int DT_OUT, int RS>
int launch_plain(const Problem& p, hipStream_t s) {
    if (tiles(p, 256) <= kCus / 2) return launch_tile<DT, DT_OUT, EPI_NONE, RS, 128>(p, s);
    return launch_tile<DT, DT_OUT, EPI_NONE, RS, 256>(p, s);
}

template <int DT, int DT_OUT>
int launch_typed(const Problem& p, hipStream_t s) {
    if (p.row_scale != nullptr) {
        if (p.epi == EPI_SILU_MUL) return launch_tile<DT, DT_OUT, EPI_SILU_MUL, 1, 256>(p, s);
        return launch_plain<DT, DT_OUT, 1>(p, s);
    }
    if (p.epi == EPI_SILU_MUL) return launch_tile<DT, DT_OUT, EPI_SILU_MUL, 0, 256>(p, s);
    return launch_plain<DT, DT_OUT, 0>(p, s);
}

}  // namespace

// Which grids take them (bf16, us, against mfma_staged's form of the same tile
// or of 128 x 128 where that was the choice):
//   * more than half a round of 128 x 256 tiles: 2048 x 4096 x 1024 20.7 -> 18.3,
//     x 4096 62.7 -> 54.1, 2048 x 2304 x 1024 (144 tiles) 15.8 -> 14.9, 8192 x 1024
//     x 3584 55.5 -> 48.2; beyond one round where 256 x 256 do not pay (that rule
//     comes first): 3072 x 6144 x 1024 49.4 -> 44.4, 4096 x 6144 x 3072 137 ->
//     119; but not from 257 tiles while those of 128 x 128 are at most 512, two
//     to each CU (1579 x 4992 x 1024 21.6 against 28.6);
//   * half a round to a round of 128 x 128: 4096 x 1024 x 3584 33.9 -> 30.1 (fp16
//     36.1 -> 32.0), 2048 x 2048 x 1024 13.0 -> 11.7, x 264 7.8 -> 7.3; on 128 x
//     256 these take 15.1 (2048 x 2048 x 1024).  Gate/up pairs of a wave need 64
//     W rows, so they have no 128 x 128.
bool mfma_mid_pays(const Problem& p) {
    if (p.b_layout != NANOVLLM_GEMM_B_NK || p.k < 4 * kBK || p.k > (int64_t(1) << 30)) return false;
    if (p.epi != EPI_NONE && p.epi != EPI_SILU_MUL) return false;
    // 32-bit byte offsets from a tile's first rows.
    constexpr int64_t kRange = int64_t(1) << 31;
    const int64_t w_rows = p.epi == EPI_SILU_MUL ? p.n + 256 : 256;
    if (p.lda >= kRange / (2 * kBM) || p.ldb >= kRange / (2 * w_rows)) return false;
    const int64_t t256 = tiles(p, 256), t128 = tiles(p, 128);
    if (t256 > kCus / 2) return t256 <= kCus || t128 > 2 * kCus;
    return p.epi == EPI_NONE && t128 > kCus / 2;
}

int launch_mfma_mid(const Problem& p, hipStream_t s) {
    if (p.dtype_in == NANOVLLM_GEMM_BF16) {
        if (p.dtype_out == NANOVLLM_GEMM_BF16) return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_BF16>(p, s);
        return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_F32>(p, s);
    }
    if (p.dtype_out == NANOVLLM_GEMM_F16) return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F16>(p, s);
    return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F32>(p, s);
}

}  // namespace nvg
