// mfma_ragged: mfma_direct's form for problems whose rows are no aligned
// 16-byte chunks (odd K or N, odd leading dimensions, unaligned pointers), for
// either B layout.  Reading MFMA operands of such rows straight from memory
// takes one load per element; here
//   * operands are read 8 elements at a time with 16-byte loads at their own
//     2-byte alignment, coalesced along the rows, two K-tiles ahead of the
//     multiply, through registers into a double-buffered LDS tile;
//   * a chunk that would end past its row's end (K for A and W[N,K], N for
//     B[K,N]) is read where it ends exactly there and shifted into place, so
//     no load leaves its row and elements past the end are zero; rows past M,
//     N or K are read from the last one, and k-rows past K are zeroed;
//   * LDS holds what mfma_staged and splitk_decode hold (chunk c of row r at
//     c ^ ((r >> 1) & 7); B[K,N] as panels of 64 columns read back with the
//     transposing LDS read), and v_mfma_f32_16x16x32 sums K in order.
// 333 x 1001 x 1003, bf16 to fp32: 87.8 -> 8.3 us.
#include <type_traits>

#include "gemm_common.hpp"

namespace nvg {
namespace {

typedef uint32_t u32x4_any_t __attribute__((ext_vector_type(4), aligned(2)));

// 16 bytes at 2-byte alignment.
__device__ __forceinline__ u32x4_t load16_any(const uint16_t* p) {
    return *reinterpret_cast<const u32x4_any_t*>(p);
}

// The last `keep` of 8 elements moved to the front, zeros behind them (all
// zero when keep <= 0; the chunk as it is when keep >= 8).
__device__ __forceinline__ u32x4_t keep_last(u32x4_t x, int64_t keep) {
    if (keep >= 8) return x;
    if (keep <= 0) return u32x4_t{0u, 0u, 0u, 0u};
    const int s = 16 * (8 - int(keep));   // 16 .. 112 bits
    const uint64_t lo = uint64_t(x[0]) | (uint64_t(x[1]) << 32), hi = uint64_t(x[2]) | (uint64_t(x[3]) << 32);
    const uint64_t l = s >= 64 ? hi >> (s - 64) : (lo >> s) | (hi << (64 - s));
    const uint64_t h = s >= 64 ? 0 : hi >> s;
    return u32x4_t{uint32_t(l), uint32_t(l >> 32), uint32_t(h), uint32_t(h >> 32)};
}

// Column chunks of B[K,N] k-rows within a panel of 64 columns; the key of
// splitk_decode's B[K,N] lines (conflict-free for the transposing reads).
__device__ __forceinline__ int panel_swizzle(int r) { return 2 * (((r >> 1) & 1) | ((r >> 2) & 2)); }

// BM x BN tile on WGM x WGN waves, K-tiles of KS * 64 elements.
template <int DT, int DT_OUT, int BL, int BM, int BN, int KS, int WGM, int WGN>
__global__ __launch_bounds__(WGM * WGN * 64) void mfma_ragged_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ b, void* __restrict__ c, int64_t m, int64_t n,
    int64_t k, int64_t lda, int64_t ldb, int64_t ldc, int tiles_m, int tiles_n) {
    constexpr bool KN = BL == NANOVLLM_GEMM_B_KN;
    constexpr int NT = WGM * WGN * 64;
    constexpr int BK = 64 * KS;
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int MI = WM / 16, NI = WN / 16;     // 16 x 16 blocks of a wave tile
    constexpr int ACH = KS * BM * 8;              // 16-byte chunks of A per stage
    constexpr int STAGE = ACH + KS * BN * 8;
    constexpr int LPT = STAGE / NT, LA = ACH / NT;   // loads per thread, of which A
    static_assert(LPT * NT == STAGE && LA * NT == ACH && WM % 16 == 0 && WN % 16 == 0, "whole loads and blocks");
    constexpr int PC = BN < 64 ? BN / 8 : 8;      // column chunks of a B[K,N] panel
    constexpr int OB = DT_OUT == NANOVLLM_GEMM_F32 ? 4 : 2;
    constexpr int PITCH = BN * OB + 16;
    constexpr int LDS = 2 * STAGE * 16 > BM * PITCH ? 2 * STAGE * 16 : BM * PITCH;
    __shared__ u32x4_t lds[LDS / 16];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int r16 = lane & 15, quad = lane >> 4;
    int tm, tn;
    grouped_tile(xcd_remap(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, 8, tm, tn);
    const int64_t m0 = int64_t(tm) * BM, n0 = int64_t(tn) * BN;
    const int kk = static_cast<int>(k);

    // Load j of a thread: chunk q = j NT + tid of its operand's part of a
    // K-tile.  src: its row (A, W[N,K]) or column chunk (B[K,N]); kpos: its
    // first k (or k-row) within the K-tile; dst: its place in a stage.
    const uint16_t* src[LPT];
    int kpos[LPT], dst[LPT];
#pragma unroll
    for (int j = 0; j < LPT; ++j) {
        const int q = (j < LA ? j : j - LA) * NT + tid;
        if (j < LA || !KN) {
            const int rows = j < LA ? BM : BN;
            const int sub = q / (rows * 8), r = (q >> 3) % rows, ch = q & 7;
            src[j] = j < LA ? a + min_i64(m0 + r, m - 1) * lda : b + min_i64(n0 + r, n - 1) * ldb;
            kpos[j] = 64 * sub + 8 * ch;
            dst[j] = (j < LA ? 0 : ACH) + (sub * rows + r) * 8 + (ch ^ ((r >> 1) & 7));
        } else {
            const int kr = q / (BN / 8), cc = q % (BN / 8);
            src[j] = b + min_i64(n0 + 8 * cc, n - 8);
            kpos[j] = kr;
            dst[j] = ACH + (((kr >> 6) * (BN / 8 / PC) + cc / PC) * 64 + (kr & 63)) * PC +
                     ((cc % PC) ^ (panel_swizzle(kr) & (PC - 1)));
        }
    }
    u32x4_t rs[2][LPT];
    // Every load is issued unconditionally from inside its row; what lies past
    // the ends is settled when the tile goes to LDS.
    auto load_tile = [&](int k0, auto set_c) {
        constexpr int S = decltype(set_c)::value;
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            const int kq = k0 + kpos[j];
            if (j < LA || !KN) rs[S][j] = load16_any(src[j] + (kq < kk - 8 ? kq : kk - 8));
            else rs[S][j] = load16_any(src[j] + int64_t(kq < kk - 1 ? kq : kk - 1) * ldb);
        }
    };
    const bool col_edge = KN && n0 + BN > n;   // B[K,N] column chunks that N cuts
    auto store_tile = [&](int st, int k0, auto set_c) {
        constexpr int S = decltype(set_c)::value;
        if (k0 + BK > kk || col_edge) {
#pragma unroll
            for (int j = 0; j < LPT; ++j) {
                const int left = kk - (k0 + kpos[j]);
                u32x4_t v;
                if (j < LA || !KN) v = keep_last(rs[S][j], left);
                else v = keep_last(rs[S][j], left > 0 ? n - (n0 + 8 * (((j - LA) * NT + tid) % (BN / 8))) : 0);
                lds[st * STAGE + dst[j]] = v;
            }
        } else {
#pragma unroll
            for (int j = 0; j < LPT; ++j) lds[st * STAGE + dst[j]] = rs[S][j];
        }
    };
    // This wave's LDS accesses have completed, then all waves meet;
    // __syncthreads() would also drain the global loads in flight.
    auto lds_barrier = [&] {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    f32x4_t acc[NI][MI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) acc[i][j] = f32x4_t{};

    const int swz = (r16 >> 1) & 7;
    auto multiply = [&](int st) {
        const u32x4_t* tile = lds + st * STAGE;
#pragma unroll
        for (int s = 0; s < 2 * KS; ++s) {
            const int sub = s >> 1, ch = (4 * (s & 1) + quad) ^ swz;
            u32x4_t af[MI], wf[NI];
#pragma unroll
            for (int i = 0; i < MI; ++i) af[i] = tile[(sub * BM + wm * WM + 16 * i + r16) * 8 + ch];
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if constexpr (KN) {
                    // Lane 16 g + j points at k-row 32 s + 8 g + j / 4 (+ 4 for
                    // the second read) and columns 4 (j % 4) .. + 3 of the block;
                    // lane 16 g + i receives k = 32 s + 8 g .. + 7 of column i.
                    typedef short v4i16_t __attribute__((ext_vector_type(4)));
                    typedef __attribute__((address_space(3))) v4i16_t* lds_v4;
                    const int kr = 32 * (s & 1) + 8 * quad + (r16 >> 2);
                    const int col = wn * WN + 16 * i;
                    const u32x4_t* panel = tile + ACH + (sub * (BN / 8 / PC) + col / (8 * PC)) * 64 * PC;
                    const int cc = (col / 8 % PC + ((r16 & 3) >> 1)) ^ (panel_swizzle(kr) & (PC - 1));
                    const uint32_t a0 = lds_address(panel) + uint32_t(kr * PC + cc) * 16u + 8u * (r16 & 1);
                    const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(uintptr_t)a0));
                    const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4)(uintptr_t)(a0 + 64u * PC)));
                    wf[i] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
                } else {
                    wf[i] = tile[ACH + (sub * BN + wn * WN + 16 * i + r16) * 8 + ch];
                }
            }
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < MI; ++j) acc[i][j] = mfma_16x16x32<DT>(wf[i], af[j], acc[i][j]);
        }
    };

    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, 1>;
    const int ktiles = (kk + BK - 1) / BK;
    load_tile(0, Set0{});
    if (ktiles > 1) load_tile(BK, Set1{});
    store_tile(0, 0, Set0{});
    if (ktiles > 2) load_tile(2 * BK, Set0{});
    lds_barrier();
    // K-tile t: K-tile t + 1 (in set (t + 1) % 2) goes to the free stage, its
    // registers take K-tile t + 3.
    auto step = [&](int t, auto set_c) {
        if (t + 1 < ktiles) store_tile((t + 1) & 1, (t + 1) * BK, set_c);
        if (t + 3 < ktiles) load_tile((t + 3) * BK, set_c);
        __builtin_amdgcn_s_setprio(3);
        multiply(t & 1);
        __builtin_amdgcn_s_setprio(0);
        lds_barrier();
    };
    for (int t = 0; t < ktiles; t += 2) {
        step(t, Set1{});
        if (t + 1 < ktiles) step(t + 1, Set0{});
    }

    // Output through LDS: acc[i][j][v] is row 16 j + l % 16, column 16 i +
    // 4 (l / 16) + v of the wave tile.  Rows of C have any alignment, so
    // adjacent lanes store adjacent elements.
    char* ctile = reinterpret_cast<char*>(lds);
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const f32x4_t x = acc[i][j];
            char* p = ctile + (wm * WM + 16 * j + r16) * PITCH + (wn * WN + 16 * i + 4 * quad) * OB;
            if constexpr (OB == 4) *reinterpret_cast<f32x4_t*>(p) = x;
            else *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack2<DT_OUT>(x[0], x[1]), pack2<DT_OUT>(x[2], x[3])};
        }
    __syncthreads();
    typedef std::conditional_t<OB == 4, uint32_t, uint16_t> elem_t;
    const int rows = static_cast<int>(min_i64(BM, m - m0)), cols = static_cast<int>(min_i64(BN, n - n0));
    elem_t* cp = static_cast<elem_t*>(c) + m0 * ldc + n0;
#pragma unroll 4
    for (int e = tid; e < BM * BN; e += NT) {
        const int r = e / BN, col = e % BN;
        if (r < rows && col < cols)
            __builtin_nontemporal_store(reinterpret_cast<const elem_t*>(ctile + r * PITCH)[col], cp + int64_t(r) * ldc + col);
    }
}

template <int DT, int DT_OUT, int BL, int BM, int BN, int KS, int WGM, int WGN>
int launch_tile(const Problem& p, hipStream_t s) {
    const int64_t tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
    if (tiles_m * tiles_n > INT32_MAX) return set_error(NANOVLLM_GEMM_EINVAL, "mfma_ragged: grid too large");
    hipLaunchKernelGGL((mfma_ragged_kernel<DT, DT_OUT, BL, BM, BN, KS, WGM, WGN>),
                       dim3(static_cast<uint32_t>(tiles_m * tiles_n)), dim3(WGM * WGN * 64), 0, s,
                       static_cast<const uint16_t*>(p.a), static_cast<const uint16_t*>(p.b), p.c, p.m, p.n, p.k, p.lda,
                       p.ldb, p.ldc, int(tiles_m), int(tiles_n));
    return check_launch("mfma_ragged", BM, BN);
}

// Tiles by grid size.  A CU takes these unaligned loads at about 16 bytes per
// clock, so small grids want their loads spread over as many CUs as there are,
// and large ones the reuse of a larger tile (bf16 and fp16, us):
//   * up to 512 tiles of 32 x 32: those, on K-tiles of 128 (333 x 1001 x 1003
//     8.3 against 8.8 / 10.6 on 32 x 64 / 64 x 64 tiles, 700 x 700 x 8001
//     39.7 against 41.6 / 62.9, 40 x 3000 x 1003 6.4 against 9.0 / 10.7);
//   * more of them at M <= 16: 16 x 32, which load no rows past M (14 x 15001 x
//     1003 7.6 against 9.0 / 9.1 / 12.2); with fewer 32 x 32 is level with it
//     (3 x 7000 x 7999 30.6 / 32.3, 14 x 4000 x 4031 18.5 / 17.9);
//   * up to 512 tiles of 64 x 64: 32 x 64 (130 x 6144 x 1003 12.5 against 13.3
//     on 32 x 32 and 15.3 on 64 x 64, B[K,N] 432 x 1664 x 4030 25.2 against
//     27.2 / 32.7);
//   * above: 64 x 64 (1500 x 2000 x 1502 27.3 against 30.7 on 32 x 64, 4000 x
//     1500 x 999 36.1 / 48.8; 128 x 128 tiles take 29.7 / 46.3).
template <int DT, int DT_OUT, int BL>
int launch_layout(const Problem& p, hipStream_t s) {
    const auto tiles = [&](int64_t bm, int64_t bn) { return ((p.m + bm - 1) / bm) * ((p.n + bn - 1) / bn); };
    if (p.m <= 16 && tiles(16, 32) > 256) return launch_tile<DT, DT_OUT, BL, 16, 32, 2, 1, 2>(p, s);
    if (tiles(32, 32) <= 512) return launch_tile<DT, DT_OUT, BL, 32, 32, 2, 2, 2>(p, s);
    if (tiles(64, 64) <= 512) return launch_tile<DT, DT_OUT, BL, 32, 64, 2, 2, 2>(p, s);
    return launch_tile<DT, DT_OUT, BL, 64, 64, 1, 2, 2>(p, s);
}

template <int DT, int DT_OUT>
int launch_typed(const Problem& p, hipStream_t s) {
    if (p.b_layout == NANOVLLM_GEMM_B_KN) return launch_layout<DT, DT_OUT, NANOVLLM_GEMM_B_KN>(p, s);
    return launch_layout<DT, DT_OUT, NANOVLLM_GEMM_B_NK>(p, s);
}

}  // namespace

// One whole chunk per row of every operand, and K-tiles counted in 32 bits.  On a
// K of a few elements a K-tile is mostly zeros, and mfma_direct's element loads are
// fewer (mfma_direct / these, bf16 and f16, us: 1482 x 925 x 11 (B[K,N]) 4.9 / 6.6,
// 469 x 841 x 15 4.0 / 4.5, 458 x 89 x 17 4.4 / 3.9; large grids 2499 x 1731 x 23
// (B[K,N]) 9.0 / 10.2, 2836 x 704 x 31 7.0 / 7.6, 4466 x 1677 x 33 21.6 / 12.6).
// B[K,N] behind rows of A that are aligned chunks needs more: mfma_direct reads
// those 16 bytes at a time, and its 64 x 64 tiles read B less often than 32 x 64,
// which tells while their last round is fuller than half: 284 x 5482 x 64 4.9 /
// 7.2, 7 x 4715 x 64 3.2 / 3.5, 16 x 7001 x 96 4.5 / 3.7; 646 x 2485 x 192 (429 tiles
// of 64 x 64) 8.3 / 10.1, 7672 x 119 x 256 (240) 6.7 / 7.3, 745 x 1861 x 128 (360) 6.5 /
// 5.8, 2854 x 470 x 256 9.4 / 7.3; 967 x 6951 x 72 11.2 / 14.5, 1313 x 2671 x 128 11.2
// / 8.4.
bool mfma_ragged_ok(const Problem& p) {
    const auto tiles = [&](int64_t t) { return (p.m + t - 1) / t * ((p.n + t - 1) / t); };
    const bool a_chunks = reinterpret_cast<uintptr_t>(p.a) % 16 == 0 && p.lda % 8 == 0 && p.k % 8 == 0;
    int64_t least = tiles(32) <= 512 ? 17 : 33;   // K
    if (p.b_layout == NANOVLLM_GEMM_B_KN && a_chunks) {
        const int64_t t64 = tiles(64);
        least = tiles(32) <= 512 ? 65 : t64 > 512 ? 88 : t64 <= 256 || t64 > 384 ? 257 : 65;
    }
    return p.k >= least && p.k < (int64_t(1) << 30) && (p.b_layout == NANOVLLM_GEMM_B_NK || p.n >= 8);
}

int launch_mfma_ragged(const Problem& p, hipStream_t s) {
    if (p.dtype_in == NANOVLLM_GEMM_BF16) {
        if (p.dtype_out == NANOVLLM_GEMM_BF16) return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_BF16>(p, s);
        return launch_typed<NANOVLLM_GEMM_BF16, NANOVLLM_GEMM_F32>(p, s);
    }
    if (p.dtype_out == NANOVLLM_GEMM_F16) return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F16>(p, s);
    return launch_typed<NANOVLLM_GEMM_F16, NANOVLLM_GEMM_F32>(p, s);
}

}  // namespace nvg
