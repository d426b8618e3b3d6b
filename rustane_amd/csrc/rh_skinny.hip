// rh_skinny.hip -- prefill GEMMs of few tokens (M <= SKINNY_M).
//
// A short prompt streams every weight once and does little else, so its floor
// is the weights' time from HBM, and the tile kernels leave most of that idle:
// their 128- to 256-row tiles give QKV 96 blocks and W2 32 for 256 CUs.  What
// bounds this shape is each CU's vector-memory path: loads return in order,
// so L2 hits queue behind HBM misses and a CU sustains about 45 - 50 GB/s of
// weight and token bytes together.  A block therefore owns RT row tiles of 16
// weight rows and all MT token tiles, with RT chosen so that about one block
// per CU is left (tokens are re-read once per block, MT / RT times the weight
// bytes), and its 8 waves split the block's k by 128-wide chunks, chunk c to
// wave c % 8 (a block's waves then read 32 KB runs of each row tile; a
// contiguous k range per wave measured 10 - 50% slower).  A wave keeps RING
// slices of 32 k of its rows and tokens in registers and refills a slice as
// soon as it is used (pinned: the compiler would gather the loads of a chunk
// behind all its MFMAs); weights are nontemporal.  The waves' sums meet in LDS
// in wave order (deterministic) and every wave stores a share of the tiles.
//
// S > 1: the chunks are split over S blocks per row group too, each writing an
// fp32 partial [M][N] at sk_part + s * M * N (the narrow Wo and W2, whose row
// kernel sums the partials).
//
// Measured (us, tile kernel -> this, weights from HBM): 7B, 45 tokens: QKV 36
// (stream-K and fix-up) -> 21, W1|W3 45 -> 35, W2 26 -> 19, Wo 8.7 -> 9.3 (half
// as many splits for its row kernel to read); 600M: QKV 13.5 -> 7.1, W1|W3 11.8 ->
// 7.9, W2 6.6 -> 5.5, Wo 5.0 -> 3.9.
#include <algorithm>

#include <hip/hip_ext.h>

#include "rh_device.h"
#include "rh_gemm_epi.h"
#include "rh_kernels.h"

namespace rh {
namespace {

template <int EPI, int RT, int MT, bool SPLIT>
__global__ __launch_bounds__(512) void gemm_skinny_kernel(GemmArgs a, int S) {
    constexpr int NW = 8, NH = NW / 2;
    constexpr int RING = RT * MT + 4 * (RT + MT) <= 52 ? 4 : 2;  // register slices that fit beside the sums
    __shared__ f32x4 red[NH][RT * MT][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nrt = (a.N + 15) >> 4, nxt = (a.M + 15) >> 4, nch = a.K >> 7;
    const int grp = SPLIT ? blockIdx.x / S : blockIdx.x, sp = SPLIT ? blockIdx.x - grp * S : 0;
    const int c0 = SPLIT ? sp * nch / S : 0, c1 = SPLIT ? (sp + 1) * nch / S : nch;
    const size_t rstride = (size_t)a.K * 16;  // halves of one 16-row block
    const f16 *wp[RT], *xp[MT];
    // rows and tokens past the last tile reread it; their results are not stored
#pragma unroll
    for (int t = 0; t < RT; ++t) wp[t] = a.W + (size_t)min(grp * RT + t, nrt - 1) * rstride + lane * 8;
#pragma unroll
    for (int j = 0; j < MT; ++j) xp[j] = a.X + (size_t)min(j, nxt - 1) * rstride + lane * 8;
    f32x4 acc[RT][MT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[t][j] = f32x4{};
    // this wave's chunks: c0 + w, c0 + w + NW, ... (< c1), 4 slices each
    const int n = c0 + w < c1 ? 4 * ((c1 - 1 - c0 - w) / NW + 1) : 0;
    f16x8 wb[RING][RT], xb[RING][MT];
    auto load = [&](int i, int u) {  // slice i < n of this wave
        const size_t o = (size_t)(c0 + w + (i >> 2) * NW) * 2048 + 512 * (i & 3);
#pragma unroll
        for (int t = 0; t < RT; ++t) wb[u][t] = ld_stream((const f16x8*)(wp[t] + o));
#pragma unroll
        for (int j = 0; j < MT; ++j) xb[u][j] = *(const f16x8*)(xp[j] + o);
    };
    auto slice = [&](int u) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j) acc[t][j] = mfma16(wb[u][t], xb[u][j], acc[t][j]);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (n > 0) {  // wave-uniform
#pragma unroll
        for (int u = 0; u < RING; ++u) load(u, u);
        __builtin_amdgcn_sched_barrier(0);
        for (int i = 0; i < n - 4; i += 4)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                slice(u % RING);
                load(i + u + RING, u % RING);
                __builtin_amdgcn_sched_barrier(0);
            }
        // the last chunk loads nothing past itself: with one to four chunks a
        // wave, RING slices too many are up to twice the bytes
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            slice(u % RING);
            if (u + RING < 4) {
                load(n - 4 + u + RING, u % RING);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // wave w + NH's sums join wave w's, then each tile adds NH sums in wave order
    if (w >= NH) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j) red[w - NH][t * MT + j][lane] = acc[t][j];
    }
    __syncthreads();
    if (w < NH) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < MT; ++j) red[w][t * MT + j][lane] += acc[t][j];
    }
    __syncthreads();
    GemmArgs b = a;
    if constexpr (SPLIT) {
        b.out_f32 = a.sk_part + (size_t)sp * a.M * a.N;
        b.ldo = a.N;
        b.softcap = 0.f;
        b.alpha = 0.f;  // raw partials: the row kernel applies alpha once to their sum
        b.part_cols = 0;
    }
    constexpr int PT = EPI == EPI_SWIGLU ? 2 : 1;  // row tiles stored together (W1 rows and the matching W3 rows)
    for (int x = w; x < RT / PT * MT; x += NW) {
        const int q = x / MT, j = x - q * MT;
        f32x4 s[PT];
#pragma unroll
        for (int t = 0; t < PT; ++t) {
            s[t] = red[0][(PT * q + t) * MT + j][lane];
#pragma unroll
            for (int v = 1; v < NH; ++v) s[t] += red[v][(PT * q + t) * MT + j][lane];
        }
        const int m = 16 * j + (lane & 15);
        if (m >= a.M) continue;
        if constexpr (EPI == EPI_SWIGLU) {
            const float h1[4] = {s[0][0], s[0][1], s[0][2], s[0][3]}, h3[4] = {s[1][0], s[1][1], s[1][2], s[1][3]};
            const int f = 16 * (grp * (RT / 2) + q) + 4 * (lane >> 4);
            if (f < a.ldo) store_swiglu<EPI>(b, m, f, h1, h3);
        } else {
            const int n4 = (grp * RT + q) * 16 + 4 * (lane >> 4);
            if (n4 < a.N) store4<EPI>(b, m, n4, s[0][0], s[0][1], s[0][2], s[0][3]);
        }
    }
}

// MTM: the most token tiles there is a kernel for.
template <int EPI, int RT, bool SPLIT, int MTM = 4>
hipError_t launch_rt(const GemmArgs& a, int S, hipStream_t st) {
    const dim3 grid((a.N + 16 * RT - 1) / (16 * RT) * S), blk(512);
#define RH_SKN(MT_)                                                                                              \
    case MT_:                                                                                                    \
        if constexpr (MT_ > MTM)                                                                                 \
            return hipErrorInvalidValue;                                                                         \
        else if (a.prof_start)                                                                                   \
            hipExtLaunchKernelGGL((gemm_skinny_kernel<EPI, RT, MT_, SPLIT>), grid, blk, 0, st, a.prof_start,     \
                                  a.prof_stop, 0u, a, S);                                                        \
        else                                                                                                     \
            hipLaunchKernelGGL((gemm_skinny_kernel<EPI, RT, MT_, SPLIT>), grid, blk, 0, st, a, S);               \
        break
    switch ((a.M + 15) / 16) {
        RH_SKN(1); RH_SKN(2); RH_SKN(3); RH_SKN(4);
        default: return hipErrorInvalidValue;
    }
#undef RH_SKN
    return hipGetLastError();
}

// Row tiles per block with one block per CU.
int row_tiles_per_cu(int N) { return ((N + 15) / 16 + 255) / 256; }

// Row tiles per block of the split form (about one block per CU, at most 8
// splits): 4, or 2 for narrow outputs.  3 where that gives as many splits (of
// the outputs that split, N 5441 - 6144: with 4 a third of the CUs had no block).
int split_rt(int N) {
    const int nrt = (N + 15) / 16;
    if (N < 2560) return 2;
    return 256 / ((nrt + 2) / 3) == 256 / ((nrt + 3) / 4) ? 3 : 4;
}

}  // namespace

int skinny_splits(const GemmArgs& a) {
    if (!a.sk_part || a.M > SKINNY_M) return 1;
    const int rt = split_rt(a.N), groups = (a.N + 16 * rt - 1) / (16 * rt);
    int S = std::min(std::min(256 / groups, 8), a.K / 128);
    while (S > 1 && (size_t)S * a.M * a.N > a.sk_part_floats) --S;
    return std::max(S, 1);
}

hipError_t launch_gemm_skinny_split(const GemmArgs& a, int S, hipStream_t st) {
    if (a.M <= 0 || a.M > SKINNY_M || a.K % 128 != 0 || a.N % 4 != 0 || S < 1 || S > a.K / 128 || !a.sk_part ||
        (size_t)S * a.M * a.N > a.sk_part_floats)
        return hipErrorInvalidValue;
    switch (split_rt(a.N)) {
        case 4: return launch_rt<EPI_F32, 4, true>(a, S, st);
        case 3: return launch_rt<EPI_F32, 3, true>(a, S, st);
    }
    return launch_rt<EPI_F32, 2, true>(a, S, st);
}

// The row tiles per block follow the width so that one round of blocks covers the
// rows: QKV takes 6 at 8192 wide, W1|W3 8 at 5632 wide (15104 hidden features).
// With at most 4 and 6 the blocks past 256 ran a second round.  16 | 64 tokens, us,
// tile kernel -> at most 4 and 6 -> as here: QKV 5632 wide 52 -> 44 -> 33 | 54 -> 60
// -> 42, 8192 wide 93 -> 71 -> 64 | 94 -> 89 -> 71; W1|W3 4608 wide 48 -> 54 -> 40 |
// 52 -> 64 -> 46, 5120 wide 55 -> 63 -> 49 | 61 -> 76 -> 52.
// 8 row tiles of more than 32 tokens do not fit the registers; there the tile
// kernel stays.  Wider W1|W3 run 6 row tiles in two rounds: 6144 wide 86 -> 77 | 95
// -> 91, 8192 wide 134 -> 109 | 130 -> 125 (of the widths timed only 7680 at 64
// tokens loses, 110 -> 120, beside 76 -> 65 of its QKV).
bool skinny_takes(int epi, const GemmArgs& a) {
    if (a.M > SKINNY_M) return false;
    const int per = row_tiles_per_cu(a.N);
    return !(epi == EPI_SWIGLU && (per == 7 || per == 8) && a.M > 32);
}

hipError_t launch_gemm_skinny(int epi, const GemmArgs& a, hipStream_t st) {
    if (a.M <= 0 || a.M > SKINNY_M || a.K % 128 != 0 || a.N % 4 != 0) return hipErrorInvalidValue;
    const int per = row_tiles_per_cu(a.N);
    switch (epi) {
        case EPI_QKV:
            if (per >= 6) return launch_rt<EPI_QKV, 6, false>(a, 1, st);
            if (per == 5) return launch_rt<EPI_QKV, 5, false>(a, 1, st);
            if (per == 4) return launch_rt<EPI_QKV, 4, false>(a, 1, st);
            return per == 3 ? launch_rt<EPI_QKV, 3, false>(a, 1, st) : launch_rt<EPI_QKV, 2, false>(a, 1, st);
        case EPI_SWIGLU:
            if (per == 7 || per == 8) return launch_rt<EPI_SWIGLU, 8, false, 2>(a, 1, st);
            if (per >= 5) return launch_rt<EPI_SWIGLU, 6, false>(a, 1, st);
            return per >= 3 ? launch_rt<EPI_SWIGLU, 4, false>(a, 1, st) : launch_rt<EPI_SWIGLU, 2, false>(a, 1, st);
        case EPI_F32:
            return per >= 3 ? launch_rt<EPI_F32, 4, false>(a, 1, st) : launch_rt<EPI_F32, 2, false>(a, 1, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace rh
