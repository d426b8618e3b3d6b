// rh_gemm.hip -- prefill GEMMs on fp16 MFMA (gfx950) with fused epilogues.
//
// One kernel family serves every projection of the forward token loop
// (kernels/sdpa_fwd.rs:115-117 QKV, dyn_matmul.rs:15-75 Wo, ffn_fused.rs:80-160
// W1/W3/W2, full_model.rs:555-567 tied logits):
//     Y[m][n] = sum_k X[m][k] * W[n][k]
// X is the token-major fp16 activation [M, K] and W the weight repacked at
// upload to [N, K] ("out x in"); both are stored in fragment order (frag_off:
// 1 KB pieces of 16 rows x 32 k), so both stream along k in 1 KB pieces.  The
// MFMA computes the transposed tile (A = weight rows, B = token rows): each
// lane's accumulator then holds 4 consecutive output features of one token,
// which makes the RoPE pairs (2i, 2i+1) and 16-byte fp32 stores lane-local.
//
// Tile policies: DTile (below) -- both operands in fragment order in HBM, moved
// global -> LDS by DMA through a 4-stage (192x256: 5-stage) pipeline of 32-wide k slices,
// 32x32x16 MFMA (16x16x32 for the 8-wave tiles) on fragments double-buffered
// in registers -- and PTile, the same operands with the block's two halves
// taking turns at the matrix pipes (8-wave 256x256 and 256x128).  Instantiated as
// 256x256 (8 waves of 128x64, or 4 waves of 128x128 with AGPR accumulators),
// 256x128, 192x256, 192x128 and 128x128; a cost model picks one per shape.
// Out-of-range rows are clamped, not predicated (they only feed accumulator
// entries the epilogue never stores), so the loads are branch-free.  Tiles are
// remapped so blocks sharing a weight panel run on the same XCD (one L2).
//
// Stream-K: P blocks split the tiles x k-iterations space evenly.  A
// block whose range covers only part of a tile stores its fp32 partial; a
// second kernel sums each split tile's partials in block order
// (deterministic) and runs the epilogue.  Partials are each thread's own
// accumulator quads, so both MFMA forms use the same format (the long-K
// narrow outputs take the 8-wave 16x16x32 256x128 tile).  Blocks never communicate inside a
// kernel: on this multi-XCD part the per-XCD L2s are not coherent, and a
// device-scope fence costs an L2 writeback + invalidate.
#include <algorithm>
#include <type_traits>

#include <hip/hip_ext.h>

#include "rh_device.h"
#include "rh_gemm_epi.h"
#include "rh_kernels.h"

namespace rh {
namespace {

constexpr int SK_P = 256;  // stream-K blocks: one per CU

template <int TN, int TM>
struct Frag {
    f32x16 v[TN][TM];
};
// Accumulators of the 16x16x32 form: NA x NB tiles of 16 x 16.
template <int NA, int NB>
struct Frag16 {
    f32x4 v[NA][NB];
};

// ---------------------------------------------------------------------------
// An operand of a product that contracts over tokens, C[i][j] = sum_t
// X[t][i] W[t][j], read straight from the token-major fragment order
// [tokens][features] that the forward and the backward leave it in.  A 1 KB
// unit holds 16 tokens x 32 features as 16-byte pieces (8 features of a
// token); 32 tokens x 32 features are two units, u = 2 (feature / 32) + token
// half, in the place of the two 16-row x 32-k fragments of a row-major
// operand.  The MFMA wants 8 consecutive tokens of one feature per lane: two
// transposing LDS reads (ds_read_b64_tr_b16), each of 4 tokens x 16 features
// per 16 lanes.  The DMA stores the pieces of odd 8-feature columns with their
// tokens XOR 4, so the 16 lanes' two columns fall into different banks, and so
// do those of lane groups 0, 1 and 2, 3.
//
// This replaces a transposed copy of every operand (one read and one write of
// each, a launch for every pair); the products' values and order are the same.
// Forward + backward with copies -> without, accumulating, ms: 20 layers of
// 4096, 8 x 512 tokens 98.2 -> 95.3, 1 x 512 23.7 -> 23.0; 20 of 2304, 8 x 512
// 39.2 -> 37.7; 16 of 1024, 8 x 512 9.97 -> 9.60; 8 of 512, 8 x 512 3.24 ->
// 3.16, 1 x 512 1.68 -> 1.72.
struct TrOperand {
    // source offset (halves) within a unit of what DMA lane l stores at 8 l
    __device__ static int src(int lane) { return (lane ^ (((lane >> 4) & 1) << 2)) * 8; }
    // lane's address (halves) in a unit pair, units KD * 512 apart, for tokens
    // 8g + 4hh + 0..3 of features 0..15 (features 16..31: + 256)
    __device__ static int base(int lane, int hh, int kd) {
        const int g = lane >> 4, r = lane & 15, b = (r >> 1) & 1;
        return (g >> 1) * kd * 512 + b * 128 + 64 * (g & 1) + 32 * (hh ^ b) + 8 * (r >> 2) + 4 * (r & 1);
    }
    __device__ static f16x8 read(const f16* p0, const f16* p1) {
        const f16x4 lo = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                       (__attribute__((address_space(3))) s16x4*)p0));
        const f16x4 hi = __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                       (__attribute__((address_space(3))) s16x4*)p1));
        return f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
    // source of unit f of a tile whose first feature is x0 of the product's
    // count, at token 0, in rows of nf features (units past the last feature
    // repeat it)
    __device__ static const f16* unit(const f16* p, int x0, int f, int count, int nf, int lane) {
        const int fg = min((x0 >> 5) + (f >> 1), ((count + 31) >> 5) - 1);
        return p + ((size_t)(f & 1) * (nf >> 5) + fg) * 512 + src(lane);
    }
};

// ---------------------------------------------------------------------------
// Tile policy (DTile): operands go global -> LDS by DMA
// (global_load_lds_dwordx4: 16 bytes per lane land at LDS base + 16 * lane),
// so no registers stage them and NS = 4 stages of 32 k are in flight (5 for
// the 192x256 tile: its long-K and 5120-token shapes gain from the depth).  A
// stage holds BN/16 weight fragments and BM/16 activation fragments of 1 KB
// each; both operands are stored in fragment order in HBM (the activations by
// the kernels that produce them), so every DMA instruction reads 1 KB
// contiguous.  The 32x32x16 MFMA operand of lane 32h + r
// at k16-step s is then lane 16(2s + h) + r%16 of fragment r/16: 16 lanes read
// 256 contiguous bytes, conflict-free without padding.  One barrier per stage:
// each wave waits for its own DMA of the stage (an explicit vmcnt, since the
// stages behind it stay in flight), then the barrier publishes every wave's.
// The stages are separate LDS arrays so the compiler's own wait-count
// tracking can tell them apart and adds no drain of its own.
//
// M16 selects the MFMA shape.  false: 32x32x16 (a 32x32 output tile per
// instruction; operand lane 32h + r reads lane 16(2s + h) + r%16 of
// fragment r/16 at k16-step s).  true: 16x16x32, whose operand layout is the
// fragment itself (lane l: row l%16, k 8(l/16)..+7), so each operand is one
// 1 KB fragment read as is; same tile sizes, operand bytes and accumulator
// registers, a different output layout (epilogue16).
//
// TR: the operands are token-major matrices [K tokens][features] in fragment
// order (see TrOperand), for the weight gradients, which contract over tokens.
template <int WGN, int WGM, int TN, int TM, bool M16 = false, int NS_ = 4, bool TR = false>
struct DTile {
    static_assert(NS_ == 4 || NS_ == 5, "4 or 5 stages");
    static_assert(!TR || M16, "transposing reads feed 16x16x32 operands");
    static constexpr bool kM16 = M16;
    static constexpr int NA = 2 * TN, NB = 2 * TM;  // 16-wide A / B tiles per wave (M16)
    static constexpr int BN = 32 * TN * WGN, BM = 32 * TM * WGM, NT = 64 * WGN * WGM;
    static constexpr int FTN = TN, FTM = TM, KI = 32, NS = NS_;
    static constexpr int NWF = BN / 16, NXF = BM / 16, NWAVE = WGN * WGM;
    // DMA instructions per wave per stage; when the fragments do not split
    // evenly, surplus slots repeat the last fragment (identical bytes to the
    // same LDS place), so every wave issues the same count and vmcnt stays exact.
    static constexpr int LPS = (NWF + NXF + NWAVE - 1) / NWAVE;
    static constexpr int SH = (NWF + NXF) * 512;     // halves per stage
    using Acc = std::conditional_t<M16, Frag16<NA, NB>, Frag<TN, TM>>;
    struct Smem {};
    __device__ static int nw(int n0) { return n0 + ((threadIdx.x >> 6) % WGN) * 32 * TN; }
    __device__ static int mw(int m0) { return m0 + ((threadIdx.x >> 6) / WGN) * 32 * TM; }
    // s_waitcnt with vmcnt <= n (expcnt, lgkmcnt left at their maximum)
    static constexpr int vm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
    // s_waitcnt with vmcnt <= n and lgkmcnt == 0: this wave's LDS reads are done
    static constexpr int vm_lgkm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

    __device__ static void run(const GemmArgs& a, int n0, int m0, int kb, int ke, Acc& acc, Smem&) {
        __shared__ __attribute__((aligned(1024))) f16 st0[SH], st1[SH], st2[SH], st3[SH];
        // The fifth stage exists only in five-stage tiles, so the four-stage
        // ones keep their LDS size (two blocks per CU where they fit); there
        // buf(4) is never used and st4 merely names st3.
        f16* st4 = st3;
        if constexpr (NS > 4) {
            __shared__ __attribute__((aligned(1024))) f16 st4s[SH];
            st4 = st4s;
        }
        const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
        const int wn = wv % WGN, wm = wv / WGN;
        const int K = a.K;
        // this wave's DMA fragments: f = wv * LPS + q over [weight frags | activation frags]
        const f16* gp[LPS];
        int gstep[LPS], loff[LPS];
#pragma unroll
        for (int q = 0; q < LPS; ++q) {
            const int f = min(wv * LPS + q, NWF + NXF - 1);
            loff[q] = f * 512;
            if constexpr (TR) {
                gp[q] = f < NWF ? TrOperand::unit(a.W, n0, f, a.N, a.trw, lane)
                                : TrOperand::unit(a.X, m0, f - NWF, a.M, a.trx, lane);
                gstep[q] = (f < NWF ? a.trw : a.trx) * 32;  // two 16-token unit rows
            } else if (f < NWF) {
                const int rb = min((n0 >> 4) + f, ((a.N + 15) >> 4) - 1);
                gp[q] = a.W + (size_t)rb * K * 16 + lane * 8;
                gstep[q] = 512;  // one 32-k fragment column of the 16-row block
            } else {
                const int rb = min((m0 >> 4) + f - NWF, ((a.M + 15) >> 4) - 1);
                gp[q] = a.X + (size_t)rb * K * 16 + lane * 8;
                gstep[q] = 512;
            }
        }
        const int r = lane & 31, h = lane >> 5;
        constexpr int AO = M16 ? NA : TN, BO = M16 ? NB : TM;
        int ao[AO], bo[BO];
        // TR: this wave's first A and B unit pairs, per token quad (hh); fragment
        // x is features 16 (x % 2) of the pair x / 2 further on
        const int ta0 = wn * NA * 512 + TrOperand::base(lane, 0, 1), ta1 = wn * NA * 512 + TrOperand::base(lane, 1, 1);
        const int tb = (NWF + wm * NB - wn * NA) * 512;
        if constexpr (M16) {
#pragma unroll
            for (int i = 0; i < NA; ++i) ao[i] = (wn * NA + i) * 512 + 8 * lane;
#pragma unroll
            for (int j = 0; j < NB; ++j) bo[j] = (NWF + wm * NB + j) * 512 + 8 * lane;
        } else {
#pragma unroll
            for (int i = 0; i < TN; ++i)
                ao[i] = (((wn * 32 * TN + 32 * i) >> 4) + (r >> 4)) * 512 + 128 * h + 8 * (r & 15);
#pragma unroll
            for (int j = 0; j < TM; ++j)
                bo[j] = (NWF + ((wm * 32 * TM + 32 * j) >> 4) + (r >> 4)) * 512 + 128 * h + 8 * (r & 15);
        }
        auto buf = [&](int s) -> f16* { return s == 0 ? st0 : s == 1 ? st1 : s == 2 ? st2 : s == 3 ? st3 : st4; };
        auto issue = [&](int kt, f16* st) {
#pragma unroll
            for (int q = 0; q < LPS; ++q)
                __builtin_amdgcn_global_load_lds((const void*)(gp[q] + (size_t)kt * gstep[q]),
                                                 (__attribute__((address_space(3))) void*)(st + loff[q]), 16, 0, 0);
        };
        // fragments of one stage: 32x32: [k16 step][tile]; 16x16: [tile] (one k32)
        struct Frags32 { f16x8 a[2][TN], b[2][TM]; };
        struct Frags16 { f16x8 a[NA], b[NB]; };
        using Frags = std::conditional_t<M16, Frags16, Frags32>;
        // operand m of a stage, in the order the interleaved step reads them
        constexpr int NR = M16 ? NA + NB : 2 * (TN + TM);
        auto read1 = [&](const f16* st, Frags& f, int m) {
            if constexpr (TR) {
                const int x = m < NA ? m : m - NA, o = (x & ~1) * 512 + (x & 1) * 256;
                if (m < NA) f.a[x] = TrOperand::read(st + ta0 + o, st + ta1 + o);
                else f.b[x] = TrOperand::read(st + (ta0 + tb) + o, st + (ta1 + tb) + o);
            } else if constexpr (M16) {
                if (m < NA) f.a[m] = *(const f16x8*)&st[ao[m]];
                else f.b[m - NA] = *(const f16x8*)&st[bo[m - NA]];
            } else {
                const int rks = m / (TN + TM), rr = m % (TN + TM);
                if (rr < TN) f.a[rks][rr] = *(const f16x8*)&st[ao[rr] + 256 * rks];
                else f.b[rks][rr - TN] = *(const f16x8*)&st[bo[rr - TN] + 256 * rks];
            }
        };
        auto readf = [&](const f16* st, Frags& f) {
#pragma unroll
            for (int m = 0; m < NR; ++m) read1(st, f, m);
        };
        // MFMA m of a stage
        constexpr int NM = M16 ? NA * NB : 2 * TN * TM;
        auto mfma1 = [&](const Frags& f, int m) {
            if constexpr (M16) {
                const int i = m / NB, j = m % NB;
                acc.v[i][j] = mfma16(f.a[i], f.b[j], acc.v[i][j]);
            } else {
                const int ks = m / (TN * TM), i = (m / TM) % TN, j = m % TM;
                acc.v[i][j] = mfma32(f.a[ks][i], f.b[ks][j], acc.v[i][j]);
            }
        };
        auto mfmas = [&](const Frags& f) {
#pragma unroll
            for (int m = 0; m < NM; ++m) mfma1(f, m);
        };
        if constexpr (M16) {
#pragma unroll
            for (int i = 0; i < NA; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) acc.v[i][j] = f32x4{};
        } else {
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int j = 0; j < TM; ++j) acc.v[i][j] = f32x16{};
        }
        // no wave may still read the stages from a previous call
        __builtin_amdgcn_s_waitcnt(vm_lgkm_wait(63));
        __builtin_amdgcn_s_barrier();
        const int n = ke - kb;
#pragma unroll
        for (int p = 0; p < NS - 1; ++p) issue(kb + min(p, n - 1), buf(p));
        // Stage t sits in buffer t % NS.  Step t: publish stage t+1, refill the
        // buffer stage t came from (its fragments are already in registers),
        // read stage t+1's fragments, then run stage t's MFMAs under those reads.
        Frags f0, f1;
        __builtin_amdgcn_s_waitcnt(vm_lgkm_wait((NS - 2) * LPS));
        __builtin_amdgcn_s_barrier();
        issue(kb + min(NS - 1, n - 1), buf(NS - 1));
        readf(buf(0), f0);
        // A full step, issued interleaved and pinned in that order: MFMA m,
        // then LDS read m, then DMA m.  With one or two waves per SIMD a
        // wave's in-order issue blocks whenever the vector-memory queue is
        // full; spreading the reads and DMAs between MFMAs keeps the matrix
        // pipe fed through those stalls (issued in bulk they idle it).
        auto step_il = [&](int t, Frags& cur, Frags& nxt, f16* refill, const f16* next) {
            __builtin_amdgcn_s_waitcnt(vm_lgkm_wait((NS - 2) * LPS));
            __builtin_amdgcn_s_barrier();
            const int kt = kb + min(t + NS, n - 1);
            constexpr int NG = NM > NR ? (NM > LPS ? NM : LPS) : (NR > LPS ? NR : LPS);
#pragma unroll
            for (int m = 0; m < NG; ++m) {
                if (m < NM) mfma1(cur, m);
                if (m < NR) read1(next, nxt, m);
                if (m < LPS)
                    __builtin_amdgcn_global_load_lds((const void*)(gp[m] + (size_t)kt * gstep[m]),
                                                     (__attribute__((address_space(3))) void*)(refill + loff[m]),
                                                     16, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // Tail step (past the last stage: a harmless read of a stale buffer,
        // MFMAs skipped).
        auto step = [&](int t, Frags& cur, Frags& nxt, f16* refill, const f16* next) {
            __builtin_amdgcn_s_waitcnt(vm_lgkm_wait((NS - 2) * LPS));
            __builtin_amdgcn_s_barrier();
            issue(kb + min(t + NS, n - 1), refill);
            readf(next, nxt);
            if (t < n) mfmas(cur);
        };
        // Whole groups of NS steps run interleaved; the remainder runs one
        // more group of predicated steps.  Every step issues LPS DMAs, so the
        // vmcnt bookkeeping stays uniform.
        int t0 = 0;
        if constexpr (NS == 4) {
            for (; t0 + NS <= n; t0 += NS) {
                step_il(t0, f0, f1, buf(0), buf(1));
                step_il(t0 + 1, f1, f0, buf(1), buf(2));
                step_il(t0 + 2, f0, f1, buf(2), buf(3));
                step_il(t0 + 3, f1, f0, buf(3), buf(0));
            }
            if (t0 < n) {
                step(t0, f0, f1, buf(0), buf(1));
                step(t0 + 1, f1, f0, buf(1), buf(2));
                step(t0 + 2, f0, f1, buf(2), buf(3));
                step(t0 + 3, f1, f0, buf(3), buf(0));
            }
        } else {  // 5 stages: groups of 10 steps bring both the buffers and the fragment sets back around
            for (; t0 + 10 <= n; t0 += 10) {
                step_il(t0, f0, f1, buf(0), buf(1));
                step_il(t0 + 1, f1, f0, buf(1), buf(2));
                step_il(t0 + 2, f0, f1, buf(2), buf(3));
                step_il(t0 + 3, f1, f0, buf(3), buf(4));
                step_il(t0 + 4, f0, f1, buf(4), buf(0));
                step_il(t0 + 5, f1, f0, buf(0), buf(1));
                step_il(t0 + 6, f0, f1, buf(1), buf(2));
                step_il(t0 + 7, f1, f0, buf(2), buf(3));
                step_il(t0 + 8, f0, f1, buf(3), buf(4));
                step_il(t0 + 9, f1, f0, buf(4), buf(0));
            }
            if (t0 < n) {
                step(t0, f0, f1, buf(0), buf(1));
                step(t0 + 1, f1, f0, buf(1), buf(2));
                step(t0 + 2, f0, f1, buf(2), buf(3));
                step(t0 + 3, f1, f0, buf(3), buf(4));
                step(t0 + 4, f0, f1, buf(4), buf(0));
                step(t0 + 5, f1, f0, buf(0), buf(1));
                step(t0 + 6, f0, f1, buf(1), buf(2));
                step(t0 + 7, f1, f0, buf(2), buf(3));
                step(t0 + 8, f0, f1, buf(3), buf(4));
                step(t0 + 9, f1, f0, buf(4), buf(0));
            }
        }
        // the trailing (unused) stage loads must land before the LDS is reused
        __builtin_amdgcn_s_waitcnt(vm_wait(0));
    }
};

// ---------------------------------------------------------------------------
// Ping-pong tile (PTile): the same operands, fragments and DMA as DTile, but
// the block's 8 waves form two groups of 4 (one wave of each per SIMD) that
// take turns.  While one group runs a stage's MFMAs with nothing else in its
// instruction stream, the other reads its next fragments from LDS and issues
// its share of the next DMA; a barrier swaps them.  DTile instead has both
// waves of a SIMD do everything at once, and whenever the vector-memory queue
// is full their in-order issue holds the MFMAs back: at 8192 x 4096 x 11008
// its 256x256 tile keeps the matrix pipes 68% busy (1.60 GHz), this one 79%
// (1.62 GHz), and what is left is the two barriers per stage and the
// prologue and epilogue of each tile.  The part is power-limited at these
// sizes, so the order of the MFMAs counts too: consecutive ones share one
// operand (every other row of B tiles runs backwards: +1.5%), and handing the
// matrix pipe over 4 MFMAs before the end of a stage (so that the two waves'
// MFMAs mix) costs 6%.  Measured at M = 8192 (7B, us, DTile 256x256 -> this):
// QKV 739 -> 623, W1|W3 1220 -> 1050, W2 623 -> 524, Wo 260 -> 225, logits
// 1856 -> 1635; 4096 x 4096 x 22016 594 -> 487 (1.52 PFLOP/s).
//
// A stage is KD slices of 32 k.  NS stages ring in LDS: at stage t each wave
// reads stage t, issues stage t + NS - 1 into the buffer stage t - 1 came
// from, and waits for its own part of stage t + 1.  Group 1 runs one barrier
// interval behind group 0, so group 0 fetches stage t in interval 2t and group
// 1 in 2t + 1; stage t - 1 was last read in interval 2t - 1, before either
// group refills its buffer, and both groups' parts of stage t + 1 have landed
// by the barrier that ends interval 2t + 1.  Every wave executes the same
// number of barriers (group 1 one extra at the start, group 0 at the end).
// The small tiles gain nothing from this (their stages hold too few MFMAs
// between barriers): 192x128 and 128x128 stay DTiles.  256x128 runs two k
// slices a stage (32 MFMAs between barriers, as 256x256): 163 -> 157 us at
// 2048 x 4096 x 11008, 132 -> 129 at 512 x 32000 x 4096.
template <int WGN, int WGM, int NA_, int NB_, int KD, int NS_, bool TR = false>
struct PTile {
    static_assert(WGN * WGM == 8 && NA_ % 2 == 0 && (NS_ == 3 || NS_ == 4), "8 waves, 3 or 4 stages");
    static constexpr bool kM16 = true;
    static constexpr int NA = NA_, NB = NB_, BN = 16 * NA * WGN, BM = 16 * NB * WGM, NT = 512;
    static constexpr int FTN = NA / 2, FTM = NB / 2, KI = 32 * KD, NS = NS_;
    static constexpr int NWF = BN / 16, NF = NWF + BM / 16, LPS = NF * KD / 8, SH = NF * KD * 512;
    static_assert(NF * KD % 8 == 0, "the DMA of a stage splits evenly over the waves");
    using Acc = Frag16<NA, NB>;
    struct Smem {};
    __device__ static int nw(int n0) { return n0 + ((threadIdx.x >> 6) % WGN) * 16 * NA; }
    __device__ static int mw(int m0) { return m0 + ((threadIdx.x >> 6) / WGN) * 16 * NB; }
    // s_waitcnt with vmcnt <= n; the same with lgkmcnt == 0
    static constexpr int vm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
    static constexpr int vm_lgkm_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

    __device__ static void run(const GemmArgs& a, int n0, int m0, int kb, int ke, Acc& acc, Smem&) {
        __shared__ __attribute__((aligned(1024))) f16 st0[SH], st1[SH], st2[SH];
        f16* st3 = st0;  // names no fourth buffer when NS == 3
        if constexpr (NS > 3) {
            __shared__ __attribute__((aligned(1024))) f16 st3s[SH];
            st3 = st3s;
        }
        auto buf = [&](int s) -> f16* { return s == 0 ? st0 : s == 1 ? st1 : s == 2 ? st2 : st3; };
        const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
        const int wn = wv % WGN, wm = wv / WGN, grp = wv >> 2;
        // this wave's DMA units: u = wv * LPS + q over [weight fragments | activation fragments] x KD slices
        const f16* gp[LPS];
        int gstep[LPS];
#pragma unroll
        for (int q = 0; q < LPS; ++q) {
            const int u = wv * LPS + q, f = u / KD, d = u % KD;
            if constexpr (TR) {
                const int nf = f < NWF ? a.trw : a.trx;
                gp[q] = (f < NWF ? TrOperand::unit(a.W, n0, f, a.N, nf, lane)
                                 : TrOperand::unit(a.X, m0, f - NWF, a.M, nf, lane)) +
                        (size_t)d * nf * 32;
                gstep[q] = nf * 32 * KD;
                continue;
            }
            gstep[q] = 512 * KD;
            const int rb = f < NWF ? min((n0 >> 4) + f, ((a.N + 15) >> 4) - 1)
                                   : min((m0 >> 4) + f - NWF, ((a.M + 15) >> 4) - 1);
            gp[q] = (f < NWF ? a.W : a.X) + (size_t)rb * a.K * 16 + d * 512 + lane * 8;
        }
        auto dma = [&](int kt, f16* st, int q) {
            __builtin_amdgcn_global_load_lds(
                (const void*)(gp[q] + (size_t)kt * (TR ? gstep[q] : 512 * KD)),
                (__attribute__((address_space(3))) void*)(st + (wv * LPS + q) * 512), 16, 0, 0);
        };
        const int lo = TR ? 0 : 8 * lane;
        const int ao = wn * NA * KD * 512 + lo, bo = (NWF + wm * NB) * KD * 512 + lo;
        const int tr0 = TrOperand::base(lane, 0, KD), tr1 = TrOperand::base(lane, 1, KD);
        // fragment x (k slice d) of the operand at o
        auto frag = [&](const f16* st, int o, int x, int d) -> f16x8 {
            if constexpr (TR) {
                const f16* p = st + o + ((x & ~1) * KD + d) * 512 + (x & 1) * 256;
                return TrOperand::read(p + tr0, p + tr1);
            }
            return *(const f16x8*)&st[o + (x * KD + d) * 512];
        };
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) acc.v[i][j] = f32x4{};
        // no wave may still read the stages from a previous call
        __builtin_amdgcn_s_waitcnt(vm_lgkm_wait(63));
        __builtin_amdgcn_s_barrier();
        const int n = ke - kb;
#pragma unroll
        for (int p = 0; p < NS - 1; ++p)
#pragma unroll
            for (int q = 0; q < LPS; ++q) dma(kb + min(p, n - 1), buf(p), q);
        __builtin_amdgcn_s_waitcnt(vm_wait((NS - 2) * LPS));
        __builtin_amdgcn_s_barrier();
        if (grp == 1) __builtin_amdgcn_s_barrier();
        // Stage t from st; stage t + NS - 1 (clamped: past the end a reload of
        // the last one that nobody reads) into refill.
        auto stage = [&](int t, const f16* st, f16* refill) {
            f16x8 fa[KD][NA], fb[KD][NB];
            const int kt = kb + min(t + NS - 1, n - 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = 0; d < KD; ++d) {
#pragma unroll
                for (int j = 0; j < NB; ++j) fb[d][j] = frag(st, bo, j, d);
#pragma unroll
                for (int i = 0; i < NA; ++i) fa[d][i] = frag(st, ao, i, d);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < LPS; ++q) dma(kt, refill, q);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_waitcnt(vm_lgkm_wait((NS - 2) * LPS));
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int d = 0; d < KD; ++d)
#pragma unroll
                for (int m = 0; m < NA * NB; ++m) {
                    const int i = m / NB, j = i & 1 ? NB - 1 - m % NB : m % NB;
                    acc.v[i][j] = mfma16(fa[d][i], fb[d][j], acc.v[i][j]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int t0 = 0; t0 < n; t0 += NS) {
            stage(t0, st0, buf(NS - 1));
            if (t0 + 1 < n) stage(t0 + 1, st1, st0);
            if (t0 + 2 < n) stage(t0 + 2, st2, st1);
            if constexpr (NS > 3)
                if (t0 + 3 < n) stage(t0 + 3, st3, st2);
        }
        if (grp == 0) __builtin_amdgcn_s_barrier();
        // the trailing (unused) stage loads must land before the LDS is reused
        __builtin_amdgcn_s_waitcnt(vm_wait(0));
    }
};

// 32x32 tiles.  (nw, mw): the wave's first feature row and token.  Lane holds
// token m = mw + j*32 + lane%32 and, per q4, the four consecutive features
// n = nw + i*32 + 8*q4 + 4*(lane/32) + (0..3).
template <int TN, int TM, int EPI>
__device__ __forceinline__ void epilogue(const GemmArgs& a, int nw, int mw, const Frag<TN, TM>& acc) {
    const int lane = threadIdx.x & 63;
    const int N = a.N, M = a.M;
#pragma unroll
    for (int j = 0; j < TM; ++j) {
        const int m = mw + j * 32 + (lane & 31);
        if (m >= M) continue;
        if constexpr (EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_SAVE) {
            // W1|W3 is interleaved in 16-row groups: rows 0..15 of 32-row tile T
            // are W1 rows of features 16T.., rows 16..31 the matching W3 rows,
            // and row r + 16 sits in the same lane as row r (accumulator + 8).
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int T = (nw + i * 32) >> 5;
#pragma unroll
                for (int q4 = 0; q4 < 2; ++q4) {
                    const int f = 16 * T + 8 * q4 + 4 * (lane >> 5);
                    if (f >= a.ldo) continue;
                    float h1[4], h3[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        h1[r] = acc.v[i][j][4 * q4 + r];
                        h3[r] = acc.v[i][j][4 * q4 + 8 + r];
                    }
                    store_swiglu<EPI>(a, m, f, h1, h3);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < TN; ++i)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    const int n = nw + i * 32 + 8 * q4 + 4 * (lane >> 5);
                    if (n >= N) continue;
                    store4<EPI>(a, m, n, acc.v[i][j][4 * q4 + 0], acc.v[i][j][4 * q4 + 1], acc.v[i][j][4 * q4 + 2],
                                acc.v[i][j][4 * q4 + 3]);
                }
        }
    }
}

// 16x16 tiles: lane l holds token m = mw + 16j + l%16 and the four
// consecutive features n = nw + 16i + 4(l/16) + (0..3) of A tile i, B tile j.
template <int NA, int NB, int EPI>
__device__ __forceinline__ void epilogue(const GemmArgs& a, int nw, int mw, const Frag16<NA, NB>& acc) {
    const int lane = threadIdx.x & 63;
    const int N = a.N, M = a.M;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int m = mw + 16 * j + (lane & 15);
        if (m >= M) continue;
        if constexpr (EPI == EPI_SWIGLU || EPI == EPI_SWIGLU_SAVE) {
            // A tiles 2p and 2p + 1 are the W1 rows of features 16T..16T+15 and
            // the matching W3 rows (T = (nw + 32p) / 32; nw is a multiple of 32)
#pragma unroll
            for (int p = 0; p < NA / 2; ++p) {
                const int f = 16 * ((nw + 32 * p) >> 5) + 4 * (lane >> 4);
                if (f >= a.ldo) continue;
                float h1[4], h3[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    h1[r] = acc.v[2 * p][j][r];
                    h3[r] = acc.v[2 * p + 1][j][r];
                }
                store_swiglu<EPI>(a, m, f, h1, h3);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const int n = nw + 16 * i + 4 * (lane >> 4);
                if (n >= N) continue;
                store4<EPI>(a, m, n, acc.v[i][j][0], acc.v[i][j][1], acc.v[i][j][2], acc.v[i][j][3]);
            }
        }
    }
}

template <class Tl, int EPI>
__device__ __forceinline__ void run_epilogue(const GemmArgs& a, int nw, int mw, const typename Tl::Acc& acc) {
    if constexpr (Tl::kM16)
        epilogue<Tl::NA, Tl::NB, EPI>(a, nw, mw, acc);
    else
        epilogue<Tl::FTN, Tl::FTM, EPI>(a, nw, mw, acc);
}

// The accumulators of a thread as TN*TM*4 quads of 4 floats (the stream-K
// partial format; the same thread stores and reloads them).  32x32: quad
// (i*TM + j)*4 + q = acc.v[i][j][4q..4q+3]; 16x16: quad a*NB + b = acc.v[a][b].
template <int TN, int TM>
__device__ __forceinline__ f32x4 get_quad(const Frag<TN, TM>& f, int x) {
    const f32x16& v = f.v[x / (TM * 4)][(x / 4) % TM];
    const int e = 4 * (x % 4);
    return f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]};
}
template <int TN, int TM>
__device__ __forceinline__ void set_quad(Frag<TN, TM>& f, int x, f32x4 q) {
    f32x16& v = f.v[x / (TM * 4)][(x / 4) % TM];
    const int e = 4 * (x % 4);
    v[e] = q[0]; v[e + 1] = q[1]; v[e + 2] = q[2]; v[e + 3] = q[3];
}
template <int NA, int NB>
__device__ __forceinline__ f32x4 get_quad(const Frag16<NA, NB>& f, int x) { return f.v[x / NB][x % NB]; }
template <int NA, int NB>
__device__ __forceinline__ void set_quad(Frag16<NA, NB>& f, int x, f32x4 q) { f.v[x / NB][x % NB] = q; }
// The quads of 32-row slice s of a wave's tile and the type holding them:
// 32x32: row tile s (TM tiles x 4 quads); 16x16: A tiles 2s, 2s+1 (2 x NB).
template <class Tl>
struct Slice {
    static constexpr int NQ = Tl::FTM * 4;
    using Acc = std::conditional_t<Tl::kM16, Frag16<2, Tl::NB>, Frag<1, Tl::FTM>>;
    __device__ static int quad_of(int s, int x) { return s * NQ + x; }  // both layouts: slice-major
};

// MODE: MODE_DP one block per tile; MODE_SK stream-K over P blocks (T =
// tiles x k-iterations); MODE_SPLIT P even k-splits per tile, each storing its
// fp32 partial [M][N] at sk_part + split * M * N.
enum { MODE_DP = 0, MODE_SK = 1, MODE_SPLIT = 2 };

template <class Tl, int EPI, int MODE>
__global__ __launch_bounds__(Tl::NT) void gemm_kernel(GemmArgs a, int P, long long T) {
    __shared__ __attribute__((aligned(16))) typename Tl::Smem sm;
    const int nbN = (a.N + Tl::BN - 1) / Tl::BN, nbM = (a.M + Tl::BM - 1) / Tl::BM;
    const int KT = a.K / Tl::KI;
    typename Tl::Acc acc;
    if constexpr (MODE == MODE_DP) {
        const int t = xcd_remap(blockIdx.x, nbN * nbM);
        // Consecutive tiles (run together on one XCD) walk groups of up to
        // 8 M-tiles x every N panel, M fastest: the 32 tiles an XCD runs at
        // a time then share 4 weight panels and 8 activation row blocks in
        // its L2, instead of one panel and 32 row blocks (7B batch 16: QKV
        // 785 -> 753 us, W2 870 -> 746 us, prefill 108.4 -> 101.5 ms).
        int nb, mb;
        if (nbM <= 8) {
            nb = t / nbM;
            mb = t - nb * nbM;
        } else {
            const int g = t / (8 * nbN), r = t - g * 8 * nbN, gm = min(8, nbM - g * 8);
            mb = g * 8 + r % gm;
            nb = r / gm;
        }
        if constexpr (EPI == EPI_SILU_BWD && Tl::kM16 && Tl::NA * Tl::NB <= 12) {
            // The saved h1, h3 of this lane's outputs are loaded before the k
            // loop, so they arrive under it instead of stalling the epilogue
            // (2 * NA * NB registers held through the loop: the larger tiles
            // would spill).
            const int nw = Tl::nw(nb * Tl::BN), mw = Tl::mw(mb * Tl::BM), lane = threadIdx.x & 63;
            const size_t plane = (size_t)a.M * a.ldo;
            f16x4 p1[Tl::NB][Tl::NA], p3[Tl::NB][Tl::NA];
#pragma unroll
            for (int j = 0; j < Tl::NB; ++j)
#pragma unroll
                for (int i = 0; i < Tl::NA; ++i) {
                    const int m = mw + 16 * j + (lane & 15), n = nw + 16 * i + 4 * (lane >> 4);
                    p1[j][i] = p3[j][i] = f16x4{};
                    if (m < a.M && n < a.N) {
                        const size_t o = (size_t)m * a.ldo + n;
                        p1[j][i] = *(const f16x4*)(a.h13 + o);
                        p3[j][i] = *(const f16x4*)(a.h13 + plane + o);
                    }
                }
            Tl::run(a, nb * Tl::BN, mb * Tl::BM, 0, KT, acc, sm);
#pragma unroll
            for (int j = 0; j < Tl::NB; ++j)
#pragma unroll
                for (int i = 0; i < Tl::NA; ++i) {
                    const int m = mw + 16 * j + (lane & 15), n = nw + 16 * i + 4 * (lane >> 4);
                    if (m < a.M && n < a.N)
                        silu_bwd4(a, m, n, acc.v[i][j][0], acc.v[i][j][1], acc.v[i][j][2], acc.v[i][j][3], p1[j][i],
                                  p3[j][i]);
                }
        } else {
            Tl::run(a, nb * Tl::BN, mb * Tl::BM, 0, KT, acc, sm);
            run_epilogue<Tl, EPI>(a, Tl::nw(nb * Tl::BN), Tl::mw(mb * Tl::BM), acc);
        }
    } else if constexpr (MODE == MODE_SPLIT) {
        // Blocks go round-robin to the 8 XCDs (block b on XCD b % 8).  When P
        // divides 8 and the tiles share out evenly, XCD x runs split x % P of
        // its 1/(8/P) of the tiles, panel by panel: each XCD's L2 then fetches
        // only its k-slice of the activation (which every tile reads) and
        // each weight slice once for all M-tiles of its panel.  Otherwise the
        // splits of one tile and the tiles of one weight panel share an XCD.
        const int tiles = nbN * nbM;
        int tile, sp;
        if (8 % P == 0 && tiles % (8 / P) == 0) {
            const int x = blockIdx.x & 7;
            sp = x % P;
            tile = (x / P) * (tiles / (8 / P)) + (blockIdx.x >> 3);
        } else {
            const int v = xcd_remap(blockIdx.x, tiles * P);
            tile = v / P;
            sp = v - tile * P;
        }
        const int nb = tile / nbM, mb = tile - nb * nbM;
        const int kb = (int)((long long)sp * KT / P), ke = (int)((long long)(sp + 1) * KT / P);
        Tl::run(a, nb * Tl::BN, mb * Tl::BM, kb, ke, acc, sm);
        GemmArgs b = a;
        b.out_f32 = a.sk_part + (size_t)sp * a.M * a.N;
        b.ldo = a.N;
        b.softcap = 0.f;
        b.alpha = 0.f;  // raw partials: the row kernel applies alpha once to their sum
        b.part_cols = 0;
        run_epilogue<Tl, EPI_F32>(b, Tl::nw(nb * Tl::BN), Tl::mw(mb * Tl::BM), acc);
    } else {
        constexpr int NT = Tl::NT;
        constexpr int NV = Tl::FTN * Tl::FTM * 4;  // f32x4 per thread per partial tile
        const int tid = threadIdx.x;
        const int lp = xcd_remap(blockIdx.x, P);
        const long long it0 = (long long)lp * T / P, it1 = (long long)(lp + 1) * T / P;
        long long it = it0;
        while (it < it1) {
            const int tile = (int)(it / KT);
            const int kb = (int)(it - (long long)tile * KT);
            const int ke = (int)((long long)KT < kb + (it1 - it) ? (long long)KT : kb + (it1 - it));
            const int nb = tile / nbM, mb = tile - nb * nbM;
            const int n0 = nb * Tl::BN, m0 = mb * Tl::BM;
            Tl::run(a, n0, m0, kb, ke, acc, sm);
            if (kb == 0 && ke == KT) {
                run_epilogue<Tl, EPI>(a, Tl::nw(n0), Tl::mw(m0), acc);
            } else {
                // A block's first segment goes to slot 0, its last to slot 1;
                // the fixup kernel merges them once this kernel has finished.
                const int slot = (it == it0) ? 0 : 1;
                f32x4* mine = (f32x4*)a.sk_part + ((size_t)(lp * 2 + slot) * NV) * NT + tid;
#pragma unroll
                for (int x = 0; x < NV; ++x) mine[(size_t)x * NT] = get_quad(acc, x);
            }
            it = (long long)tile * KT + ke;
        }
    }
}

// Stream-K fixup: one block per (tile, 32-row tile of every wave).  A tile covered
// by a single block was finished by gemm_kernel; for a split tile, sum the
// partials of its contributing blocks in block order (deterministic) and run
// the epilogue on the slice.
template <class Tl, int EPI>
__global__ __launch_bounds__(Tl::NT) void gemm_fixup_kernel(GemmArgs a, int P, long long T) {
    using Sl = Slice<Tl>;
    constexpr int NT = Tl::NT, NV = Tl::FTN * Tl::FTM * 4, NQ = Sl::NQ;
    const int nbM = (a.M + Tl::BM - 1) / Tl::BM;
    const int KT = a.K / Tl::KI;
    const int tile = blockIdx.x, i0 = blockIdx.y, tid = threadIdx.x;
    const long long tb = (long long)tile * KT, te = tb + KT;
    const int pf = (int)(((tb + 1) * P - 1) / T), pl = (int)((te * P - 1) / T);
    if (pf == pl) return;
    typename Sl::Acc acc;
#pragma unroll
    for (int x = 0; x < NQ; ++x) set_quad(acc, x, f32x4{});
    for (int c = pf; c <= pl; ++c) {
        // with fewer iterations than blocks some blocks own none and wrote nothing
        if ((long long)c * T / P == (long long)(c + 1) * T / P) continue;
        const int cslot = ((long long)c * T / P >= tb) ? 0 : 1;
        const f32x4* part = (const f32x4*)a.sk_part + ((size_t)(c * 2 + cslot) * NV) * NT + tid;
#pragma unroll
        for (int x = 0; x < NQ; ++x) set_quad(acc, x, get_quad(acc, x) + part[(size_t)Sl::quad_of(i0, x) * NT]);
    }
    const int nb = tile / nbM, mb = tile - nb * nbM;
    const int nw = Tl::nw(nb * Tl::BN) + 32 * i0, mw = Tl::mw(mb * Tl::BM);
    if constexpr (Tl::kM16)
        epilogue<2, Tl::NB, EPI>(a, nw, mw, acc);
    else
        epilogue<1, Tl::FTM, EPI>(a, nw, mw, acc);
}

template <class Tl, int EPI>
hipError_t launch_dp(const GemmArgs& a, hipStream_t st) {
    const int tiles = ((a.N + Tl::BN - 1) / Tl::BN) * ((a.M + Tl::BM - 1) / Tl::BM);
    const long long T = (long long)tiles * (a.K / Tl::KI);
    if (a.prof_start)
        hipExtLaunchKernelGGL((gemm_kernel<Tl, EPI, MODE_DP>), dim3(tiles), dim3(Tl::NT), 0, st, a.prof_start,
                              a.prof_stop, 0u, a, 1, T);
    else
        hipLaunchKernelGGL((gemm_kernel<Tl, EPI, MODE_DP>), dim3(tiles), dim3(Tl::NT), 0, st, a, 1, T);
    return hipGetLastError();
}

template <class Tl, int EPI>
hipError_t launch_tile(const GemmArgs& a, bool sk, hipStream_t st) {
    if (!sk) return launch_dp<Tl, EPI>(a, st);
    const int nbN = (a.N + Tl::BN - 1) / Tl::BN, nbM = (a.M + Tl::BM - 1) / Tl::BM;
    const int tiles = nbN * nbM;
    const long long T = (long long)tiles * (a.K / Tl::KI);
    if (!a.sk_part || (size_t)SK_P * 2 * Tl::BN * Tl::BM > a.sk_part_floats) return hipErrorInvalidValue;
    if (a.prof_start && hipEventRecord(a.prof_start, st) != hipSuccess) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_kernel<Tl, EPI, MODE_SK>), dim3(SK_P), dim3(Tl::NT), 0, st, a, SK_P, T);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((gemm_fixup_kernel<Tl, EPI>), dim3(tiles, Tl::FTN), dim3(Tl::NT), 0, st, a, SK_P, T);
    if (a.prof_stop && hipEventRecord(a.prof_stop, st) != hipSuccess) return hipErrorInvalidValue;
    return hipGetLastError();
}

// S-way split-K of a residual GEMM: partials only (the row kernel reduces).
template <class Tl>
hipError_t launch_split(const GemmArgs& a, int S, hipStream_t st) {
    const int tiles = ((a.N + Tl::BN - 1) / Tl::BN) * ((a.M + Tl::BM - 1) / Tl::BM);
    if (S < 1 || S > a.K / Tl::KI || !a.sk_part || (size_t)S * a.M * a.N > a.sk_part_floats)
        return hipErrorInvalidValue;
    if (a.prof_start && hipEventRecord(a.prof_start, st) != hipSuccess) return hipErrorInvalidValue;
    hipLaunchKernelGGL((gemm_kernel<Tl, EPI_F32, MODE_SPLIT>), dim3(tiles * S), dim3(Tl::NT), 0, st, a, S, 0LL);
    if (a.prof_stop && hipEventRecord(a.prof_stop, st) != hipSuccess) return hipErrorInvalidValue;
    return hipGetLastError();
}

// Weight-gradient GEMM (K = the token count, short; fp32 output, as large
// as the weights): persistent blocks of 8 compute waves running the 8-wave
// 16x16x32 128x128 DTile k loop and WG_SW store waves.  A tile's
// accumulators go to an LDS staging tile; the store waves write it out to
// HBM while the compute waves run the next tile, so the output stores
// overlap the MFMAs.  The compute waves issue no stores at all: on gfx950
// stores and the operand DMAs share one in-order vmcnt, so stores in the
// compute waves would make every later stage wait hold for them.
//
// Barriers: every wave of the block executes the same s_barrier sequence.
// Per tile the compute waves run Tl::run (2 + NS * ceil(KT / NS) barriers),
// then X (the store waves are done reading the staging tile), write the
// staging tile, then Y (published).  The store waves mirror that count,
// storing the previous tile in 16 rounds spread over the k loop's barriers,
// and the block's last tile after its Y.
//
// Tiles: block b runs on XCD b % 8 and takes every (gridDim / 8)-th tile of
// that XCD's contiguous share; tiles are numbered in groups of 8 M-tiles x all
// N panels (so 32 tiles in flight on an XCD span 4 panels x 8 M-tiles).
constexpr int WG_SW = 4;     // store waves
constexpr int WG_SP = 132;   // staging row pitch in floats (conflict-free b128 access)
template <class Tl, bool ACC>
__global__ __launch_bounds__(Tl::NT + 64 * WG_SW) void gemm_wgrad_kernel(GemmArgs a) {
    static_assert(Tl::kM16 && Tl::BN == 128 && Tl::BM == 128 && Tl::NWAVE == 8, "8-wave 128x128 tile");
    __shared__ __attribute__((aligned(16))) float stg[128 * WG_SP];
    typename Tl::Smem sm;
    const int nbN = (a.N + 127) / 128, nbM = (a.M + 127) / 128, T = nbN * nbM;
    const int KT = a.K / Tl::KI;
    const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3, per = gridDim.x >> 3;
    const int t0 = (int)((long long)xcd * T / 8), t1 = (int)((long long)(xcd + 1) * T / 8);
    const int mine = (t1 - t0 > k) ? (t1 - t0 - k + per - 1) / per : 0;
    const int nbar = 2 + Tl::NS * ((KT + Tl::NS - 1) / Tl::NS);  // barriers of one Tl::run
    auto tile_at = [&](int i, int& n0, int& m0) {
        const int t = t0 + k + i * per;
        const int mg = t / (nbN * 8), rem = t - mg * nbN * 8, gsz = min(8, nbM - mg * 8);
        n0 = (rem / gsz) * 128;
        m0 = (mg * 8 + rem % gsz) * 128;
    };
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (wv < Tl::NWAVE) {
        typename Tl::Acc acc;
        for (int i = 0; i < mine; ++i) {
            int n0, m0;
            tile_at(i, n0, m0);
            Tl::run(a, n0, m0, 0, KT, acc, sm);
            __builtin_amdgcn_s_barrier();  // X
            const int nl = Tl::nw(n0) - n0, ml = Tl::mw(m0) - m0;
#pragma unroll
            for (int i2 = 0; i2 < Tl::NA; ++i2)
#pragma unroll
                for (int j = 0; j < Tl::NB; ++j)
                    *(f32x4*)&stg[(ml + 16 * j + (lane & 15)) * WG_SP + nl + 16 * i2 + 4 * (lane >> 4)] = acc.v[i2][j];
            lds_barrier();  // Y
        }
    } else {
        const int sw = wv - Tl::NWAVE;
        int pn0 = 0, pm0 = 0;  // the staged tile
        // round r: rows 2 (4r + sw) + lane / 32 of the staged tile, 4 columns per lane
        auto store_round = [&](int r) {
            const int ml = 2 * (WG_SW * r + sw) + (lane >> 5), nl = 4 * (lane & 31);
            const int m = pm0 + ml, n = pn0 + nl;
            if (m < a.M && n < a.N) {
                f32x4 v = *(const f32x4*)&stg[ml * WG_SP + nl];
                float* po = a.out_f32 + (size_t)m * a.ldo + n;
                if constexpr (ACC) {
                    f32x4 x = *(const f32x4*)po;
                    x[0] = v[0] * a.alpha + x[0]; x[1] = v[1] * a.alpha + x[1];
                    x[2] = v[2] * a.alpha + x[2]; x[3] = v[3] * a.alpha + x[3];
                    v = x;
                } else if (a.alpha != 0.f) {
                    v[0] *= a.alpha; v[1] *= a.alpha; v[2] *= a.alpha; v[3] *= a.alpha;
                }
                // the gradients are read only by the optimizer: streaming stores
                // keep them from evicting the other stream's operands
                __builtin_nontemporal_store(v, (f32x4*)po);
            }
        };
        constexpr int NR = 128 / (2 * WG_SW);  // rounds per tile
        for (int i = 0; i < mine; ++i) {
            for (int bar = 0; bar < nbar; ++bar) {
                __builtin_amdgcn_s_barrier();
                if (i > 0)
                    for (int r = bar * NR / nbar; r < (bar + 1) * NR / nbar; ++r) store_round(r);
            }
            __builtin_amdgcn_s_waitcnt(Tl::vm_lgkm_wait(63));  // staging reads done before X
            __builtin_amdgcn_s_barrier();  // X
            __builtin_amdgcn_s_barrier();  // Y
            tile_at(i, pn0, pm0);
        }
        if (mine > 0)
            for (int r = 0; r < NR; ++r) store_round(r);
    }
}

// Data-parallel tiles: estimated time = rounds of one block per CU x
// tile FLOPs / that tile's per-CU rate.  The rates of 192x256, 192x128 and
// 128x128 are fitted to MI355X timings of every tile on 27 GEMM shapes of the 7B
// forward and training step (M 512 - 8192, random fp16 operands), those of
// 256x256 and 256x128 to the ping-pong tiles: at M = 8192 a 256x256 tile takes
// 1.20 times a 192x256 one's time for 1.33 times its work, at M = 512 1.09 times
// for a tile of W1|W3.  The estimate trades wave quantization (e.g. 172 vs 230
// tiles at M = 512) against per-tile efficiency and knows nothing of the
// epilogue's bytes, which count at a short K.  Two rounds of 256x256 and three of
// 256x128 come out even (257 - 384 tiles of 256x256, whose second round is at
// most half full); the three rounds measure faster: logits 3072 x 8192 x 1024 82 ->
// 70 us, x 3072 171 -> 145, W2 6144 x 4096 x 11008 503 -> 470, QKV 3200 x 7680 x
// 2560 157 -> 143.  Token-major operands take 256x256 there (forward + backward
// 3072 wide, 768 - 8192 tokens, 1 - 4% faster: the smaller tile pays more
// transposing reads).  Narrow outputs (Wo) and long K (W2) use stream-K instead,
// when every block gets at least two 32-wide k-iterations.  *cost: the pick's
// estimate (per unit of K).
int tile_pick(int M, int N, bool tokens, float* cost) {
    struct Cand { int cfg, bn, bm; float rate; };
    constexpr Cand dp[] = {{GCFG_D8_256x128, 256, 128, 3.75f}, {GCFG_D8_256x256, 256, 256, 5.0f},
                           {GCFG_D8_192x256, 192, 256, 4.35f}, {GCFG_D8_192x128, 192, 128, 3.7f},
                           {GCFG_D8_128x128, 128, 128, 3.0f}};
    float best = 3.0e38f;
    int cfg = 0;
    for (const Cand& c : dp) {
        const long long tiles = (long long)((N + c.bn - 1) / c.bn) * ((M + c.bm - 1) / c.bm);
        const float t = (float)((tiles + SK_P - 1) / SK_P) * (float)c.bn * (float)c.bm / c.rate;
        if (t < best || (tokens && t == best && c.cfg == GCFG_D8_256x256)) { best = t; cfg = c.cfg; }
    }
    if (cost) *cost = best;
    return cfg;
}

using Tile256x256 = PTile<2, 4, 8, 4, 1, 4>;
using Tile256x128 = PTile<4, 2, 4, 4, 2, 3>;

template <int EPI>
hipError_t launch_epi(const GemmArgs& a, hipStream_t st) {
    int cfg = a.force_cfg;
    if constexpr (EPI == EPI_F32 || EPI == EPI_SWIGLU || EPI == EPI_QKV) {
        if (cfg == GCFG_AUTO && skinny_takes(EPI, a)) return launch_gemm_skinny(EPI, a, st);
    }
    if (cfg == GCFG_AUTO) {
        const long long KT = a.K / 32;
        const int t256x128 = ((a.N + 255) / 256) * ((a.M + 127) / 128);
        const int t128 = ((a.N + 127) / 128) * ((a.M + 127) / 128);
        const bool sk_ok = a.sk_part && (size_t)SK_P * 2 * 256 * 256 <= a.sk_part_floats;
        if (sk_ok && a.K >= 8192 && t256x128 < 160 && t256x128 * KT >= 2 * SK_P) {
            cfg = GCFG_D8_256x128_SK;
        } else if (sk_ok && t128 < 160 && t128 * KT >= 2 * SK_P && KT * (SK_P - t128) >= 28 * SK_P) {
            // stream-K saves the idle CUs' share of one tile's k loop (about
            // 0.36 us per 32-k step) but pays a fix-up launch (about 9 us): at
            // 600M, M = 512, QKV (144 tiles, K 1536) one round of whole tiles is
            // faster (15.3 + 8.5 us stream-K + fix-up against one 17.5 us round)
            cfg = GCFG_D8_128x128_SK;
        } else {
            cfg = tile_pick(a.M, a.N, false, nullptr);
            // Of 8 - 16 stages of 64 k the ping-pong tile's longer ramp is too
            // large a share.  us, DTile | ping-pong: logits 256 x 32000 x 512 16.5 |
            // 20.6, 256 x 32000 x 768 20 | 24, 1024 x 8192 x 768 20 | 23, 200 x 32000
            // x 1024 24 | 26.6; K = 1536 34.0 | 34.9, K = 2048 even, more: slower.
            if (cfg == GCFG_D8_256x128 && a.K <= 1024) cfg = GCFG_DT_256x128;
        }
    }
    // The 8-wave 192x256, 192x128 and 128x128 tiles run the 16x16x32 form: at
    // M = 512 (7B) W1|W3 takes 84.5 us as 8-wave 16x16x32 192x256, against 87.8
    // as a 4-wave 16x16x32 tile and 91.4 as 8-wave 32x32x16; QKV 60.4 us as
    // 8-wave 16x16x32 192x128 against 64.7 as 4-wave 32x32x16; the 8-wave
    // 128x128 tile is 1-6% faster in that form than its 32x32x16 twin on every
    // shape timed.  8-wave 256x256 and 256x128 are ping-pong tiles.  The 4-wave
    // tiles and the stream-K forms that GCFG_AUTO does not name above are taken
    // only by force_cfg.
    switch (cfg) {
        case GCFG_D8_256x256: return launch_tile<Tile256x256, EPI>(a, false, st);
        case GCFG_D8_256x256_SK: return launch_tile<Tile256x256, EPI>(a, true, st);
        case GCFG_D4_128x128: return launch_tile<DTile<2, 2, 2, 2>, EPI>(a, false, st);
        case GCFG_D4_128x128_SK: return launch_tile<DTile<2, 2, 2, 2>, EPI>(a, true, st);
        case GCFG_D8_256x128: return launch_tile<Tile256x128, EPI>(a, false, st);
        case GCFG_D8_256x128_SK: return launch_tile<Tile256x128, EPI>(a, true, st);
        case GCFG_DT_256x128: return launch_dp<DTile<4, 2, 2, 2, true>, EPI>(a, st);
        case GCFG_D4_256x256: return launch_tile<DTile<2, 2, 4, 4>, EPI>(a, false, st);
        case GCFG_D4_256x256_SK: return launch_tile<DTile<2, 2, 4, 4>, EPI>(a, true, st);
        case GCFG_D4_256x128: return launch_tile<DTile<2, 2, 4, 2>, EPI>(a, false, st);
        case GCFG_D4_256x128_SK: return launch_tile<DTile<2, 2, 4, 2>, EPI>(a, true, st);
        case GCFG_D4_192x128: return launch_tile<DTile<2, 2, 3, 2>, EPI>(a, false, st);
        case GCFG_D8_192x128: return launch_tile<DTile<2, 4, 3, 1, true>, EPI>(a, false, st);
        case GCFG_D8_192x128_SK: return launch_tile<DTile<2, 4, 3, 1, true>, EPI>(a, true, st);
        case GCFG_D8_128x128: return launch_tile<DTile<2, 4, 2, 1, true>, EPI>(a, false, st);
        case GCFG_D8_128x128_SK: return launch_tile<DTile<2, 4, 2, 1, true>, EPI>(a, true, st);
        case GCFG_D4_192x128_SK: return launch_tile<DTile<2, 2, 3, 2>, EPI>(a, true, st);
        case GCFG_D8_192x256: return launch_tile<DTile<2, 4, 3, 2, true, 5>, EPI>(a, false, st);
        case GCFG_D8_192x256_SK: return launch_tile<DTile<2, 4, 3, 2, true, 5>, EPI>(a, true, st);
        case GCFG_D4_192x256: return launch_tile<DTile<2, 2, 3, 4>, EPI>(a, false, st);
        case GCFG_D4_192x256_SK: return launch_tile<DTile<2, 2, 3, 4>, EPI>(a, true, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace

size_t gemm_sk_part_floats() { return (size_t)SK_P * 2 * 256 * 256; }

namespace {
template <class Tl, bool ACC>
hipError_t launch_wgrad(const GemmArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((gemm_wgrad_kernel<Tl, ACC>), dim3(SK_P), dim3(Tl::NT + 64 * WG_SW), 0, st, a);
    return hipGetLastError();
}

template <int EPI>
hipError_t launch_tokens(const GemmArgs& a, hipStream_t st) {
    auto go = [&](auto T) {
        using Tl = decltype(T);
        const int tiles = ((a.N + Tl::BN - 1) / Tl::BN) * ((a.M + Tl::BM - 1) / Tl::BM);
        hipLaunchKernelGGL((gemm_kernel<Tl, EPI, MODE_DP>), dim3(tiles), dim3(Tl::NT), 0, st, a, 1, 0LL);
        return hipGetLastError();
    };
    switch (a.force_cfg ? a.force_cfg : tile_pick(a.M, a.N, true, nullptr)) {
        case GCFG_D8_256x256: return go(PTile<2, 4, 8, 4, 1, 4, true>{});
        case GCFG_D8_256x128: return go(PTile<4, 2, 4, 4, 2, 3, true>{});
        case GCFG_D8_192x256: return go(DTile<2, 4, 3, 2, true, 4, true>{});
        case GCFG_D8_192x128: return go(DTile<2, 4, 3, 1, true, 4, true>{});
        case GCFG_D8_128x128: return go(DTile<2, 4, 2, 1, true, 4, true>{});
    }
    return hipErrorInvalidValue;
}

bool tr_ok(const GemmArgs& a) { return a.trx >= a.M && a.trw >= a.N && a.trx % 128 == 0 && a.trw % 128 == 0; }
}  // namespace

hipError_t launch_gemm_wgrad(const GemmArgs& a, bool accumulate, hipStream_t st) {
    if (a.K % 128 != 0 || a.N % 4 != 0 || a.M <= 0 || a.N <= 0 || a.ldo < a.N || !a.out_f32)
        return hipErrorInvalidValue;
    if (a.trx || a.trw) return hipErrorInvalidValue;
    using Tl = DTile<2, 4, 2, 1, true>;
    return accumulate ? launch_wgrad<Tl, true>(a, st) : launch_wgrad<Tl, false>(a, st);
}

namespace {

// Few tokens: the skinny kernel's own splits.  Else split K when the output has
// too few tiles to fill the CUs: S splits per tile, at most 8 and at least 8
// k-iterations each, within the workspace; 1 = no split.
int split_count(const GemmArgs& a) {
    if (a.force_cfg == GCFG_AUTO && a.M <= SKINNY_M) return skinny_splits(a);
    const int bn = a.K >= 8192 ? 256 : 128, bm = 128;
    const int tiles = ((a.N + bn - 1) / bn) * ((a.M + bm - 1) / bm);
    int S = 1;
    if (a.force_cfg == GCFG_AUTO && a.sk_part && tiles < 160) {
        S = std::min(std::min(SK_P / tiles, 8), a.K / 32 / 8);
        while (S > 1 && (size_t)S * a.M * a.N > a.sk_part_floats) --S;
    }
    return S;
}

// Up to SKINNY_M tokens the few-token kernel.  Else K >= 8192 (W2): 256x128
// tiles as 8 waves of 16x16x32 (50.3 vs 52.9 us as 4 waves of 32x32x16 at 7B,
// M = 512; the ping-pong 256x128 tile measures the same there); otherwise
// 128x128 (the two forms measure the same there)
hipError_t launch_split_any(const GemmArgs& a, int S, hipStream_t st) {
    if (a.M <= SKINNY_M) return launch_gemm_skinny_split(a, S, st);
    return a.K >= 8192 ? launch_split<DTile<4, 2, 2, 2, true>>(a, S, st) : launch_split<DTile<2, 2, 2, 2>>(a, S, st);
}

}  // namespace

hipError_t launch_gemm_partials(const GemmArgs& a, int* nsplit, hipStream_t st) {
    *nsplit = 0;
    if (a.K % 128 != 0 || a.N % 8 != 0 || a.M <= 0) return hipErrorInvalidValue;
    const int S = split_count(a);
    if (S < 2) return hipSuccess;
    const hipError_t e = launch_split_any(a, S, st);
    if (e == hipSuccess) *nsplit = S;
    return e;
}

hipError_t launch_gemm_resid_norm(const GemmArgs& a, const float* gamma, float eps, f16* xn, hipStream_t st) {
    if (a.K % 128 != 0 || a.N % 8 != 0 || a.N > 8192 || a.M <= 0 || a.ldo != a.N) return hipErrorInvalidValue;
    const int S = split_count(a);
    if (S >= 2) {
        const hipError_t e = launch_split_any(a, S, st);
        if (e != hipSuccess) return e;
        return launch_resid_norm(a.resid_in ? a.resid_in : a.out_f32, a.out_f32, a.sk_part, S, (size_t)a.M * a.N,
                                 a.alpha, gamma, eps, xn, a.M, a.N, st);
    }
    const hipError_t e = launch_epi<EPI_RESID>(a, st);
    if (e != hipSuccess || !gamma) return e;
    return launch_rmsnorm(a.out_f32, gamma, xn, a.M, a.N, eps, st, true);
}

float gemm_tile_cost(int M, int N) {
    float c = 0.f;
    (void)tile_pick(M, N, true, &c);
    return c;
}

hipError_t launch_gemm(int epi, const GemmArgs& a, hipStream_t st) {
    if (a.K % 128 != 0 || a.N % 4 != 0 || a.M <= 0) return hipErrorInvalidValue;
    if (a.part_cols && ((epi != EPI_F32 && epi != EPI_RESID) || a.part_cols % 4 != 0 || a.N > 3 * a.part_cols ||
                        a.ldo != a.part_cols || a.resid_in || !a.out_part1 ||
                        (a.N > 2 * a.part_cols && !a.out_part2)))
        return hipErrorInvalidValue;
    if (a.trx || a.trw) {
        if (!tr_ok(a)) return hipErrorInvalidValue;
        if (epi == EPI_F32) return launch_tokens<EPI_F32>(a, st);
        return epi == EPI_RESID ? launch_tokens<EPI_RESID>(a, st) : hipErrorInvalidValue;
    }
    switch (epi) {
        case EPI_F32: return launch_epi<EPI_F32>(a, st);
        case EPI_RESID: return launch_epi<EPI_RESID>(a, st);
        case EPI_SWIGLU:
            if (a.N % 32 != 0) return hipErrorInvalidValue;
            return launch_epi<EPI_SWIGLU>(a, st);
        case EPI_QKV:
            if (a.hd <= 0 || (a.hd & (a.hd - 1)) != 0 || a.N != 3 * a.D || a.S <= 0) return hipErrorInvalidValue;
            return launch_epi<EPI_QKV>(a, st);
        case EPI_SWIGLU_SAVE:
            if (a.N % 32 != 0 || !a.h13) return hipErrorInvalidValue;
            return launch_epi<EPI_SWIGLU_SAVE>(a, st);
        case EPI_SILU_BWD:
            if (a.N % 128 != 0 || a.ldo != a.N || !a.h13 || !a.out_f16) return hipErrorInvalidValue;
            return launch_epi<EPI_SILU_BWD>(a, st);
    }
    return hipErrorInvalidValue;
}

}  // namespace rh
