// gemm_rows.hip - prefill kernel for calls whose 64-row x 16/32/64-column pieces fill one round of workgroups
// (17 .. 64 rows on outputs from 1024 columns up - up to 32 they are fp32 rows -, up to 512 rows on narrow ones),
// FAST mode (f16 operands).
//
// With so little work per CU (64 rows x 56 columns at N = 14336) what the tiled kernels of gemm.hip spend
// per K tile - a barrier, every weight operand read from LDS by every multiplying wave - no longer hides
// behind arithmetic: their K loop costs 0.45 - 0.6 us per K tile whatever the tile holds, and narrow outputs
// make them split K over workgroups and add the slabs in a second pass.
//
// Here the waves of a workgroup share nothing until the end.  The workgroup owns MF row blocks of 16
// (blockIdx.y: which) and NF column blocks of 16; wave w takes the K tiles w, w + WAVES, ... and, for those,
// multiplies ALL its rows against ALL its column blocks (MF x NF accumulator blocks per wave).  A weight tile
// is then needed by exactly one wave: global memory -> registers -> dequantised in registers
// (round_f16(scale * q), the operand of FAST mode) -> MFMA B operand, no LDS, no barrier; and every row of X
// enters the CU once (staged operand order, 1 KB per load) and meets all NF column blocks from registers.  One
// wave per SIMD owns the register file (accumulators, a K tile of X and four K tiles of packed weights in
// flight).  At the end the waves' partial sums meet through LDS and are added in wave order (fixed order:
// results are reproducible and a row's bits do not depend on the other rows of the batch).
// Epilogues: residual add, folded RMSNorm / widened rows (a factor per row on the finished sums), SwiGLU (gate and
// up column blocks sit side by side in a workgroup: 4096 -> 28672 at 24 .. 64 rows 27 - 33 us against 47 - 48).
//
// What bounds it is what a CU takes in: all its rows of X (512 KB for 64 rows at K = 4096) plus its column
// blocks' weights, through an L1 that delivers 64 bytes a cycle (a workgroup per CU that does nothing but read
// the same 512 KB with 1-KB wave instructions reaches 21 - 31 TB/s over the chip with four waves, 33 with
// eight; this kernel takes in 156 MB in 16 us).  Hence: the fewest column blocks that still fit one round of
// workgroups, and only as many row blocks as the call has (two or three up to 48 rows: a row block costs
// 1.1 - 1.3 us).  Per call with the staging pass, bf16 rows, against the tiled kernels (up to 64 rows on small
// weights: against two passes of the batched-rows decode kernel):
//   4096 -> 14336 at 33 .. 48 / 64 rows  17.8 / 19.1 us against 21.5 / 22.1   4096 -> 28672   31 - 33 against 38 - 39
//   4096 ->  8192 at 33 / 64 / 128 rows  13.3 / 14.7 / 19.5 against 20.6 / 21.2 / 25.5
//   4096 ->  4096 at 64 / 128 / 256 rows 12.8 / 14.3 / 19.8 against 14.5 / 25.5 / 22.3
//   4096 ->  6144 at 64 / 128 rows       14.3 / 17.6 against 19.3 / 26.8     8192 -> 14336 at 33 .. 64 rows 30 - 32 against 36.5 - 38
//   4096 ->  1024 at 128 / 256 / 512 rows 12.9 / 14.2 / 20.7 against 18.7 / 21.6 / 27.6
//   fp32 rows, 17 .. 32: 4096 -> 14336 15.9 against 21, 4096 -> 4096 10.7 against 18
// Not kept, us per call there / here: 32x32x16 MFMAs (the same to 0.3 on every shape: the MFMAs are a quarter of a wave's cycles); two waves
// per SIMD by scale groups of a K tile 14.2 / 13.1 (4096 -> 4096 at 64 rows); eight column blocks for 65 .. 128 rows 31.4 / the tiled
// kernel's 27.6, eight row blocks 27.5 / 27.4; rows read where the caller has them, without the staging launch, 23.7 / 18.3 (sixteen
// 64-byte runs per operand load instead of one KB).
#include <algorithm>
#include <type_traits>

#include "cybq_device.h"
#include "cybq_internal.h"

namespace cybq {

namespace {

#include "gemm_parts.h"

template <int I, int N, class F>
__device__ __forceinline__ void static_for_r(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for_r<I + 1, N>(f);
    }
}

// group j of a native tile -> the FAST-mode B operand round_f16(scale * q), in registers
template <int BITS>
__device__ __forceinline__ void dequant_group(const WRegs<BITS>& r, int j, uint32_t magic, Frag16& b)
{
    uint32_t bw[4];
    if (BITS == 4) unpack_q4_f16(r.q[0][2 * (j >> 1)], r.q[0][2 * (j >> 1) + 1], j & 1, magic, bw);
    else unpack_q8_f16(r.q[(BITS == 4) ? 0 : (j >> 1)][(j & 1) * 2], r.q[(BITS == 4) ? 0 : (j >> 1)][(j & 1) * 2 + 1], bw);
    const uint32_t sb = (j & 1) ? (r.s[j >> 1] >> 16) : (r.s[j >> 1] & 0xffffu);
    const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)sb);
    const half2_t s2 = {sh, sh};
#pragma unroll
    for (int p = 0; p < 4; p++) b.u[p] = as_u32(as_h2(bw[p]) * s2);
}

// the finished sums of one row block (first row m0) on their way to y: row factors, SwiGLU, residual.  stats: row m0 + lane % 16's, res: the
// block's residual, both asked for before the waves' sums meet
template <int NF>
__device__ __forceinline__ void finish_row_block(float4_t (&tot)[1][NF], float* stg, int m0, int nt0, int M, const WeightView& w, void* y, int ydt, int K,
                                                 const Epilogue& epi, const NormStats& ns, const RowStats& stats, const Residual<1, NF>& res, int lane)
{
    if (epi.gamma || ns.unscale) {
        const float mine = row_factor(stats, ns, epi.gamma != nullptr, min(m0 + (lane & 15), M - 1), K, epi.eps);
#pragma unroll
        for (int r4 = 0; r4 < 4; r4++) {
            const float rs = __shfl(mine, (lane >> 4) * 4 + r4, 64);
#pragma unroll
            for (int f = 0; f < NF; f++) tot[0][f][r4] *= rs;
        }
    }
    if constexpr (NF >= 2) {
        if (epi.kind == kEpiSwiglu) {      // column blocks 2p / 2p+1 are gate / up of output block (nt0 >> 1) + p
            float4_t act[1][NF / 2];
#pragma unroll
            for (int p = 0; p < NF / 2; p++)
#pragma unroll
                for (int r4 = 0; r4 < 4; r4++) act[0][p][r4] = silu_mul(tot[0][2 * p][r4], tot[0][2 * p + 1][r4]);
            const Epilogue plain = {kEpiNone, nullptr, nullptr, 0, 0.f};
            write_rows<1, NF / 2>(act, stg, m0, nt0 >> 1, M, w.N >> 1, y, ydt, 1.0f, plain, lane);
            return;
        }
    }
    write_rows<1, NF>(tot, res, stg, m0, nt0, M, w.N, y, ydt, 1.0f, epi, lane);
}

// MF row blocks of 16 per workgroup (blockIdx.y-th MF * 16 rows of the call), NF column blocks per workgroup, WAVES
// waves that split K, DEPTH K tiles of packed weights and XD K tiles of X in flight per wave.
// OCC: workgroups per CU.
// SHARES: the K tiles are cut into `shares` runs of kt_per_share, and a wave walks one run (number blockIdx.z * WAVES + wave)
// from the tile and in the order in which the tiled kernels' K split walks it; the runs' sums are added in their order, the
// first four here, the others (blockIdx.z = 1: a slab each) with the first four's slab by the slab-adding pass.
// The result is that of the tiled kernels bit for bit.
template <int BITS, int MF, int NF, int WAVES, int DEPTH, int XD, int OCC = 1, bool SHARES = false>
__global__ __launch_bounds__(WAVES * 64) __attribute__((amdgpu_waves_per_eu(OCC * WAVES / 4, OCC * WAVES / 4))) void gemm_rows_kernel(
    const uint8_t* __restrict__ wbase, const u32x4_t* __restrict__ x, int KT_, int NT_, int x_row_blocks, int M, int N_,
    void* __restrict__ y, int ydt, int K_, Epilogue epi, NormStats ns, int shares, int kt_per_share, float* __restrict__ slabs)
{
    const WeightView w = {wbase, N_, K_, NT_, KT_, BITS};
    constexpr int FR = MF * NF;                        // accumulator blocks per wave
    static_assert(DEPTH % XD == 0 && MF >= 1 && MF <= WAVES, "shape");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    float4_t* part = reinterpret_cast<float4_t*>(smem);                                    // [WAVES][FR][64]
    float* stg = reinterpret_cast<float*>(smem + (size_t)WAVES * FR * 1024);               // [MF][16 * NF * 16]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt0 = (int)blockIdx.x * NF;
    const int K = w.K, G = K / kGroup;
    const int share = (int)blockIdx.z * WAVES + wv;
    const int kt_lo = SHARES ? min(share * kt_per_share, w.KT - 1) : 0;
    const int KT = SHARES ? min(kt_per_share, w.KT - kt_lo) : w.KT;      // my K tiles (SHARES: mine alone): kt_lo ..
    const uint32_t magic = q4_magic_vgpr();
    // my K tiles: number t is tile wv + WAVES * t
    const int T = SHARES ? (share < shares ? KT : 0) : KT > wv ? (KT - wv + WAVES - 1) / WAVES : 0;
    // Workgroups that run side by side read the same rows of X: walking K in the same order they would all
    // ask the same L2 channels for the same lines at the same moment, so every column tile starts its walk
    // at another K tile and wraps around (the order depends on the column tile only, not on M).
    const int kt0 = SHARES ? (nt0 >> 3) % KT : (int)blockIdx.x % KT;      // (the tiled kernels' column tiles: eight blocks)
    // (a tile number past my last one is clamped to the last K tile: loaded again, never used)
    auto tile_of = [&](int t) __attribute__((always_inline)) {
        const int kt = min(SHARES ? t : wv + WAVES * t, KT - 1) + kt0;
        return kt_lo + (kt >= KT ? kt - KT : kt);
    };
    // (row blocks and column blocks past the end are clamped to the last real one: computed again, never
    // stored; the offsets are wave-uniform, the lane's part of an address is one register)
    const u32x4_t* xl = x + lane;
    int xrow[MF];
    const int rb0 = (int)blockIdx.y * MF;              // my first row block (blockIdx.y: which MF * 16 rows of the call)
#pragma unroll
    for (int i = 0; i < MF; i++) xrow[i] = __builtin_amdgcn_readfirstlane(min(rb0 + i, x_row_blocks - 1) * G * 64);
    int64_t wtile[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) wtile[f] = (int64_t)min(nt0 + f, w.NT - 1) * w.KT;
    auto load_x = [&](Frag16 (&dst)[MF], int t, int j) __attribute__((always_inline)) {
        const int g = min(tile_of(t) * 4 + j, G - 1);
#pragma unroll
        for (int i = 0; i < MF; i++) dst[i].u = xl[xrow[i] + g * 64];
    };
    auto fetch = [&](WRegs<BITS> (&dst)[NF], int t) __attribute__((always_inline)) {
        const int kt = tile_of(t);
#pragma unroll
        for (int f = 0; f < NF; f++) load_wtile<BITS>(dst[f], w, wtile[f] + kt, lane);
    };

    float4_t acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[i][f] = (float4_t){0.f, 0.f, 0.f, 0.f};

    WRegs<BITS> wreg[DEPTH][NF];
    Frag16 xa[XD][4][MF];
#pragma unroll
    for (int d = 0; d < DEPTH; d++) fetch(wreg[d], d);
#pragma unroll
    for (int d = 0; d < XD; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) load_x(xa[d][j], d, j);

    // my K tile number t (register sets R = t % DEPTH, R % XD): multiply; its X registers take the rows of tile
    // t + XD group by group as they fall free; its weight registers take tile t + DEPTH
    auto k_tile = [&](int t, auto residue) __attribute__((always_inline)) {
        constexpr int R = decltype(residue)::value;
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
            for (int f = 0; f < NF; f++) {
                Frag16 b;
                dequant_group<BITS>(wreg[R][f], j, magic, b);
#pragma unroll
                for (int i = 0; i < MF; i++) acc[i][f] = mma<0>(xa[R % XD][j][i], b, acc[i][f]);
            }
            load_x(xa[R % XD][j], t + XD, j);
        }
        fetch(wreg[R], t + DEPTH);
    };
    int t = 0;
    for (; t + DEPTH <= T; t += DEPTH)
        static_for_r<0, DEPTH>([&](auto i) __attribute__((always_inline)) { k_tile(t + decltype(i)::value, i); });
    static_for_r<0, DEPTH - 1>([&](auto i) __attribute__((always_inline)) {
        if (t + decltype(i)::value < T) k_tile(t + decltype(i)::value, i);
    });

    const Epilogue plain = {kEpiNone, nullptr, nullptr, 0, 0.f};
    if constexpr (SHARES) {
        if (blockIdx.z > 0) {
            if (share < shares)
                write_rows<MF, NF>(acc, reinterpret_cast<float*>(smem) + wv * (16 * NF * 16), rb0 * 16, nt0, M, w.N,
                                   slabs + (int64_t)(share - WAVES + 1) * M * w.N, kF32, 1.0f, plain, lane);
            return;
        }
    }
    // ---- the partial sums meet: every wave leaves all of its blocks, waves 0 .. MF-1 finish a row block each
    // (what that takes from memory is asked for first; ahead of the K loop it cost registers: 4096 -> 14336 at 64 rows 16.9 -> 17.2 us)
    const int mb = (rb0 + min(wv, MF - 1)) * 16;               // first row of the block I finish
    const bool finishes = !SHARES || shares <= WAVES;          // (else the pass that adds the slabs does, and asks for it)
    RowStats stats = {};
    Residual<1, NF> res;
    if (finishes) {
        stats = load_row_stats(ns, epi.gamma != nullptr, min(mb + (lane & 15), M - 1), wbase);
        if (wv < MF) load_residual(res, mb, nt0, M, w.N, y, ydt, epi, lane);
    }
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) part[(wv * FR + i * NF + f) * 64 + lane] = acc[i][f];
    __syncthreads();
    if (wv >= MF) return;
    float4_t tot[1][NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int blk = wv * NF + f;
        float4_t s = part[blk * 64 + lane];
#pragma unroll
        for (int p = 1; p < WAVES; p++) s += part[(p * FR + blk) * 64 + lane];
        tot[0][f] = s;
    }
    if constexpr (SHARES) {
        if (!finishes) {
            write_rows<1, NF>(tot, stg + wv * (16 * NF * 16), (rb0 + wv) * 16, nt0, M, w.N, slabs, kF32, 1.0f, plain, lane);
            return;
        }
    }
    finish_row_block<NF>(tot, stg + wv * (16 * NF * 16), mb, nt0, M, w, y, ydt, K, epi, ns, stats, res, lane);
}

// The same sums for outputs of more than a round of workgroups (up to 64 rows, four column blocks each): one workgroup of eight
// waves does the work of two, column groups g and g + D.  D is a multiple of KT, so both walk the K tiles from the same one on and
// wave wv of either half multiplies the same rows of X by its own weights: X comes once, by copies into LDS (a ring of RING steps
// of four K tiles, each half of a tile copied by the two waves that use it), and the stream into the CUs is half of what two
// workgroups draw.  What bounds it then is issue: per K tile a wave makes 16 operands of 13 vector instructions each, next to 32,
// 48 or 64 MFMAs (4096 -> 28672 at 45 rows: 3.4 us before the first step, 8 steps of 3690 cycles in 15.4, 1.9 after).  Bit for
// bit the result of gemm_rows_kernel.
// (wbase without __restrict__: the waits below count the weight loads, so none of them may move over an asm that clobbers memory.  A load
// whose value nobody reads is removed, and a wait that counted it lets the copies pass: the last DEPTH steps ask for no weights and
// wait for the copies alone.)
template <int BITS, int MF, int DEPTH, int RING>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_rows_pair_kernel(
    const uint8_t* wbase, const uint8_t* x, int KT_, int NT_, int x_row_blocks, int M, int N_,
    void* __restrict__ y, int ydt, int K_, int D, Epilogue epi, NormStats ns)
{
    const WeightView w = {wbase, N_, K_, NT_, KT_, BITS};
    constexpr int NF = 4, FR = MF * NF;
    constexpr int XC = 2 * MF;                         // copies of X per wave and step
    constexpr int WL = NF * (BITS == 4 ? 2 : 3);       // weight loads per wave and step
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w8 = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = w8 >> 2, wv = w8 & 3;
    const int nt0 = ((int)blockIdx.x + half * D) * NF;         // (a second half past the last column group computes and stores nothing of use)
    const int K = w.K, G = K / kGroup, KT = w.KT;
    const uint32_t magic = q4_magic_vgpr();
    const int steps = (KT + 3) / 4, T = KT > wv ? (KT - wv + 3) / 4 : 0;
    const int kt0 = (int)blockIdx.x % KT;
    auto tile_of = [&](int t) __attribute__((always_inline)) {
        const int kt = min(wv + 4 * t, KT - 1) + kt0;
        return kt >= KT ? kt - KT : kt;
    };
    // block e of a K tile of X = row block e / 4, group e % 4; this wave copies 2 * MF of its tile's 4 * MF
    uint32_t xrow[XC];
#pragma unroll
    for (int c = 0; c < XC; c++) xrow[c] = (uint32_t)min((half * XC + c) >> 2, x_row_blocks - 1) * (uint32_t)(G * 1024);
    auto copy_x = [&](int t, int ring) __attribute__((always_inline)) {
        const int kt = tile_of(t);
#pragma unroll
        for (int c = 0; c < XC; c++) {
            const int e = half * XC + c;
            copy_to_lds((ring * 4 + wv) * (MF * 4096) + e * 1024, x, xrow[c] + (uint32_t)min(kt * 4 + (e & 3), G - 1) * 1024u + (uint32_t)lane * 16u);
        }
    };
    int64_t wtile[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) wtile[f] = (int64_t)min(nt0 + f, w.NT - 1) * w.KT;
    auto fetch = [&](WRegs<BITS> (&dst)[NF], int t) __attribute__((always_inline)) {
        const int kt = tile_of(t);
#pragma unroll
        for (int f = 0; f < NF; f++) load_wtile<BITS>(dst[f], w, wtile[f] + kt, lane);
    };
    float4_t acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[i][f] = (float4_t){0.f, 0.f, 0.f, 0.f};

    WRegs<BITS> wreg[DEPTH][NF];
#pragma unroll
    for (int r = 0; r < RING - 1; r++) copy_x(r, r);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int d = 0; d < DEPTH; d++) fetch(wreg[d], d);
    // (a wait for all but the weights asked for behind it)
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(DEPTH * WL > 63 ? 63 : DEPTH * WL) : "memory");

    int ring = 0;
    auto step = [&](int t, auto residue, auto more, bool mine) __attribute__((always_inline)) {
        constexpr int R = decltype(residue)::value;
        constexpr bool MORE = decltype(more)::value;           // there are weights left to ask for
        const int far = ring == 0 ? RING - 1 : ring - 1;       // the step before this one's place: X of step t + RING - 1
        copy_x(t + RING - 1, far);
        asm volatile("" ::: "memory");                         // (the weights behind the copies)
        const uint8_t* xl = smem + (ring * 4 + wv) * (MF * 4096) + lane * 16;
        if (mine) {
            Frag16 xa[2][MF];
#pragma unroll
            for (int i = 0; i < MF; i++) xa[0][i].u = *reinterpret_cast<const u32x4_t*>(xl + i * 4096);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                if (j < 3) {
#pragma unroll
                    for (int i = 0; i < MF; i++) xa[(j + 1) & 1][i].u = *reinterpret_cast<const u32x4_t*>(xl + i * 4096 + (j + 1) * 1024);
                }
#pragma unroll
                for (int f = 0; f < NF; f++) {
                    Frag16 b;
                    dequant_group<BITS>(wreg[R][f], j, magic, b);
#pragma unroll
                    for (int i = 0; i < MF; i++) acc[i][f] = mma<0>(xa[j & 1][i], b, acc[i][f]);
                }
                __builtin_amdgcn_sched_barrier(0);             // (left alone the scheduler makes all operands of a K tile first and spills)
            }
        }
        if constexpr (MORE) fetch(wreg[R], t + DEPTH);
        // X of the next step is there: newer than its copies are the weights of this step and, with three places, of the one before
        // and the copies of this step; without weights those copies alone
        constexpr int NEWER = !MORE ? (RING - 2) * XC : RING == 2 ? WL : (RING - 1) * WL + (RING - 2) * XC;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NEWER) : "memory");
        ring = ring + 1 == RING ? 0 : ring + 1;
    };
    int t = 0;
    for (; t + DEPTH < steps; t += DEPTH)
        static_for_r<0, DEPTH>([&](auto i) __attribute__((always_inline)) { step(t + decltype(i)::value, i, std::true_type{}, true); });
    static_for_r<0, DEPTH>([&](auto i) __attribute__((always_inline)) {       // (in the last step not every wave has a K tile)
        if (t + decltype(i)::value < steps) step(t + decltype(i)::value, i, std::false_type{}, t + decltype(i)::value < T);
    });

    // ---- as in gemm_rows_kernel, each half for itself
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");       // (copies past the last step)
    float4_t* const part = reinterpret_cast<float4_t*>(smem) + half * (4 * FR * 64);
    float* const stg = reinterpret_cast<float*>(smem + 8 * FR * 1024) + half * (MF * 16 * NF * 16);
    const int mb = min(wv, MF - 1) * 16;
    const RowStats stats = load_row_stats(ns, epi.gamma != nullptr, min(mb + (lane & 15), M - 1), wbase);
    Residual<1, NF> res;
    if (wv < MF) load_residual(res, mb, nt0, M, w.N, y, ydt, epi, lane);
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) part[(wv * FR + i * NF + f) * 64 + lane] = acc[i][f];
    __syncthreads();
    if (wv >= MF) return;
    float4_t tot[1][NF];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        const int blk = wv * NF + f;
        float4_t s = part[blk * 64 + lane];
#pragma unroll
        for (int p = 1; p < 4; p++) s += part[(p * FR + blk) * 64 + lane];
        tot[0][f] = s;
    }
    finish_row_block<NF>(tot, stg + wv * (16 * NF * 16), wv * 16, nt0, M, w, y, ydt, K, epi, ns, stats, res, lane);
}

template <int BITS, int MF, int DEPTH, int RING>
hipError_t launch_pair_t(const WeightView& w, const void* x, int M, void* y, int ydt, const Epilogue& epi, const NormStats& ns, hipStream_t st)
{
    constexpr int lds_ring = RING * 4 * MF * 4096, lds_end = 8 * MF * 4 * 1024 + 2 * MF * 16 * 64 * 4;
    constexpr int lds = lds_ring > lds_end ? lds_ring : lds_end;
    static_assert(lds <= 160 * 1024, "LDS");
    (void)LdsRequest<&gemm_rows_pair_kernel<BITS, MF, DEPTH, RING>, lds>::registered;
    const int groups = (w.NT + 3) / 4, D = ((groups + 1) / 2 + w.KT - 1) / w.KT * w.KT;
    hipLaunchKernelGGL((gemm_rows_pair_kernel<BITS, MF, DEPTH, RING>), dim3((unsigned)D), dim3(512), lds, st, w.base,
                       static_cast<const uint8_t*>(x), w.KT, w.NT, (M + 15) / 16, M, w.N, y, ydt, w.K, D, epi, ns);
    return hipGetLastError();
}

template <int BITS, int MF, int NF, int WAVES, int DEPTH, int XD, int OCC = 1, bool SHARES = false>
hipError_t launch_rows_t(const WeightView& w, const void* x, int M, void* y, int ydt, const Epilogue& epi, const NormStats& ns, hipStream_t st,
                         int shares = 0, float* slabs = nullptr)
{
    constexpr int lds = WAVES * MF * NF * 1024 + MF * 16 * NF * 16 * 4;
    (void)LdsRequest<&gemm_rows_kernel<BITS, MF, NF, WAVES, DEPTH, XD, OCC, SHARES>, lds>::registered;
    const unsigned groups = (unsigned)((w.NT + NF - 1) / NF), row_parts = (unsigned)((M + 16 * MF - 1) / (16 * MF));
    hipLaunchKernelGGL((gemm_rows_kernel<BITS, MF, NF, WAVES, DEPTH, XD, OCC, SHARES>),
                       dim3(groups, row_parts, SHARES ? (unsigned)((shares + WAVES - 1) / WAVES) : 1u), dim3(WAVES * 64), lds, st,
                       w.base, reinterpret_cast<const u32x4_t*>(x), w.KT, w.NT, (M + 15) / 16, M, w.N, y, ydt, w.K, epi, ns,
                       shares, SHARES ? (w.KT + shares - 1) / shares : 0, slabs);
    return hipGetLastError();
}

}  // namespace

// Column blocks per workgroup (1, 2 or 4) for a call of M rows, or 0 when the kernel does not take it.
// A call takes about 1.6 us per K tile of a wave whatever the number of workgroups, and less per K tile the fewer
// column blocks a wave carries, so: the fewest column blocks that still fit one round of workgroups
// (4096 -> 4096 at 128 rows: 256 workgroups of two column blocks 14.3 us, 128 of four 17.0; 4096 -> 2048 at 24
// rows: 128 of one 11.6, the tiled kernels 17.5), at least a quarter of a round (4096 -> 1024 at 24 rows, 64
// workgroups: 11.4 against 17.4), K of at least 16 tiles.  More than 64 rows are one workgroup per 64 rows and column
// group: narrow outputs only, where all of them fit one round.
// (A longer K: gemm_rows_plan_long_k and gemm_cols.hip.)
RowsPlan gemm_rows_plan(const WeightView& w, int M, int num_cus, const Epilogue& epi, bool any_width)
{
    if (M <= 16 || M > 512 || w.KT < 16 || w.KT > 64) return {0};
    const int64_t parts = (M + 63) / 64;
    for (int nf : {1, 2, 4}) {
        if (any_width) break;
        if (nf == 1 && epi.kind == kEpiSwiglu) continue;        // (a gate block and its up block sit in one workgroup)
        const int64_t groups = (w.NT + nf - 1) / nf * parts;
        if (groups <= num_cus) return {groups * 4 >= num_cus ? nf : 0};
    }
    // up to 64 rows a wide output may take more than one round.  Up to 48 rows two workgroups share a CU then (two or three
    // packed weight tiles in flight per wave instead of four, 256 registers): one's start and end overlap the other's
    // K loop (4096 -> 28672 bf16 norm + SwiGLU at 45 rows 35.0 -> 30.2 us, fp32 at 24 rows 28.3 -> 25.6, 2048 -> 20000 at 40
    // rows 20.5 -> 17.6, 2048 -> 128256 at 40 rows 71.0 -> 51.1).
    // Beyond 48 rows one workgroup of eight waves does two column groups that share X (gemm_rows_pair_kernel): 4096 -> 28672 norm +
    // SwiGLU at 64 rows 36.5 -> 34.1 us, Q8 45.0 -> 38.5, 2048 -> 20000 Q8 25.3 -> 20.6, 4096 -> 128256 122.5 -> 116.3.  Its workgroups are
    // a multiple of the K tiles, and a round of them takes 1.7 times as long as one of single groups: not where the multiple, or
    // the last round, costs the rounds it saves (single groups / pairs, rounds in brackets, Q4: 5120 -> 32000 at 63 rows 41 (2) / 61 (2), 2176 ->
    // 33882 at 54 rows 36.8 (3) / 41.5 (2), 4256 -> 40987 at 61 rows 55.1 (3) / 63.8 (2); 49 - 64 rows by rounds 2 / 1 0.92, 4 / 2 0.88, 6 / 3 0.92, 7 / 4
    // 0.91, Q8 0.85, 0.83, 0.83, 0.91).  Up to 48 rows it pays where the groups fit one round and a step is long, Q8 or many K tiles (Q8 4096 ->
    // 28672 at 45 rows 41.0 -> 38.0, Q8 8192 -> 16640 at 40 rows 59.7 -> 49.1, Q4 44.1 -> 40.6); not else (Q4 4096 -> 28672 at 45 rows
    // 29.6 / 29.7, 2048 -> 128256 at 40 rows 49.5 / 62.9, Q8 76.2 / 81.6).
    const int groups4 = (w.NT + 3) / 4, pair_groups = ((groups4 + 1) / 2 + w.KT - 1) / w.KT * w.KT;
    const int rounds = (groups4 + num_cus - 1) / num_cus, pair_rounds = (pair_groups + num_cus - 1) / num_cus;
    const bool pairs = parts == 1 && !any_width && (M > 48 ? pair_rounds * 17 <= rounds * 10 : pair_rounds == 1 && (w.bits == 8 || w.KT > 48));
    return {parts == 1 ? 4 : 0, parts == 1 && M <= 48 && !pairs, pairs};
}

// K of more than 64 tiles (plan_gemm_cols_long_k says which calls): a share of K per wave where a round of workgroups has one column
// block each, or two of Q4, and the rows are few: nothing to share X with then, and five slabs instead of eight.  The same bits.  us per
// call, weights in the L2s (from HBM), eight strips side by side / here, Q4 fp32 rows: 11136 -> 192 at 19 rows 14.9 / 13.2 (0.95 of the
// time), 10592 -> 496 at 28 15.3 / 13.3 (0.90), 13216 -> 368 at 21 16.2 / 14.8 (0.97), Q8 10400 -> 656 at 31 15.6 / 13.5 (0.93), 10208 -> 400 at 43
// 16.5 / 14.7 (0.93), two blocks: 10944 -> 3856 at 32 17.9 / 16.3 (0.96).  Not there: pairs 13664 -> 320 at 31 rows 16.6 / 16.1 (1.03), Q8 11808 ->
// 1344 at 34 17.3 / 17.8 (1.14); a longer K with more to take in, Q8 12544 -> 160 at 33 17.0 / 16.9 (1.08), 14144 -> 2272 at 28 18.0 / 17.3 (1.05);
// 49 rows and more, 13440 -> 256 at 49 19.8 / 19.9 (1.06); four blocks 11072 -> 4896 at 18 19.0 / 21.6 (1.13).
RowsPlan gemm_rows_plan_long_k(const WeightView& w, int M, int num_cus, const Epilogue& epi)
{
    const ColsPlan cols = plan_gemm_cols_long_k(w, M, num_cus, epi);
    if (!cols.rb || M > 48 || epi.kind == kEpiSwiglu) return {0};
    const int parts = (cols.splits + 3) / 4;               // workgroups per column group, four shares each
    if (w.NT * parts <= num_cus && (M <= 32 || w.KT <= 96)) return {1, false, false, cols.splits};
    if ((w.NT + 1) / 2 * parts <= num_cus && w.bits == 4 && M <= 32 && w.KT <= 96) return {2, false, false, cols.splits};
    return {0};
}

hipError_t launch_gemm_rows(const WeightView& w, const void* x_staged, int M, void* y, int ydt, const Epilogue& epi,
                            const float* ssq_part, int ssq_blocks, const float* unscale, const RowsPlan& plan, float* slabs, hipStream_t st)
{
    const NormStats ns = {ssq_part, ssq_blocks, unscale};
    // four waves, one per SIMD with the whole register file: four K tiles of packed weights and one K tile of
    // X in flight per wave.  Measured against it on 4096 -> 14336 at 64 bf16 rows (19.1 us per call with the
    // staging pass; the tiled kernel 22.1): eight waves with two / three weight tiles in flight 22.8 / 20.2;
    // X two / four K tiles ahead 21.7 / 20.4; eight weight tiles ahead 23.9; MFMAs and dequantisation
    // interleaved by scheduling hints 21.2; four staging + four multiplying waves sharing K slots through
    // LDS 26.7.
    // Up to 48 rows the workgroup carries two or three row blocks instead of four: the rows of X are most of what
    // a CU takes in, and its L1 delivers 64 bytes a cycle.
    const int mf = M > 48 ? 4 : M > 32 ? 3 : 2;
    auto go = [&](auto bits, auto nfc) {
        constexpr int B = decltype(bits)::value, F = decltype(nfc)::value;
        if (mf == 2) return launch_rows_t<B, 2, F, 4, 4, 1>(w, x_staged, M, y, ydt, epi, ns, st);
        if (mf == 3) return launch_rows_t<B, 3, F, 4, 4, 1>(w, x_staged, M, y, ydt, epi, ns, st);
        return launch_rows_t<B, 4, F, 4, 4, 1>(w, x_staged, M, y, ydt, epi, ns, st);
    };
    auto with_bits = [&](auto nfc) {
        if (w.bits == 8) return go(std::integral_constant<int, 8>{}, nfc);
        return go(std::integral_constant<int, 4>{}, nfc);
    };
    if (plan.shares) {
        if (plan.nf == 2) return launch_rows_t<4, 2, 2, 4, 4, 1, 1, true>(w, x_staged, M, y, ydt, epi, ns, st, plan.shares, slabs);
        if (w.bits == 8) {
            if (mf == 2) return launch_rows_t<8, 2, 1, 4, 4, 1, 1, true>(w, x_staged, M, y, ydt, epi, ns, st, plan.shares, slabs);
            return launch_rows_t<8, 3, 1, 4, 4, 1, 1, true>(w, x_staged, M, y, ydt, epi, ns, st, plan.shares, slabs);
        }
        if (mf == 2) return launch_rows_t<4, 2, 1, 4, 4, 1, 1, true>(w, x_staged, M, y, ydt, epi, ns, st, plan.shares, slabs);
        return launch_rows_t<4, 3, 1, 4, 4, 1, 1, true>(w, x_staged, M, y, ydt, epi, ns, st, plan.shares, slabs);
    }
    if (plan.pairs) {
        if (w.bits == 4) {
            if (mf == 2) return launch_pair_t<4, 2, 4, 3>(w, x_staged, M, y, ydt, epi, ns, st);
            if (mf == 3) return launch_pair_t<4, 3, 4, 3>(w, x_staged, M, y, ydt, epi, ns, st);
            return launch_pair_t<4, 4, 4, 2>(w, x_staged, M, y, ydt, epi, ns, st);
        }
        if (mf == 2) return launch_pair_t<8, 2, 3, 3>(w, x_staged, M, y, ydt, epi, ns, st);
        if (mf == 3) return launch_pair_t<8, 3, 3, 3>(w, x_staged, M, y, ydt, epi, ns, st);
        return launch_pair_t<8, 4, 2, 2>(w, x_staged, M, y, ydt, epi, ns, st);
    }
    if (plan.two_per_cu) {
        if (w.bits == 8) {
            if (mf == 2) return launch_rows_t<8, 2, 4, 4, 2, 1, 2>(w, x_staged, M, y, ydt, epi, ns, st);
            return launch_rows_t<8, 3, 4, 4, 2, 1, 2>(w, x_staged, M, y, ydt, epi, ns, st);
        }
        if (mf == 2) return launch_rows_t<4, 2, 4, 4, 3, 1, 2>(w, x_staged, M, y, ydt, epi, ns, st);
        return launch_rows_t<4, 3, 4, 4, 3, 1, 2>(w, x_staged, M, y, ydt, epi, ns, st);
    }
    if (plan.nf == 1) return with_bits(std::integral_constant<int, 1>{});
    if (plan.nf == 2) return with_bits(std::integral_constant<int, 2>{});
    return with_bits(std::integral_constant<int, 4>{});
}

}  // namespace cybq
