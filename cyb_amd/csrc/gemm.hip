// gemm.hip - prefill kernel: Y[M,N] = X[M,K] * W^T for M > 16 on MFMA.
//
// Workgroup = 8 waves, output tile 256 (or 512) rows x (16*NF) columns; wave w owns
// two (four) row blocks of 16 against all NF column blocks.  Fewer rows: gemm_rows.hip and gemm_cols.hip.
//
//   X  never touches LDS.  An MFMA A operand is 16 rows x 32 k with lane l
//      holding row l%16, k 8*(l/16)..+8.  Read straight from a row-major X that is
//      64 separate 16 B accesses per load (neighbouring lanes are different rows),
//      which saturates the address path long before the matrix cores.  So a small
//      kernel first restages X once per call in operand order - row block, scale
//      group, lane - and the multiply streams it global -> registers with
//      contiguous 1 KB loads, one K tile (four scale groups) ahead of its use.
//      The same pass turns bf16 / fp32 rows into f16 operands for FAST mode.
//   W  is shared by the waves of a workgroup: per K tile (128 k = 4 groups) the NF native
//      weight tiles are read once with 128-bit loads and dequantised to
//      w = f32(scale) * q, which is exact in fp32 (11-bit x 4-bit significand).
//      A 16-bit MFMA operand cannot hold those 15 bits, so w is split without
//      loss into hi = round16(w) and lo = w - hi (both exactly representable)
//      and written to LDS as two operands, already in MFMA B-operand order.
//      LDS is double buffered, one barrier per K tile.
//   The inner loop is nothing but LDS operand reads and v_mfma_f32_16x16x32
//      accumulating hi and lo products in fp32: no per-group scaling on the
//      vector ALU, accumulators stay inside the matrix pipeline until the
//      epilogue.  The price is two MFMAs per scale group; the gain is that the
//      weights enter the contraction exactly, so the result differs from the
//      fp32 CPU path only by accumulation order.  (Q8 weights need 18 bits; lo
//      is then rounded and the split is exact to 2^-17 relative.)
//
// Two modes share this kernel:
//   EXACT  as described above: two MFMAs per scale group in the type of X.
//   FAST   one f16 MFMA per scale group.  The weight operand is round_f16(scale * q)
//          (one rounding, relative error <= 2^-11, about 2e-4 relative L2 on Y -
//          inside the operator's 1e-3 tolerance); bf16 and fp32 activations become
//          f16 operands in the staging pass behind a power-of-two scale per row that is
//          undone in the epilogue.
//
// Shapes with fewer tiles than CUs split K over workgroups: each split leaves fp32
// partial sums in its own slab of the workspace and a last kernel adds the slabs in a
// fixed order, so results are reproducible (no atomics).
//
// Out-of-range rows / columns / k are clamped to valid addresses inside the hot
// loop (their results are never stored, padded weights are zero); the loop has
// no branches, so the compiler can count outstanding loads exactly.
#include <algorithm>
#include <type_traits>

#include "cybq_device.h"
#include "cybq_internal.h"

namespace cybq {

int g_rows_kernel = 0;        // (set_gemm_tuning: 2 = the tiled kernels of this file alone in FAST mode, 3 = in both modes, 1 = the few-rows kernel whatever the width)
static bool g_role_ranges = true;     // (7 = as 2, and ranges of K stay with gemm_kernel)

namespace {

#include "gemm_parts.h"

// gamma[k0 .. k0+8) (k0 a multiple of 8, gamma 16-byte aligned) as loaded: two loads whatever its type, so that a kernel can ask for it next
// to its rows without a branch around the loads (16-bit types: the second repeats the first), and as fp32
struct Gamma8 {
    u32x4_t v[2];
};

__device__ __forceinline__ Gamma8 load_gamma8(const void* g, int gdt, int k0)
{
    const char* const p = static_cast<const char*>(g) + (int64_t)k0 * (gdt == kF32 ? 4 : 2);
    return {{*reinterpret_cast<const u32x4_t*>(p), *reinterpret_cast<const u32x4_t*>(p + (gdt == kF32 ? 16 : 0))}};
}

__device__ __forceinline__ void gamma8_values(const Gamma8& c, int gdt, float out[8])
{
    if (gdt == kF32) {
#pragma unroll
        for (int i = 0; i < 8; i++) out[i] = __builtin_bit_cast(float, (uint32_t)c.v[i >> 2][i & 3]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (gdt == kF16) {
                const half2_t h = as_h2(c.v[0][i]);
                out[2 * i] = (float)h.x;
                out[2 * i + 1] = (float)h.y;
            } else {
                out[2 * i] = __builtin_bit_cast(float, c.v[0][i] << 16);
                out[2 * i + 1] = __builtin_bit_cast(float, c.v[0][i] & 0xffff0000u);
            }
        }
    }
}

// (w0, w1) fp32 -> packed 16-bit hi pair and lo pair with hi + lo == w
template <int XBF>
__device__ __forceinline__ void split_pair(float w0, float w1, uint32_t& hi, uint32_t& lo)
{
    if (XBF) {
        bf16x2_t h = __builtin_convertvector((float2_t){w0, w1}, bf16x2_t);
        hi = __builtin_bit_cast(uint32_t, h);
        float h0 = __builtin_bit_cast(float, hi << 16);
        float h1 = __builtin_bit_cast(float, hi & 0xffff0000u);
        bf16x2_t l = __builtin_convertvector((float2_t){w0 - h0, w1 - h1}, bf16x2_t);
        lo = __builtin_bit_cast(uint32_t, l);
    } else {
        half2_t h = {(_Float16)w0, (_Float16)w1};
        hi = as_u32(h);
        half2_t l = {(_Float16)(w0 - (float)h.x), (_Float16)(w1 - (float)h.y)};
        lo = as_u32(l);
    }
}

// group j of a native tile -> B operand(s) in LDS: hi and lo (EXACT) or one rounded f16 operand
template <int BITS, int XBF, bool EXACT>
__device__ __forceinline__ void dequant_group_to_lds(const WRegs<BITS>& r, int j, uint32_t magic, u32x4_t* dst,
                                                     int lane)
{
    uint32_t bw[4];
    if (BITS == 4) unpack_q4_f16(r.q[0][2 * (j >> 1)], r.q[0][2 * (j >> 1) + 1], j & 1, magic, bw);
    else unpack_q8_f16(r.q[(BITS == 4) ? 0 : (j >> 1)][(j & 1) * 2], r.q[(BITS == 4) ? 0 : (j >> 1)][(j & 1) * 2 + 1], bw);
    const uint32_t sb = (j & 1) ? (r.s[j >> 1] >> 16) : (r.s[j >> 1] & 0xffffu);
    if (!EXACT) {
        const _Float16 sh = __builtin_bit_cast(_Float16, (uint16_t)sb);
        const half2_t s2 = {sh, sh};
        uint32_t o[4];
#pragma unroll
        for (int p = 0; p < 4; p++) o[p] = as_u32(as_h2(bw[p]) * s2);     // round_f16(scale * q)
        dst[j * 64 + lane] = (u32x4_t){o[0], o[1], o[2], o[3]};
        return;
    }
    const float sc = f16_bits_to_f32(sb);
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        half2_t qv = as_h2(bw[p]);
        split_pair<XBF>(sc * (float)qv.x, sc * (float)qv.y, hi[p], lo[p]);
    }
    dst[(j * 2 + 0) * 64 + lane] = (u32x4_t){hi[0], hi[1], hi[2], hi[3]};
    dst[(j * 2 + 1) * 64 + lane] = (u32x4_t){lo[0], lo[1], lo[2], lo[3]};
}

// XBF = 1: X is bf16, 0: X is f16.  EXACT: see the header comment.
// Wave wv of eight owns MF row blocks of 16 against all NF column blocks.
template <int BITS, int XBF, int NF, bool EXACT, int MF>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_kernel(const uint8_t* __restrict__ wbase, const u32x4_t* __restrict__ x, int KT_, int NT_, int x_row_blocks, int M,
                                                   int n_tiles, int m_tiles, int splits, int kt_per_split, int groups, int K_,
                                                   int N_, void* __restrict__ y, int ydt, float out_scale,
                                                   float* __restrict__ part, Epilogue epi, NormStats ns)
{
    // (leading scalar arguments in the order of their first use: they arrive in registers at wave start.  With K behind the output's address, us per call: here no
    // difference, 14336 -> 4096 at 1000 rows 119.8 / 119.8; in gemm_roles_kernel 14336 -> 4096 at 512 rows 67.2 / 66.8, 10240 -> 3136 46.2 / 45.8, 4096 -> 6144 with
    // a norm 37.3 / 37.1.)
    const WeightView w = {wbase, N_, K_, NT_, KT_, BITS};
    // Workgroups are handed to the 8 XCDs round-robin (id % 8) and every XCD has
    // its own L2.  Give each XCD a contiguous run of tiles in row-block-major
    // order, so the workgroups sharing an L2 read the same rows of X and X is
    // fetched into every L2 once instead of once per column tile.
    const int per_xcd = groups >> 3;
    const int item = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
    if (item >= n_tiles * m_tiles * splits) return;
    // split-major: workgroups that run side by side share a K range of X
    const int split = item / (n_tiles * m_tiles);
    const int tile_m = (item - split * (n_tiles * m_tiles)) / n_tiles;
    const int tile_n = item - (split * m_tiles + tile_m) * n_tiles;
    constexpr int WAVES = 8;
    constexpr int BM = WAVES * MF * 16;               // MF = row blocks (of 16) per wave
    constexpr int WT = (NF + WAVES - 1) / WAVES;      // weight tiles a wave stages per K tile
    constexpr int OPS = EXACT ? 2 : 1;                // B operands per scale group
    constexpr int TILE16 = 4 * OPS * 64;              // u32x4 per column block per K tile
    constexpr int BUF16 = NF * TILE16;                // u32x4 per LDS buffer
    constexpr int MMA_BF = EXACT ? XBF : 0;           // FAST always multiplies in f16
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    u32x4_t* ws = reinterpret_cast<u32x4_t*>(smem);   // [2][NF][4][OPS][64]
    const uint32_t magic = q4_magic_vgpr();

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row16 = lane & 15;
    const int oct = lane >> 4;
    const int nt0 = tile_n * NF;
    const int m0 = tile_m * BM + wv * (MF * 16);
    const int K = w.K;
    // this workgroup's K tiles: [kt_lo, kt_lo + KT) of the weight's w.KT (all of them unless K is split)
    const int kt_lo = split * kt_per_split;
    const int KT = min(kt_per_split, w.KT - kt_lo);
    // Workgroups that run side by side share rows of X.  Walking K in the same order
    // they would all ask the same few L2 channels for the same lines at the same
    // moment (a row of X is a multiple of the channel interleave long), so each
    // column tile starts its walk at a different K tile and wraps around.  The
    // order depends on the column tile only: a row of Y does not depend on M.
    const int kt0 = tile_n % KT;
    auto rot = [&](int kt) {
        const int r = min(kt, KT - 1) + kt0;
        return kt_lo + (r >= KT ? r - KT : r);
    };

    // X arrives staged in A-operand order (stage_x_kernel): row block rb, scale group
    // g is one contiguous KB, lane after lane, so a load is one wave-uniform base
    // plus lane * 16 B and adjacent lanes read adjacent memory.  Row blocks past the
    // last are clamped to it (never stored); a scale group past K (padding, zero
    // weights) reads the last real group instead.
    const int G = K / kGroup;
    const u32x4_t* xb[MF];
#pragma unroll
    for (int i = 0; i < MF; i++)
        xb[i] = x + ((int64_t)min(m0 / 16 + i, x_row_blocks - 1) * G) * 64 + lane;
    auto load_x = [&](Frag16 (&dst)[MF], int kt, int j) {
        const int g = min(rot(kt) * 4 + j, G - 1);
#pragma unroll
        for (int i = 0; i < MF; i++) dst[i].u = xb[i][g * 64];
    };

    // The weight tiles this wave stages: column block f = wv + WAVES*t (clamped: a wave
    // past the end stages a neighbour's block again with identical values, no branch).
    int64_t wtile[WT];
    int wdst[WT];
#pragma unroll
    for (int t = 0; t < WT; t++) {
        const int f = min(wv + WAVES * t, NF - 1);
        wdst[t] = f * TILE16;
        wtile[t] = (int64_t)min(nt0 + f, w.NT - 1) * w.KT;
    }
    auto load_units = [&](WRegs<BITS> (&dst)[WT], int kt) {
#pragma unroll
        for (int t = 0; t < WT; t++) load_wtile<BITS>(dst[t], w, wtile[t] + rot(kt), lane);
    };
    auto stage_units = [&](WRegs<BITS> (&src)[WT], int j, u32x4_t* buf) {
#pragma unroll
        for (int t = 0; t < WT; t++) dequant_group_to_lds<BITS, XBF, EXACT>(src[t], j, magic, buf + wdst[t], lane);
    };

    float4_t acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[i][f] = (float4_t){0.f, 0.f, 0.f, 0.f};

    // ---- prologue: first K tile of X, W tile 0 -> LDS buffer 0, W tiles 1 .. SETS-1 -> registers
    Frag16 xa[4][MF];          // one K tile (four scale groups) of X in flight
#pragma unroll
    for (int j = 0; j < 4; j++) load_x(xa[j], 0, j);
    RowStats stats = {};                            // (512-row tiles have no registers for them: 4096 -> 14336 at 2048 rows 240 -> 250 us)
    if constexpr (MF <= 2) stats = load_row_stats(ns, epi.gamma != nullptr, min(m0 + min(lane, MF * 16 - 1), M - 1), wbase);
    // Packed weights wait in registers: K tile t sits in wreg[t % SETS], requested SETS - 1
    // iterations before it is dequantised.  Loads retire in order and every iteration
    // also requests X, so two sets leave a weight tile one iteration (about 2 us) to
    // arrive - enough from cache, short for a first touch in HBM; Q4 FAST has the
    // registers for four.
    constexpr int SETS = (BITS == 4 && !EXACT) ? 4 : 2;
    WRegs<BITS> wreg[SETS][WT];
    {
        WRegs<BITS> w0[WT];
        load_units(w0, 0);
#pragma unroll
        for (int t = 1; t < SETS; t++) load_units(wreg[t], t);
#pragma unroll
        for (int j = 0; j < 4; j++) stage_units(w0, j, ws);
    }
    __syncthreads();

    // One K tile.  R = kt % SETS is a compile-time constant (the loop below is unrolled
    // SETS times), so LDS buffers (R & 1) and register sets alternate without copies
    // or selects:  multiply from LDS buffer R & 1;  dequantise tile kt+1 from its
    // register set into the other buffer;  request tile kt+SETS into the set tile kt
    // left free.  Past the end indices are clamped: a tile is staged again but never read.
    auto k_tile = [&](int kt, auto residue) {
        constexpr int R = decltype(residue)::value;
        constexpr int P = R & 1;
        const u32x4_t* wcur = ws + P * BUF16;
        u32x4_t* wnxt = ws + (1 - P) * BUF16;
        load_units(wreg[R], kt + SETS);

#pragma unroll
        for (int j = 0; j < 4; j++) {
            const Frag16 (&a)[MF] = xa[j];
#pragma unroll
            for (int f = 0; f < NF; f++) {
                Frag16 b[OPS];
#pragma unroll
                for (int o = 0; o < OPS; o++) b[o].u = wcur[f * TILE16 + (j * OPS + o) * 64 + lane];
#pragma unroll
                for (int o = 0; o < OPS; o++)
#pragma unroll
                    for (int i = 0; i < MF; i++) acc[i][f] = mma<MMA_BF>(a[i], b[o], acc[i][f]);
            }
            // After an odd group its pair of operand sets is free: refill both with
            // the same groups of the next K tile.
            if (j & 1) {
                load_x(xa[j - 1], kt + 1, j - 1);
                load_x(xa[j], kt + 1, j);
            }
            // a quarter of the next tile's dequantisation rides along with every group
            stage_units(wreg[(R + 1) % SETS], j, wnxt);
        }
        // Order inside the K tile (two waves per SIMD): the dequantisation of the next tile is
        // spread between the MFMAs.  A wave issues in order: arithmetic queued behind a run of
        // MFMAs waits for all of them and the matrix pipe idles while it runs afterwards; and the
        // barrier keeps the two waves of a SIMD in the same phase, so they do not cover for each
        // other.
        if constexpr (!EXACT) {
            constexpr int READS = 4 * NF * OPS;
            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);          // LDS reads run two ahead of their MFMAs
#pragma unroll
            for (int i = 0; i < READS; i++) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // one LDS read
                __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);     // its MFMAs, one per row block
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);      // two vector ALU instructions
            }
        }
        __syncthreads();
    };
    for (int kt = 0; kt < KT; kt += SETS) {
        k_tile(kt, std::integral_constant<int, 0>{});
        if (kt + 1 < KT) k_tile(kt + 1, std::integral_constant<int, 1>{});
        if constexpr (SETS == 4) {
            if (kt + 2 < KT) k_tile(kt + 2, std::integral_constant<int, 2>{});
            if (kt + 3 < KT) k_tile(kt + 3, std::integral_constant<int, 3>{});
        }
    }

    // ---- epilogue: a K split leaves its partial sums in fp32 for splitk_reduce_kernel (whole runs of a row
    // through LDS, like the final sums)
    if (splits > 1) {
        const Epilogue plain = {kEpiNone, nullptr, nullptr, 0, 0.f};
        write_rows<MF, NF>(acc, reinterpret_cast<float*>(smem) + wv * (16 * NF * 16), m0, nt0, M, w.N, part + (int64_t)split * M * w.N, kF32,
                           1.0f, plain, lane);
        return;
    }
    if (epi.gamma || ns.unscale) {     // folded RMSNorm: rstd of the row; widened activations: the row's power of two
        float mine = 0.f;
        if constexpr (MF <= 2) mine = row_factor(stats, ns, epi.gamma != nullptr, min(m0 + min(lane, MF * 16 - 1), M - 1), K, epi.eps);
#pragma unroll
        for (int i = 0; i < MF; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float rs = MF <= 2 ? __shfl(mine, i * 16 + oct * 4 + r, 64)
                                         : row_factor(ns, epi.gamma != nullptr, min(m0 + i * 16 + oct * 4 + r, M - 1), K, epi.eps);
#pragma unroll
                for (int f = 0; f < NF; f++) acc[i][f][r] *= rs;
            }
    }
    if (epi.kind == kEpiSwiglu) {      // column blocks 2p / 2p+1 are gate / up of output block (nt0 >> 1) + p
        const int n_out = w.N >> 1;
#pragma unroll
        for (int i = 0; i < MF; i++)
#pragma unroll
            for (int p = 0; p < NF / 2; p++) {
                const int n = ((nt0 >> 1) + p) * 16 + row16;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m0 + i * 16 + oct * 4 + r;
                    if (m < M && n < n_out)
                        store_out_g(y, ydt, (int64_t)m * n_out + n,
                                    silu_mul(acc[i][2 * p][r] * out_scale, acc[i][2 * p + 1][r] * out_scale));
                }
            }
        return;
    }
    write_rows<MF, NF>(acc, reinterpret_cast<float*>(smem) + wv * (16 * NF * 16), m0, nt0, M, w.N, y, ydt, out_scale, epi, lane);
}

// The same multiply (FAST mode, f16 operands) with the work of a workgroup split by role:
// MW waves only multiply - each owns MF row blocks against all NF column blocks, streams its X
// from global memory XD K tiles ahead and reads the weight operands from LDS - and four waves
// only fetch packed weight tiles and dequantise them into LDS, several K tiles ahead.  Loads
// retire in order within a wave: in gemm_kernel the wait for the next rows of X is also a wait
// for every weight tile requested before them, and a first touch in HBM holds the matrix pipe
// up; here the multiplying waves never wait for HBM.  Waves are dealt to the four SIMDs in turn,
// so every SIMD carries one staging wave: the dequantisation runs in the issue slots the MFMAs
// leave free.  MW*MF*16 x NF*16 outputs per workgroup, one barrier per K tile.  SPLIT: K over workgroups, partial sums as in gemm_kernel.
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

template <int BITS, int NF, int MF, int MW, int XD, bool SPLIT>
__global__ __launch_bounds__((MW + 4) * 64) __attribute__((amdgpu_waves_per_eu((MW + 7) / 4, (MW + 7) / 4))) void gemm_roles_kernel(
    const uint8_t* __restrict__ wbase, const u32x4_t* __restrict__ x, int KT_, int NT_, int x_row_blocks, int M, int n_tiles,
    int m_tiles, int groups, int K_, int splits, int kt_per_split, int N_, void* __restrict__ y, int ydt, float out_scale, float* __restrict__ part,
    Epilogue epi, NormStats ns)
{
    const WeightView w = {wbase, N_, K_, NT_, KT_, BITS};
    constexpr int SW = 4;                             // staging waves
    constexpr bool HALF = NF % SW == 2;
    constexpr int WT = HALF ? NF / SW : (NF + SW - 1) / SW;            // weight tiles a staging wave handles per K tile (and half of one)
    constexpr int TILE16 = 4 * 64;                    // u32x4 per column block per K tile
    constexpr int BUF16 = NF * TILE16;
    // K tiles of packed weights in flight per staging wave (8 measured the same at 64 and 128 rows, 16
    // slower: 23 -> 30 us at 64 rows)
    constexpr int DEPTH = 4;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    u32x4_t* ws = reinterpret_cast<u32x4_t*>(smem);   // [2][NF][4][64]

    const int per_xcd = groups >> 3;                  // (same tile order as gemm_kernel)
    const int item = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
    if (item >= n_tiles * m_tiles * (SPLIT ? splits : 1)) return;
    const int row = item / n_tiles, tile_n = item - row * n_tiles;
    const int split = SPLIT ? row / m_tiles : 0, tile_m = row - split * m_tiles;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt0 = tile_n * NF;
    const int K = w.K;
    const int kt_lo = SPLIT ? split * kt_per_split : 0;              // my K tiles: [kt_lo, kt_lo + KT)
    const int KT = SPLIT ? min(kt_per_split, w.KT - kt_lo) : w.KT;
    const int kt0 = tile_n % KT;
    auto rot = [&](int kt) {
        const int r = min(kt, KT - 1) + kt0;
        return kt_lo + (r >= KT ? r - KT : r);
    };

    if (wave >= MW) {
        // ---- staging waves ----------------------------------------------------------------
        const int pw = wave - MW;
        const uint32_t magic = q4_magic_vgpr();
        int64_t wtile[WT];
        int wdst[WT];
#pragma unroll
        for (int t = 0; t < WT; t++) {
            const int f = min(pw + SW * t, NF - 1);     // (past the end: a neighbour's block again, same values)
            wdst[t] = f * TILE16;
            wtile[t] = (int64_t)min(nt0 + f, w.NT - 1) * w.KT;
        }
        // Six blocks: the last two in halves (two scale groups each).  A K tile waits for the last of these waves, and two blocks to a wave were
        // eight's work.  us per call, before / after, bf16: 4096 -> 6144 at 512 rows 43.4 / 41.2, Q8 44.5 / 41.7, 4096 -> 12288 at 256 rows 41.1 / 39.3,
        // 2048 -> 3072 at 1000 rows 25.3 / 24.1, 2880 -> 5760 at 512 rows 30.3 / 28.7.  (Seven blocks in equal parts, three groups of a block to
        // three waves and their fourth groups to the last: 4096 -> 14336 at 512 rows 69.0 / 69.0, with a norm 69.7 / 70.9; not done.  Eight
        // staging waves: 41.5 / 42.0, 4096 -> 6144 at 256 rows 27.6 / 28.5.)
        const int half = pw & 1, hf = min(WT * SW + (pw >> 1), NF - 1), hdst = hf * TILE16 + half * 128;
        const int64_t htile = (int64_t)min(nt0 + hf, w.NT - 1) * w.KT;
        struct Staged {
            WRegs<BITS> whole[WT];
            WRegs<BITS> half;             // (its first two groups' registers)
        };
        Staged wreg[DEPTH];
        auto fetch = [&](Staged& dst, int kt) {
#pragma unroll
            for (int t = 0; t < WT; t++) load_wtile<BITS>(dst.whole[t], w, wtile[t] + rot(kt), lane);
            if constexpr (HALF) {
                const int64_t tile = htile + rot(kt);
                if constexpr (BITS == 4) {
                    const u32x2_t q = reinterpret_cast<const u32x2_t*>(tile_q<BITS>(w, tile))[lane * 2 + half];
                    dst.half.q[0][0] = q[0];
                    dst.half.q[0][1] = q[1];
                } else {
                    dst.half.q[0] = tile_q<BITS>(w, tile)[half * 64 + lane];
                }
                dst.half.s[0] = reinterpret_cast<const uint32_t*>(tile_s<BITS>(w, tile))[(lane & 15) * 2 + half];
            }
        };
        auto stage = [&](Staged& src, u32x4_t* buf) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
#pragma unroll
                for (int t = 0; t < WT; t++) dequant_group_to_lds<BITS, 0, false>(src.whole[t], j, magic, buf + wdst[t], lane);
                if constexpr (HALF) {
                    if (j < 2) dequant_group_to_lds<BITS, 0, false>(src.half, j, magic, buf + hdst, lane);
                }
            }
        };
#pragma unroll
        for (int d = 0; d < DEPTH; d++) fetch(wreg[d], d);
        stage(wreg[0], ws);
        fetch(wreg[0], DEPTH);
        __syncthreads();
        // during K tile kt: tile kt + 1 (register set (kt + 1) % DEPTH) -> the other LDS buffer, then that
        // set is refilled with tile kt + 1 + DEPTH
        auto k_tile = [&](int kt, auto residue) {
            constexpr int R = decltype(residue)::value;            // = (kt + 1) % DEPTH
            stage(wreg[R], ws + ((R & 1) ? BUF16 : 0));
            fetch(wreg[R], kt + 1 + DEPTH);
            __syncthreads();
        };
        // Whole rounds in the loop, the remainder behind it: a tile skipped inside the loop is a path
        // into the loop head with fewer loads outstanding, the one wait count an instruction carries has
        // to be safe for that path, and the first use of a tile then also waits for the newest request.
        // With few rows there is little arithmetic per K tile to hide that behind (4096 -> 14336 at 64
        // rows 26.1 -> 22.8 us); the 256-row kernel measured better with the tighter counts (60.5 against
        // 63 us at 512 rows).
        int kt = 0;
        if constexpr (MW <= 4) {
            for (; kt + DEPTH <= KT; kt += DEPTH)
                static_for<0, DEPTH>([&](auto i) { k_tile(kt + decltype(i)::value, std::integral_constant<int, (decltype(i)::value + 1) % DEPTH>{}); });
            static_for<0, DEPTH - 1>([&](auto i) {
                if (kt + decltype(i)::value < KT) k_tile(kt + decltype(i)::value, std::integral_constant<int, (decltype(i)::value + 1) % DEPTH>{});
            });
            return;
        } else {
            for (; kt < KT; kt += DEPTH) {
                k_tile(kt, std::integral_constant<int, 1>{});
                if (kt + 1 < KT) k_tile(kt + 1, std::integral_constant<int, 2>{});
                if (kt + 2 < KT) k_tile(kt + 2, std::integral_constant<int, 3>{});
                if (kt + 3 < KT) k_tile(kt + 3, std::integral_constant<int, 0>{});
            }
            return;
        }
    }

    // ---- multiplying waves --------------------------------------------------------------------
    const int m0 = tile_m * (MW * MF * 16) + wave * (MF * 16);
    const int G = K / kGroup;
    const u32x4_t* xb[MF];
#pragma unroll
    for (int i = 0; i < MF; i++) xb[i] = x + ((int64_t)min(m0 / 16 + i, x_row_blocks - 1) * G) * 64 + lane;
    auto load_x = [&](Frag16 (&dst)[MF], int kt, int j) {
        const int g = min(rot(kt) * 4 + j, G - 1);
#pragma unroll
        for (int i = 0; i < MF; i++) dst[i].u = xb[i][g * 64];
    };
    float4_t acc[MF][NF];
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) acc[i][f] = (float4_t){0.f, 0.f, 0.f, 0.f};
    Frag16 xa[XD][4][MF];          // XD K tiles of X in flight
#pragma unroll
    for (int d = 0; d < XD; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) load_x(xa[d][j], d, j);
    const RowStats stats = load_row_stats(ns, epi.gamma != nullptr, min(m0 + min(lane, MF * 16 - 1), M - 1), wbase);
    __syncthreads();
    auto k_tile = [&](int kt, auto residue) {
        constexpr int D = decltype(residue)::value;                 // = kt % XD
        const u32x4_t* wcur = ws + ((kt & 1) ? BUF16 : 0);
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
            for (int f = 0; f < NF; f++) {
                Frag16 b;
                b.u = wcur[f * TILE16 + j * 64 + lane];
#pragma unroll
                for (int i = 0; i < MF; i++) acc[i][f] = mma<0>(xa[D][j][i], b, acc[i][f]);
            }
            load_x(xa[D][j], kt + XD, j);      // this group's operands are free: those of K tile kt + XD take their place
        }
        constexpr int READS = 4 * NF;
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);          // LDS reads run two ahead of their MFMAs
#pragma unroll
        for (int i = 0; i < READS; i++) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, MF, 0);
            // (a group's X operands are requested again as soon as its last MFMA is out: left to itself
            // the scheduler moves all of a tile's requests to its end, one K tile less of lead)
            if (i % NF == NF - 1) __builtin_amdgcn_sched_group_barrier(0x020, MF, 0);
        }
        __syncthreads();
    };
    int kt = 0;
    if constexpr (MW <= 4) {                       // (whole rounds in the loop: see the staging waves)
        for (; kt + XD <= KT; kt += XD) {
            k_tile(kt, std::integral_constant<int, 0>{});
            if constexpr (XD > 1) k_tile(kt + 1, std::integral_constant<int, 1>{});
            if constexpr (XD > 2) k_tile(kt + 2, std::integral_constant<int, 2>{});
            if constexpr (XD > 3) k_tile(kt + 3, std::integral_constant<int, 3>{});
        }
    }
    for (; kt < KT; kt += XD) {
        k_tile(kt, std::integral_constant<int, 0>{});
        if constexpr (XD > 1) {
            if (kt + 1 < KT) k_tile(kt + 1, std::integral_constant<int, 1>{});
        }
        if constexpr (XD > 2) {
            if (kt + 2 < KT) k_tile(kt + 2, std::integral_constant<int, 2>{});
        }
        if constexpr (XD > 3) {
            if (kt + 3 < KT) k_tile(kt + 3, std::integral_constant<int, 3>{});
        }
    }
    if constexpr (SPLIT) {
        const Epilogue plain = {kEpiNone, nullptr, nullptr, 0, 0.f};
        write_rows<MF, NF>(acc, reinterpret_cast<float*>(smem) + wave * (16 * NF * 16), m0, nt0, M, w.N, part + (int64_t)split * M * w.N, kF32, 1.0f, plain,
                           lane);
        return;
    }
    if (epi.gamma || ns.unscale) {
        const float mine = row_factor(stats, ns, epi.gamma != nullptr, min(m0 + min(lane, MF * 16 - 1), M - 1), K, epi.eps);
#pragma unroll
        for (int i = 0; i < MF; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float rs = __shfl(mine, i * 16 + (lane >> 4) * 4 + r, 64);
#pragma unroll
                for (int f = 0; f < NF; f++) acc[i][f][r] *= rs;
            }
    }
    if constexpr (NF % 2 == 0) {
        if (epi.kind == kEpiSwiglu) {      // column blocks 2p / 2p+1 are gate / up of output block (nt0 >> 1) + p
            float4_t act[MF][NF / 2];
#pragma unroll
            for (int i = 0; i < MF; i++)
#pragma unroll
                for (int p = 0; p < NF / 2; p++)
#pragma unroll
                    for (int r = 0; r < 4; r++) act[i][p][r] = silu_mul(acc[i][2 * p][r] * out_scale, acc[i][2 * p + 1][r] * out_scale);
            const Epilogue plain = {kEpiNone, nullptr, nullptr, 0, 0.f};
            write_rows<MF, NF / 2>(act, reinterpret_cast<float*>(smem) + wave * (16 * NF * 16), m0, nt0 >> 1, M, w.N >> 1, y, ydt, 1.0f, plain, lane);
            return;
        }
    }
    write_rows<MF, NF>(acc, reinterpret_cast<float*>(smem) + wave * (16 * NF * 16), m0, nt0, M, w.N, y, ydt, out_scale, epi, lane);
}

constexpr int kMaxSplits = 8;

// y = epilogue(out_scale * (part[0] + part[1] + ... + part[splits-1])), slabs added in that order.
// One thread per output element; N = columns of a slab (for SwiGLU y has N / 2).
__global__ void splitk_reduce_kernel(const float* __restrict__ part, int splits, int M, int N, void* __restrict__ y, int ydt,
                                     float out_scale, Epilogue epi, NormStats ns, int K)
{
    const int64_t slab = (int64_t)M * N;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (epi.kind == kEpiSwiglu) {
        const int n_out = N >> 1;
        if (i >= (int64_t)M * n_out) return;
        const int m = (int)(i / n_out), n = (int)(i - (int64_t)m * n_out);
        const int64_t ig = (int64_t)m * N + (n >> 4) * 32 + (n & 15);
        float g = part[ig], u = part[ig + 16];
        for (int s = 1; s < splits; s++) {
            g += part[s * slab + ig];
            u += part[s * slab + ig + 16];
        }
        const float sc = out_scale * row_factor(ns, epi.gamma != nullptr, m, K, epi.eps);
        store_out_g(y, ydt, i, silu_mul(g * sc, u * sc));
        return;
    }
    if (i >= slab) return;
    float v = part[i];
    for (int s = 1; s < splits; s++) v += part[s * slab + i];
    v *= out_scale;
    if (epi.gamma || ns.unscale) v *= row_factor(ns, epi.gamma != nullptr, (int)(i / N), K, epi.eps);
    if (epi.kind == kEpiAdd) v += load_out_g(epi.residual, ydt, i);
    store_out_g(y, ydt, i, v);
}

// The same sum for N of four or more, four neighbouring elements of a row per thread.  The pass is latency: everything a
// thread needs - its pieces of all the slabs, its residual, its row's factors - is requested before anything is used, and
// the row is the workgroup's (blockIdx.y), not a division per element.  (Before: slab after slab, then four 64-bit
// divisions, each in front of its own loads of the row's factor and the residual.)
// 14336 -> 4096, bf16 rows with a residual, us per call with staging and multiply: 45 rows 36.5 -> 33.9, 128 rows 38.6 -> 36.9,
// 512 rows 76.0 -> 74.1.
// RAGGED: N is no multiple of four.  Rows start at any multiple of four bytes (which 128-bit loads and stores of floats take), and
// the last thread of a row steps back to its last four elements and stores those that are its own.  us per call, against one
// thread per element (with a 64-bit division each): 14336 -> 4090 at 512 rows 77.5 -> 74.9, -> 2050 at 256 rows 43.4 -> 40.7, with a norm
// -> 4094 at 512 rows 81.9 -> 78.1, fp32 10240 -> 3507 at 444 rows 57.4 -> 54.8.
typedef float4_t float4_any __attribute__((aligned(4)));

template <int SPLITS, bool SWIGLU, bool RAGGED>
__global__ __launch_bounds__(256) void splitk_reduce4_kernel(const float* __restrict__ part, int M, int N, void* __restrict__ y, int ydt,
                                                             float out_scale, Epilogue epi, NormStats ns, int K)
{
    const int n_out = SWIGLU ? N >> 1 : N;
    const int first = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4, m = blockIdx.y;
    if (first >= n_out) return;
    const int n = RAGGED ? min(first, n_out - 4) : first;
    const int64_t slab = (int64_t)M * N, at = (int64_t)m * n_out + n;
    // (a pair's 16 gate columns sit in front of its 16 up columns)
    const float* const p0 = part + (int64_t)m * N + (SWIGLU ? (n >> 4) * 32 + (n & 15) : n);
    float4_t g[SPLITS], u[SWIGLU ? SPLITS : 1];
#pragma unroll
    for (int s = 0; s < SPLITS; s++) {
        if constexpr (RAGGED) g[s] = *reinterpret_cast<const float4_any*>(p0 + s * slab);
        else g[s] = *reinterpret_cast<const float4_t*>(p0 + s * slab);
        if (SWIGLU) u[SWIGLU ? s : 0] = *reinterpret_cast<const float4_t*>(p0 + s * slab + 16);
    }
    const uintptr_t mask = ydt == kF32 ? 15u : 7u;
    const bool aligned = !RAGGED && ((reinterpret_cast<uintptr_t>(y) | (epi.kind == kEpiAdd ? reinterpret_cast<uintptr_t>(epi.residual) : 0u)) & mask) == 0;
    float4_t res = {0.f, 0.f, 0.f, 0.f};
    if (epi.kind == kEpiAdd) {
        if (!aligned) {
#pragma unroll
            for (int e = 0; e < 4; e++) res[e] = load_out_g(epi.residual, ydt, at + e);
        } else if (ydt == kF32) {
            res = *reinterpret_cast<const float4_t*>(static_cast<const float*>(epi.residual) + at);
        } else {
            const u32x2_t r = *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(epi.residual) + at);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t h = (e & 1) ? r[e >> 1] >> 16 : r[e >> 1] & 0xffffu;
                res[e] = ydt == kF16 ? f16_bits_to_f32(h) : __builtin_bit_cast(float, h << 16);
            }
        }
    }
    const float f = out_scale * (epi.gamma || ns.unscale ? row_factor(ns, epi.gamma != nullptr, m, K, epi.eps) : 1.0f);
    float4_t v = g[0];
#pragma unroll
    for (int s = 1; s < SPLITS; s++) v += g[s];
    if (SWIGLU) {
        float4_t w = u[0];
#pragma unroll
        for (int s = 1; s < SPLITS; s++) w += u[SWIGLU ? s : 0];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = silu_mul(v[e] * f, w[e] * f);
    } else {
        {
            // (scaled, rounded, then added: with and without the residual the scaled sum has the same bits)
#pragma clang fp contract(off)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                v[e] *= f;
                if (epi.kind == kEpiAdd) v[e] += res[e];
            }
        }
    }
    if (RAGGED && ydt == kF32 && n == first) {
        *reinterpret_cast<float4_any*>(static_cast<float*>(y) + at) = v;
    } else if (!aligned) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (!RAGGED || n + e >= first) store_out_g(y, ydt, at + e, v[e]);
    } else if (ydt == kF32) {
        *reinterpret_cast<float4_t*>(static_cast<float*>(y) + at) = v;
    } else {
        u32x2_t o;
        if (ydt == kF16) {
            const half2_t a = {(_Float16)v[0], (_Float16)v[1]}, b = {(_Float16)v[2], (_Float16)v[3]};
            o = (u32x2_t){as_u32(a), as_u32(b)};
        } else {
            o = (u32x2_t){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
        *reinterpret_cast<u32x2_t*>(static_cast<uint16_t*>(y) + at) = o;
    }
}

template <bool SWIGLU, bool RAGGED>
hipError_t launch_reduce4(const float* part, int splits, int M, int N, void* y, int ydt, float out_scale, const Epilogue& epi, const NormStats& ns,
                          int K, hipStream_t st)
{
    const dim3 grid((unsigned)(((SWIGLU ? N / 2 : N) + 1023) / 1024), (unsigned)M);
    auto go = [&](auto count) {
        hipLaunchKernelGGL((splitk_reduce4_kernel<decltype(count)::value, SWIGLU, RAGGED>), grid, dim3(256), 0, st, part, M, N, y, ydt, out_scale, epi, ns, K);
        return hipGetLastError();
    };
    switch (splits) {
        case 2: return go(std::integral_constant<int, 2>{});
        case 3: return go(std::integral_constant<int, 3>{});
        case 4: return go(std::integral_constant<int, 4>{});
        case 5: return go(std::integral_constant<int, 5>{});
        case 6: return go(std::integral_constant<int, 6>{});
        case 7: return go(std::integral_constant<int, 7>{});
        case 8: return go(std::integral_constant<int, 8>{});
    }
    return hipErrorInvalidValue;               // kMaxSplits
}

// adds the slabs of a K split (2 .. kMaxSplits of them) and applies the epilogue
hipError_t launch_reduce(const float* part, int splits, int M, int N, void* y, int ydt, float out_scale, const Epilogue& epi, const NormStats& ns,
                         int K, hipStream_t st)
{
    const bool rows_fit = M <= 65535;          // the grid's second dimension
    if (rows_fit && epi.kind == kEpiSwiglu) return launch_reduce4<true, false>(part, splits, M, N, y, ydt, out_scale, epi, ns, K, st);
    if (rows_fit && N % 4 == 0) return launch_reduce4<false, false>(part, splits, M, N, y, ydt, out_scale, epi, ns, K, st);
    if (rows_fit && N > 4) return launch_reduce4<false, true>(part, splits, M, N, y, ydt, out_scale, epi, ns, K, st);
    const int64_t total = (int64_t)M * N;
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, part, splits, M, N, y, ydt, out_scale, epi, ns, K);
    return hipGetLastError();
}

template <int BITS, int NF, int MF, int MW, int XD, bool SPLIT = false>
hipError_t launch_roles(const WeightView& w, const void* x, int M, void* y, int ydt, float out_scale, const Epilogue& epi,
                        const NormStats& ns, hipStream_t st, float* part = nullptr, int splits = 1)
{
    constexpr int lds = 2 * NF * (4 * 64) * 16;
    constexpr int BM = MW * MF * 16;
    (void)LdsRequest<&gemm_roles_kernel<BITS, NF, MF, MW, XD, SPLIT>, lds>::registered;
    const int n_tiles = (w.NT + NF - 1) / NF, m_tiles = (M + BM - 1) / BM;
    const unsigned groups = (unsigned)(((int64_t)n_tiles * m_tiles * splits + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_roles_kernel<BITS, NF, MF, MW, XD, SPLIT>), dim3(groups), dim3((MW + 4) * 64), lds, st, w.base,
                       reinterpret_cast<const u32x4_t*>(x), w.KT, w.NT, (M + 15) / 16, M, n_tiles, m_tiles, (int)groups, w.K, splits,
                       (w.KT + splits - 1) / splits, w.N, y, ydt, out_scale, part, epi, ns);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || !SPLIT) return e;
    return launch_reduce(part, splits, M, w.N, y, ydt, out_scale, epi, ns, w.K, st);
}

template <int BITS, int XBF, int NF, bool EXACT, int MF>
hipError_t launch_m(const WeightView& w, const void* x, int M, void* y, int ydt, float out_scale, float* part, int splits, const Epilogue& epi,
                    const NormStats& ns, hipStream_t st)
{
    constexpr int BM = 8 * MF * 16;
    constexpr int lds = 2 * NF * (4 * (EXACT ? 2 : 1) * 64) * 16;     // operand buffers, 56 .. 128 KB
    auto kern = gemm_kernel<BITS, XBF, NF, EXACT, MF>;
    (void)LdsRequest<&gemm_kernel<BITS, XBF, NF, EXACT, MF>, lds>::registered;
    const int n_tiles = (w.NT + NF - 1) / NF, m_tiles = (M + BM - 1) / BM;
    const int kt_per_split = (w.KT + splits - 1) / splits;
    const unsigned groups = (unsigned)(((int64_t)n_tiles * m_tiles * splits + 7) / 8 * 8);
    hipLaunchKernelGGL(kern, dim3(groups), dim3(512), lds, st, w.base, reinterpret_cast<const u32x4_t*>(x), w.KT, w.NT,
                       (M + 15) / 16, M, n_tiles, m_tiles, splits, kt_per_split, (int)groups, w.K, w.N, y, ydt, out_scale, part, epi, ns);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || splits == 1) return e;
    return launch_reduce(part, splits, M, w.N, y, ydt, out_scale, epi, ns, w.K, st);
}

// What multiplies a staged chunk of M rows.
//   kRoles   gemm_roles_kernel, mw multiplying waves (32 rows each), nf column blocks, with eight of them K split over `splits` workgroups
//   kTiles   gemm_kernel, mf row blocks per wave (256 or 512 rows), nf column blocks, K split over `splits` workgroups
//   kCols    gemm_cols_kernel (gemm_cols.hip)
struct TilePlan {
    enum { kRoles, kTiles, kCols } kind;
    int nf, mw, mf, splits;
    ColsPlan cols;
};

// The tiled kernels' way with a call, and an estimate of its time behind the staging pass in us (< 0: whatever the others take).
// The estimates are fits to 1900 calls of 33 .. 600 rows on N of 512 .. 32768, K of 512 .. 14336 (Q4 and Q8, bf16; 4 - 8 % rms): a
// round of workgroups costs a fixed part and so much per K tile, whatever the number of workgroups in it.
// For the K ranges of the role-split kernel it is gemm_kernel's line, 7 % too long (52 calls: 0.81 - 0.99 of gemm_kernel's time, about 1.12 per K tile instead of
// 1.29).  It stays for what it decides, against gemm_cols.hip, whose line is off by as much: of 36 calls drawn from those that 1.12 would move from there,
// 18 take 4.7 % less in the mean (Q8 8480 -> 7056 at 182 bf16 rows 47.9 / 42.2) and 18 up to 19 % more (f16 rows, which have no staging launch there: Q8 12032 -> 1007
// at 1298 rows 46.1 / 54.9, Q4 7744 -> 1663 at 1502 49.4 / 56.6).
static float tiled_plan(const WeightView& w, int M, bool exact, int num_cus, size_t part_bytes, const Epilogue& epi, TilePlan& plan)
{
    const int64_t cus = num_cus;
    const float out_mb = 4e-6f * (float)M * (float)w.N, kt = (float)w.KT;
    auto roles = [&](int nf, int mw) { plan = {TilePlan::kRoles, nf, mw, 2, 1, {}}; };
    if (!exact && epi.kind != kEpiSwiglu) {
        const int64_t tiles64 = (w.NT + 3) / 4;                  // 64-column tiles
        // up to 128 rows on a wide output: one round of 128 x 64 tiles (at least half of one where K is short) needs no K
        // split and no second pass over partial sums; 64 rows where those cover the batch (every workgroup streams all the
        // rows of X from the L2).  More than a round of them, or a long K, is gemm_cols.hip's: 4096 -> 28672 at 64 / 96 / 128 rows
        // 32.7 / 42.5 / 46.6 -> 28.9 / 33.5 / 39.9 us, 14336 -> 14336 at 40 / 64 / 96 rows 58.5 / 56.4 / 64.7 -> 44.1 / 48.2 / 56.2
        if (M <= 128 && tiles64 <= cus && w.KT <= 64 && (tiles64 * 4 >= 3 * cus || (tiles64 * 2 >= cus && w.KT <= 48))) {
            roles(4, M <= 64 ? 2 : 4);
            return -1.f;
        }
        // A narrow output with a short K (the attention projections at a prefill chunk): 256 x 112 tiles
        // would leave most CUs idle and get a K split with its second pass over the partial sums.
        // One round of 128-row tiles of the role-split kernel, as wide as still gives every CU a tile,
        // does without (X then crosses from the L2 once per column tile: K stays short for this).
        if (w.KT <= 48 && M > 128 && (int64_t)((w.NT + 6) / 7) * ((M + 255) / 256) < cus) {
            // (128-row tiles first, 64-row ones for batches they cannot spread over the chip; the
            // width that fills most of one round, at least three quarters of it)
            int best_nf = 0, best_mw = 0;
            int64_t best_groups = 0;
            for (int mw : {4, 2})
                for (int nf : {8, 6, 4}) {
                    const int64_t g = (int64_t)((M + mw * 32 - 1) / (mw * 32)) * ((w.NT + nf - 1) / nf);
                    if (g <= cus && g * 4 >= 3 * cus && (best_mw == 0 || (mw == best_mw && g > best_groups))) {
                        best_nf = nf;
                        best_mw = mw;
                        best_groups = g;
                    }
                }
            if (best_mw) {
                roles(best_nf, best_mw);
                const float fixed = best_nf == 4 ? 1.4f : best_nf == 6 ? 2.0f : 2.4f;
                const float per_kt = best_mw == 4 ? (best_nf == 4 ? 0.48f : best_nf == 6 ? 0.73f : 0.84f) : (best_nf == 4 ? 0.45f : best_nf == 6 ? 0.62f : 0.75f);
                return fixed + per_kt * kt + 0.27f * out_mb;
            }
        }
    }
    // 7 column blocks (BN = 112) tile N = 14336 = 128 * 112 exactly: with M = 512
    // that is 256 workgroups, one per CU; 8 column blocks otherwise
    const int nf = w.NT % 7 == 0 && epi.kind != kEpiSwiglu ? 7 : 8;      // gate / up pairs need an even number of column blocks
    // 512-row workgroups (four row blocks per wave: half the LDS operand reads per MFMA) once they
    // fill the chip by themselves (eight column blocks x four row blocks spill)
    if (!exact && nf == 7) {
        const int64_t tiles512 = (int64_t)((w.NT + 6) / 7) * ((M + 511) / 512);
        const int rem = M % 512;                       // (a last tile at most half full: 256-row tiles waste less)
        if (tiles512 >= cus && (rem == 0 || rem > 256)) {
            plan = {TilePlan::kTiles, 7, 8, 4, 1, {}};
            return -1.f;
        }
    }
    const int64_t tiles = (int64_t)((w.NT + nf - 1) / nf) * ((M + 255) / 256);
    // enough 256-row tiles to fill the chip without a K split: the role-split kernel
    if (!exact && tiles >= cus) {
        roles(nf, 8);
        return (float)((tiles + cus - 1) / cus) * (0.4f + 1.43f * kt) + 0.27f * out_mb;
    }
    // Too few tiles to fill the chip: split K over workgroups.  Every split adds its
    // K range in fp32 into its own slab of `part`; a second kernel adds the slabs in
    // a fixed order (no atomics: results are reproducible).
    int splits = (int)std::min<int64_t>(kMaxSplits, cus / tiles);
    splits = std::min(splits, w.KT / 4);                         // at least 4 K tiles per split
    while (splits > 1 && (size_t)splits * M * w.N * 4 > part_bytes) splits--;
    if (splits < 1) splits = 1;
    const int per = (w.KT + splits - 1) / splits;
    splits = (w.KT + per - 1) / per;                             // no empty split
    plan = {TilePlan::kTiles, nf, 8, 2, splits, {}};
    // Their K ranges go to the role-split kernel where they are long and there are three of them or up to three row tiles; the bits are the same (a tuning
    // value keeps them in gemm_kernel, and a test compares).  us per
    // call, gemm_kernel / role-split: 14336 -> 4096 at 512 rows 68.5 / 66.3, Q8 70.6 / 68.8, 10240 -> 3136 at 512 rows 46.3 / 44.9, 12288 -> 8192 at 256 rows
    // 59.4 / 57.9, Q8 11168 -> 2145 at 1020 rows 69.3 / 65.2.  Two ranges of more row tiles: 14336 -> 4096 at 1000 rows 121.3 / 123.0, 5760 -> 1959 at 1551 rows
    // 54.2 / 54.9; short ranges: Q8 14336 -> 1024 at 700 rows (14 K tiles) 39.4 / 40.0.
    if (!exact && splits > 1 && per >= 16 && (splits >= 3 || M <= 768) && g_role_ranges) plan.kind = TilePlan::kRoles;
    const float rounds = (float)((tiles * splits + cus - 1) / cus);
    // (EXACT: fits to 254 calls of 33 .. 2048 rows on N of 256 .. 32768, 10 - 12 % rms, taken when gemm_cols.hip went over to integer operands; with
    // the lines from before, 0.9 + 2.75 per K tile, wide outputs of a short K and the odd large call stayed here that are quicker there.  us per
    // call here / there: f16 640 -> 14364 at 327 rows 27.7 / 21.1, 1120 -> 7768 at 1015 rows 46.6 / 37.2, bf16 Q8 1248 -> 30164 at 174 rows 43.7 /
    // 32.6, Q4 4544 -> 13471 at 452 rows 124 / 104)
    const float round = exact ? (nf == 7 ? 2.4f + 2.77f * (float)per : 2.7f + 3.03f * (float)per) : 1.4f + 1.29f * (float)per;
    return rounds * round +
           (splits > 1 ? 2.2f + 0.5f * ((float)splits + 0.5f) * out_mb : 0.27f * out_mb);
}

// The quicker of the tiled kernels and the one whose waves stand side by side (gemm_cols.hip), by their estimates
static TilePlan plan_tiles(const WeightView& w, int M, bool exact, bool bf16, int num_cus, size_t part_bytes, const Epilogue& epi)
{
    TilePlan plan = {};
    if (!exact && g_rows_kernel < 2) {
        const ColsPlan cols = plan_gemm_cols_long_k(w, M, num_cus, epi);
        if (cols.rb) return {TilePlan::kCols, 0, 0, 0, cols.splits, cols};
    }
    const float tiled = tiled_plan(w, M, exact, num_cus, part_bytes, epi, plan);
    if (tiled < 0.f || g_rows_kernel == 3 || (g_rows_kernel == 2 && !exact)) return plan;
    const ColsPlan cols = plan_gemm_cols(w, !exact ? 0 : bf16 ? 2 : 1, M, num_cus, part_bytes);
    if (cols.us < 0.97f * tiled) plan = {TilePlan::kCols, 0, 0, 0, cols.splits, cols};
    return plan;
}

template <int BITS, int XBF>
hipError_t launch_tiles(const TilePlan& p, const WeightView& w, const void* x, bool raw, int M, void* y, int ydt, bool exact, float out_scale, float* part,
                        const Epilogue& epi, const NormStats& ns, hipStream_t st)
{
    if (p.kind == TilePlan::kCols) {
        const hipError_t e = launch_gemm_cols(w, x, raw, !exact ? 0 : XBF ? 2 : 1, M, y, ydt, p.cols, epi, ns.part, ns.nblk, ns.unscale, part, st);
        if (e != hipSuccess || p.splits == 1) return e;
        return launch_reduce(part, p.splits, M, w.N, y, ydt, out_scale, epi, ns, w.K, st);
    }
    if (exact) {
        if (p.nf == 7) return launch_m<BITS, XBF, 7, true, 2>(w, x, M, y, ydt, out_scale, part, p.splits, epi, ns, st);
        return launch_m<BITS, XBF, 8, true, 2>(w, x, M, y, ydt, out_scale, part, p.splits, epi, ns, st);
    }
    if constexpr (XBF == 0) {       // FAST multiplies in f16: bf16 activations were widened by the staging pass
        if (p.kind == TilePlan::kRoles) {
            if (p.splits > 1) {
                if (p.nf == 7) return launch_roles<BITS, 7, 2, 8, 2, true>(w, x, M, y, ydt, out_scale, epi, ns, st, part, p.splits);
                return launch_roles<BITS, 8, 2, 8, 2, true>(w, x, M, y, ydt, out_scale, epi, ns, st, part, p.splits);
            }
            if (p.mw == 8 && p.nf == 7) return launch_roles<BITS, 7, 2, 8, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            if (p.mw == 8) return launch_roles<BITS, 8, 2, 8, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            if (p.mw == 4 && p.nf == 8) return launch_roles<BITS, 8, 2, 4, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            if (p.mw == 4 && p.nf == 6) return launch_roles<BITS, 6, 2, 4, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            if (p.mw == 4) return launch_roles<BITS, 4, 2, 4, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            if (p.nf == 8) return launch_roles<BITS, 8, 2, 2, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            if (p.nf == 6) return launch_roles<BITS, 6, 2, 2, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
            return launch_roles<BITS, 4, 2, 2, 2>(w, x, M, y, ydt, out_scale, epi, ns, st);
        }
        if (p.mf == 4) return launch_m<BITS, 0, 7, false, 4>(w, x, M, y, ydt, out_scale, part, 1, epi, ns, st);
        if (p.nf == 7) return launch_m<BITS, 0, 7, false, 2>(w, x, M, y, ydt, out_scale, part, p.splits, epi, ns, st);
        return launch_m<BITS, 0, 8, false, 2>(w, x, M, y, ydt, out_scale, part, p.splits, epi, ns, st);
    }
    return hipErrorInvalidValue;
}

// The multiply that follows a staging launch starts on weights that come from HBM for the first time (2.4 of the
// 14.5 us of a 64-row call on 4096 -> 14336 pass before its K loops start).  Extra workgroups of the staging launch,
// which leaves most of the chip idle, ask for the first K tiles of every column group ahead of it - one dword per
// 128-byte line, nothing kept: workgroup number b here asks for what workgroup b of the multiply reads first (the
// hardware deals workgroups to the eight XCDs in turn, so with first_group a multiple of eight the lines land in
// that workgroup's L2; anywhere else they land in the memory-side cache).
struct Touch {
    const uint8_t* base;          // the weight tensor (first_group past the grid: nothing to do)
    int first_group, NT, KT, NF, tile_bytes, ahead;
    int per_xcd, tiles;           // the tiled kernels' order: workgroup b works on column tile (b % 8) * per_xcd + b / 8 of `tiles` (0: on b)
};

__device__ __forceinline__ void touch_weights(const Touch& tc, int b, int tid, int nthreads)
{
    const int lines = (tc.tile_bytes + 127) >> 7;
    if (tc.per_xcd) {
        b = (b & 7) * tc.per_xcd + (b >> 3);
        if (b >= tc.tiles) return;
    }
    const int kt0 = b % tc.KT;                     // (the multiply's workgroups start their K walk there)
    uint32_t acc = 0;
    for (int idx = tid; idx < tc.NF * tc.ahead * lines; idx += nthreads) {
        const int line = idx % lines, ft = idx / lines, t = ft % tc.ahead, f = ft / tc.ahead;
        const int nt = min(b * tc.NF + f, tc.NT - 1);
        int kt = kt0 + t;
        if (kt >= tc.KT) kt -= tc.KT;
        acc ^= *reinterpret_cast<const uint32_t*>(tc.base + ((int64_t)nt * tc.KT + kt) * tc.tile_bytes + min(line * 128, tc.tile_bytes - 4));
    }
    asm volatile("" ::"v"(acc));                   // (the loads have to be issued and waited for; nothing is stored)
}

// op over the 64 lanes, in the order of a butterfly over lane distances 32, 16, 8, 4, 2, 1, without a trip through LDS per step: halves and
// rows of 16 lanes are swapped in the registers, and from distance 8 on a rotation by n within a row meets the lane at distance n, or
// one that holds the same value by then.  A wave has nothing else to do meanwhile: six trips through LDS were 0.25 us of the pass.  us per call, before /
// after: 4096 -> 1024 at 512 rows with a norm 20.6 / 20.3, lists of six layers at 45 / 64 / 100 / 128 rows 456 / 453, 500 / 496, 616 / 613, 638 / 634.
template <class Op>
__device__ __forceinline__ float butterfly(float v, Op op)
{
    const auto bits = [](float f) { return __builtin_bit_cast(uint32_t, f); };
    const auto value = [](uint32_t b) { return __builtin_bit_cast(float, b); };
    const auto halves = __builtin_amdgcn_permlane32_swap(bits(v), bits(v), false, false);
    v = op(value(halves[0]), value(halves[1]));
    const auto rows = __builtin_amdgcn_permlane16_swap(bits(v), bits(v), false, false);
    v = op(value(rows[0]), value(rows[1]));
    v = op(v, value(__builtin_amdgcn_update_dpp(0, bits(v), 0x128, 0xf, 0xf, true)));       // row_ror:8
    v = op(v, value(__builtin_amdgcn_update_dpp(0, bits(v), 0x124, 0xf, 0xf, true)));
    v = op(v, value(__builtin_amdgcn_update_dpp(0, bits(v), 0x122, 0xf, 0xf, true)));
    return op(v, value(__builtin_amdgcn_update_dpp(0, bits(v), 0x121, 0xf, 0xf, true)));
}

// X [M, K] row major (16-bit elements, used as they are) -> A-operand order: for row block rb
// (16 rows, zero padded) and scale group g, 64 x 16 B where slot (oct, r) = oct*16 + r holds row
// 16*rb + r, k = 32*g + 8*oct .. +8.  A workgroup moves one row block x 16 groups through LDS:
// waves read 1 KB runs of a row and write whole 1 KB units.
constexpr int kStageGroups = 16;                       // scale groups per workgroup
constexpr int kStagePitch = kStageGroups * 4 + 1;      // 16 B slots per LDS row (odd: no bank conflicts)

// NORM: RMSNorm folded in.  x * gamma is formed in fp32 and rounded once to the operand type (XBF:
// bf16, else f16); the squares of the unscaled row are summed per (row, workgroup) in a fixed
// butterfly order into ssq_part[row * gridDim.y + blockIdx.y].
template <bool XBF, bool NORM>
__global__ __launch_bounds__(256) void stage_x_kernel(const u32x4_t* __restrict__ src, u32x4_t* __restrict__ dst, int M, int K8,
                                                      Epilogue epi, float* __restrict__ ssq_part)
{
    __shared__ u32x4_t tile[16 * kStagePitch];
    const int rb = blockIdx.x;
    const int c0 = blockIdx.y * (kStageGroups * 4);     // first 16 B chunk of the row handled here
    const int t = threadIdx.x;
    Gamma8 graw = {};
    if (NORM) graw = load_gamma8(epi.gamma, epi.gamma_dt, min(c0 + (t & 63), K8 - 1) * 8);
#pragma unroll
    for (int it = 0; it < 4; it++) {
        const int r = it * 4 + (t >> 6), c = c0 + (t & 63);
        const int row = rb * 16 + r;
        Frag16 a;
        a.u = (u32x4_t){0u, 0u, 0u, 0u};
        if (row < M && c < K8) a.u = src[(int64_t)row * K8 + c];
        if (NORM) {
            float sq = 0.f;
            if (c < K8) {
                float g[8];
                gamma8_values(graw, epi.gamma_dt, g);
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    float v0, v1;
                    if (XBF) {
                        v0 = __builtin_bit_cast(float, a.u[p] << 16);
                        v1 = __builtin_bit_cast(float, a.u[p] & 0xffff0000u);
                    } else {
                        const half2_t h = as_h2(a.u[p]);
                        v0 = (float)h.x;
                        v1 = (float)h.y;
                    }
                    sq = fmaf(v1, v1, fmaf(v0, v0, sq));
                    v0 *= g[2 * p];
                    v1 *= g[2 * p + 1];
                    if (XBF) {
                        a.u[p] = pack_bf16x2(v0, v1);
                    } else {
                        const half2_t h = {(_Float16)v0, (_Float16)v1};
                        a.u[p] = as_u32(h);
                    }
                }
            }
            sq = butterfly(sq, [](float u, float v) { return u + v; });
            if ((t & 63) == 0) ssq_part[(int64_t)row * gridDim.y + blockIdx.y] = sq;      // (rows past M: zeros, never read)
        }
        tile[r * kStagePitch + (t & 63)] = a.u;
    }
    __syncthreads();
    const int G = K8 >> 2;
#pragma unroll
    for (int it = 0; it < 4; it++) {
        const int gl = it * 4 + (t >> 6), slot = t & 63;        // group within the workgroup, (oct, r)
        const int g = blockIdx.y * kStageGroups + gl;
        if (g < G) dst[((int64_t)rb * G + g) * 64 + slot] = tile[(slot & 15) * kStagePitch + gl * 4 + (slot >> 4)];
    }
}

// The same restaging for FAST mode when the activations are not f16 (bf16 or fp32 in, f16 operands
// out), with a power-of-two scale PER ROW: a workgroup owns four rows.  First a row is read for the
// largest magnitude (of x, or of x * gamma with a folded norm, whose sum of squares is also taken),
// which picks the power of two s that brings it just under 2^14 and leaves 1 / s in `unscale` for
// the multiply's epilogue; then the four rows go through LDS in pieces of 512 k, every value
// multiplied by its row's s on the way to f16, and leave as 64-byte runs (four neighbouring rows of
// one k octet in operand order).
// Whatever the magnitude of a row, its largest element lands in [2^13, 2^14) and elements down to
// 2^-27 of it stay normal f16 numbers.  Rows of up to PW * CH * 512 elements stay in registers
// between the two steps (CH chunks of 8 values per lane in each of a row's PW waves, all requested
// at once); longer rows are read again (the second read hits the L2).
template <int XT>
struct RowChunk {                 // 8 consecutive activations of a row as loaded
    u32x4_t v[XT == 2 ? 2 : 1];
};

template <int XT>
__device__ __forceinline__ RowChunk<XT> load_row_chunk(const void* src, int64_t row, int K, int c)
{
    RowChunk<XT> o;
    if (XT == 2) {
        const u32x4_t* p = reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(src) + row * K + c * 8);
        o.v[0] = p[0];
        o.v[XT == 2 ? 1 : 0] = p[1];
    } else {
        o.v[0] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint16_t*>(src) + row * K + c * 8);
    }
    return o;
}

template <int XT>
__device__ __forceinline__ void row_chunk_values(const RowChunk<XT>& c, float v[8])
{
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (XT == 2) {
            v[e] = __builtin_bit_cast(float, (uint32_t)c.v[0][e]);
            v[4 + e] = __builtin_bit_cast(float, (uint32_t)c.v[XT == 2 ? 1 : 0][e]);
        } else {
            v[2 * e] = __builtin_bit_cast(float, c.v[0][e] << 16);
            v[2 * e + 1] = __builtin_bit_cast(float, c.v[0][e] & 0xffff0000u);
        }
    }
}

// A workgroup of sixteen waves owns ROWS rows (8, 4, 2 or 1) and gives every row PW = 16 / ROWS waves: wave (r, p) takes the
// pieces of 512 k numbered p, p + PW, ... of row r (CH of them at most stay in registers between the two steps), the parts
// of a row meet once through LDS for the row's largest magnitude (and sum of squares).  One wave per row took 5 - 7 us for
// 512 rows of 4096 and 10 - 12 us for rows of 14336, most of it the latency of one wave walking its row.
template <int XT, bool NORM, int CH, int ROWS, bool GKEEP = (CH * XT <= 4)>
__global__ __launch_bounds__(1024) void stage_rows_kernel(const void* __restrict__ src, u32x4_t* __restrict__ dst, int M, int K, int first_group,
                                                          int gamma_dt, const void* __restrict__ gamma, float* __restrict__ unscale,
                                                          float* __restrict__ ssq, Touch touch)
{
    static_assert(XT == 1 || XT == 2, "bf16 or fp32 activations");
    if ((int)blockIdx.x >= first_group) {
        touch_weights(touch, (int)blockIdx.x - first_group, (int)threadIdx.x, 1024);
        return;
    }
    if ((int)blockIdx.x * ROWS >= M) return;                   // (rows past M; padding up to first_group)
    constexpr int PW = 16 / ROWS;                              // waves per row
    __shared__ u32x4_t tile[PW][2][ROWS * kStagePitch];
    __shared__ float amax_part[ROWS][PW];
    __shared__ float sq_part[ROWS][PW];
    const int rb = (int)blockIdx.x * ROWS >> 4, r0 = (int)blockIdx.x * ROWS & 15;      // row block, first of this workgroup's rows in it
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int r = wv % ROWS, part = wv / ROWS;                           // my row of the workgroup's, my part of the row
    const int64_t row = min(rb * 16 + r0 + r, M - 1);      // (rows past M repeat the last one and are never read back)
    const int K8 = K >> 3, G = K8 >> 2;
    const int pieces = (K8 + 63) >> 6;                     // pieces of 64 chunks (512 k) in a row
    const bool resident = pieces <= PW * CH;

    // ---- the row's largest magnitude (and sum of squares)
    // What the pass waits for is latency: rows and gamma are asked for together and without branches, two pieces share a barrier on their way out.  us per
    // call with its multiply, without the three / with them, bf16: 14336 -> 1024 at 512 rows 35.0 / 33.9, 14336 -> 4096 at 45 rows 22.6 / 22.2, Q8 at 2048 rows
    // 214.2 / 209.6, 4096 -> 1024 with a norm at 512 rows 20.2 / 20.0, 8192 -> 1024 with a norm at 300 rows 26.2 / 25.5, 4096 -> 28672 norm + SwiGLU at 45 rows 27.7 /
    // 26.9.  One of them taken out of the three: gamma kept 25.9 / 25.5, 27.7 / 26.8 in the last two (19.7 / 19.9 at 512 rows of 4096); the shared barrier 34.6 /
    // 34.4, 22.6 / 22.4, 209.5 / 208.8 in the first three; what is left there is the loads'.  (The first touching workgroup's number comes in a register too, ahead
    // of what only that one reads: 4096 -> 14336 at 64 rows 16.9 / 16.4, 4096 -> 28672 SwiGLU at 64 rows 28.4 / 27.2.)
    // Pieces past the end of the row are its last chunk again (no branches around the loads); gamma stays with a piece where there are registers
    // for it (GKEEP) - elsewhere it is loaded again for the conversion - and is asked for next to it.
    RowChunk<XT> keep[CH];
    Gamma8 gk[NORM && GKEEP ? CH : 1];
    auto chunk_at = [&](int p0, int i) { return (p0 + i * PW + part) * 64 + lane; };
    auto load = [&](int p0) {
#pragma unroll
        for (int i = 0; i < CH; i++) keep[i] = load_row_chunk<XT>(src, row, K, min(chunk_at(p0, i), K8 - 1));
        if constexpr (NORM && GKEEP) {
#pragma unroll
            for (int i = 0; i < CH; i++) gk[i] = load_gamma8(gamma, gamma_dt, min(chunk_at(p0, i), K8 - 1) * 8);
        }
    };
    auto scaled = [&](int i, int c, float v[8]) {
        float g[8];
        gamma8_values(GKEEP ? gk[GKEEP ? i : 0] : load_gamma8(gamma, gamma_dt, min(c, K8 - 1) * 8), gamma_dt, g);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] *= g[e];
    };
    // (a folded norm's sum of squares is formed in an order that goes with PW = 4: the launcher keeps to it)
    static_assert(!NORM || ROWS == 4, "one order for the sums of squares");
    float amax = 0.f, sq = 0.f;
    for (int p0 = 0; p0 < pieces; p0 += PW * CH) {
        load(p0);
#pragma unroll
        for (int i = 0; i < CH; i++) {
            const int c = chunk_at(p0, i);
            if (p0 + i * PW + part >= pieces) break;
            float v[8];
            row_chunk_values<XT>(keep[i], v);
            if (NORM) {
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const float x = c < K8 ? v[e] : 0.f;
                    sq = fmaf(x, x, sq);
                }
                scaled(i, c, v);
            }
#pragma unroll
            for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
        }
    }
    amax = butterfly(amax, [](float u, float v) { return fmaxf(u, v); });
    if (NORM) sq = butterfly(sq, [](float u, float v) { return u + v; });
    if (lane == 0) {
        amax_part[r][part] = amax;
        if (NORM) sq_part[r][part] = sq;
    }
    __syncthreads();
    amax = amax_part[r][0];
#pragma unroll
    for (int p = 1; p < PW; p++) amax = fmaxf(amax, amax_part[r][p]);
    if constexpr (NORM) sq = ((sq_part[r][0] + sq_part[r][1]) + sq_part[r][2]) + sq_part[r][3];
    // amax = f * 2^e with f in [0.5, 1): s = 2^(14 - e) puts it in [2^13, 2^14); zero, Inf and NaN rows keep s = 1
    float s = 1.0f;
    if (amax > 0.f && amax < __builtin_inff()) {
        int e;
        (void)frexpf(amax, &e);
        s = ldexpf(1.0f, min(14 - e, 126));        // (rows below 2^-112: 2^126 keeps s and 1 / s normal numbers)
    }
    if (lane == 0 && part == 0 && rb * 16 + r0 + r < M) {
        unscale[row] = 1.0f / s;
        if (NORM) ssq[row] = sq;
    }

    // ---- scale, round to f16, through LDS into operand order, two pieces at a time (one to each of a part's tiles)
    const int tp = r * 64 + lane;                           // my place among the threads of my part
    const int gl = tp / (4 * ROWS), oct = tp / ROWS & 3, rr = tp % ROWS;  // when writing out: group within the piece, k octet, row
    for (int p0 = 0; p0 < pieces; p0 += PW * CH) {
        if (!resident) load(p0);
#pragma unroll
        for (int i0 = 0; i0 < CH; i0 += 2) {
            if (p0 + i0 * PW < pieces) {                     // (uniform over the workgroup: some part has this piece)
                if (p0 + i0 > 0) __syncthreads();            // (the tiles have been read)
#pragma unroll
                for (int i = i0; i < i0 + 2 && i < CH; i++) {
                    if (p0 + i * PW + part >= pieces) break;
                    float v[8];
                    row_chunk_values<XT>(keep[i], v);
                    if (NORM) scaled(i, chunk_at(p0, i), v);
                    Frag16 a;
#pragma unroll
                    for (int p = 0; p < 4; p++) {
                        const half2_t h = {(_Float16)(v[2 * p] * s), (_Float16)(v[2 * p + 1] * s)};
                        a.u[p] = as_u32(h);
                    }
                    tile[part][i - i0][r * kStagePitch + lane] = a.u;
                }
                __syncthreads();
#pragma unroll
                for (int i = i0; i < i0 + 2 && i < CH; i++) {
                    const int g = (p0 + i * PW + part) * 16 + gl;
                    if (g < G) dst[((int64_t)rb * G + g) * 64 + oct * 16 + r0 + rr] = tile[part][i - i0][rr * kStagePitch + gl * 4 + oct];
                }
            }
        }
    }
}

}  // namespace

static bool g_raw = true;     // (4 = gemm_cols.hip reads staged rows only)
static int g_touch = 2;       // (5 = the staging launch asks for no weights ahead of the multiply, 6 = only ahead of the few-rows kernel)
void set_gemm_tuning(int rows_kernel)
{
    g_rows_kernel = rows_kernel == 7 ? 2 : rows_kernel >= 4 ? 0 : rows_kernel;
    g_role_ranges = rows_kernel != 7;
    g_raw = rows_kernel != 4;
    g_touch = rows_kernel == 5 ? 0 : rows_kernel == 6 ? 1 : 2;
}

static RowsPlan rows_plan(const WeightView& w, int M, int num_cus, const Epilogue& epi)
{
    if (g_rows_kernel == 2 || g_rows_kernel == 3) return {0};
    return gemm_rows_plan(w, M, num_cus, epi, g_rows_kernel == 1);
}

bool gemm_rows_takes(const WeightView& w, int M, int num_cus, const Epilogue& epi)
{
    return rows_plan(w, M, num_cus, epi).nf != 0;
}

// whether tiled_plan gives a FAST-mode call of M rows the 64-column tiles
static bool few_rows_tiles64(const WeightView& w, int M, int num_cus, const Epilogue& epi)
{
    TilePlan plan = {};
    if (M > 128 || epi.kind == kEpiSwiglu) return false;
    return tiled_plan(w, M, false, num_cus, 0, epi, plan) < 0.f && plan.kind == TilePlan::kRoles && plan.nf == 4;
}

// the extra workgroups of a staging launch (grid_x grows by them) for a call of 33 rows or more that goes through the
// row-scaling pass (bf16 / fp32 rows) and on to the few-row kernel or to the tiled kernels' 64-column tiles: up to
// 16 MB of the tensor, from the K tile every column group starts at.  Per call: 4096 -> 14336 at 64 rows 19.6 -> 18.7
// us with 16 of the 32 K tiles (no gain with all of them: the launch then takes as long as the reads), 4096 -> 4096
// at 64 / 128 rows 13.6 / 14.6 -> 12.4 / 13.4, 4096 -> 1024 13.1 -> 11.7, 8192 -> 4096 at 128 rows 25.1 -> 22.9.  Not
// for f16 rows (their pass only reorders and is over before the reads are: 4096 -> 14336 at 64 rows 18.6 -> 19.1),
// for 17 .. 32 fp32 rows (12.5 -> 13.4 on 4096 -> 8192) or for K up to 2048.
static Touch plan_touch(const WeightView& w, int mc, int num_cus, const Epilogue& ec, bool exact, unsigned& grid_x)
{
    Touch tc = {nullptr, 0x7fffffff, w.NT, w.KT, 1, tile_bytes(w.bits), 0, 0, 0};
    if (g_touch == 0 || exact || mc < 33 || w.KT < 32) return tc;
    const int64_t per_k_tile = (int64_t)w.NT * tile_bytes(w.bits);
    int nf = 0, groups = 0;
    const RowsPlan plan = rows_plan(w, mc, num_cus, ec);
    if (plan.nf) {
        nf = plan.nf;
        groups = (w.NT + nf - 1) / nf;
    } else if (g_touch >= 2 && per_k_tile * w.KT <= ((int64_t)40 << 20) && few_rows_tiles64(w, mc, num_cus, ec)) {
        // the 128 x 64 / 64 x 64 tiles of the tiled kernels (65 .. 128 rows on wide outputs; 4096 -> 14336 at 128 rows:
        // 27.5 us, 24.3 with the same tensor every call): 4096 -> 14336 at 65 / 100 / 128 rows 25.3 / 27.1 / 28.1 ->
        // 23.9 / 26.0 / 27.3 us, 4096 -> 11008 23.9 / 25.5 / 26.5 -> 23.3 / 24.6 / 25.2; nothing on tensors of 66 MB
        nf = 4;
        tc.tiles = (w.NT + 3) / 4;
        groups = (tc.tiles + 7) / 8 * 8;
        tc.per_xcd = groups / 8;
    } else {
        return tc;
    }
    tc.base = w.base;
    tc.NF = nf;
    tc.ahead = (int)std::min<int64_t>(w.KT, std::max<int64_t>(4, ((int64_t)16 << 20) / per_k_tile));
    tc.first_group = (int)((grid_x + 7) / 8 * 8);
    grid_x = (unsigned)(tc.first_group + groups);
    return tc;
}

// The last MiB of the scratch's first half: per-row statistics - partial sums of squares of a folded
// RMSNorm (rows of a chunk x K / 512 floats: less than half / 256 bytes) and, in its last
// quarter, the per-row power of two of widened activations (at most 65536 rows per chunk).
constexpr size_t kStatsBytes = (size_t)1 << 20;

// rows of K 16-bit elements the first half holds in front of them, in whole row tiles
static int64_t staged_rows(const WeightView& w, size_t workspace_bytes)
{
    const size_t half = workspace_bytes / 2;
    if (half <= kStatsBytes) return 0;
    return std::min<int64_t>(65536, (int64_t)((half - kStatsBytes) / ((size_t)w.K * 2)) / 256 * 256);
}

bool gemm_stages(const WeightView& w, size_t workspace_bytes) { return staged_rows(w, workspace_bytes) >= 256; }

// Rows per workgroup of sixteen waves: with few of them one workgroup per four rows leaves the chip idle and a
// row's waves walk it piece after piece; with many, the shorter runs in which the operands leave cost more (64, 32, 16
// bytes).  us per call, 4 / 2 / 1 rows, bf16 unless noted.  K over 8192: 14336 -> 4096 at 45 rows 28.0 / 26.5 / 25.8, 128 rows
// 39.6 / 37.1 / 35.8, 160 rows 49.3 / 47.9 / 47.4, 256 rows 47.3 / 45.9 / 47.5, 300 rows 66.5 / 64.7 / 67.3, 384 rows 68.3 / 67.8 /
// 70.9, 448 rows 69.5 / 69.6 / 73.9, 512 rows 72.6 / 73.4 / 78.6; 9216 -> 4096 at 300 / 384 rows 48.9 / 47.5 / 48.8, 49.9 / 49.4 / 51.2;
// 10240 -> 4096 at 384 rows 53.4 / 52.9 / 54.9; 14336 -> 1024 at 384 / 512 rows 39.6 / 40.4 / 42.0, 38.0 / 39.5 / 44.6; fp32 (twice the bytes to a row), 4 / 2 rows, 14336 -> 4096 at
// 512 / 640 rows 76.0 / 74.4, 106.9 / 107.4, 10240 -> 14336 and 9216 -> 4096 at 512 rows 134.0 / 132.8, 54.6 / 54.3.  Shorter K:
// 8192 -> 4096 at 45 rows 18.7 / 17.2 / 17.1, at 64 rows 21.4 / 20.0 / 19.8, at 100 rows 21.8 / 21.6 / 21.6; 4096 -> 4096 at 45 rows
// 11.2 / 10.9 / 11.3, fp32 at 24 rows 10.5 / 10.1 / 10.4; 4096 -> 14336 at 45 / 64 rows 17.2 / 17.2 / 17.6, 18.8 / 19.0 / 19.4.
// (A folded norm: always four, one order of its sums.)
// Eight where that makes one workgroup per CU of a second round of four-row ones: all rows go at once then, and out in whole 128-byte
// lines.  bf16 of K up to 4096 at more than 6 and up to 8 rows per CU, us per call, 4 / 8 rows: 4096 -> 4096 at 1900 / 2048 rows 70.4 /
// 68.8, 70.5 / 69.1, 4096 -> 1024 at 1560 / 2048 rows 31.8 / 29.8, 35.6 / 31.5 (the pass alone 15.1 / 9.7), 2048 -> 4096 44.4 / 42.9,
// 2048 -> 1024 21.3 / 20.5, 22.7 / 21.4, 4096 -> 14336 at 2048 rows 211.6 / 211.0; 30 calls of the range on N of 256 .. 8192: 5 % in the
// mean, none slower.  Outside: 4096 -> 1024 at 1400 / 1500 / 2100 / 2700 rows
// 29.7 / 31.5, 30.5 / 32.6, 38.1 / 40.8, 44.2 / 45.3, 14336 -> 1024 at 3000 rows 135 / 155, fp32 4096 -> 1024 at 2048 rows 33.3 / 34.1.
static int rows_per_staging_workgroup(const WeightView& w, int xdt, int mc, int num_cus, bool norm)
{
    if (!norm && xdt == kBF16 && w.K <= 4096 && mc > 6 * num_cus && mc <= 8 * num_cus) return 8;
    if (norm) return 4;
    if (w.K <= 8192) return mc <= 48 ? 2 : 4;
    return mc <= 128 ? 1 : mc <= (xdt == kF32 ? 512 : 384) ? 2 : 4;
}

// What multiplies a chunk of mc rows that fits the scratch (part_bytes: its second half): the kernel of gemm_rows.hip where rows.nf is not 0, else tiles
struct ChunkPlan {
    RowsPlan rows;
    TilePlan tiles;
};

static ChunkPlan plan_chunk(const WeightView& w, int xdt, int mc, int num_cus, bool exact, size_t part_bytes, const Epilogue& epi)
{
    ChunkPlan p = {};
    // few rows on a wide output, FAST mode: the kernel of gemm_rows.hip (waves split K, no LDS on the way)
    if (!exact) p.rows = rows_plan(w, mc, num_cus, epi);
    if (!p.rows.nf && !exact && g_rows_kernel < 2) p.rows = gemm_rows_plan_long_k(w, mc, num_cus, epi);
    if (!p.rows.nf) p.tiles = plan_tiles(w, mc, exact, exact && xdt == kBF16, num_cus, part_bytes, epi);
    return p;
}

hipError_t launch_gemm(const WeightView& w, const void* x, int xdt, int M, void* y, int ydt,
                       int num_cus, bool exact, void* workspace, size_t workspace_bytes, const Epilogue& epi,
                       hipStream_t st)
{
    if (xdt == kF32 && exact) return hipErrorNotSupported;   // api.hip walks exact fp32 prefill through the decode kernel
    // FAST multiplies in f16: bf16 activations are widened, fp32 activations rounded to f16
    // (both behind a power-of-two scale per row that the epilogue undoes)
    const bool widen = !exact && xdt != kF16;
    const float out_scale = 1.0f;
    const int kdt = widen ? kF16 : xdt;
    // Rows are staged through the workspace in chunks that fit it; work on one stream is
    // ordered, so a chunk's multiply is done before the next chunk overwrites the stage.
    // First half of the workspace: staged X; second half: partial sums of a K split.
    const size_t half = workspace_bytes / 2;
    float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) + half);
    const int64_t max_rows = staged_rows(w, workspace_bytes);
    if (!workspace || max_rows < 256) return hipErrorOutOfMemory;
    float* ssq_part = reinterpret_cast<float*>(static_cast<char*>(workspace) + half - kStatsBytes);
    float* unscale = reinterpret_cast<float*>(static_cast<char*>(workspace) + half - kStatsBytes / 4);
    const int64_t row_bytes = (int64_t)w.K * (xdt == kF32 ? 4 : 2);        // a row of the caller's X
    const size_t ysize = ydt == kF32 ? 4 : 2;
    for (int64_t m_lo = 0; m_lo < M; m_lo += max_rows) {
        const int mc = (int)((M - m_lo) < max_rows ? (M - m_lo) : max_rows);
        const u32x4_t* xs = reinterpret_cast<const u32x4_t*>(static_cast<const char*>(x) + m_lo * row_bytes);
        const int64_t n_out = epi.kind == kEpiSwiglu ? w.N / 2 : w.N;
        void* yc = static_cast<char*>(y) + (size_t)m_lo * n_out * ysize;
        Epilogue ec = epi;                 // this row chunk's slice of the residual
        if (epi.kind == kEpiAdd) ec.residual = static_cast<const char*>(epi.residual) + (size_t)m_lo * n_out * ysize;
        const ChunkPlan chunk = plan_chunk(w, xdt, mc, num_cus, exact, half, ec);
        const RowsPlan& plan = chunk.rows;
        const TilePlan& tp = chunk.tiles;
        // gemm_cols.hip takes rows that are operands as they stand from where the caller has them: no staging launch (not where y is
        // written over them).  us per call with / without it, EXACT: bf16 4096 -> 14336 at 64 / 256 rows 26.8 / 23.5, 57.7 / 53.9, 512 -> 1000
        // at 100 rows 9.9 / 7.6, 7008 -> 800 at 200 rows 17.8 / 14.0, f16 4096 -> 6144 at 512 rows 51.9 / 45.6; FAST f16 14336 -> 4096 at 45 / 128
        // rows 21.2 / 17.6, 30.9 / 26.6.
        const char *xb = reinterpret_cast<const char*>(xs), *yb = static_cast<const char*>(yc);
        const bool apart = xb + (size_t)mc * w.K * 2 <= yb || yb + (size_t)mc * n_out * ysize <= xb;
        const bool raw = !plan.nf && tp.kind == TilePlan::kCols && !widen && !epi.gamma && apart && g_raw;
        const int K8 = w.K / 8;
        const dim3 grid((unsigned)((mc + 15) / 16), (unsigned)((K8 / 4 + kStageGroups - 1) / kStageGroups));
        u32x4_t* xst = reinterpret_cast<u32x4_t*>(workspace);
        NormStats ns = {ssq_part, (int)grid.y, nullptr};
        if (raw) {
            ns = NormStats{nullptr, 0, nullptr};
        } else if (widen) {
            // per-row scaled f16 operands; one sum of squares per row
            ns = NormStats{ssq_part, 1, unscale};
            const int stage_rows = rows_per_staging_workgroup(w, xdt, mc, num_cus, epi.gamma != nullptr);
            dim3 rgrid((unsigned)((mc + 15) / 16) * (16 / stage_rows));
            const Touch touch = plan_touch(w, mc, num_cus, ec, exact, rgrid.x);
            // pieces of 512 k a lane keeps in registers: the whole row when it has at most 16384 (bf16) or 8192 (fp32)
            // elements, 16384 with two rows per workgroup, 32768 with one
            const int per_row = 16 / stage_rows, batches = ((K8 + 63) / 64 + per_row - 1) / per_row;
#define CYBQ_STAGE_ROWS(XT, NORM, CH, ...) \
    hipLaunchKernelGGL((stage_rows_kernel<XT, NORM, CH, __VA_ARGS__>), rgrid, dim3(1024), 0, st, xs, xst, mc, w.K, touch.first_group, epi.gamma_dt, epi.gamma, unscale, ssq_part, touch)
#define CYBQ_STAGE_ROWS_CH(XT, NORM, ROWS, C1, C2, C3)              \
    do {                                                            \
        if (batches <= C1) CYBQ_STAGE_ROWS(XT, NORM, C1, ROWS);     \
        else if (batches <= C2) CYBQ_STAGE_ROWS(XT, NORM, C2, ROWS); \
        else CYBQ_STAGE_ROWS(XT, NORM, C3, ROWS);                   \
    } while (0)
#define CYBQ_STAGE_ROWS_N(XT, NORM)                                                        \
    do {                                                                                   \
        if (stage_rows == 1) CYBQ_STAGE_ROWS_CH(XT, false, 1, 1, 2, 4);                    \
        else if (stage_rows == 2) CYBQ_STAGE_ROWS_CH(XT, false, 2, 1, 2, 4);               \
        else CYBQ_STAGE_ROWS_CH(XT, NORM, 4, (XT == 2 ? 1 : 2), (XT == 2 ? 2 : 4), (XT == 2 ? 4 : 8)); \
    } while (0)
            if (stage_rows == 8) {
                if (batches <= 2) CYBQ_STAGE_ROWS(1, false, 2, 8);
                else CYBQ_STAGE_ROWS(1, false, 4, 8);
            } else if (xdt == kF32 && epi.gamma) CYBQ_STAGE_ROWS_N(2, true);
            else if (xdt == kF32) CYBQ_STAGE_ROWS_N(2, false);
            // bf16 rows of K over 4096 with a norm: with gamma kept (79 registers, not 47) a CU has room for one workgroup, which is all there is for it
            // up to four rows per CU, and not beyond.  us per call, kept / loaded twice: 6144 -> 1024 at 768 / 1024 rows 30.3 / 30.9, 33.3 / 34.2, at 1040 /
            // 1100 / 2048 / 4096 rows 36.6 / 35.7, 38.4 / 36.0, 45.4 / 42.1, 88.0 / 83.6; 8192 -> 4096 at 2048 rows 128.4 / 125.6.
            else if (epi.gamma && batches > 2 && batches <= 4 && mc > 4 * num_cus) CYBQ_STAGE_ROWS(1, true, 4, 4, false);
            else if (epi.gamma) CYBQ_STAGE_ROWS_N(1, true);
            else CYBQ_STAGE_ROWS_N(1, false);
#undef CYBQ_STAGE_ROWS_N
#undef CYBQ_STAGE_ROWS_CH
#undef CYBQ_STAGE_ROWS
        } else if (epi.gamma) {
            if (xdt == kBF16) hipLaunchKernelGGL((stage_x_kernel<true, true>), grid, dim3(256), 0, st, xs, xst, mc, K8, epi, ssq_part);
            else hipLaunchKernelGGL((stage_x_kernel<false, true>), grid, dim3(256), 0, st, xs, xst, mc, K8, epi, ssq_part);
        } else {
            hipLaunchKernelGGL((stage_x_kernel<false, false>), grid, dim3(256), 0, st, xs, xst, mc, K8, epi, ssq_part);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (plan.nf) {
            e = launch_gemm_rows(w, workspace, mc, yc, ydt, ec, ns.part, ns.nblk, ns.unscale, plan, part, st);
            if (e == hipSuccess && plan.shares > 4) e = launch_reduce(part, plan.shares - 3, mc, w.N, yc, ydt, out_scale, ec, ns, w.K, st);
            if (e != hipSuccess) return e;
            continue;
        }
        const void* const from = raw ? static_cast<const void*>(xs) : workspace;
        if (w.bits == 4) {
            e = kdt == kBF16 ? launch_tiles<4, 1>(tp, w, from, raw, mc, yc, ydt, exact, out_scale, part, ec, ns, st)
                             : launch_tiles<4, 0>(tp, w, from, raw, mc, yc, ydt, exact, out_scale, part, ec, ns, st);
        } else {
            e = kdt == kBF16 ? launch_tiles<8, 1>(tp, w, from, raw, mc, yc, ydt, exact, out_scale, part, ec, ns, st)
                             : launch_tiles<8, 0>(tp, w, from, raw, mc, yc, ydt, exact, out_scale, part, ec, ns, st);
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

PrefillRoute prefill_route(const WeightView& w, int xdt, int M, int num_cus, bool exact, size_t workspace_bytes, const Epilogue& epi)
{
    const int64_t max_rows = staged_rows(w, workspace_bytes);
    if (max_rows < 256 || (xdt == kF32 && exact)) return {};
    const int mc = (int)std::min<int64_t>(M, max_rows);
    const ChunkPlan p = plan_chunk(w, xdt, mc, num_cus, exact, workspace_bytes / 2, epi);
    PrefillRoute r = {};
    if (!exact && xdt != kF16) r.stage_rows = rows_per_staging_workgroup(w, xdt, mc, num_cus, epi.gamma != nullptr);
    if (p.rows.nf) {
        r.kernel = 1;
        r.nf = p.rows.nf;
        r.splits = 1;
    } else {
        r.kernel = p.tiles.kind == TilePlan::kTiles ? 2 : p.tiles.kind == TilePlan::kRoles ? 3 : 4;
        r.nf = p.tiles.nf;
        r.splits = p.tiles.splits;
    }
    return r;
}

}  // namespace cybq
