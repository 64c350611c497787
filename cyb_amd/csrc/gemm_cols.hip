// gemm_cols.hip - prefill kernel whose waves stand side by side along the columns and share out every K tile.
//
// Workgroup = 8 waves, output tile 16 * RB rows x 64 * CS columns (KH = 2).  Wave (col, kh) owns CS strips of 16 columns against ALL rows and,
// of every K tile, the two scale groups of half kh; the halves' sums meet in LDS once at the end.  KH = 1: eight waves side by side,
// whole K tiles (a long K on few rows, plan_gemm_cols_long_k).
//
//   W  a native tile is multiplied by the two waves that hold its groups and by nobody else: its words go from LDS to registers,
//      are dequantised there and are MFMA operands as they stand - no operand goes through LDS, none is made twice.
//   X  is shared by the four columns of waves: copied to LDS once, read by each.  Rows that are operands as they stand (16-bit, no norm,
//      FAST mode: f16) come from where the caller has them (RAW), whole lines of a row per copy, their pieces permuted so that
//      reads meet no bank conflicts: as quick as copies of staged operands, and the staging launch (2.4 us and 1 us a megabyte) is gone.
//   Both come by global_load_lds, which needs no registers while in flight: 3 - 5 K tiles of X and up to 10 of packed weights
//      are on their way, counted by hand (s_waitcnt vmcnt: copies retire in order), one barrier per K tile in its middle - the first
//      half's operands are in registers when it is passed, the second half's arithmetic covers the reads behind it.
//   EXACT mode: the operands are the integers q (bf16 rows: times the power of two of the group's scale, so that no sum leaves fp32's range
//      before the scale is on it), one MFMA of a strip and group starts from zero and its sums are scaled on their way into the fp32
//      accumulators, two MFMAs later: four FMAs per MFMA.  Nothing is rounded before fp32.  (w = scale * q cut into two operands took
//      twice the MFMAs and 18 (f16) to 43 (bf16) vector instructions to make them.)
//      f16 integers take 10 vector instructions per eight weights (Q8: 8), bf16 operands 16.
//
// What bounds it: a SIMD's issue slots and LDS.  Per 16x16x32 MFMA (16 cycles of the matrix pipe) a SIMD issues two other vector
// instructions for free, whatever the number of waves; per strip and group FAST has 14 of them and EXACT 11 - 18 and four per row block.
// So the gain is where the tiled kernels of gemm.hip have few rows (their waves own 32 each, and every weight operand crosses LDS for
// each of them) or EXACT's operands to make.  A K tile of 128 rows x 128 columns takes 1700 cycles in FAST, 1024 of them MFMAs.
// us per call, weights from HBM, hi / lo operands with a staging launch -> now, EXACT: bf16 Q4 4096 -> 14336 at 40 / 64 / 256 rows 27.6 / 28.7 / 60.2 ->
// 20.6 / 22.1 / 45.3, 14336 -> 4096 at 128 rows 39.8 -> 31.0, 4096 -> 4096 at 256 rows 27.8 -> 19.4, 4096 -> 6144 at 512 rows 59.1 -> 43.4; Q8
// 4096 -> 14336 at 64 / 256 rows 30.0 / 68.9 -> 24.4 / 54.1; f16 Q4 4096 -> 14336 at 256 rows 61.0 -> 49.5, 4096 -> 4096 at 256 rows 26.5 -> 21.1.  (The
// powers of two: nothing to 4 %, 40 rows 19.7 -> 20.6, Q8 53.1 -> 54.1.)  Relative L2 against float64, same calls and Q8: bf16 1.2e-7 -
// 3e-7 (Q8 1.7e-6) -> 6e-8 - 1.4e-7, f16 1.4e-7 - 3.9e-7 -> 6e-8 - 1.4e-7.  FAST, tiled kernels -> this one, both behind a staging launch: 4096 ->
// 28672 at 96 / 128 rows 42.5 / 46.6 -> 33.5 / 39.9, with SwiGLU 48.9 / 49.8 -> 33.3 / 39.5, 14336 -> 14336 at 40 / 192 rows 58.5 / 124.5 -> 44.1 / 92.8,
// 4096 -> 14336 at 192 rows 39.4 -> 33.7, 1024 -> 4096 at 128 rows 15.7 -> 10.1.
// Tried: four waves of 128 x 64 on 32x32x16 MFMAs, every weight of a K tile dequantised by its wave (one wave per SIMD: MFMAs and
// vector instructions add up, 2900 cycles a K tile for 2048 of MFMAs; 4096 -> 14336 at 512 rows 77 us against 60 of the role-split
// kernel); deeper rings for the few-row forms (no change); words read from LDS a K tile earlier (3 % slower).
#include <algorithm>
#include <type_traits>

#include "cybq_device.h"
#include "cybq_internal.h"

namespace cybq {

namespace {

#include "gemm_parts.h"

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// the same from the lanes of `lanes` alone (all 64 lanes are active around it; a branch would cut the scheduling region)
__device__ __forceinline__ void copy_to_lds(uint32_t lds_off, const void* base, uint32_t off, uint64_t lanes)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1" ::"s"(__builtin_amdgcn_readfirstlane(lds_off)), "v"(off), "s"(base), "s"(lanes));
}
template <int N>
__device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// MODE 0: FAST (operands round_f16(scale * q)), 1 / 2: EXACT with f16 / bf16 rows (operands q / q * 2^e, the scale / the rest of it on each
// group's sums)
template <int BITS, int MODE, int RB, int CS, int KH>
struct ColsShape {
    static constexpr int COLS = 8 / KH;                                    // waves side by side
    static constexpr int STRIPS = COLS * CS;
    static constexpr int GROUPS = 4 / KH;                                  // scale groups of a K tile per wave
    static constexpr int WORDS = BITS / 2 * GROUPS / 2;                    // and packed words per lane
    static constexpr int XTILE = RB * 4096;                                // bytes of a K tile of X
    static constexpr int WSCALES = STRIPS * 1024 * (BITS / 4);             // scales behind the q words
    static constexpr int WTILE = WSCALES + STRIPS * 128;
    static constexpr bool FOLDED = BITS == 4 && STRIPS == 4;               // four waves copy q words, the other four scales
    static constexpr int XCOPIES = (RB * 4 + 7) / 8;                       // per wave and K tile
    static constexpr int QCOPIES = FOLDED ? 1 : STRIPS * (BITS / 4) / 8;
    static constexpr int WCOPIES = FOLDED ? 1 : QCOPIES + 1;
    static constexpr int BUDGET = 156 * 1024;
    // K tiles of X in flight: three where a tile is long, up to five where it is short; weights get the rest
    static constexpr int NX = RB >= 8 ? 3 : RB >= 6 ? (BITS * STRIPS > 32 ? 3 : 4) : RB >= 4 && BITS * STRIPS > 32 ? 4 : 5;
    static constexpr int NWFIT = (BUDGET - NX * XTILE) / WTILE;
    static constexpr int NW = NWFIT > 10 ? 10 : NWFIT;
    // copies that may be outstanding when a K tile's X and words have to be there, `newer` batches behind the one with its X
    static constexpr int allowed(int newer) { return newer * (XCOPIES + WCOPIES) + (NW > NX ? WCOPIES : 0); }
    static constexpr int WBASE = NX * XTILE;
    static constexpr int PITCH = STRIPS * 16 + 4;                          // floats, finished tile
    static constexpr int TILE = RB * 16 * PITCH * 4;
    static constexpr int LDS = WBASE + NW * WTILE > TILE + RB * 64 ? WBASE + NW * WTILE : TILE + RB * 64;
    static_assert(NW >= NX && LDS <= 160 * 1024, "LDS");
};

// RAW: X as the caller has it, row major, of the operands' type (no staging launch before the multiply)
template <int BITS, int MODE, int RB, int CS, int KH, bool RAW>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_cols_kernel(
    const uint8_t* __restrict__ wbase, const uint8_t* __restrict__ x, int K, int N, int M, int n_tiles, int m_tiles, int splits, int kt_per_split, int groups,
    void* __restrict__ y, int ydt, float* __restrict__ part, Epilogue epi, NormStats ns)
{
    // (the arguments up to ydt come in registers at wave start, sixteen words of them, so what follows from K, N and M is not one.  With tile counts
    // handed over and y behind the sixteen, us per call: EXACT f16 4096 -> 14336 at 64 rows 21.5 / 20.5, bf16 320 -> 19224 at 51 rows with a residual 40.9 /
    // 38.7, f16 8384 -> 528 at 225 rows 11.7 / 11.5; with K behind y, 8224 -> 1920 Q8 bf16 at 119 rows 23.4 / 22.7, FAST 14336 -> 4096 at 45 rows 23.3 / 23.0)
    const int KT_ = (K + kTileK - 1) / kTileK, NT = (N + kTileN - 1) / kTileN, x_row_blocks = (M + 15) / 16;
    using S = ColsShape<BITS, MODE, RB, CS, KH>;
    constexpr int NX = S::NX, NW = S::NW, XC = S::XCOPIES, WC = S::WCOPIES, GROUPS = S::GROUPS, WORDS = S::WORDS;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int per_xcd = groups >> 3;
    const int item = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
    if (item >= n_tiles * m_tiles * splits) return;
    // (divisions leave their results in vector registers: back to scalars, the copies' bases hang on them)
    const int split = __builtin_amdgcn_readfirstlane(item / (n_tiles * m_tiles));
    const int rest = item - split * (n_tiles * m_tiles);
    const int tile_n = __builtin_amdgcn_readfirstlane(rest / m_tiles), tile_m = rest - tile_n * m_tiles;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = wave % S::COLS, kh = wave / S::COLS;       // my strips, my half of every K tile (KH = 1: all of it)
    const int m0 = tile_m * (RB * 16);
    const int nt0 = tile_n * S::STRIPS;                        // first strip of the workgroup
    const int kt_lo = split * kt_per_split;
    const int KT = min(kt_per_split, KT_ - kt_lo);
    const int kt0 = __builtin_amdgcn_readfirstlane(tile_n % KT);
    const int G = K / kGroup;
    auto rot = [&](int kt) {
        const int r = min(kt, KT - 1) + kt0;
        return kt_lo + (r >= KT ? r - KT : r);
    };

    // ---- copies into LDS.  X: block e = row block e / 4, group e % 4 of the K tile.  RAW: block e = rows 8 * (e / 2) .. + 8, half e % 2 of
    // the K tile: whole 128-byte lines, eight lanes to a row, with piece p of row r in slot p ^ (r & 7) of the row: eight lanes in a row that
    // read one piece of their rows then meet eight different slots, all 128 bytes that LDS gives in a cycle.  (Rows r and r + 8 meet the same
    // banks, a cycle apart: 0.24 M conflict cycles over the chip at 256 rows of 4096 -> 14336, as many as with staged operands.)
    const int raw_row = lane >> 3, raw_piece = (lane & 7) ^ raw_row;
    uint32_t xrow[XC];
    int xblk[XC];
#pragma unroll
    for (int c = 0; c < XC; c++) {
        if constexpr (RAW) {
            xblk[c] = min(c * 8 + wave, RB * 4 - 2 + (wave & 1));
            xrow[c] = (uint32_t)min(m0 + (xblk[c] >> 1) * 8 + raw_row, M - 1) * (uint32_t)(K * 2) + (uint32_t)(raw_piece & 3) * 16u;
        } else {
            xblk[c] = min(c * 8 + wave, RB * 4 - 1);
            xrow[c] = (uint32_t)min(m0 / 16 + (xblk[c] >> 2), x_row_blocks - 1) * (uint32_t)(G * 1024);
        }
    }
    auto copy_x = [&](int kt, int buf, int c) {
        if constexpr (RAW) {
            // (groups past the end of a row: its last one, against weights of zero)
            const int g = min(rot(kt) * 4 + ((wave & 1) * 2 + (raw_piece >> 2)), G - 1);
            copy_to_lds(buf * S::XTILE + (xblk[c] & 1) * (RB * 2048) + (xblk[c] >> 1) * 1024, x, xrow[c] + (uint32_t)g * 64u);
        } else {
            const int g = min(rot(kt) * 4 + (xblk[c] & 3), G - 1);
            copy_to_lds(buf * S::XTILE + xblk[c] * 1024, x, xrow[c] + (uint32_t)g * 1024u + (uint32_t)lane * 16u);
        }
    };
    const int ntb = min(nt0, NT - 1);
    const uint8_t* const wsrc = wbase + (int64_t)ntb * KT_ * kTileBytes<BITS>;
    auto strip_at = [&](int s) { return (uint32_t)((min(nt0 + s, NT - 1) - ntb) * KT_) * (uint32_t)kTileBytes<BITS>; };
    constexpr int PER_WAVE = S::STRIPS / 8 > 0 ? S::STRIPS / 8 : 1;                 // strips whose scales a wave copies
    const int sfirst = (wave * PER_WAVE) % S::STRIPS;
    const uint32_t sc_off = strip_at(sfirst + min(lane >> 3, PER_WAVE - 1)) + (uint32_t)(kTileQBytes<BITS> + (lane & 7) * 16);
    uint32_t q_off[S::QCOPIES];
    int q_dst[S::QCOPIES];
#pragma unroll
    for (int c = 0; c < S::QCOPIES; c++) {
        const int e = S::FOLDED ? (wave & 3) : c * 8 + wave;                        // 1-KB block of the q words
        q_dst[c] = e * 1024;
        q_off[c] = strip_at(e / (BITS / 4)) + (uint32_t)(e % (BITS / 4)) * 1024u + (uint32_t)lane * 16u;
    }
    auto copy_w = [&](int kt, int buf, int c) {
        const uint32_t at = (uint32_t)rot(kt) * (uint32_t)kTileBytes<BITS>;
        const int dst = S::WBASE + buf * S::WTILE;
        if (S::FOLDED) {
            const bool sc = wave >= 4;
            copy_to_lds(dst + (sc ? S::WSCALES + (wave - 4) * 128 : q_dst[0]), wsrc, (sc ? sc_off : q_off[0]) + at, sc ? 0xffull : ~0ull);
        } else if (c < S::QCOPIES) {
            copy_to_lds(dst + q_dst[c < S::QCOPIES ? c : 0], wsrc, q_off[c < S::QCOPIES ? c : 0] + at);
        } else {
            copy_to_lds(dst + S::WSCALES + sfirst * 128, wsrc, sc_off + at, (1ull << (8 * PER_WAVE)) - 1);
        }
    };

    // ---- LDS -> registers
    Frag16 a[2][RB], b[2][CS];
    uint32_t wq[CS][WORDS], wn[CS][WORDS], sq[CS][GROUPS / 2], sn[CS][GROUPS / 2];     // packed weights and scales of my groups: this K tile's, the next one's
    const uint32_t raw_lane = (uint32_t)(((lane >> 3) & 1) * 1024 + (lane & 7) * 128 + (((lane >> 4) ^ (lane & 7)) * 16));
    auto read_a = [&](Frag16& dst, int buf, int j, int i) {               // j: which of my groups
        if constexpr (RAW) {
            const int half = KH == 2 ? kh : j >> 1;
            dst.u = *reinterpret_cast<const u32x4_t*>(smem + buf * S::XTILE + half * (RB * 2048) + i * 2048 + ((j & 1) ? raw_lane ^ 64u : raw_lane));
        } else dst.u = *reinterpret_cast<const u32x4_t*>(smem + buf * S::XTILE + kh * (GROUPS * 1024) + lane * 16 + (i * 4 + j) * 1024);
    };
    auto read_w = [&](int buf, uint32_t (&q)[CS][WORDS], uint32_t (&sc)[CS][GROUPS / 2]) {
        const uint8_t* p = smem + S::WBASE + buf * S::WTILE;
#pragma unroll
        for (int s = 0; s < CS; s++) {
            const int strip = col * CS + s;
            if constexpr (BITS == 4 && KH == 2) {
                const u32x2_t v = *reinterpret_cast<const u32x2_t*>(p + strip * 1024 + lane * 16 + kh * 8);
                q[s][0] = v[0];
                q[s][1] = v[1];
            } else {
#pragma unroll
                for (int h = 0; h < WORDS / 4; h++) {
                    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(p + strip * (1024 * (BITS / 4)) + (kh + h) * 1024 + lane * 16);
#pragma unroll
                    for (int e = 0; e < 4; e++) q[s][(h * 4 + e) & (WORDS - 1)] = v[e];
                }
            }
            const uint32_t* sp = reinterpret_cast<const uint32_t*>(p + S::WSCALES + strip * 128 + (lane & 15) * 8 + kh * 4);
#pragma unroll
            for (int g = 0; g < GROUPS / 2; g++) sc[s][g] = sp[g];
        }
    };
    uint32_t magic_lo, magic_hi;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic_lo));
    asm volatile("v_mov_b32 %0, 0x54005400" : "=v"(magic_hi));
    // slots 2p, 2p + 1 of my group j in f16, plus a bias (kBias): 1024 + u, 64 + u (odd group of Q4) or 1024 + u with u = q + 128 (Q8)
    auto biased = [&](const uint32_t (&q)[WORDS], int j, int p) {
        if constexpr (BITS == 4) {
            const uint32_t src = q[(2 * (j >> 1) + (p >> 1)) & (WORDS - 1)] >> (8 * (p & 1));
            return as_h2((j & 1) ? (src & 0x00F000F0u) | magic_hi : (src & 0x000F000Fu) | magic_lo);
        } else {
            return as_h2(__builtin_amdgcn_perm(0x64646464u, q[(2 * j + (p >> 1)) & (WORDS - 1)], (p & 1) ? 0x04030402u : 0x04010400u));
        }
    };
    auto scale_of = [&](const uint32_t (&sc)[GROUPS / 2], int j) {
        return __builtin_bit_cast(_Float16, (uint16_t)((j & 1) ? sc[j >> 1] >> 16 : sc[j >> 1] & 0xffffu));
    };
    // bf16 rows: a group's operands are q * 2^e with 2^e the power of two of its scale (exact: eight significant bits), its sums are multiplied
    // by scale / 2^e, 1 to 2: they leave fp32's range where the group's own contribution to y does.  (Sums of q itself were Inf from |x| of
    // 8e34 on, whatever the scale.)  Q4: |q| up to 8 fits the upper byte of an f16 number, and a pair of such bytes is converted with the
    // exponent of the scale (zero: 2^-127) in one instruction; 16 vector instructions per eight weights.  Q8: one fma to fp32 each, 16.
    uint32_t pend[2] = {};
    auto operand = [&](const uint32_t (&q)[WORDS], const uint32_t (&sc)[GROUPS / 2], int j, int p, int buf, int s) {
        const float bias = BITS == 8 ? -1152.0f : (j & 1) ? -72.0f : -1032.0f;
        auto integers = [&]() { return biased(q, j, p) + (half2_t){(_Float16)bias, (_Float16)bias}; };          // exact
        if constexpr (MODE == 2 && BITS == 4) {
            pend[p & 1] = as_u32(integers());
            if (p & 1) {
                const uint32_t bytes = __builtin_amdgcn_perm(pend[1], pend[0], 0x07050301u);
                const float f = (float)scale_of(sc, j);
                b[buf][s].u[p - 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(bytes, f, false));
                b[buf][s].u[p] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(bytes, f, true));
            }
        } else if constexpr (MODE == 2) {
            const half2_t v = biased(q, j, p);
            const float f = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, (float)scale_of(sc, j)) & 0x7f800000u), c = bias * f;
            const float w0 = fmaf((float)v.x, f, c), w1 = fmaf((float)v.y, f, c);
            b[buf][s].u[p] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, w1), __builtin_bit_cast(uint32_t, w0), 0x07060302u);
        } else {
            half2_t n = integers();
            if constexpr (MODE == 0) {
                const _Float16 sh = scale_of(sc, j);
                n *= (half2_t){sh, sh};
            }
            b[buf][s].u[p] = as_u32(n);
        }
    };

    float4_t acc[RB][CS];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
        for (int s = 0; s < CS; s++) acc[i][s] = (float4_t){0.f, 0.f, 0.f, 0.f};
    // EXACT: the sums of one strip and group, on their way for two MFMAs before the scale is applied, and the scales of this group and the last
    float4_t d[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    float scf[2][CS] = {};
    auto apply = [&](float4_t& sum, float f, const float4_t& v) {
#pragma unroll
        for (int r = 0; r < 4; r++) sum[r] = fmaf(f, v[r], sum[r]);
    };

    // ---- prologue: batch -n of the copies holds X of K tile NX - n and the weights of K tile NW - n
    static_for<0, NW>([&](auto n_) {
        constexpr int back = NW - decltype(n_)::value;         // NW .. 1
        if constexpr (back <= NX) {
#pragma unroll
            for (int c = 0; c < XC; c++) copy_x(NX - back, NX - back, c);
        }
#pragma unroll
        for (int c = 0; c < WC; c++) copy_w(NW - back, NW - back, c);
    });
    wait_copies<S::allowed(NX - 1)>();
    asm volatile("s_barrier" ::: "memory");
    read_w(0, wq, sq);
#pragma unroll
    for (int i = 0; i < RB; i++) read_a(a[0][i], 0, 0, i);
#pragma unroll
    for (int s = 0; s < CS; s++)
#pragma unroll
        for (int p = 0; p < 4; p++) operand(wq[s], sq[s], 0, p, 0, s);

    int xbuf = 0, wbuf = 0;
    // PHASE 0: copies of X and weights go out, 1: of X alone (the last NW K tiles), 2: none (the last NX)
    auto k_tile = [&](int kt, auto phase_) {
        constexpr int PHASE = decltype(phase_)::value;
        const int xnext = xbuf + 1 == NX ? 0 : xbuf + 1, wnext = wbuf + 1 == NW ? 0 : wbuf + 1;
        static_for<0, GROUPS>([&](auto j_) {
            constexpr int j = decltype(j_)::value, cur = j & 1, nxt = 1 - cur;
            constexpr bool last = j == GROUPS - 1;
            if constexpr (last) {
                // all copies of the next K tile are in LDS, and nobody reads this one's any more
                if constexpr (PHASE == 0) {
                    wait_copies<S::allowed(NX - 2)>();
                } else if constexpr (PHASE == 1) {
                    wait_copies<(NX - 2) * XC>();
                } else {
                    const int left = min(NX - 2, KT - 2 - kt);         // K tiles of X requested after the next one's
                    if (left == 3) wait_copies<3 * XC>();
                    else if (left == 2) wait_copies<2 * XC>();
                    else if (left == 1) wait_copies<XC>();
                    else wait_copies<0>();
                }
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                read_w(wnext, wn, sn);
            }
            constexpr int MMAS = RB * CS, PAIRS = 4 * CS;
            if constexpr (MODE != 0) {
#pragma unroll
                for (int s = 0; s < CS; s++) {
                    const float f = (float)scale_of(sq[s], j);
                    scf[cur][s] = MODE == 1 ? f : 2.0f * __builtin_amdgcn_frexp_mantf(f);
                }
            }
            static_for<0, MMAS>([&](auto m_) {
                constexpr int m = decltype(m_)::value, i = m / CS, s = m % CS;
                if constexpr (MODE == 0) {
                    acc[i][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[cur][i].h, b[cur][s].h, acc[i][s], 0, 0, 0);
                } else {
                    constexpr int slot = (j * MMAS + m) & 1, before = (m + MMAS - 2) % MMAS;      // two MFMAs ago: perhaps of the last group
                    apply(acc[before / CS][before % CS], scf[m < 2 ? nxt : cur][before % CS], d[slot]);
                    d[slot] = mma<MODE == 2>(a[cur][i], b[cur][s], (float4_t){0.f, 0.f, 0.f, 0.f});
                }
                if constexpr (s == 0) read_a(a[nxt][i], last ? xnext : xbuf, last ? 0 : j + 1, i);
                // (the next K tile's words have just been asked for: the second half of the group is theirs; a form that read them a
                // K tile earlier and spread their arithmetic over the whole group was 3 % slower)
                constexpr int F = last ? MMAS / 2 : 0, p0 = m < F ? 0 : (m - F) * PAIRS / (MMAS - F), p1 = m < F ? 0 : (m - F + 1) * PAIRS / (MMAS - F);
                static_for<p0, p1>([&](auto q_) {
                    constexpr int q = decltype(q_)::value, ds = q / 4, p = q & 3;
                    if constexpr (last) operand(wn[ds], sn[ds], 0, p, nxt, ds);
                    else operand(wq[ds], sq[ds], j + 1, p, nxt, ds);
                });
                if constexpr (last && PHASE < 2) {
                    constexpr int ALL = PHASE == 0 ? XC + WC : XC;
                    static_for<m * ALL / MMAS, (m + 1) * ALL / MMAS>([&](auto c_) {
                        constexpr int c = decltype(c_)::value;
                        if constexpr (c < XC) copy_x(kt + NX, xbuf, c);
                        else copy_w(kt + NW, wbuf, c - XC);
                    });
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        xbuf = xnext;
        wbuf = wnext;
#pragma unroll
        for (int s = 0; s < CS; s++) {
#pragma unroll
            for (int g = 0; g < GROUPS / 2; g++) sq[s][g] = sn[s][g];
#pragma unroll
            for (int e = 0; e < WORDS; e++) wq[s][e] = wn[s][e];
        }
    };
    int kt = 0;
    for (; kt + NW < KT; kt++) k_tile(kt, std::integral_constant<int, 0>{});
    for (; kt + NX < KT; kt++) k_tile(kt, std::integral_constant<int, 1>{});
    for (; kt < KT; kt++) k_tile(kt, std::integral_constant<int, 2>{});
    if constexpr (MODE != 0) {
#pragma unroll
        for (int m = RB * CS - 2; m < RB * CS; m++) apply(acc[m / CS][m % CS], scf[(GROUPS - 1) & 1][m % CS], d[((GROUPS - 1) * RB * CS + m) & 1]);
    }

    // ---- the two halves of K meet in LDS; then whole runs of a row, four elements per thread
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float* const tile = reinterpret_cast<float*>(smem);
    float* const rowf = reinterpret_cast<float*>(smem + S::TILE);
    const bool slab = splits > 1;
    const int row16 = lane & 15, oct = lane >> 4;
    if (tid < RB * 16) rowf[tid] = slab || !(epi.gamma || ns.unscale) ? 1.0f : row_factor(ns, epi.gamma != nullptr, min(m0 + tid, M - 1), K, epi.eps);
    if (kh == KH - 1) {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
            for (int s = 0; s < CS; s++)
#pragma unroll
                for (int r = 0; r < 4; r++) tile[(i * 16 + oct * 4 + r) * S::PITCH + (col * CS + s) * 16 + row16] = acc[i][s][r];
    }
    __syncthreads();
    if constexpr (KH == 2) {
        if (kh == 0) {
#pragma unroll
            for (int i = 0; i < RB; i++)
#pragma unroll
                for (int s = 0; s < CS; s++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        float* t = &tile[(i * 16 + oct * 4 + r) * S::PITCH + (col * CS + s) * 16 + row16];
                        *t = acc[i][s][r] + *t;
                    }
        }
        __syncthreads();
    }
    const bool swiglu = !slab && epi.kind == kEpiSwiglu, add = !slab && epi.kind == kEpiAdd;
    if (slab) {
        y = part + (int64_t)split * M * N;
        ydt = kF32;
    }
    const int n_out = swiglu ? N >> 1 : N, n0 = swiglu ? nt0 * 8 : nt0 * 16;
    const uintptr_t amask = ydt == kF32 ? 15u : 7u;
    const bool aligned = (n_out & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & amask) == 0 &&
                         (!add || (reinterpret_cast<uintptr_t>(epi.residual) & amask) == 0);
    auto store4 = [&](float4_t v, int m, int n) {
        const int64_t at = (int64_t)m * n_out + n;
        if (!aligned) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < n_out) {
                    float o = v[e];
                    if (add) o += load_out_g(epi.residual, ydt, at + e);
                    store_out_g(y, ydt, at + e, o);
                }
        } else if (n < n_out) {
            if (ydt == kF32) {
                if (add) v += *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(epi.residual) + at);
                *reinterpret_cast<float4_t*>(reinterpret_cast<float*>(y) + at) = v;
            } else {
                if (add) {
                    const u32x2_t rr = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const uint16_t*>(epi.residual) + at);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t h = (e & 1) ? rr[e >> 1] >> 16 : rr[e >> 1] & 0xffffu;
                        v[e] += ydt == kF16 ? f16_bits_to_f32(h) : __builtin_bit_cast(float, h << 16);
                    }
                }
                u32x2_t o;
                if (ydt == kF16) {
                    const half2_t p = {(_Float16)v[0], (_Float16)v[1]}, q = {(_Float16)v[2], (_Float16)v[3]};
                    o = (u32x2_t){as_u32(p), as_u32(q)};
                } else {
                    o = (u32x2_t){pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
                }
                *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(y) + at) = o;
            }
        }
    };
    const int rows = min(RB * 16, M - m0);
    if (swiglu) {                          // strips 2p / 2p + 1 are gate / up of output block (nt0 >> 1) + p
        constexpr int V4 = S::STRIPS * 2;
        for (int p = tid; p < rows * V4; p += 512) {
            const int row = p / V4, c4 = p % V4;
            const float* t = tile + row * S::PITCH + (c4 >> 2) * 32 + (c4 & 3) * 4;
            const float f = rowf[row];
            float4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = silu_mul(t[e] * f, t[16 + e] * f);
            store4(v, m0 + row, n0 + c4 * 4);
        }
    } else {
        constexpr int V4 = S::STRIPS * 4;
        for (int p = tid; p < rows * V4; p += 512) {
            const int row = p / V4, c4 = p % V4;
            store4(*reinterpret_cast<const float4_t*>(tile + row * S::PITCH + c4 * 4) * rowf[row], m0 + row, n0 + c4 * 4);
        }
    }
}

template <int BITS, int MODE, int RB, int CS, int KH, bool RAW>
hipError_t launch_cols_t(const WeightView& w, const void* x, int M, void* y, int ydt, int splits, const Epilogue& epi, const NormStats& ns,
                         float* part, hipStream_t st)
{
    using S = ColsShape<BITS, MODE, RB, CS, KH>;
    (void)LdsRequest<&gemm_cols_kernel<BITS, MODE, RB, CS, KH, RAW>, S::LDS>::registered;
    const int n_tiles = (w.NT + S::STRIPS - 1) / S::STRIPS, m_tiles = (M + 16 * RB - 1) / (16 * RB);
    const int kt_per_split = (w.KT + splits - 1) / splits;
    const unsigned groups = (unsigned)(((int64_t)n_tiles * m_tiles * splits + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_cols_kernel<BITS, MODE, RB, CS, KH, RAW>), dim3(groups), dim3(512), S::LDS, st, w.base, static_cast<const uint8_t*>(x),
                       w.K, w.N, M, n_tiles, m_tiles, splits, kt_per_split, (int)groups, y, ydt, part, epi, ns);
    return hipGetLastError();
}

constexpr int kColsSplits = 8;               // the slab-adding pass takes as many

}  // namespace

// Row blocks, strips per wave and splits with the shortest estimate.  A round of workgroups costs a fixed part and so much per K
// tile (below, us; fits to 9000 forced calls of 33 .. 600 rows, N of 512 .. 32768, K of 512 .. 14336, Q4 and Q8), a split its slabs' way
// through memory.  FAST: 3 - 5 % rms, choosing by it costs 0.5 % against the best of all forms on these calls.  EXACT: the fits are those of
// two operands per weight, which had twice the MFMAs.  Calls of 65 .. 2048 rows on the integer operands take 0.9 - 2.3 times the estimate (143
// calls; in the mean 1.36 / 1.23 times with one / two strips and f16 rows, 1.23 / 1.06 with bf16 rows), so it ranks these forms no more than
// roughly; against the kernels before (same choice, staged rows) none of 210 EXACT calls is slower, in the mean they are 1.2 times as fast.
ColsPlan plan_gemm_cols(const WeightView& w, int mode, int M, int num_cus, size_t part_bytes)
{
    struct Form {
        int rb, cs;
        float fixed[3], per_kt[3];           // FAST, EXACT f16, EXACT bf16
    };
    static const Form forms[] = {
        {3, 1, {1.4f, 2.1f, 2.1f}, {0.384f, 0.407f, 0.527f}}, {4, 1, {1.7f, 1.8f, 1.9f}, {0.390f, 0.480f, 0.583f}},
        {6, 1, {1.75f, 2.2f, 2.2f}, {0.450f, 0.550f, 0.656f}}, {8, 1, {1.9f, 2.2f, 2.2f}, {0.530f, 0.680f, 0.790f}},
        {3, 2, {2.1f, 3.0f, 2.9f}, {0.516f, 0.620f, 0.900f}}, {4, 2, {2.2f, 2.5f, 2.5f}, {0.555f, 0.745f, 1.020f}},
        {6, 2, {2.6f, 2.9f, 3.2f}, {0.650f, 0.910f, 1.150f}}, {8, 2, {3.0f, 3.0f, 3.3f}, {0.760f, 1.170f, 1.370f}},
    };
    const int need = (M + 15) / 16;          // row blocks
    const float out_mb = 4e-6f * (float)M * (float)w.N;
    ColsPlan best = {0, 0, 1, false, 1e30f};
    for (const Form& f : forms) {
        // up to 128 rows one row tile, the smallest that holds them; beyond, neither 48 rows nor many row tiles of 64
        if (need <= 8 ? (f.rb < need || (f.rb > 3 && f.rb - (f.rb > 4 ? 2 : 1) >= need)) : (f.rb == 3 || (f.rb == 4 && need > 16))) continue;
        const int64_t tiles = (int64_t)((w.NT + 4 * f.cs - 1) / (4 * f.cs)) * ((need + f.rb - 1) / f.rb);
        for (int splits = 1; splits <= kColsSplits; splits++) {
            const int per = (w.KT + splits - 1) / splits;
            if (splits > 1 && (per < 4 || (w.KT + per - 1) / per != splits || (splits - 1) * tiles > num_cus ||
                               (size_t)splits * M * w.N * 4 > part_bytes)) continue;
            const float rounds = (float)((tiles * splits + num_cus - 1) / num_cus);
            const float us = rounds * (f.fixed[mode] + f.per_kt[mode] * (float)per) +
                             (splits > 1 ? 2.2f + 0.5f * ((float)splits + 0.5f) * out_mb : 0.27f * out_mb);
            if (us < best.us) best = {f.rb, f.cs, splits, false, us};
        }
    }
    return best;
}

// K of more than 64 tiles, up to 128 rows, where the tiled kernels split K three ways or more: that split, eight waves of one strip
// that take whole K tiles of their share in the tiled kernels' order - their bits - and all shares as slabs.  A CU then takes in one
// share of X for eight strips.  (Sums in another order are up to 5 % quicker, but through 32 layers of bf16 activations two such runs
// end 1.3 % apart.)  us per call with all passes, against waves of the few-row kernel with a share each (X once per two strips): 14336 -> 4096
// bf16 at 45 / 64 / 100 / 128 rows 25.8 / 28.7 / 33.3 / 35.8 -> 23.5 / 24.9 / 30.9 / 33.0, Q8 29.1 / 32.7 / 38.9 / 42.8 -> 25.0 / 26.5 / 32.3 / 34.2, fp32 at 24
// rows 20.9 -> 20.5; 14336 -> 8192 35.1 / 41.1 / 45.5 / 49.3 -> 30.7 / 33.7 / 44.4 / 46.5; 12288 -> 6144 SwiGLU at 45 / 64 rows 33.8 / 37.7 -> 26.4 / 28.2.
// Two row tiles beyond 64 rows where both fit one round: 9216 -> 1030 at 100 / 128 rows 22.9 / 24.8 -> 19.7 / 21.0.
ColsPlan plan_gemm_cols_long_k(const WeightView& w, int M, int num_cus, const Epilogue& epi)
{
    const ColsPlan none = {0, 0, 1, false, 0.f};
    const bool pairs = epi.kind == kEpiSwiglu;
    if (M <= 16 || M > 128 || w.KT <= 64) return none;
    if ((w.NT % 7 == 0 && !pairs) || (!pairs && (w.NT + 3) / 4 * 4 >= 3 * num_cus)) return none;
    const int tiles = (w.NT + 7) / 8;
    int shares = std::min(kColsSplits, num_cus / tiles);                  // the tiled kernels' K split
    if (shares < 3) return none;
    const int per = (w.KT + shares - 1) / shares;
    shares = (w.KT + per - 1) / per;
    const int need = (M + 15) / 16;
    const int rb = need <= 2 ? 2 : need <= 4 ? need : 2 * tiles * shares <= num_cus ? (need <= 6 ? 3 : 4) : need <= 6 ? 6 : 8;
    return {rb, 1, shares, true, 0.f};
}

hipError_t launch_gemm_cols(const WeightView& w, const void* x, bool raw, int mode, int M, void* y, int ydt, const ColsPlan& plan, const Epilogue& epi,
                            const float* ssq_part, int ssq_blocks, const float* unscale, float* part, hipStream_t st)
{
    const NormStats ns = {ssq_part, ssq_blocks, unscale};
    auto go = [&](auto bits, auto md, auto r, auto c, auto kh) {
        constexpr int B = decltype(bits)::value, MD = decltype(md)::value, R = decltype(r)::value, C = decltype(c)::value, KH = decltype(kh)::value;
        return raw ? launch_cols_t<B, MD, R, C, KH, true>(w, x, M, y, ydt, plan.splits, epi, ns, part, st)
                   : launch_cols_t<B, MD, R, C, KH, false>(w, x, M, y, ydt, plan.splits, epi, ns, part, st);
    };
    using i0 = std::integral_constant<int, 0>;
    using i1 = std::integral_constant<int, 1>;
    using i2 = std::integral_constant<int, 2>;
    using i3 = std::integral_constant<int, 3>;
    using i4 = std::integral_constant<int, 4>;
    using i6 = std::integral_constant<int, 6>;
    using i8 = std::integral_constant<int, 8>;
    if (plan.whole_tiles) {
        auto whole = [&](auto bits) {
            if (plan.rb == 2) return go(bits, i0{}, i2{}, i1{}, i1{});
            if (plan.rb == 3) return go(bits, i0{}, i3{}, i1{}, i1{});
            if (plan.rb == 4) return go(bits, i0{}, i4{}, i1{}, i1{});
            if (plan.rb == 6) return go(bits, i0{}, i6{}, i1{}, i1{});
            return go(bits, i0{}, i8{}, i1{}, i1{});
        };
        return w.bits == 4 ? whole(i4{}) : whole(i8{});
    }
    auto rows = [&](auto bits, auto md, auto cs) {
        if (plan.rb == 3) return go(bits, md, i3{}, cs, i2{});
        if (plan.rb == 4) return go(bits, md, i4{}, cs, i2{});
        if (plan.rb == 6) return go(bits, md, i6{}, cs, i2{});
        if (plan.rb == 8) return go(bits, md, i8{}, cs, i2{});
        return hipErrorInvalidValue;
    };
    auto shape = [&](auto bits, auto md) { return plan.cs == 1 ? rows(bits, md, i1{}) : rows(bits, md, i2{}); };
    if (w.bits == 4) return mode == 0 ? shape(i4{}, i0{}) : mode == 1 ? shape(i4{}, i1{}) : shape(i4{}, i2{});
    return mode == 0 ? shape(i8{}, i0{}) : mode == 1 ? shape(i8{}, i1{}) : shape(i8{}, i2{});
}

}  // namespace cybq
