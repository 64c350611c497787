// gemv_stream.hip - 3 .. 32 rows of 16-bit activations on wide outputs: workgroups that stay and stream strips.
//
// Bound by HBM.  The batched-rows kernel of gemv.hip gives a workgroup one group of strips: it loads its rows of x,
// waits for them, streams two to eight strips, exchanges, ends - and on outputs with several rounds of workgroups per CU
// x is loaded again in every round (27 rows of K = 2560 are 138 KB, two Q8 strips 87 KB).  Here the grid is one
// workgroup per CU and a wave keeps the MFMA operands of its K tiles of x in registers for the whole call.  Strips come
// in pairs (a gate / up pair, or two neighbours): as soon as a weight tile has been multiplied, the same tile of
// the next pair is requested into its registers, so between half and all of a pair per wave is always on its
// way.  The waves' partial sums of a pair meet in one of two LDS areas - one barrier per pair - and the waves that
// add them up do so while the others are already multiplying.
//
// Which wave owns which K tile, and the order of every sum, is that of gemv.hip's kernel with the same waves, with its plain
// operands (f16 rows: exact integers) or, where that kernel shares a shape by row count and walks it by tile, with those of that
// walk (TILE): a row's bits do not depend on the batch of 3 .. 32 rows it travels in.  (With a folded norm the squares are summed as
// loaded, so they do: 3 .. 8, 9 .. 32 rows here, up to 4, 8, 16 in gemv.hip.  The operands are the plain ones then: by tile 4096 -> 32768 at 8 f16 rows takes 16.2 us
// instead of 18.0, but its sums carry the bias: 5e-7 of relative L2 against float64 where the integers have 1e-7.)
// (f16 rows, us per call before -> after: Q8 2560 -> 32003 at 8 / 27 rows 20.1 -> 16.1, 36.4 -> 17.9 (12.4 at 7 TB/s); Q4 2048 ->
// 20000 with a norm 17.6 -> 8.2, 22.0 -> 10.6; Q4 4096 -> 128256 at 27 rows 92.6 -> 66.2.  Two or three pairs ahead
// instead of one changed nothing on long outputs and cost 2 us on short ones.)
#include "gemv_parts.h"

namespace cybq {

namespace {

// TS: K tiles a wave owns at most (kt = wave, wave + 8, ...).  MB: blocks of 16 rows.
// S: strips of a step, 2 or (where the registers do not hold two) 1.
// TILE (Q4): the operands and the order of sums of the batched-rows kernel's walk by tile - the product of the activations
// with the constant that takes the bias off comes first, one for all strips of a step, and f16 activations meet subnormal
// weights (gemv_rows_kernel, SUB).  For shapes where that kernel has the calls with fewer, or more, rows: a row keeps its bits.
template <int BITS, int XMODE, int W, int TS, int MB, int XR, bool NORM, int S, bool TILE>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void gemv_stream_kernel(const uint8_t* __restrict__ wbase, const uint16_t* __restrict__ x, const void* __restrict__ gamma, int KT, int K, int NT,
                        int M, int gamma_dt, int steps, int N, void* __restrict__ y, int ydt, Epilogue epi)
{
    static_assert(W == 4 || W == 8, "a wave finishes output registers of one row in four");
    static_assert(!TILE || (BITS == 4 && !NORM), "by tile: Q4, no folded norm");
    const WeightView w = {wbase, N, K, NT, KT, BITS};
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const uint32_t magic = (BITS == 4 && XMODE == XBF16) ? q4_magic_vgpr_bf16() : q4_magic_vgpr();
    const int tid = threadIdx.x, lane = tid & 63, oct = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int AREA = S * MB * W * 4 * 64;              // floats of one exchange area
    float* const red = reinterpret_cast<float*>(smem);
    float* const ssq_part = red + 2 * AREA;                     // [wave][row]

    // my K tiles of x as MFMA operands (as in gemv_rows_kernel: a load covers XR rows x P neighbouring 16 B pieces, then
    // the pieces cross lanes), behind the gamma of those tiles: 8 values in each of 16 lanes, fp32 4 in each of 32
    constexpr int P = 64 / XR, L = 16 / P, GPL = 4 / L;         // pieces per row and load, loads per tile, groups per load
    static_assert(MB == 1 || XR == 16, "two row blocks: full loads");
    const bool gamma_h = NORM && XMODE == XF16 && gamma_dt == kF16;
    const bool gamma_f32 = NORM && gamma_dt == kF32;
    u32x4_t graw[NORM ? TS : 1];
    if constexpr (NORM) {
        const int g_count = gamma_f32 ? 4 : 8, g_first = (lane & (gamma_f32 ? 31 : 15)) * g_count;
#pragma unroll
        for (int u = 0; u < TS; u++)
            graw[u] = *reinterpret_cast<const u32x4_t*>(static_cast<const uint8_t*>(gamma) +
                                                        ((size_t)min(min(wv + W * u, KT - 1) * kTileK + g_first, K - g_count) << (gamma_f32 ? 2 : 1)));
    }
    Frag16 a[MB][TS][4];
    float ssq[MB] = {};
    const int r0 = min(lane / P, M - 1), r1 = min(16 + lane / P, M - 1);
    const uint16_t* const x0 = x + (int64_t)r0 * K + (lane % P) * 8;
    const int64_t to_second = MB > 1 ? (int64_t)(r1 - r0) * K : 0;
    const int klast = K - 8 - (lane % P) * 8;
    const int from_lane = ((((lane & 15) & (XR - 1)) * P) | oct) << 2;
#pragma unroll
    for (int u = 0; u < TS; u++) {
        const int kt = min(wv + W * u, KT - 1);
#pragma unroll
        for (int h = 0; h < L; h++)
#pragma unroll
            for (int b = 0; b < MB; b++)
                a[b][u][h].u = *reinterpret_cast<const u32x4_t*>(x0 + b * to_second + (XR == 16 ? min(kt * kTileK + h * 32, K - 32)
                                                                                               : min(kt * kTileK + h * (GPL * 32), klast)));
    }

    const int step0 = blockIdx.x, stride = gridDim.x;
    auto run = [&](auto tiles) {
        constexpr int TV = decltype(tiles)::value;             // tiles this wave owns: TS or TS - 1
        TileRegs<BITS> buf[S][TV];
        auto request = [&](TileRegs<BITS>& r, int step, int s, int u) {
            load_tile<BITS>(r, w, (int64_t)min(S * step + s, NT - 1) * KT + wv + W * u, lane);
        };
#pragma unroll
        for (int u = 0; u < TV; u++)
#pragma unroll
            for (int s = 0; s < S; s++) request(buf[s][u], step0, s, u);

        if constexpr (NORM) {
            // my tiles' gamma -> my LDS area, read back piece by piece: no other wave is involved
            uint8_t* const gamma_lds = reinterpret_cast<uint8_t*>(ssq_part + MB * W * 16 + (size_t)wv * TS * kTileK);
            if (gamma_h) {
                if (lane < 16) {
#pragma unroll
                    for (int u = 0; u < TV; u++) reinterpret_cast<u32x4_t*>(gamma_lds)[u * 16 + lane] = graw[u];
                }
            } else if (gamma_f32) {
                if (lane < 32) {
#pragma unroll
                    for (int u = 0; u < TV; u++) reinterpret_cast<u32x4_t*>(gamma_lds)[u * 32 + lane] = graw[u];
                }
            } else if (lane < 16) {
                const bool gh = gamma_dt == kF16;
#pragma unroll
                for (int u = 0; u < TV; u++) {
                    float g[8];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const half2_t h = as_h2(graw[u][i]);
                        g[2 * i] = gh ? (float)h.x : __builtin_bit_cast(float, graw[u][i] << 16);
                        g[2 * i + 1] = gh ? (float)h.y : __builtin_bit_cast(float, graw[u][i] & 0xffff0000u);
                    }
                    reinterpret_cast<float4_t*>(gamma_lds)[u * 32 + 2 * lane] = (float4_t){g[0], g[1], g[2], g[3]};
                    reinterpret_cast<float4_t*>(gamma_lds)[u * 32 + 2 * lane + 1] = (float4_t){g[4], g[5], g[6], g[7]};
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            auto norm_all = [&](auto packed) {
                constexpr bool GH = decltype(packed)::value;
#pragma unroll
                for (int u = 0; u < TV; u++)
#pragma unroll
                    for (int h = 0; h < L; h++) {
                        const int kt = wv + W * u;
                        const int k0 = kt * kTileK + h * (GPL * 32);
                        const int kp = k0 + (lane % P) * 8;             // my piece (one past K repeats one inside: not counted)
                        const int kk = (XR == 16 ? min(k0, K - 32) + (lane % P) * 8 : min(kp, K - 8)) - kt * kTileK + u * kTileK;
                        const GammaPiece g = gamma_piece<GH>(gamma_lds, kk);
#pragma unroll
                        for (int b = 0; b < MB; b++) norm_piece<XMODE, GH>(a[b][u][h].u, g, kp < K, ssq[b]);
                    }
            };
            if constexpr (XMODE == XF16) {
                if (gamma_h) norm_all(std::true_type{});
                else norm_all(std::false_type{});
            } else norm_all(std::false_type{});
        }
#pragma unroll
        for (int b = 0; b < MB; b++)
#pragma unroll
            for (int u = 0; u < TV; u++) {
                u32x4_t raw[L];
#pragma unroll
                for (int h = 0; h < L; h++) raw[h] = a[b][u][h].u;
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int p = 0; p < 4; p++)
                        a[b][u][j].u[p] = (uint32_t)__builtin_amdgcn_ds_bpermute(from_lane + (j % GPL) * 16, (int)raw[j / GPL][p]);
            }

        float scale[MB];                                        // 1 / rms of the rows whose outputs this wave finishes
#pragma unroll
        for (int b = 0; b < MB; b++) scale[b] = TILE && XMODE == XF16 ? kSubUnscale : 1.f;
        if constexpr (NORM) {
            // P lanes hold a row's pieces
#pragma unroll
            for (int b = 0; b < MB; b++) {
                ssq[b] += lane_cross<0xB1>(ssq[b]);
                ssq[b] += lane_cross<0x4E>(ssq[b]);
                if (P >= 8) ssq[b] += lane_cross<0x141>(ssq[b]);
                if (P >= 16) ssq[b] += lane_cross<0x140>(ssq[b]);
                if (lane % P == 0) ssq_part[(b * W + wv) * 16 + lane / P] = ssq[b];
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // (output register r of a wave's accumulators is row 4 * oct + r, and every register it finishes has r = wave % 4)
#pragma unroll
            for (int b = 0; b < MB; b++) {
                float t = 0.f;
#pragma unroll
                for (int k = 0; k < W; k++) t += ssq_part[(b * W + k) * 16 + 4 * oct + (wv & 3)];
                scale[b] = __builtin_amdgcn_rsqf(fmaf(t, __builtin_amdgcn_rcpf((float)K), epi.eps));
            }
        }

        float* area = red;
        // (the last step is code of its own: where requests hang on a condition the compiler waits for more than it has to)
        auto step = [&](int i, auto more) {
            float acc[S][MB][4];
#pragma unroll
            for (int s = 0; s < S; s++)
#pragma unroll
                for (int b = 0; b < MB; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[s][b][r] = 0.f;
#pragma unroll
            for (int u = 0; u < TV; u++) {
                float4_t bias[TILE ? MB : 1][4];
                if constexpr (TILE) {
#pragma unroll
                    for (int b = 0; b < MB; b++) tile_bias<XMODE>(a[b][u], bias[b]);
                }
#pragma unroll
                for (int s = 0; s < S; s++) {
                    Frag16 bop[4];
                    if constexpr (TILE && XMODE == XF16) tile_operands_sub(buf[s][u], bop);
                    else tile_operands<BITS, XMODE>(buf[s][u], magic, bop);
                    const u32x2_t sc = buf[s][u].s;
                    if constexpr (decltype(more)::value) request(buf[s][u], i + stride, s, u);
                    float4_t d[MB][4];
#pragma unroll
                    for (int b = 0; b < MB; b++) {
                        if constexpr (TILE) tile_multiply_from<XMODE>(a[b][u], bop, bias[b], d[b]);
                        else tile_multiply<BITS, XMODE>(a[b][u], bop, d[b]);
                    }
#pragma unroll
                    for (int b = 0; b < MB; b++) {
                        if constexpr (TILE && XMODE == XF16) tile_accum_sub(sc, d[b], acc[s][b]);
                        else tile_accum<4>(sc, d[b], acc[s][b]);
                    }
                    if (MB == 2) __builtin_amdgcn_sched_barrier(0);          // (unpacking ahead would spill)
                }
            }
#pragma unroll
            for (int s = 0; s < S; s++)
#pragma unroll
                for (int b = 0; b < MB; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) area[(((s * MB + b) * W + wv) * 4 + r) * 64 + lane] = acc[s][b][r];
            // the exchange only needs the LDS writes to have landed: requests stay in flight across the barrier
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (S == 2 && epi.kind == kEpiSwiglu) {
                const int n_out = N >> 1;
                for (int p = wv; p < MB * 4; p += W) {
                    const int r = p & 3, b = p >> 2;
                    const float sb = MB == 1 || b == 0 ? scale[0] : scale[MB - 1];
                    const float g = sum_partials(area + (b * W * 4 + r) * 64 + lane, W, 4 * 64) * sb;
                    const float v = sum_partials(area + ((MB + b) * W * 4 + r) * 64 + lane, W, 4 * 64) * sb;
                    const int n = i * 16 + (lane & 15), m = 16 * b + 4 * oct + r;
                    if (m < M && n < n_out) store_out(y, ydt, (int64_t)m * n_out + n, silu_mul(g, v));
                }
            } else {
                for (int p = wv; p < S * MB * 4; p += W) {
                    const int r = p & 3, b = (p >> 2) % MB, s = (p >> 2) / MB;
                    const float sb = MB == 1 || b == 0 ? scale[0] : scale[MB - 1];
                    const float v = sum_partials(area + ((s * MB + b) * W * 4 + r) * 64 + lane, W, 4 * 64) * sb;
                    const int n = (S * i + s) * 16 + (lane & 15), m = 16 * b + 4 * oct + r;
                    if (m < M && n < N) emit(y, ydt, epi, (int64_t)m * N + n, v);
                }
            }
            area = area == red ? red + AREA : red;             // (the barrier of the next pair separates its readers from the one after)
        };
        int i = step0;
        for (; i + stride < steps; i += stride) step(i, std::true_type{});
        step(i, std::false_type{});
    };
    if (wv + W * (TS - 1) < KT) run(std::integral_constant<int, TS>{});
    else run(std::integral_constant<int, TS - 1>{});
}

template <int BITS, int XMODE, int W, int TS, int MB, int XR, bool NORM, bool TILE = false>
hipError_t launch_k(const WeightView& w, const void* x, int M, void* y, int ydt, int num_cus, const Epilogue& epi, hipStream_t st)
{
    constexpr int S = (TS == 4 && MB == 2) ? 1 : 2;
    const int steps = (w.NT + S - 1) / S;
    // two exchange areas, the waves' sums of squares, each wave's tiles of gamma as fp32
    constexpr int lds = (2 * S * MB * W * 4 * 64 + MB * W * 16 + (NORM ? W * TS * kTileK : 0)) * (int)sizeof(float);
    auto kern = gemv_stream_kernel<BITS, XMODE, W, TS, MB, XR, NORM, S, TILE>;
    if constexpr (lds > 64 * 1024) (void)LdsRequest<&gemv_stream_kernel<BITS, XMODE, W, TS, MB, XR, NORM, S, TILE>, lds>::registered;
    hipLaunchKernelGGL(kern, dim3((unsigned)min(steps, num_cus * (8 / W))), dim3(W * 64), lds, st, w.base, static_cast<const uint16_t*>(x), epi.gamma,
                       w.KT, w.K, w.NT, M, epi.gamma_dt, steps, w.N, y, ydt, epi);
    return hipGetLastError();
}

// (the x load pattern follows the batch: up to 4, up to 8, up to 16 rows per load.  f16 rows, 4 rows, eight / four to a load: 4096 -> 6144
// 5.4 / 4.9 us.  With a folded norm the squares are summed as loaded: eight to a load, so that 3 .. 8 rows share a row's bits; Q8 8.9 / 8.5, bf16 9.6 / 9.0)
template <int BITS, int XMODE, int W, int TS, bool NORM, bool TILE>
hipError_t launch_m(const WeightView& w, const void* x, int M, void* y, int ydt, int num_cus, const Epilogue& epi, hipStream_t st)
{
    // (17 .. 32 rows: a norm only of f16 rows and up to three tiles per wave; by tile never with four waves)
    if (M > 16) {
        if constexpr (!NORM) return launch_k<BITS, XMODE, W, TS, 2, 16, false, TILE && W == 8>(w, x, M, y, ydt, num_cus, epi, st);
        else if constexpr (TS < 4 && XMODE == XF16) return launch_k<BITS, XMODE, W, TS, 2, 16, true>(w, x, M, y, ydt, num_cus, epi, st);
        else return hipErrorInvalidValue;        // gemv_stream_serves() said no
    }
    if constexpr (W == 8) {
        if constexpr (!NORM) {
            if (M <= 4) return launch_k<BITS, XMODE, W, TS, 1, 4, false, TILE>(w, x, M, y, ydt, num_cus, epi, st);
        }
        if (M <= 8) return launch_k<BITS, XMODE, W, TS, 1, 8, NORM, TILE>(w, x, M, y, ydt, num_cus, epi, st);
    }
    return launch_k<BITS, XMODE, W, TS, 1, 16, NORM, TILE>(w, x, M, y, ydt, num_cus, epi, st);
}

// the wave count the batched-rows kernel gives these K
int waves_of(const WeightView& w) { return w.KT < 16 ? 4 : 8; }
int tiles_per_wave(const WeightView& w) { return (w.KT + waves_of(w) - 1) / waves_of(w); }

// seven strips per CU, or eight and more: the batched-rows kernel goes strip by strip there
bool is_widest(const WeightView& w, int num_cus) { return w.NT >= 8 * num_cus || w.NT == 7 * num_cus; }

// Q4, four K tiles per wave: whether the batched-rows kernel's workgroups (four strips, or two) come in nearly full rounds.  It walks
// such a shape by tile (gemv_rows_kernel, BY_TILE), and so does this kernel then, whichever of the two has a call: a row keeps its bits.
bool rows_kernel_by_tile(const WeightView& w, int num_cus)
{
    if (w.bits != 4 || waves_of(w) != 8 || tiles_per_wave(w) != 4 || is_widest(w, num_cus)) return false;
    const int ns = (w.NT + num_cus / 2) / num_cus >= 3 ? 4 : 2;
    const int groups = (w.NT + ns - 1) / ns, rounds = (groups + num_cus - 1) / num_cus;
    return groups * 5 >= rounds * num_cus * 4;
}

// Whether the batched-rows kernel is the quicker one up to 16 rows.  Without a norm: nine rows or more where its workgroups are one nearly
// full round of four strips, and, but for pairs of bf16 rows, the widest outputs.  It gives every wave four K tiles to walk whether they are there
// or not, so a shorter K is never its.  us per call, this kernel / that one, f16 rows (bf16).  K = 4096: 14336 at 4 / 8 / 16 rows 8.3 / 8.3,
// 8.5 / 8.5, 9.7 / 9.0 (8.4 / 8.4, 9.0 / 9.0, 10.3 / 9.4), 16384 8.9 / 8.7, 9.0 / 9.7, 10.5 / 9.6, 28672 15.7 / 14.6, pairs at 4 / 8 / 16
// rows 16.4 / 14.6, 16.9 / 15.1, 16.7 / 16.0 (14.5 / 14.6, 14.7 / 16.0, 15.9 / 16.3), of 128256 57.1 / 51.1, 58.5 / 53.2, 56.3 / 57.5 (49.6 / 52.7,
// 51.6 / 56.4, 52.2 / 59.2).  K = 3456: 14336 at 8 / 16 rows 7.4 / 8.6, 8.9 / 8.9, 32768 14.2 / 15.0, 15.0 / 16.3; K = 3712: 28672 at 8 rows 15.3 / 14.2.
// With a norm: nearly full rounds, whatever the rows and K, and the widest outputs.
bool leaves_few_rows(const WeightView& w, int xdt, int M, int num_cus, const Epilogue& epi)
{
    if (w.bits != 4 || waves_of(w) != 8 || tiles_per_wave(w) != 4) return false;
    if (epi.gamma) {
        const int ns = (w.NT + num_cus / 2) / num_cus >= 3 ? 4 : 2;
        const int groups = (w.NT + ns - 1) / ns, rounds = (groups + num_cus - 1) / num_cus;
        return is_widest(w, num_cus) || groups * 4 >= rounds * num_cus * 3;
    }
    if (w.KT < 28) return false;
    if (is_widest(w, num_cus)) return epi.kind != kEpiSwiglu || xdt == kF16;
    return M > 8 && w.NT * 5 >= num_cus * 16 && w.NT <= num_cus * 4;
}

// By tile (TILE), besides those: gate / up pairs of four tiles per wave (17 .. 32 rows of them run the batched-rows kernel, by tile), but for
// f16 rows of the widest, which keep their integers (1.5e-7 against 8e-7 of relative L2).  f16 rows only in decode mode STREAM.  17 .. 32 rows
// go the same way and lose by it (4096 -> 14336 at 24 rows 11.8 / 12.7 us), so only the shapes whose rows that keeps together do.
bool by_tile(const WeightView& w, int xdt, int num_cus, bool exact_operands, const Epilogue& epi)
{
    if (w.bits != 4 || tiles_per_wave(w) != 4 || epi.gamma || (xdt == kF16 && exact_operands)) return false;
    if (epi.kind == kEpiSwiglu) return xdt == kBF16 || !is_widest(w, num_cus);
    return rows_kernel_by_tile(w, num_cus);
}

template <int BITS, int XMODE, int W, bool NORM>
hipError_t launch_w(const WeightView& w, const void* x, int M, void* y, int ydt, int num_cus, bool tile, const Epilogue& epi, hipStream_t st)
{
    const int ts = tiles_per_wave(w);
    if constexpr (BITS == 4 && !NORM) {
        if (ts == 4 && tile) return launch_m<BITS, XMODE, W, 4, NORM, true>(w, x, M, y, ydt, num_cus, epi, st);
    }
    if (ts == 2) return launch_m<BITS, XMODE, W, 2, NORM, false>(w, x, M, y, ydt, num_cus, epi, st);
    if (ts == 3) return launch_m<BITS, XMODE, W, 3, NORM, false>(w, x, M, y, ydt, num_cus, epi, st);
    if (ts == 4) return launch_m<BITS, XMODE, W, 4, NORM, false>(w, x, M, y, ydt, num_cus, epi, st);
    return hipErrorInvalidValue;         // gemv_stream_serves() said no
}

template <int BITS, int XMODE>
hipError_t launch_x(const WeightView& w, const void* x, int M, void* y, int ydt, int num_cus, bool tile, const Epilogue& epi, hipStream_t st)
{
    if (waves_of(w) == 4) {
        if (epi.gamma) return launch_w<BITS, XMODE, 4, true>(w, x, M, y, ydt, num_cus, tile, epi, st);
        return launch_w<BITS, XMODE, 4, false>(w, x, M, y, ydt, num_cus, tile, epi, st);
    }
    if (epi.gamma) return launch_w<BITS, XMODE, 8, true>(w, x, M, y, ydt, num_cus, tile, epi, st);
    return launch_w<BITS, XMODE, 8, false>(w, x, M, y, ydt, num_cus, tile, epi, st);
}

}  // namespace

bool gemv_stream_serves(const WeightView& w, int xdt, int M, int num_cus, const Epilogue& epi)
{
    if (M < 3 || M > 32 || xdt == kF32) return false;
    // two to four K tiles per wave: operands that fit the registers
    if (w.KT < 8 || w.KT > 32 || (int64_t)w.NT * 2 < (int64_t)num_cus * 3) return false;
    if (tiles_per_wave(w) == 4 && M > 16 && (epi.kind == kEpiSwiglu || epi.gamma)) return false;          // (pairs, or gamma, do not fit them)
    // (x * gamma is rounded to the operand type: the prefill kernels, which take these calls otherwise, round it to f16)
    if (M > 16 && epi.gamma && xdt == kBF16) return false;
    return M > 16 || !leaves_few_rows(w, xdt, M, num_cus, epi);
}

hipError_t launch_gemv_stream(const WeightView& w, const void* x, int xdt, int M, void* y, int ydt, int num_cus, bool exact_operands,
                              const Epilogue& epi, hipStream_t st)
{
    const bool tile = by_tile(w, xdt, num_cus, exact_operands, epi);
    if (w.bits == 4) {
        if (xdt == kF16) return launch_x<4, XF16>(w, x, M, y, ydt, num_cus, tile, epi, st);
        return launch_x<4, XBF16>(w, x, M, y, ydt, num_cus, tile, epi, st);
    }
    if (xdt == kF16) return launch_x<8, XF16>(w, x, M, y, ydt, num_cus, tile, epi, st);
    return launch_x<8, XBF16>(w, x, M, y, ydt, num_cus, tile, epi, st);
}

}  // namespace cybq
