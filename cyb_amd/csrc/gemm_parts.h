// gemm_parts.h - pieces shared by the prefill kernels (gemm.hip, gemm_rows.hip): output element
// access, the row statistics of a folded norm / widened activations, a weight tile in registers,
// the MFMA wrapper and the epilogue that writes a wave's finished sums.  Included inside
// namespace cybq { namespace { ... } } of each translation unit.
#ifndef CYBQ_GEMM_PARTS_H
#define CYBQ_GEMM_PARTS_H

typedef float float2_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ void store_out_g(void* y, int ydt, int64_t idx, float v)
{
    if (ydt == kF32) reinterpret_cast<float*>(y)[idx] = v;
    else if (ydt == kF16) reinterpret_cast<_Float16*>(y)[idx] = (_Float16)v;
    else reinterpret_cast<uint16_t*>(y)[idx] = f32_to_bf16_bits(v);
}


__device__ __forceinline__ float load_out_g(const void* p, int dt, int64_t idx)
{
    if (dt == kF32) return reinterpret_cast<const float*>(p)[idx];
    if (dt == kF16) return (float)reinterpret_cast<const _Float16*>(p)[idx];
    return __builtin_bit_cast(float, (uint32_t)reinterpret_cast<const uint16_t*>(p)[idx] << 16);
}

// Folded RMSNorm on the prefill path: the staging pass leaves, per row of the chunk, `nblk`
// partial sums of squares; rstd of a row adds them in index order.
// `unscale` (FAST mode with widened activations): the power of two every staged row was
// divided by on its way to f16, to be multiplied back onto the finished sums.
struct NormStats {
    const float* part;
    int nblk;
    const float* unscale;
};

__device__ __forceinline__ float rstd_of(const NormStats& ns, int row, int K, float eps)
{
    float t = 0.f;
    for (int j = 0; j < ns.nblk; j++) t += ns.part[(int64_t)row * ns.nblk + j];
    return 1.0f / sqrtf(t / (float)K + eps);
}

// what a finished sum of row `row` is multiplied by before the epilogue
__device__ __forceinline__ float row_factor(const NormStats& ns, bool norm, int row, int K, float eps)
{
    float f = ns.unscale ? ns.unscale[row] : 1.0f;
    if (norm) f *= rstd_of(ns, row, K, eps);
    return f;
}

// The same from a row's two statistics, one row per lane, asked for ahead of where they are used.  Behind the K loop with four rows per lane
// they were eight loads, eight square roots and divisions and a trip to memory with nothing left to hide it (and the residual another one
// per row block).  us per call before / after, bf16: 4096 -> 6144 with a norm at 512 rows 39.5 / 36.8, 4096 -> 28672 norm + SwiGLU 117.2 / 114.3,
// 4096 -> 4096 with a residual 30.5 / 29.3; at 45 rows 13.6 / 12.9, 26.4 / 25.3, 10.5 / 10.3; results bit for bit.  `any` is a readable
// address: what has no place in the call is loaded from there and not used.
struct RowStats {
    float unscale, ssq;
};

__device__ __forceinline__ RowStats load_row_stats(const NormStats& ns, bool norm, int row, const void* any)
{
    const float* const spare = static_cast<const float*>(any);
    const bool one = norm && ns.nblk == 1;
    const RowStats s = {ns.unscale ? ns.unscale[row] : *spare, one ? ns.part[row] : *spare};
    return s;
}

__device__ __forceinline__ float row_factor(const RowStats& s, const NormStats& ns, bool norm, int row, int K, float eps)
{
    float f = ns.unscale ? s.unscale : 1.0f;
    if (norm) f *= ns.nblk == 1 ? 1.0f / sqrtf(s.ssq / (float)K + eps) : rstd_of(ns, row, K, eps);
    return f;
}

// 16 bytes per lane from base + off (the lane's own) to LDS bytes lds_off + 16 * lane, past the registers
__device__ __forceinline__ void copy_to_lds(uint32_t lds_off, const void* base, uint32_t off)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_off)), "v"(off), "s"(base));
}

template <int BITS>
struct WRegs {               // one native weight tile as loaded by one lane, and its 4 group scales
    u32x4_t q[BITS == 4 ? 1 : 2];
    u32x2_t s;
};

template <int BITS>
__device__ __forceinline__ void load_wtile(WRegs<BITS>& r, const WeightView& w, int64_t tile, int lane)
{
    const u32x4_t* qp = tile_q<BITS>(w, tile);
    r.q[0] = qp[lane];
    if (BITS == 8) r.q[BITS == 4 ? 0 : 1] = qp[64 + lane];
    r.s = tile_s<BITS>(w, tile)[lane & 15];
}

template <int XBF>
__device__ __forceinline__ float4_t mma(const Frag16& a, const Frag16& b, float4_t c)
{
    if (XBF) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, b.b, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a.h, b.h, c, 0, 0, 0);
}

// The residual under a wave's output tile, four elements per piece as write_rows stores them (16-bit types: in the first two words).
// LATE: each piece when it is added.
template <int MF, int NF, bool LATE = false>
struct Residual {
    u32x4_t v[LATE ? 1 : MF][LATE ? 1 : NF];
};

__device__ __forceinline__ u32x4_t residual_piece(const Epilogue& epi, int ydt, int64_t at)
{
    if (ydt == kF32) return *reinterpret_cast<const u32x4_t*>(static_cast<const float*>(epi.residual) + at);
    const u32x2_t r = *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(epi.residual) + at);
    return (u32x4_t){r[0], r[1], 0u, 0u};
}

// whether write_rows stores whole pieces: output rows (and the residual's) start on a 16-byte boundary, 8 for 16-bit outputs
__device__ __forceinline__ bool rows_in_pieces(int N, const void* y, int ydt, const Epilogue& epi)
{
    const uintptr_t amask = ydt == kF32 ? 15u : 7u;
    return (N & 3) == 0 && (reinterpret_cast<uintptr_t>(y) & amask) == 0 &&
           (epi.kind != kEpiAdd || (reinterpret_cast<uintptr_t>(epi.residual) & amask) == 0);
}

// requests it (nothing where write_rows goes element by element)
template <int MF, int NF, bool LATE>
__device__ __forceinline__ void load_residual(Residual<MF, NF, LATE>& res, int m0, int nt0, int M, int N, const void* y, int ydt, const Epilogue& epi, int lane)
{
    if (LATE || epi.kind != kEpiAdd || !rows_in_pieces(N, y, ydt, epi)) return;
    constexpr int V4 = NF * 4;
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int k = 0; k < NF; k++) {
            const int p = lane + k * 64, row = p / V4, m = m0 + i * 16 + row, n = nt0 * 16 + (p - row * V4) * 4;
            if (m < M && n < N) res.v[LATE ? 0 : i][LATE ? 0 : k] = residual_piece(epi, ydt, (int64_t)m * N + n);
        }
}

// The finished sums of one wave (MF row blocks x NF column blocks, lane = column, four rows per lane;
// first row m0, first column block nt0) -> y, with the residual-add epilogue (res: load_residual's).  `stg`: 16 x NF*16
// floats of LDS that belong to this wave.
template <int MF, int NF, bool LATE>
__device__ __forceinline__ void write_rows(const float4_t (&acc)[MF][NF], const Residual<MF, NF, LATE>& res, float* stg, int m0, int nt0, int M, int N, void* y,
                                           int ydt, float out_scale, const Epilogue& epi, int lane)
{
    const int row16 = lane & 15, oct = lane >> 4;
    // Output rows that start on a 16-byte boundary (8 for 16-bit outputs): the accumulators (lane =
    // column, four rows per lane) go through LDS - the operand buffers are free after the last K
    // tile's barrier, a wave's share of them holds one of its row blocks - and leave four
    // elements per lane, 64 lanes writing whole runs of a row instead of 64-byte pieces of four rows.
    if (rows_in_pieces(N, y, ydt, epi)) {
        constexpr int ROWF = NF * 16;               // floats of a tile row
        constexpr int V4 = ROWF / 4;                // four-element pieces of a tile row
        const float4_t* stg4 = reinterpret_cast<const float4_t*>(stg);
#pragma unroll
        for (int i = 0; i < MF; i++) {
#pragma unroll
            for (int f = 0; f < NF; f++)
#pragma unroll
                for (int r = 0; r < 4; r++) stg[(oct * 4 + r) * ROWF + f * 16 + row16] = acc[i][f][r] * out_scale;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int k = 0; k < NF; k++) {
                const int p = lane + k * 64;
                const int row = p / V4, c4 = p - row * V4;
                const int m = m0 + i * 16 + row, n = nt0 * 16 + c4 * 4;
                if (m < M && n < N) {
                    float4_t v = stg4[p];
                    const int64_t at = (int64_t)m * N + n;
                    if (ydt == kF32) {
                        if (epi.kind == kEpiAdd)
                            v += LATE ? *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(epi.residual) + at)
                                      : __builtin_bit_cast(float4_t, res.v[LATE ? 0 : i][LATE ? 0 : k]);
                        *reinterpret_cast<float4_t*>(reinterpret_cast<float*>(y) + at) = v;
                    } else {
                        if (epi.kind == kEpiAdd) {
                            u32x2_t add = {};
                            if constexpr (LATE) {
                                add = *reinterpret_cast<const u32x2_t*>(reinterpret_cast<const uint16_t*>(epi.residual) + at);
                            } else {
                                add[0] = res.v[i][k][0];
                                add[1] = res.v[i][k][1];
                            }
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const uint32_t h = (e & 1) ? add[e >> 1] >> 16 : add[e >> 1] & 0xffffu;
                                v[e] += ydt == kF16 ? f16_bits_to_f32(h) : __builtin_bit_cast(float, h << 16);
                            }
                        }
                        u32x2_t o;
                        if (ydt == kF16) {
                            const half2_t a = {(_Float16)v[0], (_Float16)v[1]}, b = {(_Float16)v[2], (_Float16)v[3]};
                            o = (u32x2_t){as_u32(a), as_u32(b)};
                        } else {
                            o = (u32x2_t){(uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16),
                                          (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16)};
                        }
                        *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(y) + at) = o;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < MF; i++)
#pragma unroll
        for (int f = 0; f < NF; f++) {
            const int n = (nt0 + f) * 16 + row16;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + i * 16 + oct * 4 + r;
                if (m < M && n < N) {
                    float v = acc[i][f][r] * out_scale;
                    if (epi.kind == kEpiAdd) v += load_out_g(epi.residual, ydt, (int64_t)m * N + n);
                    store_out_g(y, ydt, (int64_t)m * N + n, v);
                }
            }
        }
}

template <int MF, int NF>
__device__ __forceinline__ void write_rows(const float4_t (&acc)[MF][NF], float* stg, int m0, int nt0, int M, int N, void* y, int ydt,
                                           float out_scale, const Epilogue& epi, int lane)
{
    Residual<MF, NF, (MF > 2)> res;                // (no registers for all of it next to so many sums)
    load_residual(res, m0, nt0, M, N, y, ydt, epi, lane);
    write_rows(acc, res, stg, m0, nt0, M, N, y, ydt, out_scale, epi, lane);
}

#endif
