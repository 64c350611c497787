// gemv_parts.h - pieces the decode kernels of gemv.hip and gemv_stream.hip share.
#pragma once

#include <type_traits>

#include "cybq_device.h"
#include "cybq_internal.h"

namespace cybq {

namespace {

constexpr int XF16 = 0, XBF16 = 1, XF32 = 2;

template <int BITS>
struct TileRegs {
    u32x4_t q[BITS == 4 ? 1 : 2];
    u32x2_t s;
};

template <int BITS>
__device__ __forceinline__ void load_tile(TileRegs<BITS>& t, const WeightView& w, int64_t tile, int lane)
{
    const u32x4_t* qp = tile_q<BITS>(w, tile);
    t.q[0] = __builtin_nontemporal_load(qp + lane);
    if (BITS == 8) t.q[BITS == 8 ? 1 : 0] = __builtin_nontemporal_load(qp + 64 + lane);
    t.s = __builtin_nontemporal_load(tile_s<BITS>(w, tile) + (lane & 15));
}

__device__ __forceinline__ void store_out(void* y, int ydt, int64_t idx, float v)
{
    if (ydt == kF32) reinterpret_cast<float*>(y)[idx] = v;
    else if (ydt == kF16) reinterpret_cast<_Float16*>(y)[idx] = (_Float16)v;
    else reinterpret_cast<uint16_t*>(y)[idx] = f32_to_bf16_bits(v);
}

__device__ __forceinline__ float load_out(const void* p, int dt, int64_t idx)
{
    if (dt == kF32) return reinterpret_cast<const float*>(p)[idx];
    if (dt == kF16) return (float)reinterpret_cast<const _Float16*>(p)[idx];
    return __builtin_bit_cast(float, (uint32_t)reinterpret_cast<const uint16_t*>(p)[idx] << 16);
}

// the same in two steps, to ask for an element ahead of its use: its bits, and their value
__device__ __forceinline__ uint32_t load_out_bits(const void* p, int dt, int64_t idx)
{
    if (dt == kF32) return reinterpret_cast<const uint32_t*>(p)[idx];
    return reinterpret_cast<const uint16_t*>(p)[idx];
}

__device__ __forceinline__ float out_value(uint32_t bits, int dt)
{
    return dt == kF32 ? __builtin_bit_cast(float, bits) : dt == kF16 ? f16_bits_to_f32(bits) : __builtin_bit_cast(float, bits << 16);
}

// one finished output element: residual add (fp32, before the single rounding to ydt), store
__device__ __forceinline__ void emit(void* y, int ydt, const Epilogue& epi, int64_t idx, float v)
{
    if (epi.kind == kEpiAdd) v += load_out(epi.residual, ydt, idx);
    store_out(y, ydt, idx, v);
}

template <int RMAX>
__device__ __forceinline__ void tile_accum(u32x2_t s, const float4_t d[4], float acc[RMAX])
{
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t sb = (j & 1) ? (s[j >> 1] >> 16) : (s[j >> 1] & 0xffffu);
        float sc = f16_bits_to_f32(sb);
#pragma unroll
        for (int r = 0; r < RMAX; r++) acc[r] = __builtin_fmaf(sc, d[j][r], acc[r]);
    }
}

// Sum of the waves' partial sums red[k * stride], k = 0 .. nwaves-1, added in wave
// order.  The reads go out eight at a time: one LDS round trip per eight waves
// instead of one per wave.  (Slots past nwaves add +0, which changes nothing: a sum
// that starts from +0 is never -0.)
__device__ __forceinline__ float sum_partials(const float* red, int nwaves, int stride)
{
    float v = 0.f;
    for (int k0 = 0; k0 < nwaves; k0 += 8) {
        float t[8];
#pragma unroll
        for (int i = 0; i < 8; i++) t[i] = red[min(k0 + i, nwaves - 1) * stride];
#pragma unroll
        for (int i = 0; i < 8; i++) v += (k0 + i < nwaves) ? t[i] : 0.f;
    }
    return v;
}

template <int BITS, int XMODE>
__device__ __forceinline__ void tile_operands(const TileRegs<BITS>& t, uint32_t magic, Frag16 (&b)[4])
{
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t bw[4];
        if (BITS == 4 && XMODE == XBF16) {
            unpack_q4_bf16_biased(t.q[0][2 * (j >> 1)], t.q[0][2 * (j >> 1) + 1], j & 1, magic, bw);
        } else if (XMODE == XBF16) {
            unpack_q8_bf16_biased(t.q[j >> 1][(j & 1) * 2], t.q[j >> 1][(j & 1) * 2 + 1], bw);
        } else {
            if (BITS == 4) unpack_q4_f16(t.q[0][2 * (j >> 1)], t.q[0][2 * (j >> 1) + 1], j & 1, magic, bw);
            else unpack_q8_f16(t.q[j >> 1][(j & 1) * 2], t.q[j >> 1][(j & 1) * 2 + 1], bw);
        }
        b[j].u = (u32x4_t){bw[0], bw[1], bw[2], bw[3]};
    }
}

template <int BITS, int XMODE>
__device__ __forceinline__ void tile_multiply(const Frag16 (&a)[4], const Frag16 (&b)[4], float4_t d[4])
{
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    Frag16 off;
    const uint32_t offw = BITS == 4 ? kBf16Neg136x2 : kBf16Neg128x2;
    off.u = (u32x4_t){offw, offw, offw, offw};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (XMODE == XBF16) {
            d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j].b, b[j].b, zero, 0, 0, 0);
            d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j].b, off.b, d[j], 0, 0, 0);
        } else d[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j].h, b[j].h, zero, 0, 0, 0);
    }
}

// ---- the walk by tile (Q4): one product of the activations with the constant(s) that take the bias off, the C operand of
// every strip's MFMAs.  f16 activations: subnormal weights, 1/16 for the odd groups on their scale, 2^22 on the final sums;
// bf16: the numbers 128 + u (tile_operands).
template <int XMODE>
__device__ __forceinline__ void tile_bias(const Frag16 (&a)[4], float4_t bias[4])
{
    const float4_t zero = {0.f, 0.f, 0.f, 0.f};
    Frag16 off, off_odd;
    const uint32_t offw = XMODE == XF16 ? kSubBiasL : kBf16Neg136x2, offw_odd = XMODE == XF16 ? kSubBiasH : offw;
    off.u = (u32x4_t){offw, offw, offw, offw};
    off_odd.u = (u32x4_t){offw_odd, offw_odd, offw_odd, offw_odd};
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if constexpr (XMODE == XF16) bias[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j].h, ((j & 1) ? off_odd : off).h, zero, 0, 0, 0);
        else bias[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j].b, off.b, zero, 0, 0, 0);
    }
}

__device__ __forceinline__ void tile_operands_sub(const TileRegs<4>& t, Frag16 (&b)[4])
{
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t bw[4];
        unpack_q4_sub(t.q[0][2 * (j >> 1)], t.q[0][2 * (j >> 1) + 1], j & 1, bw);
        b[j].u = (u32x4_t){bw[0], bw[1], bw[2], bw[3]};
    }
}

template <int XMODE>
__device__ __forceinline__ void tile_multiply_from(const Frag16 (&a)[4], const Frag16 (&b)[4], const float4_t bias[4], float4_t d[4])
{
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if constexpr (XMODE == XF16) d[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[j].h, b[j].h, bias[j], 0, 0, 0);
        else d[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[j].b, b[j].b, bias[j], 0, 0, 0);
    }
}

__device__ __forceinline__ void tile_accum_sub(u32x2_t s, const float4_t d[4], float acc[4])
{
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t sb = (j & 1) ? (s[j >> 1] >> 16) : (s[j >> 1] & 0xffffu);
        const float sf = (j & 1) ? f16_bits_to_f32(sb) * 0.0625f : f16_bits_to_f32(sb);
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(sf, d[j][r], acc[r]);
    }
}

// v as the lanes named by a DPP control see it (quad permutations, mirrors within a row of 16)
template <int CTRL>
__device__ __forceinline__ float lane_cross(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// (the LDS reads of a tile's pieces are issued together, ahead of the arithmetic)
struct GammaPiece {
    u32x4_t lo, hi;           // 8 x fp32, or (GH) 8 x f16 in lo
};

template <bool GH>
__device__ __forceinline__ GammaPiece gamma_piece(const void* gamma_lds, int k)
{
    GammaPiece g;
    if constexpr (GH) {
        g.lo = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint16_t*>(gamma_lds) + k);
        g.hi = g.lo;
    } else {
        g.lo = reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(gamma_lds) + k)[0];
        g.hi = reinterpret_cast<const u32x4_t*>(reinterpret_cast<const float*>(gamma_lds) + k)[1];
    }
    return g;
}

template <int XMODE, bool GH>
__device__ __forceinline__ void norm_piece(u32x4_t& v, const GammaPiece& gp, bool counts, float& ssq)
{
    float sq = ssq;
    if constexpr (GH) {
        const u32x4_t g = gp.lo;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const half2_t h = as_h2(v[p]);
            sq = __builtin_amdgcn_fdot2(h, h, sq, false);
            v[p] = as_u32(h * as_h2(g[p]));
        }
    } else {
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const uint32_t ua = p < 2 ? gp.lo[2 * p] : gp.hi[2 * p - 4], ub = p < 2 ? gp.lo[2 * p + 1] : gp.hi[2 * p - 3];
            const float ga = __builtin_bit_cast(float, ua), gb = __builtin_bit_cast(float, ub);
            if (XMODE == XBF16) {
                const float v0 = __builtin_bit_cast(float, v[p] << 16);
                const float v1 = __builtin_bit_cast(float, v[p] & 0xffff0000u);
                sq = fmaf(v1, v1, fmaf(v0, v0, sq));
                v[p] = pack_bf16x2(v0 * ga, v1 * gb);
            } else {
                const half2_t h = as_h2(v[p]);
                sq = __builtin_amdgcn_fdot2(h, h, sq, false);
                const half2_t o = {(_Float16)((float)h.x * ga), (_Float16)((float)h.y * gb)};
                v[p] = as_u32(o);
            }
        }
    }
    ssq = counts ? sq : ssq;
}

}  // namespace

}  // namespace cybq
