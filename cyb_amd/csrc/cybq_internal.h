// cybq_internal.h - launcher prototypes shared between the C ABI (api.hip) and
// the kernel translation units.  Every launcher validates nothing: api.hip
// checks shapes, alignment and pointers before it calls down here.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cybq_device.h"

namespace cybq {

// dtype codes mirror enum cybq_dtype
constexpr int kF32 = 0, kF16 = 1, kBF16 = 2;

// q: PLANAR q plane (4-byte aligned) with `scales`, or BLOCK_AOS blocks (16-byte aligned with 15 readable bytes behind
// them, scales unused); device memory, or pinned host memory that the kernel reads across the bus (from_host)
// wide_flag: word (device or pinned host memory) that receives 1 when some scale times the largest q leaves f16 (nullptr: no scan)
hipError_t launch_repack(int bits, int layout, bool from_host, const void* q, const void* scales, uint8_t* dst, int N, int K, int NT, int KT,
                         uint32_t* wide_flag, hipStream_t st);
hipError_t launch_dequant(const WeightView& w, float* out, hipStream_t st);

// decode path, 1 <= M <= 16 per call, and 17 .. 32 rows where gemv_serves_32 says so (api.hip
// walks the other 17..32-row calls 16 rows at a time)
bool gemv_serves_32(const WeightView& w, int xdt, int M, int num_cus, const Epilogue& epi);
bool gemv_is_automatic();            // no tuning override is set
// exact_operands: keep the weight operands exact integers for one and two f16 rows too (the LDS
// kernel) instead of the subnormal-operand kernel of gemv1.hip
// scratch: device memory the batched-rows kernel may use when it splits K over workgroups (few strips, a
// long K): a ticket word per strip group at its start - zero at rest - and the slabs of partial sums behind
// them; nullptr = never split.  Calls that share it must not overlap.
constexpr size_t kDecodeScratchBytes = (size_t)8 << 20;
hipError_t launch_gemv(const WeightView& w, const void* x, int xdt, int M, void* y, int ydt,
                       int num_cus, bool exact_operands, const Epilogue& epi, void* scratch, size_t scratch_bytes, hipStream_t st);
// 3 .. 32 rows on outputs with several pairs of strips per CU (gemv_stream.hip)
bool gemv_stream_serves(const WeightView& w, int xdt, int M, int num_cus, const Epilogue& epi);
hipError_t launch_gemv_stream(const WeightView& w, const void* x, int xdt, int M, void* y, int ydt, int num_cus, bool exact_operands,
                              const Epilogue& epi, hipStream_t st);
// decode kernel for one and two rows (f16 / bf16 activations, no folded norm): weight operands are f16 subnormals
// (bf16: 128 + u),
// the +8 / +128 bias comes off inside the MFMA accumulation (gemv1.hip)
bool gemv1_serves(const WeightView& w, int xdt, int M, const Epilogue& epi);
hipError_t launch_gemv1(const WeightView& w, const void* x, int xdt, int M, void* y, int ydt, const Epilogue& epi, hipStream_t st);
// prefill path (api.hip sends 16-bit activations with M > 32 here)
// exact: two MFMAs per group with losslessly split weights; otherwise one f16 MFMA
// per group with weights rounded once to f16
// workspace: device scratch owned by the context (activations restaged in MFMA operand
// order, fp32 slabs of a K split, per-row statistics of a folded norm)
hipError_t launch_gemm(const WeightView& w, const void* x, int xdt, int M, void* y, int ydt,
                       int num_cus, bool exact, void* workspace, size_t workspace_bytes, const Epilogue& epi,
                       hipStream_t st);

// few rows (17 .. 64 on an output wide enough, up to 512 on a narrow one), FAST mode, activations already staged as f16 operands
// (gemm_rows.hip); ssq_part / ssq_blocks / unscale: the staging pass's per-row statistics
struct RowsPlan {
    int nf;                  // column blocks of 16 per workgroup (1, 2 or 4); 0: the kernel does not take the call
    bool two_per_cu = false; // two workgroups share a CU (nf = 4, up to 48 rows)
    bool pairs = false;      // one workgroup of eight waves does two column groups (nf = 4)
    int shares = 0;          // > 0: K is cut into that many shares, one per wave; more than four go to shares - 3 slabs, fp32 [M][N]
};
// (any_width: a group to a workgroup, up to 64 rows, however many rounds that makes)
RowsPlan gemm_rows_plan(const WeightView& w, int M, int num_cus, const Epilogue& epi, bool any_width);
hipError_t launch_gemm_rows(const WeightView& w, const void* x_staged, int M, void* y, int ydt, const Epilogue& epi,
                            const float* ssq_part, int ssq_blocks, const float* unscale, const RowsPlan& plan, float* slabs, hipStream_t st);
// the calls of plan_gemm_cols_long_k (below) that are this kernel's, a share of K per wave
RowsPlan gemm_rows_plan_long_k(const WeightView& w, int M, int num_cus, const Epilogue& epi);
// whether a scratch of this size holds enough staged rows of w's K for launch_gemm (which refuses the call otherwise)
bool gemm_stages(const WeightView& w, size_t workspace_bytes);
// the prefill kernel whose waves stand side by side along the columns (gemm_cols.hip).  mode: 0 FAST, 1 / 2 EXACT with f16 / bf16
// operands; more than one split leaves fp32 slabs [splits][M][N] in `part` for the slab-adding pass
struct ColsPlan {
    int rb, cs, splits;      // row blocks of 16 per workgroup, strips per wave, workgroups that share out K (none of them empty)
    bool whole_tiles;        // eight waves of one strip that take whole K tiles: the tiled kernels' order of sums, bit for bit
    float us;                // estimate of its time behind the staging pass
};
// FAST, a long K and few rows on an output that the tiled kernels split K for three ways or more (rb = 0: another call)
ColsPlan plan_gemm_cols_long_k(const WeightView& w, int M, int num_cus, const Epilogue& epi);
ColsPlan plan_gemm_cols(const WeightView& w, int mode, int M, int num_cus, size_t part_bytes);
// raw: x is the caller's, row major in the operands' type (no norm), instead of staged operands
hipError_t launch_gemm_cols(const WeightView& w, const void* x, bool raw, int mode, int M, void* y, int ydt, const ColsPlan& plan, const Epilogue& epi,
                            const float* ssq_part, int ssq_blocks, const float* unscale, float* part, hipStream_t st);
// test/bench hook: 2 = in FAST mode the tiled kernels alone (neither the few-rows kernel nor gemm_cols.hip), 3 = in both modes,
// 1 = the few-rows kernel whatever the width, 7 = as 2 with ranges of K in gemm_kernel, 0 = automatic
void set_gemm_tuning(int rows_kernel);
// what launch_gemm does with the first rows of a call that fit its scratch (tests)
struct PrefillRoute {
    int kernel;              // what multiplies: 1 gemm_rows.hip, 2 gemm_kernel, 3 gemm_roles_kernel, 4 gemm_cols.hip; 0: launch_gemm refuses the call
    int nf, splits;          // column blocks of 16 per workgroup (kernels 1 .. 3), workgroups that share out K (1: gemm_rows.hip's shares are not counted)
    int stage_rows;          // rows per workgroup of the row-scaling pass, 0: the rows do not go through it
};
PrefillRoute prefill_route(const WeightView& w, int xdt, int M, int num_cus, bool exact, size_t workspace_bytes, const Epilogue& epi);
// whether launch_gemm hands a FAST-mode call of M rows with this epilogue to the few-rows kernel (the hook included)
bool gemm_rows_takes(const WeightView& w, int M, int num_cus, const Epilogue& epi);

hipError_t launch_quantize(int bits, const float* src, int N, int K, void* q_out, void* s_out,
                           hipStream_t st);

// Kernels that need more dynamic LDS than the default 64 KB say so when the library is loaded:
// naming LdsRequest<&kernel, bytes>::registered anywhere in a launcher puts the pair on a list
// (a static initialiser, run before any call).  cybq_init walks the list for its device, so
// no launch ever changes a function attribute: first calls behave like all others and may sit
// inside a stream capture.
void register_lds_request(const void* kernel, int bytes);
hipError_t raise_all_lds_limits();              // for the current device
template <auto Kernel, int Bytes>
struct LdsRequest {
    static inline const bool registered = (register_lds_request(reinterpret_cast<const void*>(Kernel), Bytes), true);
};

// measurement probes (debug.hip)
hipError_t launch_read_probe(const WeightView& w, bool io, const void* x, void* y, hipStream_t st);
// other pure-read patterns over the same bytes (pattern 1 .. 6, see cybq_debug.h)
hipError_t launch_read_pattern(const WeightView& w, int pattern, int num_cus, hipStream_t st);
hipError_t launch_mfma_loop(int num_cus, int waves_per_simd, int iters, float* sink, hipStream_t st);
hipError_t launch_cache_read(const void* buf, int64_t bytes, int waves, int in_flight, int iters, int num_cus, hipStream_t st);

// test/bench hook: overrides the decode kernel's launch heuristics (0 = automatic)
void set_gemv_tuning(int waves_per_group, int rows_kernel, int unroll);


}  // namespace cybq
