// Internal launchers, one per kernel family.  Arguments are validated by the C-ABI layer (api.hip);
// these only pick a kernel variant and launch it.  All return a bitnet_hip_status.
#pragma once
#include "common.hpp"
#include "ieee.hpp"

namespace bitnet {

// ---- geometry of the re-tiled weight layout (see weight_prep.hip) ----
constexpr int TILE_ROWS = 16;    // output rows per tile
constexpr int TILE_K = 256;      // input columns per tile
constexpr int TILE_BYTES = 1024; // TILE_ROWS * TILE_K / 4
inline size_t row_blocks(size_t n) { return (n + TILE_ROWS - 1) / TILE_ROWS; }
inline size_t k_tiles(size_t k) { return (k + TILE_K - 1) / TILE_K; }
inline size_t tiled_bytes(size_t n, size_t k) { return row_blocks(n) * k_tiles(k) * (size_t)TILE_BYTES; }

// act_quant.hip
// Layout of the int8 rows.  TILES16 (row stride a multiple of 256): what launch_gemv_rows reads, the 16 rows of a group
// interleaved in pieces of 16 bytes; byte b of piece c of row r lies at 16 g ldq + (c R + r % 16) 16 + b, with g = r / 16 and R the
// rows of that group (16; fewer in the last one).
enum class ActRows { ROW_MAJOR, TILES16 };
int launch_act_quant(const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode,
                     size_t gqa_group, size_t head_dim, const float *gamma, float eps, int sum_order,
                     int8_t *q, size_t ldq, float *a_scale, int32_t *a_sum, float *y, hipStream_t stream, ActRows rows = ActRows::ROW_MAJOR);
// ldq: row stride of q, k or padded_k(k).  Padded rows end in zeros, so the contraction may take padded_k(k) for k: its weight
// tiles are padded with zero weights, and every width then has the aligned rows the LDS-direct and the batched kernels need.
inline size_t padded_k(size_t k) { return (k + TILE_K - 1) / TILE_K * TILE_K; }

// absmax_quantize_activations (activations.rs:530-641): one scale per tensor; scratch of absmax_quantize_scratch_bytes(n)
// bytes; stats: 4 floats (scale, mse, min, max)
size_t absmax_quantize_scratch_bytes(size_t n);
int launch_absmax_quantize(const float *x, size_t n, int precision, void *scratch, int8_t *q, float *stats, hipStream_t stream);
// max |x| of a tensor for the waiting host, a partial maximum from each of `workgroups` (answers and ticket of a HostParts,
// staging.hpp; abs_max_workgroups: how many the tensor is worth, at most `most`), and the quantiser of
// DynamicActivationQuantizer with the scale given from outside (activations.rs:269-294, 315-360), which also stores the
// scale to scale_out unless that is null
int abs_max_workgroups(size_t n, int most);
int launch_abs_max(const float *x, size_t n, int workgroups, unsigned long long *answers, unsigned ticket, hipStream_t stream, float *parts = nullptr);
// Both at once, the scale computed on the device from the maximum and the moving average before this step.  parts: 256 floats of
// device scratch; answers receives one word (n <= DYNAMIC_SMALL) or one from each of `workgroups`.
struct DynamicScale {
    int has_average;
    float average, decay;
};
constexpr int DYNAMIC_SMALL = 32768;
int launch_dynamic_quantize(const float *x, size_t n, int precision, const DynamicScale &d, int reference_u8, int8_t *q, float *scale_out, float *parts,
                            int workgroups, unsigned long long *answers, unsigned ticket, hipStream_t stream);
int launch_scaled_quantize(const float *x, size_t n, int precision, float scale, int reference_u8, int8_t *q, float *scale_out,
                           hipStream_t stream);

// weight_prep.hip
int launch_pack_2bit(const int8_t *q, size_t count, uint8_t *packed, hipStream_t stream);
int launch_unpack_2bit(const uint8_t *packed, size_t count, int8_t *q, hipStream_t stream);
int launch_lookup_compute(int kind, const int8_t *w, const float *x, float *out, size_t n, hipStream_t stream);
// base-3 bytes (5 values each): pack, unpack, and re-code into the 2-bit bytes (4 values each)
int launch_pack_base3(const int8_t *q, size_t count, uint8_t *packed, hipStream_t stream);
int launch_unpack_base3(const uint8_t *packed, size_t count, int8_t *q, hipStream_t stream);
int launch_base3_to_2bit(const uint8_t *base3, size_t count, uint8_t *packed, hipStream_t stream);
// row_sums: device scratch of n doubles; apart: they are not where the codes go
int launch_quantize_weights(const float *w, size_t n, size_t k, int method, float threshold_factor,
                            double *row_sums, bool apart, uint8_t *packed, float *w_scale, int8_t *q_i8,
                            hipStream_t stream);
// BitNetWeightQuantizer::quantize (weights.rs:568-611): method = TernaryMethod 0..4, custom_factor <= 0 = none;
// scratch: quantize_weights_reference_scratch_bytes(n) bytes of device memory; stats: 12 floats or null
size_t quantize_weights_reference_scratch_bytes(size_t n);
int launch_quantize_weights_reference(const float *w, size_t n, size_t k, int method, int normalize, float outlier_threshold,
                                      float custom_factor, void *scratch, uint8_t *packed, float *w_scale, int8_t *q_i8,
                                      float *stats, hipStream_t stream);
// canonical (optional): the weights back in flat [n, k] order with code 3 stored as code 1; w_scale_out (optional): receives
// w_scale (a value the host holds, stored without a copy of its own)
int launch_retile(const uint8_t *packed, size_t n, size_t k, int layout, uint8_t *tiled, hipStream_t stream,
                  uint8_t *canonical = nullptr, float w_scale = 0.0f, float *w_scale_out = nullptr);
int launch_untile(const uint8_t *tiled, size_t n, size_t k, uint8_t *packed, hipStream_t stream);

// gemv_base3.hip: the decode GEMV on base-3 bytes (five values per byte) in their own streaming layout
size_t base3_tiled_bytes(size_t n, size_t k);
int launch_retile_base3(const uint8_t *flat, size_t n, size_t k, uint8_t *tiled, hipStream_t stream);
int launch_gemv_base3(const uint8_t *tiled, const int8_t *a, int32_t *acc, float *out, const float *w_scale, const float *a_scale,
                      size_t n, size_t k, hipStream_t stream);

// gemv_w2a8.hip
int launch_gemv_rowmajor(const uint8_t *packed, const int8_t *a, int32_t *out, size_t n, size_t k,
                         hipStream_t stream);
constexpr int GEMV_MAX_M = 95;       // token rows that the token GEMV takes at any width, unless the GEMM is faster
constexpr int GEMV_WIDE_MAX_M = 512; // and where its workgroups are a single round of the chip (gemv_takes)
// Between the two from 17 tokens on, by what each takes beyond what both do (launch, quantiser, weights once, outputs once), in ns.
// The token GEMV, per 16-row block and group of 16 tokens: its part of the exchange of partial results, its k-tiles up to 16 (one per
// wavefront, whose partial results are exchanged) and those beyond.  The GEMM: gemm_beyond_ns.  Fitted to the recorded times of both:
// calls of 17 to 512 tokens, 15 widths from 256 to 16384 columns by 14 from 1024 to 131072 outputs, with a pair of layers and with layers
// that outrun the last-level cache (the mean of the two); and 14 stacks of decoder blocks at 17 to 95 tokens with each launch group
// by either kernel.  Where they differ, the one chosen is behind the faster one by 0.36 % in the geometric mean of the calls and 0.39 %
// of the launches in stacks (a rule by workgroups and tiles: 2.0 and 0.6 %, at worst 2.1 times).  GEMV / GEMM, quantiser included, in us:
// 2560 -> 13824 at 48 / 49 / 95 tokens 10.2 / 10.4, 11.6 / 10.4, 14.5 / 12.7; 1536 -> 16384 at 48 / 64 / 95 7.9 / 8.9, 8.7 / 9.2, 10.7 /
// 10.3; 4096 -> 13824 at 48 / 49 / 95 12.0 / 12.5, 13.5 / 12.5, 17.6 / 15.0; 8192 -> 8192 at 32 / 48 / 95 10.2 / 13.9, 14.5 / 14.6, 19.6 /
// 18.6; 6912 -> 2560 at 95 10.1 / 12.8; 256 -> 32768 at 33 / 64 / 95 7.6 / 7.6, 8.9 / 8.2, 11.2 / 9.1; 768 -> 20480 at 33 / 64 / 95 7.3 / 8.4,
// 8.0 / 8.9, 9.6 / 9.7; 256 -> 131072 at 95 37.0 / 17.3.  A block of a stack with one group by either: 2560 -> 6912 + 6912 at 48 tokens is the
// GEMV's by 0.3, at 64 the GEMM's by 1.2; 12288 -> 4096 at 95 the GEMV's by 0.3 where the call alone is the GEMM's by 2.1.
size_t gemm_beyond_ns(size_t m, size_t k, size_t n);  // gemm_w2a8.hip
inline bool gemm_beats_token_gemv(size_t m, size_t k, size_t n_blocks, const void *a)
{
    if (m <= 16 || m > (size_t)GEMV_WIDE_MAX_M || k == 0 || k % TILE_K != 0 || n_blocks * k >= (1ull << 29) || (reinterpret_cast<uintptr_t>(a) & 15) != 0)
        return false;
    const size_t kt = k / TILE_K, blocks = n_blocks * ((m + 15) / 16), near = blocks * (kt < 16 ? kt : 16), all = blocks * kt;
    const size_t gemv_ns = blocks / 6 + near / 8 + (all - near) / 10;
    return gemv_ns > 2300 && gemm_beyond_ns(m, k, n_blocks * 16) < gemv_ns;  // the GEMM takes no less anywhere
}
// sums: the caller has the rows' sums, without which the GEMM takes a slower kernel.  Above 95 tokens (rows of up to 8192 columns) the
// GEMV is taken only while its workgroups run as a single round, row blocks per workgroup and slots as in launch_gemv_tiled: 2560 ->
// 2560 at 128 / 192 tokens 8.2 / 9.0, 8.6 / 9.3 us (GEMV / GEMM), 6912 -> 2560 at 96 10.1 / 12.8; a second round: 6912 -> 2560 at 112 13.1 / 12.9.
inline bool gemv_takes(size_t m, size_t k, size_t n_blocks, const void *a, bool sums = true)
{
    if (sums && gemm_beats_token_gemv(m, k, n_blocks, a)) return false;
    if (m <= (size_t)GEMV_MAX_M) return true;
    if (m > (size_t)GEMV_WIDE_MAX_M || k % 256 != 0 || k > 8192 || (reinterpret_cast<uintptr_t>(a) & 15) != 0) return false;
    const size_t tgroups = (m + 15) / 16, slots = k <= 3072 ? 768 : 256;
    const size_t rb = n_blocks * tgroups > 2 * slots ? 4 : (n_blocks * tgroups > slots ? 2 : 1);
    return (n_blocks + rb - 1) / rb * tgroups <= slots;
}
constexpr int GEMV_MFMA_MAX_M = 64; // rows per launch of the MFMA variant of the decode GEMV (2 and more rows)
constexpr int GEMV_MAX_PROJ = 3;  // projections sharing one input row per launch (q,k,v / gate,up)
// One projection of a decode-GEMV launch: re-tiled weights [n, k], its scale, optional bias [n] and
// residual [m, n]; out [m, n] f32 and acc [m, n] int32 are each optional.
struct GemvProj {
    const uint8_t *tiled;
    const float *w_scale;
    const float *bias;
    const float *residual;
    float *out;
    int32_t *acc;
    size_t n;
};
// activations already int8 ([m, k], a_scale [m]); any m (launched in groups of up to GEMV_MAX_M rows)
int launch_gemv_tiled(const GemvProj *projs, int nproj, const int8_t *a, const float *a_scale, size_t m, size_t k,
                      hipStream_t stream);
// the same for rows in ActRows::TILES16 order, where gemv_rows_takes says so
constexpr size_t GEMV_ROWS_MAX_BLOCKS = 0xfff0;  // 16-row blocks of a launch (counts of 16 bits in its arguments)
inline bool gemv_rows_takes(size_t m, size_t k, size_t n_blocks, const void *a)
{
    return m >= 2 && k % TILE_K == 0 && n_blocks <= GEMV_ROWS_MAX_BLOCKS && k_tiles(k) <= 0xffff && (reinterpret_cast<uintptr_t>(a) & 15) == 0 &&
           gemv_takes(m, k, n_blocks, a);
}
int launch_gemv_rows(const GemvProj *projs, int nproj, const int8_t *a, const float *a_scale, size_t m, size_t k, hipStream_t stream);
// gemv_rowq.hip: several tokens on short f32 rows, quantised by every workgroup of the one launch.  Only where gemv_rowq_takes()
// says so; blocks: 16-row blocks of all projections of the launch; alone: the launch is a call of its own, not one of a step or of a
// caller's capture.
bool gemv_rowq_takes(const float *x, size_t ldx, size_t m, size_t k, int input_mode, size_t gqa_group, size_t head_dim,
                     const float *gamma, int sum_order, size_t blocks, bool alone);
int launch_gemv_rowq(const GemvProj *projs, int nproj, const float *x, size_t m, size_t k, int input_mode, size_t gqa_group, size_t head_dim,
                     const float *gamma, float eps, hipStream_t stream);
// gemv_die.hip: several tokens in one launch, their rows quantised once on every die.  Only where gemv_die_takes() says so.
// flags: 16 dies x stride 64-bit words, none of which holds tag before the launch; clear (optional): clear_sets other sets of them, one behind
// the other, cleared for the m rows by the launch; looks: how often a workgroup looks at the flags before it quantises its rows itself.
constexpr int GEMV_DIE_MAX_M = 128;
constexpr size_t GEMV_DIE_SETS = 16;  // dies whose flags are kept apart
constexpr int GEMV_DIE_LOOKS = 4096;
struct DieFlags {
    uint64_t *flags, *clear;
    unsigned clear_sets;
    uint64_t tag;
    unsigned stride;
    int looks;
};
// blocks: 16-row blocks of all projections of the launch; alone: a call of its own, not one of a step
bool gemv_die_takes(const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode, const float *gamma, int sum_order, size_t blocks,
                    bool alone);
int launch_gemv_die(const GemvProj *projs, int nproj, const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode, const float *gamma,
                    float eps, int8_t *q, float *a_scale, const DieFlags &f, hipStream_t stream);
// clears the flags of m rows in one set
int launch_clear_die_flags(uint64_t *flags, size_t stride, size_t m, hipStream_t stream);
// f32 input quantised inside the GEMV launch; only where gemv_fused_supported() says so.  q_out / a_scale_out /
// a_sum_out (each optional) receive the quantiser's results.
bool gemv_fused_supported(const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode,
                          size_t head_dim, const float *gamma, int sum_order, size_t blocks);
size_t gemv_fused_tiles(size_t m, size_t k, size_t blocks);  // weight tiles that one workgroup of that launch walks
// blocks: 16-row blocks of all projections of the launch (of its largest launch group)
int launch_gemv_fused(const GemvProj *projs, int nproj, const float *x, const float *x2, size_t ldx, size_t m,
                      size_t k, int input_mode, size_t gqa_group, size_t head_dim, const float *gamma, float eps,
                      int sum_order, int8_t *q_out, float *a_scale_out, int32_t *a_sum_out, hipStream_t stream);

// gemm_w2a8.hip
constexpr int GEMM_MAX_PROJ = 3;  // projections sharing one activation matrix per launch of the LDS-direct kernels
// several projections in one launch; BITNET_HIP_UNSUPPORTED (no message) if the LDS-direct kernels do not apply
int launch_gemm_multi(const GemvProj *projs, int nproj, const int8_t *a, const int32_t *a_sum, const float *a_scale,
                      size_t m, size_t k, hipStream_t stream);
// a_sum (sum_k a[t, k] per row, from the activation quantiser) may be NULL: the slower kernel then computes it
int launch_gemm_tiled(const uint8_t *tiled, const int8_t *a, const int32_t *a_sum, size_t m, size_t n, size_t k,
                      int32_t *acc, const float *w_scale, const float *a_scale, const float *bias,
                      const float *residual, float *out, hipStream_t stream);

// Diagnostic: `iters` rounds of eight v_mfma_i32_16x16x64_i8 per wavefront, MFMA_RATE_THREADS / 64 wavefronts on each of
// `compute_units` workgroups, operands in registers; sink receives compute_units * MFMA_RATE_THREADS ints.
constexpr int MFMA_RATE_THREADS = 512;
constexpr int MFMA_RATE_PER_ITER = 8;
int launch_mfma_rate(bool random_operands, int iters, int compute_units, int *sink, hipStream_t stream);

}  // namespace bitnet
