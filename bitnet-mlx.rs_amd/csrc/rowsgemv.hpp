// What the GEMVs that quantise their one row share (Fused16Params, row_lane), and what the token GEMVs on interleaved rows (ActRows::TILES16) share: the products of one wavefront, and the finish of a workgroup, where
// the wavefronts' partial results meet in LDS and wavefront r stores row block r, four outputs a lane.  gemv_rows_kernel takes rows
// that a launch before it wrote; gemv_die_kernel has them quantised by the workgroups of its own die.
#pragma once
#include "kernels.hpp"
#include "rowquant.hpp"

namespace bitnet {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u_t __attribute__((ext_vector_type(4)));
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(4)));  // 16-byte accesses need four-byte alignment only
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));

constexpr int AUX_SC1 = 0x10;  // cache policy of a buffer load: device scope, not from L1

// One projection in the argument buffer: one scalar load.
struct Fused16Proj {
    const uint8_t *w;
    const float *w_scale, *bias, *residual;
    float *out;
    int32_t *acc;
    int n;
    int rb_end;  // groups of row blocks of projections 0..this one, cumulative
    uint64_t unused;
};
static_assert(sizeof(Fused16Proj) == 64, "one scalar load a block");

// The arguments behind the preloaded ones, in blocks of 64 bytes: each is one scalar load.
struct Fused16Params {
    int kt_count;
    float eps;
    uint64_t reserved;
    int8_t *q_out;  // optional copies of what the prologue produced (written by the first group of row blocks)
    float *a_scale_out;
    int32_t *a_sum_out;
    uint64_t unused[3];
    Fused16Proj proj[GEMV_MAX_PROJ];
};
static_assert(sizeof(Fused16Params) == 64 * (1 + GEMV_MAX_PROJ), "one scalar load a block");
constexpr int FUSED16_ARGS_AT = 48;  // offset of the Fused16Params in the argument buffer: three pointers and six ints before it

// One token through more row blocks than one round of workgroups takes (gemv_stream.hip); p: projections with a row block each.
bool gemv_stream_takes(size_t m, size_t k, const float *gamma, int sum_order, size_t blocks);
int launch_gemv_stream(const Fused16Params &p, int nproj, const RowSource &src, int input_mode, size_t blocks, hipStream_t stream);

// The value of a lane of the own 16 lanes (a constant once unrolled): a row broadcast, 0x150 + lane.
template <int LANE>
__device__ __forceinline__ int row_lane_at(int v) { return dpp_i32<0x150 + LANE>(v); }
__device__ __forceinline__ int row_lane(uint32_t packed, int at)
{
    const int v = (int)packed;
    switch (at) {
        case 0: return row_lane_at<0>(v); case 1: return row_lane_at<1>(v); case 2: return row_lane_at<2>(v); case 3: return row_lane_at<3>(v);
        case 4: return row_lane_at<4>(v); case 5: return row_lane_at<5>(v); case 6: return row_lane_at<6>(v); case 7: return row_lane_at<7>(v);
        case 8: return row_lane_at<8>(v); case 9: return row_lane_at<9>(v); case 10: return row_lane_at<10>(v); case 11: return row_lane_at<11>(v);
        case 12: return row_lane_at<12>(v); case 13: return row_lane_at<13>(v); case 14: return row_lane_at<14>(v); default: return row_lane_at<15>(v);
    }
}

// The A operands of the k-tiles kt0, kt0 + nw, ...: lane 16 g + r takes row r, columns 16 g .. + 15 of a tile; lanes without a row load
// nothing (the results of their row are not used).  group_rows: the first byte of the token group.
template <int NT>
__device__ __forceinline__ void rows_load_a(v4i (&af)[NT][4], global_ptr<const uint8_t> group_rows, int lane, int rows_here, int kt0, int nw, int kt_count)
{
    const global_ptr<const uint8_t> a_lane = group_rows + (unsigned)(((lane >> 4) * rows_here + (lane & 15)) * 16);
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t) asm("" : "=v"(af[u][t]));
    if ((lane & 15) < rows_here) {
#pragma unroll
        for (int u = 0; u < NT; ++u)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                af[u][t] = *(global_ptr<const v4i>)(a_lane + (unsigned)((min(kt0 + nw * u, kt_count - 1) * 4 + t) * 64 * rows_here));
    }
}
// The same for rows that workgroups of this die wrote in this launch: past the compute unit's L1, which may hold the lines from before.
template <int NT>
__device__ __forceinline__ void rows_load_a_l2(v4i (&af)[NT][4], __amdgpu_buffer_rsrc_t group_rows, int lane, int rows_here, int kt0, int nw, int kt_count)
{
    const int at = ((lane >> 4) * rows_here + min(lane & 15, rows_here - 1)) * 16;
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            af[u][t] = __builtin_amdgcn_raw_buffer_load_b128(group_rows, at, (min(kt0 + nw * u, kt_count - 1) * 4 + t) * 64 * rows_here, AUX_SC1);
}
// Their weight tiles (row blocks and tiles past the end repeat the last one; their results are not stored or not added).
template <int RB, int NT>
__device__ __forceinline__ void rows_load_w(v4u_t (&w)[NT][RB], global_ptr<const v4u_t> tiles, int rb0, int rb_count, int kt0, int nw, int kt_count)
{
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < RB; ++r)
            w[u][r] = __builtin_nontemporal_load(tiles + ((size_t)min(rb0 + r, rb_count - 1) * kt_count + min(kt0 + nw * u, kt_count - 1)) * 64);
}

// The products of the k-tiles kt0, kt0 + nw, ... that a wavefront holds.  The weights are the first operand of the MFMA, so lane l of a
// result holds four consecutive outputs, 4 (l / 16) and on, of token l % 16; the rows' sums for the code offset are one more MFMA.
template <int RB, int NT>
__device__ __forceinline__ void rows_multiply(const v4i (&a)[NT][4], const v4u_t (&wt)[NT][RB], int kt0, int nw, int kt_count, v4i (&acc)[RB], v4i &sums)
{
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        if (kt0 + nw * u >= kt_count) break;  // uniform over the wavefront
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, a[u][t], sums, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                const unsigned wd = wt[u][r][t];
                const v4i bf = {(int)(wd & 0x03030303u), (int)((wd >> 2) & 0x03030303u), (int)((wd >> 4) & 0x03030303u), (int)((wd >> 6) & 0x03030303u)};
                acc[r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bf, a[u][t], acc[r], 0, 0, 0);
            }
        }
    }
}

// The epilogue of one wavefront: row block rb0 + wave of a projection, tokens 16 tg .. of one group.
struct RowsFinish {
    global_ptr<const float> w_scale, bias, residual, scales;
    global_ptr<float> out;
    global_ptr<int32_t> acc_out;
    int P_n, n_lane, t_lane;
    bool finishing, whole, row_ok;
    float e_ws, e_scale;
    v4f_any e_bias, e_res;

    // P: the projection's block of the argument buffer
    __device__ __forceinline__ RowsFinish(const v16u &P, const float *a_scale, int rb0, int row_blocks, int wave, int lane, int tg, int rows_here)
    {
        w_scale = pointer_at<const float>(P, 2); bias = pointer_at<const float>(P, 4); residual = pointer_at<const float>(P, 6);
        scales = (global_ptr<const float>)(uintptr_t)a_scale;
        out = pointer_at<float>(P, 8);
        acc_out = pointer_at<int32_t>(P, 10);
        P_n = (int)P[12];
        finishing = wave < row_blocks;  // a workgroup has four wavefronts at least
        const int n_block = (rb0 + wave) * TILE_ROWS;
        n_lane = n_block + 4 * (lane >> 4);
        t_lane = tg * 16 + min(lane & 15, rows_here - 1);
        whole = n_block + TILE_ROWS <= P_n;
        row_ok = (lane & 15) < rows_here;
        e_ws = 0.0f; e_scale = 1.0f;
        e_bias = (v4f_any){0.0f, 0.0f, 0.0f, 0.0f}; e_res = (v4f_any){0.0f, 0.0f, 0.0f, 0.0f};
    }
    // Asks for the operands of the epilogue; the rows' scales apart, where a workgroup of the launch writes them.
    __device__ __forceinline__ void request_operands()
    {
        if (!(finishing && whole && out)) return;  // uniform over the wavefront
        int lane_zero = 0;
        asm volatile("" : "+v"(lane_zero));
        e_ws = w_scale[lane_zero];
        if (bias) e_bias = *(global_ptr<const v4f_any>)(bias + n_lane);
        if (residual) e_res = *(global_ptr<const v4f_any>)(residual + ((size_t)t_lane * P_n + n_lane));
    }
    __device__ __forceinline__ void request_scales()
    {
        if (finishing && out) e_scale = scales[t_lane];
    }
    // The same past the compute unit's L1, for scales that workgroups of this die wrote in this launch.
    __device__ __forceinline__ void request_scales_l2()
    {
        if (finishing && out) e_scale = __hip_atomic_load(reinterpret_cast<const float *>((uintptr_t)scales) + t_lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // part: [nw][RB][64] of LDS
    template <int RB>
    __device__ __forceinline__ void finish(const v4i (&acc)[RB], const v4i &sums, v4i *part, int wave, int lane, int nw)
    {
#pragma unroll
        for (int r = 0; r < RB; ++r) part[((size_t)wave * RB + r) * 64 + lane] = acc[r] - sums;
        lds_barrier();
        if (!finishing) return;
        const v4i *from = part + wave * 64 + lane;
        v4i total = {0, 0, 0, 0};
        int v = 0;
        for (; v + 4 <= nw; v += 4) {  // uniform, as the rest is
            v4i got[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) got[i] = from[(v + i) * (RB * 64)];
#pragma unroll
            for (int i = 0; i < 4; ++i) total = total + got[i];
        }
        if (v < nw) {
            v4i got[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) got[i] = from[min(v + i, nw - 1) * (RB * 64)];
#pragma unroll
            for (int i = 0; i < 3; ++i)
                if (v + i < nw) total = total + got[i];
        }
        if (!row_ok) return;
        const size_t o = (size_t)t_lane * P_n + n_lane;
        if (whole) {
            if (acc_out) *(global_ptr<v4i_any>)(acc_out + o) = total;
            if (out) {
                v4f_any y;
                bool short_ok = invariant_divisor_ok(e_scale);
                const float recip = recip_of_ok_divisor(e_scale);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float scaled = f32_mul((float)total[i], e_ws);
                    short_ok = short_ok && dividend_ok(scaled);
                    y[i] = div_by_invariant_unchecked(scaled, e_scale, recip);
                }
                if (__builtin_expect(!short_ok, 0)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] = f32_div(f32_mul((float)total[i], e_ws), e_scale);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (bias) y[i] = f32_add(y[i], e_bias[i]);
                    if (residual) y[i] = f32_add(y[i], e_res[i]);
                }
                *(global_ptr<v4f_any>)(out + o) = y;
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // the last row block of a projection
            if (n_lane + i >= P_n) break;
            if (acc_out) acc_out[o + i] = total[i];
            if (out) {
                float y = f32_div(f32_mul((float)total[i], w_scale[0]), e_scale);
                if (bias) y = f32_add(y, bias[n_lane + i]);
                if (residual) y = f32_add(y, residual[o + i]);
                out[o + i] = y;
            }
        }
    }
};

}  // namespace bitnet
