// One token through many row blocks: gemv_fused16_kernel's prologue with a workgroup that then walks its row blocks.
//
// A launch has one workgroup a compute unit, which quantises the row once (the row's pieces reach the MFMA by lane broadcasts and stay in
// registers: a wavefront has the same k-tiles of every row block) while its first weight tiles are on their way, and asks for the tiles of
// a row block D further on where it has used one.  Nothing but weights goes through memory in the loop, and nobody waits for another
// wavefront there: the partial results lie in LDS until the end.  Bound by the read of the weights once there are some 30 MB of them, by the
// chain of gemv_fused16_kernel's steps below.
// Calls, as two launches (rows above 7168 columns) or with the row quantised again for every row block or two -> here, us:
//   16384 -> 32768 24.9 -> 20.7 (134 MB: 6.5 TB/s), 16384 -> 8192 11.7 -> 7.7, 12288 -> 20000 15.1 -> 11.3, 8192 -> 13824 9.8 -> 6.7 (norm 10.7 -> 7.5),
//   6912 -> 32768 15.7 -> 10.4 (norm 26.0 -> 11.0), 6912 -> 131072 58.9 -> 36.9 (norm 99.7 -> 37.7), 5120 -> 5120 with a norm 7.2 -> 6.0.
// D: as few row blocks in flight as cover the latency.  8192 -> 20000 with 2 / 3 / 4 / 6 of them: 7.6 / 7.8 / 8.5 / 9.2 us.  Row blocks past the
// last are not walked: with D rounds to the end a small launch takes 1.5 us more.
#include "kernels.hpp"
#include "rowsgemv.hpp"

namespace bitnet {

namespace {

constexpr int AUX_NT = 2;  // cache policy of a buffer load: read once
constexpr size_t STREAM_WORKGROUPS = 256, STREAM_MOST_BLOCKS = 60;  // a compute unit each; row blocks of one whose results LDS holds

// The tiles first, first + nw, .. of a row block (of all projections one after the other); of a row block past the last, and past the row's
// end, no bytes, which come back as zeros and add nothing.
struct StreamTiles {
    uint64_t w0, w1, w2;
    int end0, end1, blocks, row_bytes;
};
template <int NCHB>
__device__ __forceinline__ void request_tiles(v4u_t (&to)[NCHB], const StreamTiles s, int block, int at_lane, int wave_step)
{
    const int pj = (block >= s.end0) + (block >= s.end1);
    const uint64_t w = pj == 0 ? s.w0 : (pj == 1 ? s.w1 : s.w2);
    const int at = block - (pj == 0 ? 0 : (pj == 1 ? s.end0 : s.end1));
    const uint64_t base = w + (uint64_t)(uint32_t)at * (uint32_t)s.row_bytes;
    const __amdgpu_buffer_rsrc_t tiles = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(base), 0, block < s.blocks ? s.row_bytes : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < NCHB; ++i) to[i] = __builtin_amdgcn_raw_buffer_load_b128(tiles, at_lane + wave_step * i, 0, AUX_NT);
}

typedef const __attribute__((address_space(4))) v16u *stream_args;

// What the epilogue of a row block takes: output n of its projection for lanes 0..15.
struct StreamFinish {
    global_ptr<const float> bias, residual;
    global_ptr<float> out;
    global_ptr<int32_t> acc_out;
    int n;
    bool stores;
    float ws, e_bias, e_res;
    __device__ __forceinline__ void request(stream_args blocks, const StreamTiles s, int block, int lane)
    {
        const int pj = (block >= s.end0) + (block >= s.end1);
        const v16u P = blocks[1 + pj];
        const global_ptr<const float> w_scale = pointer_at<const float>(P, 2);
        bias = pointer_at<const float>(P, 4); residual = pointer_at<const float>(P, 6);
        out = pointer_at<float>(P, 8);
        acc_out = pointer_at<int32_t>(P, 10);
        n = (block - (pj == 0 ? 0 : (pj == 1 ? s.end0 : s.end1))) * TILE_ROWS + (lane & 15);
        stores = lane < TILE_ROWS && n < (int)P[12];
        ws = 0.0f; e_bias = 0.0f; e_res = 0.0f;
        int lane_zero = 0;
        asm volatile("" : "+v"(lane_zero));  // a vector load, which nothing waits for before its use
        if (stores) {
            if (out) ws = w_scale[lane_zero];
            if (bias) e_bias = bias[n];
            if (residual) e_res = residual[n];
        }
    }
};

template <int MODE, bool NORM, int NCHB, int D>
__global__ __launch_bounds__(1024) void gemv_stream_kernel(const float *hot_x, const float *hot_x2, const float *hot_gamma, int hot_k, int hot_blocks,
                                                           int hot_nw, int hot_head_chunks, int hot_end0, int hot_end1, [[maybe_unused]] Fused16Params args)
{
    extern __shared__ int part[];  // [row block of this workgroup][wavefront][16]
    __shared__ float red_f[2][16];
    __shared__ int asum_s;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = hot_nw, chunks = hot_k >> 2, workgroups = (int)gridDim.x, wg = (int)blockIdx.x;

    const int in_tile = 16 * ((lane >> 2) & 3) + 4 * (lane >> 4) + (lane & 3);
    Row16<NORM, NCHB> row16;
    const uint64_t magics = MODE == BITNET_HIP_INPUT_GQA_BROADCAST ? reinterpret_cast<uintptr_t>(hot_x2) : 0;
    row16.template load<MODE>(hot_x, MODE == BITNET_HIP_INPUT_RELU2_MUL ? hot_x2 : nullptr, magics, hot_head_chunks, hot_gamma, chunks, nw, wave, tid, in_tile);
    __builtin_amdgcn_sched_barrier(0);
    const stream_args args_at = (stream_args)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + FUSED16_ARGS_AT);
    v16u common = args_at[0];
    uint64_t w0 = *(const __attribute__((address_space(4))) uint64_t *)(args_at + 1), w1 = *(const __attribute__((address_space(4))) uint64_t *)(args_at + 2),
             w2 = *(const __attribute__((address_space(4))) uint64_t *)(args_at + 3);
    if (tid < 16 && tid >= nw) red_f[1][tid] = 0.0f;  // the slots of absent wavefronts hold the neutral element
    if (tid == 0) asum_s = 0;
    float k_f = (float)hot_k, k_recip = recip_of_ok_divisor(k_f);  // k <= 16384: a divisor the short division accepts
    asm volatile("" : "+v"(k_recip));
    asm volatile("" : "+s"(common), "+s"(w0), "+s"(w1), "+s"(w2));
    const int kt_count = (int)common[0];
    const float eps = __builtin_bit_cast(float, (unsigned)common[1]);
    const global_ptr<uint32_t> q_out = pointer_at<uint32_t>(common, 4);
    const global_ptr<float> a_scale_out = pointer_at<float>(common, 6);
    const global_ptr<int32_t> a_sum_out = pointer_at<int32_t>(common, 8);

    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();  // all wavefronts have asked for the row: memory answers a compute unit in the order of its requests
    __builtin_amdgcn_sched_barrier(0);
    const StreamTiles tiles = {w0, w1, w2, hot_end0, hot_end1, hot_blocks, kt_count * 1024};
    const int at_lane = 16 * lane + 1024 * wave, wave_step = 1024 * nw;
    v4u_t wt[D][NCHB];
#pragma unroll
    for (int d = 0; d < D; ++d) request_tiles(wt[d], tiles, wg + d * workgroups, at_lane, wave_step);
    __builtin_amdgcn_sched_barrier(0);
    StreamFinish finish;  // of the first row block that this wavefront finishes
    if (wg + wave * workgroups < hot_blocks) finish.request(args_at, tiles, wg + wave * workgroups, lane);
    __builtin_amdgcn_sched_barrier(0);

    uint32_t packed[NCHB];
    const float scale = row16.quantise(chunks, k_f, k_recip, eps, wave, tid, red_f, packed);
    v4i af[NCHB][4], sums = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NCHB; ++i) {
        if (q_out && wg == 0 && row16.chunk[i] < chunks) q_out[row16.chunk[i]] = packed[i];
        const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            af[i][j] = (v4i){row_lane(packed[i], 4 * j), row_lane(packed[i], 4 * j + 1), row_lane(packed[i], 4 * j + 2), row_lane(packed[i], 4 * j + 3)};
            sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i][j], ones, sums, 0, 0, 0);
        }
    }
    if (a_sum_out && wg == 0 && lane == 0) atomicAdd(&asum_s, sums[0]);

    int *mine = part + wave * TILE_ROWS + lane;
    const auto multiply = [&](const v4u_t (&w)[NCHB]) {
        v4i acc = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < NCHB; ++i)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const unsigned c = w[i][t];
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                    af[i][t], (v4i){(int)(c & 0x03030303u), (int)((c >> 2) & 0x03030303u), (int)((c >> 4) & 0x03030303u), (int)((c >> 6) & 0x03030303u)}, acc, 0, 0, 0);
            }
        if (lane < TILE_ROWS) *mine = acc[0] - sums[0];
        mine += nw * TILE_ROWS;
    };
    int block = wg;
    for (; block + (D - 1) * workgroups < hot_blocks; block += D * workgroups) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            multiply(wt[d]);
            request_tiles(wt[d], tiles, block + (D + d) * workgroups, at_lane, wave_step);
        }
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d) {
        if (block + d * workgroups >= hot_blocks) break;
        multiply(wt[d]);
    }
    const float s_recip = recip_of_ok_divisor(scale);
    const bool divisor_fits = invariant_divisor_ok(scale);
    lds_barrier();

    // A wavefront finishes row blocks: lane 16 p + r adds up the results of wavefronts p, p + 4, ... for row r.
    for (int i = wave; wg + i * workgroups < hot_blocks; i += nw) {
        if (i != wave) finish.request(args_at, tiles, wg + i * workgroups, lane);
        int total = 0;
        for (int v = lane >> 4; v < nw; v += 4) total += part[(i * nw + v) * TILE_ROWS + (lane & 15)];
        total = sum_over_lane_groups(total);
        if (!finish.stores) continue;
        if (finish.acc_out) finish.acc_out[finish.n] = total;
        if (finish.out) {
            const float scaled = f32_mul((float)total, finish.ws);
            float y = div_by_invariant_unchecked(scaled, scale, s_recip);
            if (__builtin_expect(!(divisor_fits && dividend_ok(scaled)), 0)) y = f32_div(scaled, scale);
            if (finish.bias) y = f32_add(y, finish.e_bias);
            if (finish.residual) y = f32_add(y, finish.e_res);
            finish.out[finish.n] = y;
        }
    }
    if (wg == 0 && tid == 0) {
        if (a_scale_out) *a_scale_out = scale;
        if (a_sum_out) *a_sum_out = asum_s;
    }
}

template <int MODE, bool NORM, int NCHB, int D>
int launch(const Fused16Params &p, int nproj, const RowSource &src, size_t blocks, int nw, hipStream_t stream)
{
    const unsigned workgroups = blocks < STREAM_WORKGROUPS ? (unsigned)blocks : STREAM_WORKGROUPS;
    const size_t lds = (blocks + workgroups - 1) / workgroups * (size_t)nw * TILE_ROWS * sizeof(int);
    const float *x2 = src.x2;
    if (MODE == BITNET_HIP_INPUT_GQA_BROADCAST) {
        uint64_t magics = 0;
        if (!row16_magics(src.head_dim, src.gqa_group, &magics))
            return fail(BITNET_HIP_INVALID_CONFIG, "GQA group of %d heads of %d out of range", src.gqa_group, src.head_dim);
        x2 = reinterpret_cast<const float *>(static_cast<uintptr_t>(magics));
    }
    launch_kernel((gemv_stream_kernel<MODE, NORM, NCHB, D>), dim3(workgroups), dim3(64u * (unsigned)nw), lds, stream, src.x, x2, src.gamma, src.k,
                  (int)blocks, nw, src.head_dim / 4, nproj > 1 ? p.proj[0].rb_end : 0x7fffffff, nproj > 2 ? p.proj[1].rb_end : 0x7fffffff, p);
    BITNET_HIP_CHECK_LAUNCH("gemv_stream_kernel");
    return BITNET_HIP_OK;
}

template <int MODE>
int launch_mode(const Fused16Params &p, int nproj, const RowSource &src, size_t blocks, hipStream_t stream)
{
    const int nw = row_workgroup_waves(src.k), kt = p.kt_count;
    if (src.gamma) {  // plain rows only, and of up to 32 k-tiles: what gemv_stream_takes and the callers let through
        if constexpr (MODE == BITNET_HIP_INPUT_PLAIN)
            if (kt <= 32) return launch<MODE, true, 2, 2>(p, nproj, src, blocks, nw, stream);
        return fail(BITNET_HIP_UNSUPPORTED, "streaming GEMV: %d k-tiles of input mode %d with a norm", kt, MODE);
    }
    if (kt <= 32) return launch<MODE, false, 2, 2>(p, nproj, src, blocks, nw, stream);
    // one row block in flight while a workgroup has few of them: 16384 -> 8192 7.7 us against 8.7, -> 32768 21.6 against 20.7
    return blocks > 4 * STREAM_WORKGROUPS ? launch<MODE, false, 4, 2>(p, nproj, src, blocks, nw, stream) : launch<MODE, false, 4, 1>(p, nproj, src, blocks, nw, stream);
}

}  // namespace

bool gemv_stream_takes(size_t m, size_t k, const float *gamma, int sum_order, size_t blocks)
{
    // Rows of up to 4096 columns stay with gemv_fused16_kernel, which holds the tiles of four row blocks at once: 2560 -> 32768 4.8 us there, 6.1
    // here, 4096 -> 32768 6.5 and 8.0, and only beyond 65536 outputs less (4096 -> 131072 23.2 and 21.6).  Above, its workgroups have one row block:
    // with up to two rounds of them and no norm it is as fast (6912 -> 8192 5.0 and 5.3, -> 9000 6.6 and 6.0), with a norm slower from the second
    // round on (6912 -> 4160 7.2 and 5.8).  Above 7168 columns the other way is two launches from the second round on (8192 -> 4160 7.6 and 5.0).
    if (m != 1 || k <= 4096 || k > 16384 || blocks > STREAM_WORKGROUPS * STREAM_MOST_BLOCKS) return false;
    if (gamma && (sum_order != BITNET_HIP_SUM_BLOCK256 || k > 8192)) return false;
    return blocks > (gamma || k > 7168 ? STREAM_WORKGROUPS : 2 * STREAM_WORKGROUPS);
}

int launch_gemv_stream(const Fused16Params &p, int nproj, const RowSource &src, int input_mode, size_t blocks, hipStream_t stream)
{
    switch (input_mode) {
        case BITNET_HIP_INPUT_PLAIN: return launch_mode<BITNET_HIP_INPUT_PLAIN>(p, nproj, src, blocks, stream);
        case BITNET_HIP_INPUT_RELU2_MUL: return launch_mode<BITNET_HIP_INPUT_RELU2_MUL>(p, nproj, src, blocks, stream);
        default: return launch_mode<BITNET_HIP_INPUT_GQA_BROADCAST>(p, nproj, src, blocks, stream);
    }
}

}  // namespace bitnet
