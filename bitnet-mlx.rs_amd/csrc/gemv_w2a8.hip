// Decode GEMV kernels: int8 activations x 2-bit ternary weights -> int32, for gfx950.
//
//   acc[t, n] = sum_k a[t, k] * w[n, k]         exact in int32 (|acc| <= 127*K)
//   out[t, n] = (float(acc) * w_scale) / a_scale[t] (+ bias[n]) (+ residual[t, n])
//
// Semantics: bitnet-quant/src/simd/matrix.rs:471-490 (GEMV) with the contract of
// bitnet-cuda/src/kernels/w2a8_gemv.cu:100-105 (u8 packed weights, i8 activations, i32 output).
//
// The kernels never decode to {-1,0,+1}.  They multiply by the stored code c = w + 1 in {0,1,2}
// (two VALU operations turn a packed dword into four code bytes: shift, and with 0x03030303) and
// subtract sum_k a[t, k] once per output:  sum a*(c-1) = sum a*c - sum a.
//
// gemv_tiled_kernel streams the re-tiled layout (weight_prep.hip).  A workgroup of four wavefronts owns
// one block of 16 output rows; its wavefronts take the k-tiles round-robin, so all of a workgroup's
// weight bytes are requested in the first few instructions.  Lane l of a wavefront loads the 16 bytes at
// offset 16*l of a 1 KiB tile: row r = l mod 16, four groups of 16 columns.  Activations sit in LDS; the 16
// lanes of a group read the same LDS address (a broadcast).  Partial sums are combined with two wavefront
// shuffles (the four lanes of a row), then across the four wavefronts through LDS.
//
// Two more things are folded into the same launch, because at one token the cost of a decode step is the
// number of dependent launches, not bytes:
//   * the activation quantiser: with MODE >= 0 the workgroup reads the f32 row itself, runs RMSNorm +
//     absmax + int8 rounding (rowquant.hpp, the same code and summation order as the stand-alone
//     quantiser) and writes the int8 row straight into LDS.  The weight tiles are requested first, so
//     their HBM latency overlaps this prologue.
//   * up to three projections that share the input row (q, k, v or gate, up): the grid is the
//     concatenation of their row blocks.
// HBM traffic per call: n*k/4 weight bytes; the input row (K or 4K bytes per workgroup) comes from L2.
// gemv_fused16_kernel is this launch with up to 16 wavefronts per workgroup (the default for one token; see its comment): there the
// row reaches the MFMA by lane broadcasts, and the tiles are requested behind it.
//
// gemv_stream.hip is the same for launches of more row blocks than one round of workgroups takes, on rows above 4096 columns.
//
// gemv_rows_kernel serves several tokens whose rows the quantiser laid out for it.  gemv_mfma_kernel is the same
// weight-streaming scheme for 2..16 row-major token rows, which a caller brings or wants to see: the 16 x 16 x 64 int8 MFMA takes
// the place of the dot-product chain (its A operand is 16 token rows x 64 columns, loaded straight from the
// int8 activation matrix, which stays in L2; its B operand is a decoded weight dword, exactly as in the
// prefill GEMM), so up to 16 tokens cost what one costs in weight traffic and instructions.  A workgroup
// owns RB adjacent 16-row blocks so that the activation matrix is re-read by fewer workgroups.
#include <type_traits>

#include "kernels.hpp"
#include "rowsgemv.hpp"
#include "tiledot.hpp"
#include "ldsdma.hpp"

namespace bitnet {

namespace {

constexpr int MODE_PREQUANT = -1;
constexpr int GEMV_FUSED_MAX_ROWS = 8;   // tokens per fused quantiser + GEMV launch (a set of workgroups per token)
constexpr int GEMV_FUSED_MAX_WGS = 256;  // and its workgroups over all tokens: one per compute unit
constexpr int FUSED_NCH = 7;  // 16-byte f32 chunks per thread kept in registers: K <= 7168

struct GemvProjDev {
    const uint8_t *w;
    const float *w_scale;
    const float *bias;
    const float *residual;
    float *out;
    int32_t *acc;
    int n;
    int rb_end;  // row blocks of projections 0..this one, cumulative
};

struct GemvParams {
    GemvProjDev proj[GEMV_MAX_PROJ];
    int nproj;
    // MODE_PREQUANT: activations already int8
    const int8_t *a;
    const float *a_scale;
    // MODE >= 0: f32 input, quantised in the prologue
    RowSource src;
    int8_t *q_out;        // optional copies of what the prologue produced (written by workgroup 0)
    float *a_scale_out;
    int32_t *a_sum_out;
    int m;  // tokens in this launch (<= MB)
    int k;
    int kt_count;
};

constexpr int GEMV_PREFETCH = 4;  // tiles in flight per wavefront

template <int MB, int MODE>
__global__ __launch_bounds__(256) void gemv_tiled_kernel(GemvParams p)
{
    extern __shared__ uint4 lds_a[];  // [MB][groups]: int8 activations, 16 per uint4, zero past K / past m
    __shared__ int red[4][TILE_ROWS][MB];
    __shared__ float red_f[MB][2][4];
    __shared__ int red_i[MB][4];
    __shared__ float scale_s[MB];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int groups = p.kt_count * 16;

    // which projection, which of its row blocks
    int pj = 0;
#pragma unroll
    for (int j = 0; j < GEMV_MAX_PROJ - 1; ++j)
        if (j + 1 < p.nproj && (int)blockIdx.x >= p.proj[j].rb_end) pj = j + 1;
    const GemvProjDev &P = p.proj[pj];
    const int rb = (int)blockIdx.x - (pj ? p.proj[pj - 1].rb_end : 0);
    const uint4 *tiles = reinterpret_cast<const uint4 *>(P.w) + (size_t)rb * p.kt_count * 64;

    // Loads retire in issue order, so what the prologue waits for first is requested first: the f32 input row
    // of token 0 and the RMSNorm weights (L2 hits), then the first batch of weight tiles (HBM), whose latency
    // the quantiser prologue then hides.
    float4 v0[MODE == MODE_PREQUANT ? 1 : FUSED_NCH], gm[MODE == MODE_PREQUANT ? 1 : FUSED_NCH];
    if constexpr (MODE != MODE_PREQUANT) {
        const int chunks = p.k >> 2;
        const bool norm = p.src.gamma != nullptr;
#pragma unroll
        for (int i = 0; i < FUSED_NCH; ++i) {
            int c = tid + 256 * i;
            v0[i] = c < chunks ? load_chunk<MODE, true>(p.src, 0, c) : make_float4(0.f, 0.f, 0.f, 0.f);
            gm[i] = (norm && c < chunks) ? load_gamma_chunk(p.src, c, true) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    uint4 wbuf[GEMV_PREFETCH];
#pragma unroll
    for (int u = 0; u < GEMV_PREFETCH; ++u) {
        int kt = wave + 4 * u;
        wbuf[u] = load_weight_slot(tiles + (size_t)min(kt, p.kt_count - 1) * 64 + lane);  // unconditional: the waits can be counted
    }

    if constexpr (MODE == MODE_PREQUANT) {
        // Stage the int8 activations; every thread also accumulates sum_k a[t, k] for the code offset.
        const bool vec_ok = (p.k % 16 == 0) && ((reinterpret_cast<uintptr_t>(p.a) & 15) == 0);
#pragma unroll
        for (int t = 0; t < MB; ++t) {
            int local = 0;
            for (int g = tid; g < groups; g += 256) {
                uint4 v = make_uint4(0, 0, 0, 0);
                if (t < p.m) {
                    const int8_t *srcp = p.a + (size_t)t * p.k + 16 * (size_t)g;
                    if (vec_ok) {
                        if (16 * g < p.k) v = *reinterpret_cast<const uint4 *>(srcp);
                    } else {
                        uint32_t d[4] = {0, 0, 0, 0};
                        for (int j = 0; j < 16; ++j)
                            if (16 * g + j < p.k) d[j >> 2] |= (uint32_t)(uint8_t)srcp[j] << (8 * (j & 3));
                        v = make_uint4(d[0], d[1], d[2], d[3]);
                    }
                }
                lds_a[t * groups + g] = v;
                local = dot4(v.x, 0x01010101u, local);
                local = dot4(v.y, 0x01010101u, local);
                local = dot4(v.z, 0x01010101u, local);
                local = dot4(v.w, 0x01010101u, local);
            }
            local = wave_sum_i32(local);
            if (lane == 0) red_i[t][wave] = local;
            if (tid == 0) scale_s[t] = (t < p.m && p.a_scale) ? p.a_scale[t] : 1.0f;
        }
    } else {
        // Quantise the f32 input row(s) here: thread tid is virtual lane tid of the declared summation order.
        const RowSource &src = p.src;
        const int chunks = p.k >> 2;  // the host takes this path only when K % 4 == 0
        const int lds_words = groups * 4;
        uint32_t *lds_w = reinterpret_cast<uint32_t *>(lds_a);
        const bool norm = src.gamma != nullptr;
#pragma unroll
        for (int t = 0; t < MB; ++t) {
            if (t >= p.m) {  // uniform
                for (int c = tid; c < lds_words; c += 256) lds_w[t * lds_words + c] = 0;
                if (lane == 0) red_i[t][wave] = 0;
                if (tid == 0) scale_s[t] = 1.0f;
                continue;
            }
            float4 v[FUSED_NCH];
#pragma unroll
            for (int i = 0; i < FUSED_NCH; ++i) {
                int c = tid + 256 * i;
                if (t == 0) v[i] = v0[i];
                else v[i] = c < chunks ? load_chunk<MODE, true>(src, (size_t)t, c) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            Divisor rdiv = {1.0f, 1.0f, false};
            if (norm) {
                float ss;
                if (src.sum_order == BITNET_HIP_SUM_SEQUENTIAL) {
                    ss = sum_squares_sequential<MODE>(src, (size_t)t);
                } else {
                    float part = 0.0f;
#pragma unroll
                    for (int i = 0; i < FUSED_NCH; ++i) part = sum_squares4(part, v[i]);
                    part = wave_sum_f32(part);
                    if (lane == 0) red_f[t][0][wave] = part;
                    __syncthreads();
                    ss = f32_add(f32_add(f32_add(red_f[t][0][0], red_f[t][0][1]), red_f[t][0][2]), red_f[t][0][3]);
                }
                rdiv = make_divisor(rms_from_ss(ss, p.k, src.eps));
            }
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < FUSED_NCH; ++i) {
                int c = tid + 256 * i;
                if (norm && c < chunks) v[i] = normalize4(v[i], rdiv, gm[i]);
                amax = absmax4(amax, v[i]);
            }
            amax = wave_max_f32(amax);
            if (lane == 0) red_f[t][1][wave] = amax;
            __syncthreads();
            amax = fmaxf(fmaxf(red_f[t][1][0], red_f[t][1][1]), fmaxf(red_f[t][1][2], red_f[t][1][3]));
            const float scale = scale_from_absmax(amax);
            int isum = 0;
#pragma unroll
            for (int i = 0; i < FUSED_NCH; ++i) {
                int c = tid + 256 * i;
                if (c < chunks) {
                    uint32_t packed = quant4_packed(v[i], scale, &isum);
                    lds_w[t * lds_words + c] = packed;
                    if (p.q_out && blockIdx.x == 0) reinterpret_cast<uint32_t *>(p.q_out)[(size_t)t * chunks + c] = packed;
                } else if (c < lds_words) {
                    lds_w[t * lds_words + c] = 0;
                }
            }
            isum = wave_sum_i32(isum);
            if (lane == 0) red_i[t][wave] = isum;
            if (tid == 0) scale_s[t] = scale;
        }
    }
    __syncthreads();

    if constexpr (MODE != MODE_PREQUANT) {
        if (blockIdx.x == 0 && tid < MB && tid < p.m) {
            if (p.a_scale_out) p.a_scale_out[tid] = scale_s[tid];
            if (p.a_sum_out) p.a_sum_out[tid] = red_i[tid][0] + red_i[tid][1] + red_i[tid][2] + red_i[tid][3];
        }
    }

    int acc[MB];
#pragma unroll
    for (int t = 0; t < MB; ++t) acc[t] = 0;

    const int kq = lane >> 4;  // lane group: columns 64t + 16kq .. +15 of each tile, t = 0..3
    auto dot_batch = [&](int kt0) {
#pragma unroll
        for (int u = 0; u < GEMV_PREFETCH; ++u) {
            int kt = kt0 + 4 * u;
            if (kt < p.kt_count) {
                const uint4 *ag = lds_a + kt * 16 + kq;
#pragma unroll
                for (int t = 0; t < MB; ++t) acc[t] = dot64(wbuf[u], ag + t * groups, acc[t]);
            }
        }
    };
    for (int kt0 = wave; kt0 < p.kt_count; kt0 += 4 * GEMV_PREFETCH) {
        // two straight-line bodies: the last batch requests nothing more and waits for nothing but itself
        if (kt0 + 4 * GEMV_PREFETCH < p.kt_count) {  // uniform over the wavefront
            uint4 wnext[GEMV_PREFETCH];
#pragma unroll
            for (int u = 0; u < GEMV_PREFETCH; ++u)
                wnext[u] = load_weight_slot(tiles + (size_t)min(kt0 + 4 * (GEMV_PREFETCH + u), p.kt_count - 1) * 64 + lane);
            dot_batch(kt0);
#pragma unroll
            for (int u = 0; u < GEMV_PREFETCH; ++u) wbuf[u] = wnext[u];
        } else {
            dot_batch(kt0);
        }
    }

    // the four lanes l, l+16, l+32, l+48 hold the four column groups of row l mod 16
#pragma unroll
    for (int t = 0; t < MB; ++t) {
        acc[t] = sum_over_lane_groups(acc[t]);
    }
    if (lane < TILE_ROWS) {
#pragma unroll
        for (int t = 0; t < MB; ++t) red[wave][lane][t] = acc[t];
    }
    __syncthreads();

    if (tid < TILE_ROWS * MB) {
        const int r = tid / MB, t = tid % MB;
        const int n = rb * TILE_ROWS + r;
        if (n < P.n && t < p.m) {
            const int asum = red_i[t][0] + red_i[t][1] + red_i[t][2] + red_i[t][3];
            int total = red[0][r][t] + red[1][r][t] + red[2][r][t] + red[3][r][t] - asum;
            size_t o = (size_t)t * P.n + n;
            if (P.acc) P.acc[o] = total;
            if (P.out) {
                float v = f32_mul((float)total, *P.w_scale);
                v = f32_div(v, scale_s[t]);
                if (P.bias) v = f32_add(v, P.bias[n]);
                if (P.residual) v = f32_add(v, P.residual[o]);
                P.out[o] = v;
            }
        }
    }
}

// One token, f32 input: the quantiser runs in the prologue (see the head of this file).  Every load of the
// workgroup - input row, RMSNorm weights, all of its weight tiles - is issued up front and unconditionally
// (indices past the end are clamped and the values discarded), in the order in which the data is needed.  Loads
// return in issue order, so the compiler can wait for "all but the last n" and the weight tiles stay in
// flight while the row is normalised and quantised; the workgroup barriers order LDS traffic only, for the same
// reason.  NCH: 16-byte chunks of the row per thread, and weight tiles per wavefront (k <= 1024 * NCH).
template <int MODE, bool NORM, int NCH, int RBW>
__global__ __launch_bounds__(256) void gemv_fused_kernel(GemvParams p)
{
    extern __shared__ uint4 lds_a[];  // int8 activations, 16 per uint4, zero past K
    __shared__ int red[4][RBW][TILE_ROWS];
    __shared__ float red_f[2][4];
    __shared__ int red_i[4];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunks = p.k >> 2, lds_words = p.kt_count * 64;

    int pj = 0;
#pragma unroll
    for (int j = 0; j < GEMV_MAX_PROJ - 1; ++j)
        if (j + 1 < p.nproj && (int)blockIdx.x >= p.proj[j].rb_end) pj = j + 1;
    const GemvProjDev &P = p.proj[pj];
    const int rb0 = ((int)blockIdx.x - (pj ? p.proj[pj - 1].rb_end : 0)) * RBW;  // rb_end counts groups of RBW row blocks
    const int rb_count = (P.n + TILE_ROWS - 1) / TILE_ROWS;
    const uint4 *tiles = reinterpret_cast<const uint4 *>(P.w) + lane;

    float4 v[NCH], gm[NCH];
    uint4 wt[RBW][NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = min(tid + 256 * i, chunks - 1);
        v[i] = load_chunk<MODE, true>(p.src, 0, c);
    }
    // what the epilogue threads need from memory (weight scale, bias, residual of their output row) is requested
    // now as well, so that its latency is not paid at the end
    const int e_n = min((rb0 + (tid >> 4)) * TILE_ROWS + (tid & 15), P.n - 1);  // meaningful for tid < 16 * RBW
    const float e_ws = P.out ? *P.w_scale : 0.0f;
    const float e_bias = P.bias ? P.bias[e_n] : 0.0f;
    const float e_res = P.residual ? P.residual[e_n] : 0.0f;
    if constexpr (NORM) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) gm[i] = load_gamma_chunk(p.src, min(tid + 256 * i, chunks - 1), true);
    }
#pragma unroll
    for (int r = 0; r < RBW; ++r)
#pragma unroll
        for (int u = 0; u < NCH; ++u)  // row blocks past the end repeat the last one; their results are not stored
            wt[r][u] = load_weight_slot(tiles + ((size_t)min(rb0 + r, rb_count - 1) * p.kt_count + min(wave + 4 * u, p.kt_count - 1)) * 64);
#pragma unroll
    for (int i = 0; i < NCH; ++i)
        if (tid + 256 * i >= chunks) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);

    // thread tid is virtual lane tid of the declared summation order
    Divisor rdiv = {1.0f, 1.0f, false};
    if constexpr (NORM) {
        float ss;
        if (p.src.sum_order == BITNET_HIP_SUM_SEQUENTIAL) {
            // the reference's literal order: the squares go through LDS (the launch sizes it for them; the int8 row
            // takes the same place later, behind the barrier of the absmax reduction) and every wavefront runs the chain
            float *sq_lds = reinterpret_cast<float *>(lds_a);
#pragma unroll
            for (int i = 0; i < NCH; ++i)
                if (tid + 256 * i < chunks) store_squares4(sq_lds, tid + 256 * i, v[i]);
            lds_barrier();
            ss = sum_sequential_lds(sq_lds, p.k);
        } else {
            float part = 0.0f;
#pragma unroll
            for (int i = 0; i < NCH; ++i) part = sum_squares4(part, v[i]);
            part = wave_sum_f32(part);
            if (lane == 0) red_f[0][wave] = part;
            lds_barrier();
            ss = f32_add(f32_add(f32_add(red_f[0][0], red_f[0][1]), red_f[0][2]), red_f[0][3]);
        }
        rdiv = make_divisor(rms_from_ss(ss, p.k, p.src.eps));
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        if (NORM && tid + 256 * i < chunks) v[i] = normalize4(v[i], rdiv, gm[i]);
        amax = absmax4(amax, v[i]);
    }
    amax = wave_max_f32(amax);
    if (lane == 0) red_f[1][wave] = amax;
    lds_barrier();
    amax = fmaxf(fmaxf(red_f[1][0], red_f[1][1]), fmaxf(red_f[1][2], red_f[1][3]));
    const float scale = scale_from_absmax(amax);
    uint32_t *lds_w = reinterpret_cast<uint32_t *>(lds_a);
    int isum = 0;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = tid + 256 * i;
        if (c < chunks) {
            const uint32_t packed = quant4_packed(v[i], scale, &isum);
            lds_w[c] = packed;
            if (p.q_out && blockIdx.x == 0) reinterpret_cast<uint32_t *>(p.q_out)[c] = packed;
        } else if (c < lds_words) {
            lds_w[c] = 0;
        }
    }
    isum = wave_sum_i32(isum);
    if (lane == 0) red_i[wave] = isum;
    lds_barrier();

    const int kq = lane >> 4;  // lane group: columns 64t + 16kq .. +15 of each tile, t = 0..3
#pragma unroll
    for (int r = 0; r < RBW; ++r) {
        int acc = 0;
#pragma unroll
        for (int u = 0; u < NCH; ++u) {
            const int kt = wave + 4 * u;
            if (kt < p.kt_count) acc = dot64(wt[r][u], lds_a + kt * 16 + kq, acc);
        }
        // the four lanes l, l+16, l+32, l+48 hold the four column groups of row l mod 16
        acc = sum_over_lane_groups(acc);
        if (lane < TILE_ROWS) red[wave][r][lane] = acc;
    }
    lds_barrier();

    if (tid < TILE_ROWS * RBW) {
        const int r = tid >> 4, row = tid & 15;
        const int n = (rb0 + r) * TILE_ROWS + row;
        const int asum = red_i[0] + red_i[1] + red_i[2] + red_i[3];
        if (blockIdx.x == 0 && tid == 0) {
            if (p.a_scale_out) p.a_scale_out[0] = scale;
            if (p.a_sum_out) p.a_sum_out[0] = asum;
        }
        if (n < P.n) {
            const int total = red[0][r][row] + red[1][r][row] + red[2][r][row] + red[3][r][row] - asum;
            if (P.acc) P.acc[n] = total;
            if (P.out) {
                float y = f32_mul((float)total, e_ws);
                y = f32_div(y, scale);
                if (P.bias) y = f32_add(y, e_bias);
                if (P.residual) y = f32_add(y, e_res);
                P.out[n] = y;
            }
        }
    }
}

// The same launch with up to 16 wavefronts per workgroup: the default.  One wavefront per 256-column k-tile (nw wavefronts;
// NCHB = 2: two tiles each, w and w + nw), a lane per 16-byte chunk of the tile: the element-wise steps run once, in
// parallel, and what the launch takes is the chain of dependent steps.  At the decode shapes that chain, not memory, is
// the bound: a launch whose workgroups only read the row and their cold weight tiles behind a barrier takes 2.2 us, and the
// stack is as fast on weights that fit the last-level cache as on ones that do not.  So everything here is about the chain:
//   * All arguments are in registers before the first barrier.  Scalar loads that the compiler places at their use (the
//     width, eps, the output pointers) each cost a trip to L2 between two barriers.  What the first loads need arrives
//     preloaded; the rest is fetched while the row is on its way, and pinned.
//   * A lane's chunk is chosen so that the quantised row never goes through LDS.  Inside a tile, lane 16 kq + 4 t + u takes chunk
//     16 t + 4 kq + u (columns 64 t + 16 kq + 4 u .. + 3), so that row broadcasts bring a lane the 16 columns 64 t + 16 kq .. + 15
//     that dword t of its weight slot stands for: the A operand of MFMA t, all 16 rows of it the one row there is.  With four
//     and more row blocks per workgroup taking the codes apart is what the matrix part waits for: MFMA u then takes the codes
//     at bits 2u of all four dwords, for u < 3 in place (dword & (3 << 2u); the factor 4^u is shifted out between the
//     MFMAs), 20 vector operations a tile instead of 28, and its A operand is the broadcasts of t = 0..3 for that u.
//   * The row's sum for the code offset is an MFMA on a constant operand.
//   * Wavefront reductions end in lane 63 by DPP row broadcasts, one instruction a step.
// The sum of squares keeps the declared order: chunk c belongs to virtual lane c % 256, whose chain runs over its chunks in
// ascending order, so threads 0..255 (one per virtual lane) also fetch their lane's chunks (from L2, with the first loads of
// the kernel) and add the squares up in that order, then the four 64-lane butterflies as before.  The partial sums of a
// row meet in LDS atomics (int32: any order gives the same sum).
// A block of the 30-block stack (2560 / 6912), replayed, at one token: 16.5 us before these points, 14.8 with them; at four tokens
// 23.9 and 22.3.

template <int MODE, bool NORM, int NCHB, int RBW>
__global__ __launch_bounds__(1024) void gemv_fused16_kernel(const float *hot_x, const float *hot_x2, const float *hot_gamma, int hot_k, int hot_head_chunks,
                                                           int hot_nw, int hot_ldx, int hot_end0, int hot_end1, [[maybe_unused]] Fused16Params args)
{
    // A launch has one to eight tokens (input rows), each with its own workgroups.  Workgroup (x, y) of the grid works on
    // token x / 8 and on group 8y + x % 8 of row blocks: the workgroups of one group are neighbours in dispatch order and,
    // workgroups going to the XCDs in turn, run on the same XCD, so its L2 fetches their weight tiles once.
    // The leading scalar arguments are what the first loads need (input rows, RMSNorm weights, k): the file is compiled with
    // kernel-argument preloading, so they arrive in registers with the wavefront.
    __shared__ float red_f[2][16];
    __shared__ int tot[RBW][TILE_ROWS];
    __shared__ int asum_s;

    const size_t tok = blockIdx.x >> 3;
    const int group = (int)blockIdx.y * 8 + (int)(blockIdx.x & 7);  // may lie past the last group: such workgroups store nothing
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = hot_nw, chunks = hot_k >> 2;
    const float *row = hot_x + tok * (size_t)hot_ldx;
    const float *row2 = MODE == BITNET_HIP_INPUT_RELU2_MUL ? hot_x2 + tok * (size_t)hot_ldx : nullptr;
    const uint64_t magics = MODE == BITNET_HIP_INPUT_GQA_BROADCAST ? reinterpret_cast<uintptr_t>(hot_x2) : 0;

    // The loads that need no argument but the preloaded ones, unconditional (clamped indices, values discarded).
    const int in_tile = 16 * ((lane >> 2) & 3) + 4 * (lane >> 4) + (lane & 3);
    Row16<NORM, NCHB> row16;
    row16.template load<MODE, (RBW > 1)>(row, row2, magics, hot_head_chunks, hot_gamma, chunks, nw, wave, tid, in_tile);
    __builtin_amdgcn_sched_barrier(0);

    // The other arguments, all at once, and pinned here.  Which projection a workgroup serves it knows from the preloaded
    // ends of the first two (INT_MAX where there is no next one).
    typedef const __attribute__((address_space(4))) v16u *arg_ptr;
    const arg_ptr blocks = (arg_ptr)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + FUSED16_ARGS_AT);
    const int pj = group < hot_end0 ? 0 : (group < hot_end1 ? 1 : 2), first_group = group < hot_end0 ? 0 : (group < hot_end1 ? hot_end0 : hot_end1);
    v16u common = blocks[0], P = blocks[1 + pj];
    if (tid < RBW * TILE_ROWS) tot[tid >> 4][tid & 15] = 0;
    if (tid < 16 && tid >= nw) red_f[1][tid] = 0.0f;  // the slots of absent wavefronts hold the neutral element
    if (tid == 0) asum_s = 0;
    float k_f = (float)hot_k, k_recip = recip_of_ok_divisor(k_f);  // k <= 16384: a divisor the short division accepts
    asm volatile("" : "+s"(common), "+s"(P), "+v"(k_recip));
    const int kt_count = (int)common[0];
    const float eps = __builtin_bit_cast(float, (unsigned)common[1]);
    const global_ptr<uint32_t> q_out = pointer_at<uint32_t>(common, 4);
    const global_ptr<float> a_scale_out = pointer_at<float>(common, 6);
    const global_ptr<int32_t> a_sum_out = pointer_at<int32_t>(common, 8);
    const global_ptr<const float> absent = (global_ptr<const float>)(uintptr_t)hot_x;
    const global_ptr<const float> w_scale = pointer_at<const float>(P, 2), bias = pointer_at<const float>(P, 4), residual = pointer_at<const float>(P, 6);
    const global_ptr<float> out = pointer_at<float>(P, 8);
    const global_ptr<int32_t> acc_out = pointer_at<int32_t>(P, 10);
    const int P_n = (int)P[12];
    const int rb0 = (group - first_group) * RBW;  // rb_end counts groups of RBW row blocks
    const int rb_count = (P_n + TILE_ROWS - 1) / TILE_ROWS;
    // Epilogue operands, fetched by the wavefronts that store; absent ones read the input row instead (always there) and are
    // not used.  The weight scale goes through a per-lane address so that it is a vector load, which nothing waits for
    // before the epilogue.
    float e_ws = 0.0f, e_bias = 0.0f, e_res = 0.0f;
    if (64 * wave < TILE_ROWS * RBW) {
        const int e_n = min((rb0 + (tid >> 4)) * TILE_ROWS + (tid & 15), P_n - 1);
        int lane_zero = 0;
        asm volatile("" : "+v"(lane_zero));
        e_ws = (out ? w_scale : absent)[lane_zero];
        e_bias = *(bias ? bias + e_n : absent);
        e_res = *(residual ? residual + (tok * (size_t)P_n + e_n) : absent);
    }
    // The weight tiles (tiles and row blocks past the end repeat the last one; their results are not added), non-temporal.
    // The vector memory of a compute unit answers in the order of the requests, whichever wavefront they are from: a tile
    // that comes from memory would hold up the input row of a wavefront that asked a little later.  So all wavefronts meet
    // once their row is requested, and ask for the tiles then.
    const global_ptr<const v4u_t> tiles = pointer_at<const v4u_t>(P, 0) + lane;
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    v4u_t wt[RBW][NCHB];
#pragma unroll
    for (int r = 0; r < RBW; ++r)
#pragma unroll
        for (int i = 0; i < NCHB; ++i)
            wt[r][i] = __builtin_nontemporal_load(tiles + ((size_t)min(rb0 + r, rb_count - 1) * kt_count + min(wave + nw * i, kt_count - 1)) * 64);
    __builtin_amdgcn_sched_barrier(0);
    uint32_t packed[NCHB];
    const float scale = row16.quantise(chunks, k_f, k_recip, eps, wave, tid, red_f, packed);

    v4i acc[RBW], sums = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < RBW; ++r) acc[r] = (v4i){0, 0, 0, 0};
    constexpr bool IN_PLACE = RBW >= 4;
#pragma unroll
    for (int i = 0; i < NCHB; ++i) {
        if (NCHB > 1 && wave + nw * i >= kt_count) break;  // uniform over the wavefront
        if (q_out && group == 0 && row16.chunk[i] < chunks) q_out[tok * (size_t)chunks + row16.chunk[i]] = packed[i];
        const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
        v4i af[4];  // the A operands: chunk (t, u) of a column group is in its lane 4t + u
#pragma unroll
        for (int j = 0; j < 4; ++j)
            af[j] = IN_PLACE ? (v4i){row_lane(packed[i], j), row_lane(packed[i], 4 + j), row_lane(packed[i], 8 + j), row_lane(packed[i], 12 + j)}
                             : (v4i){row_lane(packed[i], 4 * j), row_lane(packed[i], 4 * j + 1), row_lane(packed[i], 4 * j + 2), row_lane(packed[i], 4 * j + 3)};
#pragma unroll
        for (int j = 0; j < 4; ++j) sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[j], ones, sums, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < RBW; ++r) {
            const v4u_t w4 = wt[r][i];
            if constexpr (IN_PLACE) {
                auto codes = [&](unsigned mask, int shift) {
                    return (v4i){(int)((w4[0] >> shift) & mask), (int)((w4[1] >> shift) & mask), (int)((w4[2] >> shift) & mask), (int)((w4[3] >> shift) & mask)};
                };
                v4i part = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[2], codes(0x30303030u, 0), (v4i){0, 0, 0, 0}, 0, 0, 0);
                part[0] >>= 2;  // 16 times the sum; only the first result register is used
                part = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[1], codes(0x0c0c0c0cu, 0), part, 0, 0, 0);
                part[0] >>= 2;
                part = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[0], codes(0x03030303u, 0), part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[3], codes(0x03030303u, 6), part, 0, 0, 0);
                acc[r][0] += part[0];
            } else {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[t], (v4i){(int)(w4[t] & 0x03030303u), (int)((w4[t] >> 2) & 0x03030303u),
                                                                                (int)((w4[t] >> 4) & 0x03030303u), (int)((w4[t] >> 6) & 0x03030303u)},
                                                                   acc[r], 0, 0, 0);
            }
        }
    }
    if (wave < kt_count && lane < TILE_ROWS) {  // wavefronts beyond the row's tiles hold a repeated tile: nothing of theirs is added
#pragma unroll
        for (int r = 0; r < RBW; ++r) atomicAdd(&tot[r][lane], acc[r][0] - sums[0]);
        if (a_sum_out && lane == 0) atomicAdd(&asum_s, sums[0]);
    }
    const float s_recip = recip_of_ok_divisor(scale);
    const bool divisor_fits = invariant_divisor_ok(scale);
    lds_barrier();

    if (tid < TILE_ROWS * RBW) {
        const int r = tid >> 4, rw = tid & 15;
        const int n = (rb0 + r) * TILE_ROWS + rw;
        const int total = tot[r][rw];
        const float scaled = f32_mul((float)total, e_ws);
        float y = div_by_invariant_unchecked(scaled, scale, s_recip);
        if (__builtin_expect(!(divisor_fits && dividend_ok(scaled)), 0)) y = f32_div(scaled, scale);
        if (bias) y = f32_add(y, e_bias);
        if (residual) y = f32_add(y, e_res);
        if (n < P_n) {
            if (acc_out) acc_out[tok * (size_t)P_n + n] = total;
            if (out) out[tok * (size_t)P_n + n] = y;
        }
        if (group == 0 && tid == 0) {
            if (a_scale_out) a_scale_out[tok] = scale;
            if (a_sum_out) a_sum_out[tok] = asum_s;
        }
    }
}

struct GemvMfmaParams {
    GemvProjDev proj[GEMV_MAX_PROJ];  // rb_end counts groups of RB row blocks
    int nproj;
    const int8_t *a;       // [m, k] int8
    const float *a_scale;  // [m]
    int m;                 // 1..16
    int k;
    int kt_count;
};

// MT: groups of 16 token rows (m <= 16 * MT); a decoded weight dword then feeds MT MFMAs.
// FAST: k is a multiple of 256 and the activations are 16-byte aligned.  Every load is then unconditional
// (indices past the end are clamped, the values discarded), so the compiler can count the loads in flight
// and the next batch of tiles really stays outstanding while the current one is multiplied.
// ONE: the wavefront's k-tiles (at most 8: k <= 8192) form a single batch, requested as a whole at the start: one
// memory latency instead of one per batch (RB = MT = 1 only, where the registers allow it).
template <int RB, int MT, bool FAST, bool ONE = false>
__global__ __launch_bounds__(256) void gemv_mfma_kernel(const int8_t *hot_a, int hot_k, int hot_m, int hot_kt_count, GemvMfmaParams p)
{
    // the leading scalar arguments repeat the fields a, k, m and kt_count of p, which the first address computations need;
    // they are preloaded into registers (see the Makefile) and used in place of the fields throughout
    __shared__ int red[4][RB][MT][64][4];  // partial accumulators of the four wavefronts
    __shared__ int red_sum[4][MT][16];     // per wavefront: sum_k a[t, k] over its k-tiles

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 15, lg = lane >> 4;

    // A operand of this lane in token group g: token row 16g + lr, the 16 columns 64t + 16lg of each k-tile
    // (rows past m read as zero)
    const bool a_vec = (hot_k % 16 == 0) && ((reinterpret_cast<uintptr_t>(hot_a) & 15) == 0);
    bool row_ok[MT];
    const int8_t *arow[MT];
#pragma unroll
    for (int g = 0; g < MT; ++g) {
        row_ok[g] = 16 * g + lr < hot_m;
        arow[g] = hot_a + (size_t)(row_ok[g] ? 16 * g + lr : 0) * hot_k + lg * 16;
    }
    auto load_a = [&](int g, int kt, int t) -> v4i {
        if constexpr (FAST) {
            const v4i v = *reinterpret_cast<const v4i *>(arow[g] + min(kt, hot_kt_count - 1) * TILE_K + t * 64);
            return row_ok[g] ? v : (v4i){0, 0, 0, 0};
        }
        v4i v = (v4i){0, 0, 0, 0};
        const int col = kt * TILE_K + t * 64 + lg * 16;
        if (row_ok[g] && col < hot_k) {
            const int8_t *src = arow[g] + kt * TILE_K + t * 64;
            if (a_vec) {
                v = *reinterpret_cast<const v4i *>(src);
            } else {
                int d[4] = {0, 0, 0, 0};
                for (int j = 0; j < 16; ++j)
                    if (col + j < hot_k) d[j >> 2] |= (int)((uint32_t)(uint8_t)src[j] << (8 * (j & 3)));
                v = (v4i){d[0], d[1], d[2], d[3]};
            }
        }
        return v;
    };
    static_assert(!ONE || MT == 1, "single batch: one token group");
    constexpr int PF = ONE ? (RB == 1 ? 8 : (RB == 2 ? 4 : 3))
                           : (RB * MT == 1 ? 4 : (RB * MT == 2 ? 3 : (MT <= 2 ? 2 : 1)));  // bounded by the register file
    // All loads of a batch of PF k-tiles are issued before the first MFMA of the batch, and the next
    // batch is requested while the current one is computed: the weight stream is what the kernel waits for.
    uint4 wcur[PF][RB], wnxt[ONE ? 1 : PF][RB];
    v4i acur[PF][MT][4], anxt[ONE ? 1 : PF][MT][4];
    // The first batch: the activations are addressed by the preloaded arguments alone, so with FAST they are requested
    // before anything reads the argument buffer (the weights' address comes from there).
    if constexpr (FAST) {
#pragma unroll
        for (int u = 0; u < PF; ++u)
#pragma unroll
            for (int g = 0; g < MT; ++g)
#pragma unroll
                for (int t = 0; t < 4; ++t) acur[u][g][t] = load_a(g, wave + 4 * u, t);
    }
    __builtin_amdgcn_sched_barrier(0);  // nothing below moves above: the first wait for the argument buffer comes here

    int pj = 0;
#pragma unroll
    for (int j = 0; j < GEMV_MAX_PROJ - 1; ++j)
        if (j + 1 < p.nproj && (int)blockIdx.x >= p.proj[j].rb_end) pj = j + 1;
    const GemvProjDev &P = p.proj[pj];
    const int grp = (int)blockIdx.x - (pj ? p.proj[pj - 1].rb_end : 0);
    const int rb0 = grp * RB;
    const int rb_count = (P.n + TILE_ROWS - 1) / TILE_ROWS;
    const uint4 *wbase = reinterpret_cast<const uint4 *>(P.w) + lane;


    auto load_w = [&](int kt, uint4 (&w)[RB]) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int rb = rb0 + r;
            if constexpr (FAST)  // results of row blocks past the end are never stored
                w[r] = load_weight_slot(wbase + ((size_t)min(rb, rb_count - 1) * hot_kt_count + min(kt, hot_kt_count - 1)) * 64);
            else
                w[r] = rb < rb_count ? load_weight_slot(wbase + ((size_t)rb * hot_kt_count + kt) * 64)
                                     : make_uint4(0x55555555u, 0x55555555u, 0x55555555u, 0x55555555u);
        }
    };

    constexpr int NFRAG = RB * MT, FPW = (NFRAG + 3) / 4;  // fragments, fragments per wavefront
    v4i acc[RB][MT];
    int rowsum[MT];
#pragma unroll
    for (int g = 0; g < MT; ++g) {
        rowsum[g] = 0;
#pragma unroll
        for (int r = 0; r < RB; ++r) acc[r][g] = (v4i){0, 0, 0, 0};
    }

    auto load_batch = [&](int kt0, uint4 (&w)[PF][RB], v4i (&a)[PF][MT][4]) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            const int kt = kt0 + 4 * u;
            if (FAST || kt < hot_kt_count) {
                load_w(kt, w[u]);
#pragma unroll
                for (int g = 0; g < MT; ++g)
#pragma unroll
                    for (int t = 0; t < 4; ++t) a[u][g][t] = load_a(g, kt, t);
            }
        }
    };
    if constexpr (FAST) {  // the activations of the first batch are on their way already
#pragma unroll
        for (int u = 0; u < PF; ++u) load_w(wave + 4 * u, wcur[u]);
    } else {
        load_batch(wave, wcur, acur);
    }
    __builtin_amdgcn_sched_barrier(0);

    auto compute_batch = [&](int kt0) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            if (kt0 + 4 * u >= hot_kt_count) continue;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int g = 0; g < MT; ++g) {
                    const v4i af = acur[u][g][t];
                    rowsum[g] = __builtin_amdgcn_sdot4(af[0], 0x01010101, rowsum[g], false);
                    rowsum[g] = __builtin_amdgcn_sdot4(af[1], 0x01010101, rowsum[g], false);
                    rowsum[g] = __builtin_amdgcn_sdot4(af[2], 0x01010101, rowsum[g], false);
                    rowsum[g] = __builtin_amdgcn_sdot4(af[3], 0x01010101, rowsum[g], false);
                }
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    const uint4 w4 = wcur[u][r];
                    const uint32_t wd = t == 0 ? w4.x : (t == 1 ? w4.y : (t == 2 ? w4.z : w4.w));
                    v4i bf;
                    bf[0] = (int)(wd & 0x03030303u);
                    bf[1] = (int)((wd >> 2) & 0x03030303u);
                    bf[2] = (int)((wd >> 4) & 0x03030303u);
                    bf[3] = (int)((wd >> 6) & 0x03030303u);
#pragma unroll
                    for (int g = 0; g < MT; ++g)
                        acc[r][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(acur[u][g][t], bf, acc[r][g], 0, 0, 0);
                }
            }
        }
    };
    // The RB * MT fragments (row block, token group) are finished by the wavefronts in turn: fragment
    // q = wave + 4 * f is (row block q / MT, token group q % MT); result register i of a lane belongs to token
    // 16g + 4*(lane/16) + i.  Scales, bias and residuals are requested now, behind the first batch of the main loads, so
    // that their latency is not paid at the end.  Absent operands read the weight tiles instead (always there; the
    // values are not used), which keeps this part free of branches, and the weight scale goes through a per-lane address:
    // a vector load, which nothing waits for before the epilogue.
    const float *absent = reinterpret_cast<const float *>(P.w);
    int lane_zero = 0;
    asm volatile("" : "+v"(lane_zero));
    const float ws = (P.out ? P.w_scale : absent)[lane_zero];
    float e_bias[FPW], e_scale[FPW][4], e_res[FPW][4];
#pragma unroll
    for (int f = 0; f < FPW; ++f) {
        const int q = min(wave + 4 * f, NFRAG - 1), fr = q / MT, fg = q % MT;
        const int e_n = min((rb0 + fr) * TILE_ROWS + lr, P.n - 1);
        e_bias[f] = *(P.bias ? P.bias + e_n : absent);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = min(16 * fg + lg * 4 + i, hot_m - 1);
            e_scale[f][i] = *(P.out ? p.a_scale + t : absent);
            e_res[f][i] = *(P.residual ? P.residual + ((size_t)t * P.n + e_n) : absent);
        }
    }

    if constexpr (ONE) {
        compute_batch(wave);
    } else
    for (int kt0 = wave; kt0 < hot_kt_count; kt0 += 4 * PF) {
        // two straight-line bodies, so that the wait before the MFMAs is for this batch only in both of them
        if constexpr (!ONE) {
            if (kt0 + 4 * PF < hot_kt_count) {  // uniform over the wavefront
                load_batch(kt0 + 4 * PF, wnxt, anxt);
                compute_batch(kt0);
#pragma unroll
                for (int u = 0; u < PF; ++u) {
#pragma unroll
                    for (int r = 0; r < RB; ++r) wcur[u][r] = wnxt[u][r];
#pragma unroll
                    for (int g = 0; g < MT; ++g)
#pragma unroll
                        for (int t = 0; t < 4; ++t) acur[u][g][t] = anxt[u][g][t];
                }
            } else {
                compute_batch(kt0);
            }
        }
    }

    // sum_k a[row, k] over this wavefront's tiles: lanes lr, lr+16, lr+32, lr+48 hold the four column groups
#pragma unroll
    for (int g = 0; g < MT; ++g) {
        rowsum[g] = sum_over_lane_groups(rowsum[g]);
        if (lane < 16) red_sum[wave][g][lane] = rowsum[g];
    }
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int g = 0; g < MT; ++g)
            *reinterpret_cast<v4i *>(&red[wave][r][g][lane][0]) = acc[r][g];
    lds_barrier();
#pragma unroll
    for (int f = 0; f < FPW; ++f) {
        if (wave + 4 * f >= NFRAG) break;  // uniform over the wavefront
        const int q = wave + 4 * f, fr = q / MT, fg = q % MT;
        const int n = (rb0 + fr) * TILE_ROWS + lr;  // result register i of lane l is C[4*(l/16) + i][l mod 16]
        const v4i s0 = *reinterpret_cast<const v4i *>(&red[0][fr][fg][lane][0]), s1 = *reinterpret_cast<const v4i *>(&red[1][fr][fg][lane][0]);
        const v4i s2 = *reinterpret_cast<const v4i *>(&red[2][fr][fg][lane][0]), s3 = *reinterpret_cast<const v4i *>(&red[3][fr][fg][lane][0]);
        const v4i sum = s0 + s1 + s2 + s3;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tl = lg * 4 + i, t = 16 * fg + tl;
            if (n < P.n && t < hot_m) {
                const int asum = red_sum[0][fg][tl] + red_sum[1][fg][tl] + red_sum[2][fg][tl] + red_sum[3][fg][tl];
                const int total = sum[i] - asum;
                const size_t o = (size_t)t * P.n + n;
                if (P.acc) P.acc[o] = total;
                if (P.out) {
                    float v = f32_div(f32_mul((float)total, ws), e_scale[f][i]);
                    if (P.bias) v = f32_add(v, e_bias[f]);
                    if (P.residual) v = f32_add(v, e_res[f][i]);
                    P.out[o] = v;
                }
            }
        }
    }
}

// gemv_mfma_kernel for up to 16 tokens with the activations staged through LDS.  There every wavefront gathers its A
// fragments straight from memory: 16 bytes per lane from 16 different rows, four loads per k-tile, and the address
// unit of the compute unit spends more time on those gathers than the weight stream needs.  Here the workgroup copies
// the m rows into LDS once with dense loads (thread t takes the 16-byte chunks t, t + 256, .. of every row) and the
// fragments are LDS reads.  Rows are k + 16 bytes apart in LDS.  KCLASS 0: k <= 3072 (one chunk column per thread,
// three k-tiles per wavefront), KCLASS 1: k <= 8192 and m <= 8 (two chunk columns, eight k-tiles).  k % 256 == 0, the
// activations 16-byte aligned, m * (k + 16) bytes of dynamic LDS.
template <int RB, int KCLASS>
__global__ __launch_bounds__(256) void gemv_mfma_lds_kernel(const int8_t *hot_a, int hot_k, int hot_m, int hot_kt_count, GemvMfmaParams p)
{
    constexpr int JN = KCLASS == 0 ? 1 : 2, NT = KCLASS == 0 ? 3 : 8;
    extern __shared__ uint4 lds_act[];        // [m][k / 16 + 1] chunks of 16 int8
    __shared__ int red[4][RB][64][4];         // partial accumulators of the four wavefronts
    __shared__ int red_sum[4][16];            // per wavefront: sum_k a[t, k] over its k-tiles

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int cpr = hot_k >> 4, stride = cpr + 1;  // chunks per row in memory and in LDS

    // the copy's loads first: they are addressed by the preloaded arguments alone (unconditional: rows past m repeat
    // the last row, chunks past the row its last chunk; those are not stored)
    v4i stage[16];
    const v4i *a_chunks = reinterpret_cast<const v4i *>(hot_a);
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int r = min(s / JN, hot_m - 1), cc = min(tid + 256 * (s % JN), cpr - 1);
        stage[s] = a_chunks[(size_t)r * cpr + cc];
    }
    __builtin_amdgcn_sched_barrier(0);  // nothing below moves above: the first wait for the argument buffer comes here

    int pj = 0;
#pragma unroll
    for (int j = 0; j < GEMV_MAX_PROJ - 1; ++j)
        if (j + 1 < p.nproj && (int)blockIdx.x >= p.proj[j].rb_end) pj = j + 1;
    const GemvProjDev &P = p.proj[pj];
    const int rb0 = ((int)blockIdx.x - (pj ? p.proj[pj - 1].rb_end : 0)) * RB;
    const int rb_count = (P.n + TILE_ROWS - 1) / TILE_ROWS;
    const uint4 *wbase = reinterpret_cast<const uint4 *>(P.w) + lane;
    __builtin_amdgcn_sched_barrier(0);
    // The copy's stores, then everyone may read the rows.  The weight stream is requested only now: megabytes from all
    // workgroups at once, behind which the activations (and the argument buffers of workgroups that start a little
    // later) would queue in the memory system; this way they arrive about as early as they can, and the weights about
    // when they would have anyway.
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int r = s / JN, cc = tid + 256 * (s % JN);
        if (r < hot_m && cc < cpr) reinterpret_cast<v4i *>(lds_act)[r * stride + cc] = stage[s];
    }
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
    // all k-tiles of this wavefront (kt = wave + 4u) in one batch; tiles and row blocks past the end repeat the last one
    uint4 w[NT][RB];
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < RB; ++r)
            w[u][r] = load_weight_slot(wbase + ((size_t)min(rb0 + r, rb_count - 1) * hot_kt_count + min(wave + 4 * u, hot_kt_count - 1)) * 64);

    // Row block q = wave + 4f of the workgroup is finished by this wavefront; scales, bias and residuals are requested now
    // (absent operands read the weight tiles instead, the values are not used; the weight scale goes through a per-lane
    // address: a vector load, which nothing waits for before the epilogue).
    constexpr int FPW = (RB + 3) / 4;
    const float *absent = reinterpret_cast<const float *>(P.w);
    int lane_zero = 0;
    asm volatile("" : "+v"(lane_zero));
    const float ws = (P.out ? P.w_scale : absent)[lane_zero];
    float e_bias[FPW], e_scale[FPW][4], e_res[FPW][4];
#pragma unroll
    for (int f = 0; f < FPW; ++f) {
        const int fr = min(wave + 4 * f, RB - 1);
        const int e_n = min((rb0 + fr) * TILE_ROWS + lr, P.n - 1);
        e_bias[f] = *(P.bias ? P.bias + e_n : absent);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = min(lg * 4 + i, hot_m - 1);
            e_scale[f][i] = *(P.out ? p.a_scale + t : absent);
            e_res[f][i] = *(P.residual ? P.residual + ((size_t)t * P.n + e_n) : absent);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    v4i acc[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[r] = (v4i){0, 0, 0, 0};
    int rowsum = 0;
    const bool row_ok = lr < hot_m;
    const uint4 *arow = lds_act + (row_ok ? lr : 0) * stride + lg;  // A operand: token row lr, columns 64t + 16lg .. +15 of a k-tile
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int kt = wave + 4 * u;
        if (kt < hot_kt_count) {  // uniform over the wavefront
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v4i af = (v4i){0, 0, 0, 0};
                if (row_ok) af = *reinterpret_cast<const v4i *>(arow + kt * 16 + t * 4);
                rowsum = __builtin_amdgcn_sdot4(af[0], 0x01010101, rowsum, false);
                rowsum = __builtin_amdgcn_sdot4(af[1], 0x01010101, rowsum, false);
                rowsum = __builtin_amdgcn_sdot4(af[2], 0x01010101, rowsum, false);
                rowsum = __builtin_amdgcn_sdot4(af[3], 0x01010101, rowsum, false);
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    const uint4 w4 = w[u][r];
                    const uint32_t wd = t == 0 ? w4.x : (t == 1 ? w4.y : (t == 2 ? w4.z : w4.w));
                    v4i bf;
                    bf[0] = (int)(wd & 0x03030303u);
                    bf[1] = (int)((wd >> 2) & 0x03030303u);
                    bf[2] = (int)((wd >> 4) & 0x03030303u);
                    bf[3] = (int)((wd >> 6) & 0x03030303u);
                    acc[r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, bf, acc[r], 0, 0, 0);
                }
            }
        }
    }

    // sum_k a[row, k] over this wavefront's tiles: lanes lr, lr+16, lr+32, lr+48 hold the four column groups
    rowsum = sum_over_lane_groups(rowsum);
    if (lane < 16) red_sum[wave][lane] = rowsum;
#pragma unroll
    for (int r = 0; r < RB; ++r) *reinterpret_cast<v4i *>(&red[wave][r][lane][0]) = acc[r];
    lds_barrier();
#pragma unroll
    for (int f = 0; f < FPW; ++f) {
        if (wave + 4 * f >= RB) break;  // uniform over the wavefront
        const int fr = wave + 4 * f;
        const int n = (rb0 + fr) * TILE_ROWS + lr;  // result register i of lane l is C[4*(l/16) + i][l mod 16]
        const v4i s0 = *reinterpret_cast<const v4i *>(&red[0][fr][lane][0]), s1 = *reinterpret_cast<const v4i *>(&red[1][fr][lane][0]);
        const v4i s2 = *reinterpret_cast<const v4i *>(&red[2][fr][lane][0]), s3 = *reinterpret_cast<const v4i *>(&red[3][fr][lane][0]);
        const v4i sum = s0 + s1 + s2 + s3;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = lg * 4 + i;
            if (n < P.n && t < hot_m) {
                const int asum = red_sum[0][t] + red_sum[1][t] + red_sum[2][t] + red_sum[3][t];
                const int total = sum[i] - asum;
                const size_t o = (size_t)t * P.n + n;
                if (P.acc) P.acc[o] = total;
                if (P.out) {
                    float v = f32_div(f32_mul((float)total, ws), e_scale[f][i]);
                    if (P.bias) v = f32_add(v, e_bias[f]);
                    if (P.residual) v = f32_add(v, e_res[f][i]);
                    P.out[o] = v;
                }
            }
        }
    }
}

// 17 and more tokens: gemv_mfma_lds_kernel's scheme with the tokens cut into groups of 16, one workgroup per
// (group of RB row blocks, token group).  gemv_mfma_kernel gives every workgroup ALL token rows (16 * MT of them) for
// its 16 * RB output rows, gathered per wavefront straight from memory: at 64 tokens that is 164 KB (k = 2560) to
// 442 KB (k = 6912) through the one L1 of a compute unit for 32 output rows, 70 MB of L2 traffic per launch for a
// 4.4 MB weight matrix, and the kernel takes 11 to 15 us.  Here a workgroup copies only its 16 token rows into LDS
// (dense 16-byte loads, rows k + 16 bytes apart) and the weight tiles are read once per token group: with the token
// groups of a row-block group placed on the same XCD, from HBM once and from that XCD's L2 afterwards.
// The copy is made by LDS-direct loads, all in flight at once, and the wavefront's k-tiles (kt = wave + 4u, at most NT of
// them) are requested as one batch right behind it, so the two latencies overlap.  k % 256 == 0, activations 16-byte
// aligned, m * k < 4 GiB, 16 * (k + 16) bytes of dynamic LDS rounded up to a whole KiB (the copy stores whole loads).
template <int RB, int NT>
__global__ __launch_bounds__(256) void gemv_mfma_tg_kernel(const int8_t *hot_a, int hot_k, int hot_m, int hot_kt_count, int hot_groups,
                                                           int hot_tgroups, GemvMfmaParams p)
{
    extern __shared__ uint4 lds_act[];        // [16][k / 16 + 1] chunks of 16 int8
    __shared__ int red[4][RB][64][4];         // partial accumulators of the four wavefronts
    __shared__ int red_sum[4][16];            // per wavefront: sum_k a[t, k] over its k-tiles

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lg = lane >> 4;
    const int cpr = hot_k >> 4, stride = cpr + 1;  // chunks per row in memory and in LDS

    // Workgroups go to the eight XCDs in turn: the ids that share an XCD walk the (row-block group, token group) pairs
    // with the token group fastest, so the token groups of one row-block group meet in one L2.
    const int total = hot_groups * hot_tgroups;
    const int per_xcd = (total + 7) >> 3;
    const int idx = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (idx >= total) return;  // uniform over the workgroup
    const int grp_all = idx / hot_tgroups, tg = idx - grp_all * hot_tgroups;
    const int t0 = tg * 16, rows_here = min(16, hot_m - t0);

    // The copy, by LDS-direct loads (no registers, every load of the wavefront in flight at once): load q of the
    // workgroup fills the LDS chunks 64q .. 64q + 63, lane l the chunk L = 64q + l = (row L / stride, column chunk
    // L % stride); it fetches that chunk of its token row (rows past the end repeat the last one, the pad chunk of a
    // row repeats the chunk before it: neither is ever read).
    {
        const uint32_t lds_base = (uint32_t)(uintptr_t)lds_act;
        const int nl = 16 * stride;
        const uint32_t row_bytes = (uint32_t)hot_k;
        const uint32_t base_off = (uint32_t)t0 * row_bytes;  // the launcher keeps m * k below 4 GiB
        for (int q = wave; q * 64 < nl; q += 4) {
            const int L = min(q * 64 + lane, nl - 1);
            const int r = L / stride, cc = L - r * stride;
            dma16(hot_a, base_off + (uint32_t)min(r, rows_here - 1) * row_bytes + (uint32_t)min(cc, cpr - 1) * 16u,
                  lds_base + (uint32_t)q * 1024u);
        }
    }

    int pj = 0;
#pragma unroll
    for (int j = 0; j < GEMV_MAX_PROJ - 1; ++j)
        if (j + 1 < p.nproj && grp_all >= p.proj[j].rb_end) pj = j + 1;
    const GemvProjDev &P = p.proj[pj];
    const int rb0 = (grp_all - (pj ? p.proj[pj - 1].rb_end : 0)) * RB;
    const int rb_count = (P.n + TILE_ROWS - 1) / TILE_ROWS;
    const uint4 *wbase = reinterpret_cast<const uint4 *>(P.w) + lane;
    // all k-tiles of this wavefront in one batch, requested right behind the copy; tiles and row blocks past the end
    // repeat the last one.  The weights are read by the other token groups too, so these loads keep their cache lines
    // (no non-temporal hint).
    uint4 w[NT][RB];
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < RB; ++r)
            w[u][r] = wbase[((size_t)min(rb0 + r, rb_count - 1) * hot_kt_count + min(wave + 4 * u, hot_kt_count - 1)) * 64];
    __builtin_amdgcn_sched_barrier(0);
    wait_vm<NT * RB>();  // loads return in order: the copy has landed, the weight tiles may still be in flight
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);

    constexpr int FPW = (RB + 3) / 4;
    const float *absent = reinterpret_cast<const float *>(P.w);
    int lane_zero = 0;
    asm volatile("" : "+v"(lane_zero));
    const float ws = (P.out ? P.w_scale : absent)[lane_zero];
    float e_bias[FPW], e_scale[FPW][4], e_res[FPW][4];
#pragma unroll
    for (int f = 0; f < FPW; ++f) {
        const int fr = min(wave + 4 * f, RB - 1);
        const int e_n = min((rb0 + fr) * TILE_ROWS + lr, P.n - 1);
        e_bias[f] = *(P.bias ? P.bias + e_n : absent);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = t0 + min(lg * 4 + i, rows_here - 1);
            e_scale[f][i] = *(P.out ? p.a_scale + t : absent);
            e_res[f][i] = *(P.residual ? P.residual + ((size_t)t * P.n + e_n) : absent);
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    v4i acc[RB];
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[r] = (v4i){0, 0, 0, 0};
    int rowsum = 0;
    const bool row_ok = lr < rows_here;
    const uint4 *arow = lds_act + (row_ok ? lr : 0) * stride + lg;  // A operand: token row lr, columns 64t + 16lg .. +15 of a k-tile
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int kt = wave + 4 * u;
        if (kt < hot_kt_count) {  // uniform over the wavefront
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                v4i af = (v4i){0, 0, 0, 0};
                if (row_ok) af = *reinterpret_cast<const v4i *>(arow + kt * 16 + t * 4);
                rowsum = __builtin_amdgcn_sdot4(af[0], 0x01010101, rowsum, false);
                rowsum = __builtin_amdgcn_sdot4(af[1], 0x01010101, rowsum, false);
                rowsum = __builtin_amdgcn_sdot4(af[2], 0x01010101, rowsum, false);
                rowsum = __builtin_amdgcn_sdot4(af[3], 0x01010101, rowsum, false);
#pragma unroll
                for (int r = 0; r < RB; ++r) {
                    const uint4 w4 = w[u][r];
                    const uint32_t wd = t == 0 ? w4.x : (t == 1 ? w4.y : (t == 2 ? w4.z : w4.w));
                    v4i bf;
                    bf[0] = (int)(wd & 0x03030303u);
                    bf[1] = (int)((wd >> 2) & 0x03030303u);
                    bf[2] = (int)((wd >> 4) & 0x03030303u);
                    bf[3] = (int)((wd >> 6) & 0x03030303u);
                    acc[r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, bf, acc[r], 0, 0, 0);
                }
            }
        }
    }

    rowsum = sum_over_lane_groups(rowsum);
    if (lane < 16) red_sum[wave][lane] = rowsum;
#pragma unroll
    for (int r = 0; r < RB; ++r) *reinterpret_cast<v4i *>(&red[wave][r][lane][0]) = acc[r];
    lds_barrier();
#pragma unroll
    for (int f = 0; f < FPW; ++f) {
        if (wave + 4 * f >= RB) break;  // uniform over the wavefront
        const int fr = wave + 4 * f;
        const int n = (rb0 + fr) * TILE_ROWS + lr;  // result register i of lane l is C[4*(l/16) + i][l mod 16]
        const v4i s0 = *reinterpret_cast<const v4i *>(&red[0][fr][lane][0]), s1 = *reinterpret_cast<const v4i *>(&red[1][fr][lane][0]);
        const v4i s2 = *reinterpret_cast<const v4i *>(&red[2][fr][lane][0]), s3 = *reinterpret_cast<const v4i *>(&red[3][fr][lane][0]);
        const v4i sum = s0 + s1 + s2 + s3;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int tl = lg * 4 + i;
            if (n < P.n && tl < rows_here) {
                const int asum = red_sum[0][tl] + red_sum[1][tl] + red_sum[2][tl] + red_sum[3][tl];
                const int total_acc = sum[i] - asum;
                const size_t o = (size_t)(t0 + tl) * P.n + n;
                if (P.acc) P.acc[o] = total_acc;
                if (P.out) {
                    float v = f32_div(f32_mul((float)total_acc, ws), e_scale[f][i]);
                    if (P.bias) v = f32_add(v, e_bias[f]);
                    if (P.residual) v = f32_add(v, e_res[f][i]);
                    P.out[o] = v;
                }
            }
        }
    }
}

// Several tokens on rows that the quantiser laid out for it (ActRows::TILES16): a workgroup of up to 16 wavefronts takes RB row
// blocks and one group of up to 16 tokens, a wavefront the k-tiles wave, wave + nw, ... of them.  The tile of a token group by 64
// columns is contiguous, so an A operand is one dense load into the registers the MFMA reads: no copy through LDS, no
// gathers of 16 bytes per row, and no barrier before the products.  NT tiles are requested at once (LOOP: more than 16 NT tiles,
// in batches of NT with the next batch in flight).  The rows' sums for the code offset are an MFMA on a constant operand and
// leave the wavefront subtracted; the partial results of the wavefronts meet in LDS, and wavefront r finishes row block r, four
// outputs a lane.  What a launch takes is one trip to memory, the MFMAs of a wavefront and that exchange, and, with more than one
// workgroup a compute unit, the issue of vector instructions: 10 wavefronts of some 400 hold the four SIMDs for 2 us.  6912 -> 2560, 16
// tokens: 4.1 us (gathering the rows from memory 7.6).  A block of the 30-block stack with this kernel for qkv, gate + up and down: 24.8 us at 8
// tokens, 29.2 at 24, 33.1 at 42 (with a thread per output, which took a third more instructions and, with four row blocks, 80 registers, so that
// a compute unit held two workgroups instead of three: 24.9, 30.6 and 35.0; rows copied to LDS first 30.0 at 8 and 50.2 at 42; with
// gemv_die_kernel where that takes the launch, as now: 21.3, 26.3 and 31.5).
// Everything that the loads need arrives preloaded, the weights' addresses too: a scalar load of an argument takes as long as
// the weights do, and the two would add up (2560 columns, 160 row blocks: 0.55 us of 3.4).  Counts of row blocks and their
// groups are packed, 16 bits each: rows and k-tiles; groups of projection 0, and of 0 and 1 (0xffff where there is no next
// projection); row blocks of projections 0 and 1; row blocks of projection 2 and the wavefronts.
struct RowsParams {
    Fused16Proj proj[GEMV_MAX_PROJ];  // rb_end counts groups of RB row blocks
    int kt_count;
};
constexpr int ROWS_ARGS_AT = 56;  // its offset in the argument buffer: five pointers and four ints before it

template <int RB, int NT, bool LOOP>
__global__ __launch_bounds__(1024) void gemv_rows_kernel(const int8_t *hot_a, const uint8_t *hot_w0, const uint8_t *hot_w1, const uint8_t *hot_w2, unsigned hot_m_kt,
                                                        unsigned hot_ends, unsigned hot_blocks, unsigned hot_blocks_nw, const float *a_scale,
                                                        [[maybe_unused]] RowsParams args)
{
    extern __shared__ v4i part[];  // [nw][RB][64]
    // workgroup (x, y): token group x / 8, group 8y + x % 8 of row blocks, as in gemv_fused16_kernel: the token groups of one group
    // of row blocks run on the same XCD
    const int tg = (int)(blockIdx.x >> 3);
    const int group = (int)blockIdx.y * 8 + (int)(blockIdx.x & 7);  // may lie past the last group: such workgroups store nothing
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = (int)(hot_m_kt & 0xffffu), kt_count = (int)(hot_m_kt >> 16), nw = (int)(hot_blocks_nw >> 16);
    const int end0 = (int)(hot_ends & 0xffffu), end1 = (int)(hot_ends >> 16);
    const int pj = group < end0 ? 0 : (group < end1 ? 1 : 2);
    // the other arguments: asked for first, used once all loads of the products are on their way
    typedef const __attribute__((address_space(4))) v16u *arg_ptr;
    v16u P = ((arg_ptr)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + ROWS_ARGS_AT))[pj];
    __builtin_amdgcn_sched_barrier(0);
    const int rows_here = min(16, m - tg * 16);
    const global_ptr<const uint8_t> group_rows = (global_ptr<const uint8_t>)(uintptr_t)hot_a + (size_t)tg * 16 * TILE_K * kt_count;
    auto load_a = [&](v4i (&af)[NT][4], int kt0) { rows_load_a<NT>(af, group_rows, lane, rows_here, kt0, nw, kt_count); };
    v4i af[NT][4];
    load_a(af, wave);
    __builtin_amdgcn_sched_barrier(0);

    const int rb0 = (group - (pj == 0 ? 0 : (pj == 1 ? end0 : end1))) * RB;
    const int rb_count = (int)(pj == 0 ? hot_blocks & 0xffffu : (pj == 1 ? hot_blocks >> 16 : hot_blocks_nw & 0xffffu));
    const global_ptr<const v4u_t> tiles = (global_ptr<const v4u_t>)(uintptr_t)(pj == 0 ? hot_w0 : (pj == 1 ? hot_w1 : hot_w2)) + lane;
    auto load_w = [&](v4u_t (&w)[NT][RB], int kt0) { rows_load_w<RB, NT>(w, tiles, rb0, rb_count, kt0, nw, kt_count); };
    v4u_t w[NT][RB];
    load_w(w, wave);
    __builtin_amdgcn_sched_barrier(0);

    // The epilogue's operands are requested behind the tiles, or, where the registers are full of tiles, behind the products.
    asm volatile("" : "+s"(P));
    constexpr bool REQUEST_EARLY = RB < 4 && !LOOP;
    RowsFinish end(P, a_scale, rb0, RB, wave, lane, tg, rows_here);
    auto request = [&]() {
        end.request_operands();
        end.request_scales();
    };
    if constexpr (REQUEST_EARLY) request();
    __builtin_amdgcn_sched_barrier(0);

    v4i acc[RB], sums = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[r] = (v4i){0, 0, 0, 0};
    if constexpr (LOOP) {
        for (int kt0 = wave; kt0 < kt_count; kt0 += nw * NT) {  // uniform over the wavefront
            v4i a_next[NT][4];
            v4u_t w_next[NT][RB];
            load_a(a_next, kt0 + nw * NT);
            load_w(w_next, kt0 + nw * NT);
            rows_multiply<RB, NT>(af, w, kt0, nw, kt_count, acc, sums);
#pragma unroll
            for (int u = 0; u < NT; ++u) {
#pragma unroll
                for (int t = 0; t < 4; ++t) af[u][t] = a_next[u][t];
#pragma unroll
                for (int r = 0; r < RB; ++r) w[u][r] = w_next[u][r];
            }
        }
    } else {
        rows_multiply<RB, NT>(af, w, wave, nw, kt_count, acc, sums);
    }
    if constexpr (!REQUEST_EARLY) {
        __builtin_amdgcn_sched_barrier(0);
        request();
    }
    end.template finish<RB>(acc, sums, part, wave, lane, nw);
}

// The reference's flat row-major packing, any n and k (rows need not start on a byte boundary).
// One wavefront per output row; lane l takes columns 4l..4l+3, 4l+256.., gathers their codes one by one.
__global__ __launch_bounds__(256) void gemv_rowmajor_kernel(const uint8_t *packed, const int8_t *a,
                                                            int32_t *out, size_t n, size_t k)
{
    const int lane = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * blockDim.y + threadIdx.y;
    if (row >= n) return;
    int acc = 0;
    if (k % 16 == 0 && (reinterpret_cast<uintptr_t>(packed) & 3) == 0 &&
        (reinterpret_cast<uintptr_t>(a) & 3) == 0) {
        // rows are dword aligned: 16 weights per load
        const uint32_t *wr = reinterpret_cast<const uint32_t *>(packed) + row * (k / 16);
        const uint32_t *ad = reinterpret_cast<const uint32_t *>(a);
        for (size_t g = lane; g < k / 16; g += 64) {
            uint32_t w = wr[g];
            w &= ~((w & (w >> 1) & 0x55555555u) << 1);  // code 3 -> code 1 (both are weight 0)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                uint32_t byte = (w >> (8 * b)) & 0xffu;
                uint32_t c = (byte & 3u) | ((byte & 0xcu) << 6) | ((byte & 0x30u) << 12) | ((byte & 0xc0u) << 18);
                uint32_t av = ad[4 * g + b];
                acc = dot4(av, c, acc) - dot4(av, 0x01010101u, 0);  // codes are w + 1: take sum(a) off
            }
        }
    } else {
        for (size_t k0 = 4 * (size_t)lane; k0 < k; k0 += 256) {
            for (int j = 0; j < 4; ++j) {
                size_t kk = k0 + j;
                if (kk >= k) break;
                size_t e = row * k + kk;
                unsigned code = (packed[e >> 2] >> (2 * (e & 3))) & 3u;
                int w = code == 0 ? -1 : (code == 2 ? 1 : 0);
                acc += w * (int)a[kk];
            }
        }
    }
    acc = wave_sum_i32(acc);
    if (lane == 0) out[row] = acc;
}

template <int MB, int MODE>
int launch_mb_mode(const GemvParams &p, hipStream_t stream)
{
    size_t lds = (size_t)MB * p.kt_count * 16 * sizeof(uint4);
    dim3 grid((unsigned)p.proj[p.nproj - 1].rb_end);
    launch_kernel((gemv_tiled_kernel<MB, MODE>), grid, dim3(256), lds, stream, p);
    BITNET_HIP_CHECK_LAUNCH("gemv_tiled_kernel");
    return BITNET_HIP_OK;
}

template <int MODE>
int launch_mode(const GemvParams &p, hipStream_t stream)
{
    return launch_mb_mode<1, MODE>(p, stream);  // one token row per launch; 2..16 rows take gemv_mfma_kernel
}

template <int MODE, int RBW>
int launch_fused_mode(const GemvParams &p, hipStream_t stream)
{
    const bool norm = p.src.gamma != nullptr, small = p.k <= 3 * 1024;
    // the int8 row, or (first) the f32 squares of the row for the literal summation order
    const size_t lds_q = (size_t)p.kt_count * 16 * sizeof(uint4), lds_sq = squares_lds_bytes(p.k);
    const size_t lds = (norm && p.src.sum_order == BITNET_HIP_SUM_SEQUENTIAL && lds_sq > lds_q) ? lds_sq : lds_q;
    const dim3 grid((unsigned)p.proj[p.nproj - 1].rb_end);
    if (norm && small) launch_kernel((gemv_fused_kernel<MODE, true, 3, RBW>), grid, dim3(256), lds, stream, p);
    else if (norm) launch_kernel((gemv_fused_kernel<MODE, true, FUSED_NCH, RBW>), grid, dim3(256), lds, stream, p);
    else if (small) launch_kernel((gemv_fused_kernel<MODE, false, 3, RBW>), grid, dim3(256), lds, stream, p);
    else launch_kernel((gemv_fused_kernel<MODE, false, FUSED_NCH, RBW>), grid, dim3(256), lds, stream, p);
    BITNET_HIP_CHECK_LAUNCH("gemv_fused_kernel");
    return BITNET_HIP_OK;
}

template <int MODE, int RBW>
int launch_fused16_mode(const Fused16Params &p, int nproj, const RowSource &src, int m, hipStream_t stream)
{
    const bool norm = src.gamma != nullptr;
    const dim3 grid(8u * (unsigned)m, ((unsigned)p.proj[nproj - 1].rb_end + 7u) / 8u);
    // One wavefront per k-tile (at least the four of the summation order) for rows of up to 16 k-tiles, one chunk per
    // thread; 16 wavefronts and two or four chunks per thread above.
    const int nchb = p.kt_count <= 16 ? 1 : (p.kt_count <= 32 ? 2 : 4);
    const int nw = p.kt_count <= 16 ? row_workgroup_waves(src.k) : 16;
    const dim3 block(64u * (unsigned)nw);
    const float *x2 = src.x2;
    if (MODE == BITNET_HIP_INPUT_GQA_BROADCAST) {
        uint64_t magics = 0;
        if (!row16_magics(src.head_dim, src.gqa_group, &magics))
            return fail(BITNET_HIP_INVALID_CONFIG, "GQA group of %d heads of %d out of range", src.gqa_group, src.head_dim);
        x2 = reinterpret_cast<const float *>(static_cast<uintptr_t>(magics));
    }
    const int end0 = nproj > 1 ? p.proj[0].rb_end : 0x7fffffff, end1 = nproj > 2 ? p.proj[1].rb_end : 0x7fffffff;
#define BITNET_HOT_ARGS src.x, x2, src.gamma, src.k, src.head_dim / 4, nw, (int)src.ldx, end0, end1
#define BITNET_F16_LAUNCH(NCHB) \
    do { \
        if (norm) launch_kernel((gemv_fused16_kernel<MODE, true, NCHB, RBW>), grid, block, 0, stream, BITNET_HOT_ARGS, p); \
        else launch_kernel((gemv_fused16_kernel<MODE, false, NCHB, RBW>), grid, block, 0, stream, BITNET_HOT_ARGS, p); \
    } while (0)
    // rows of more than 16 k-tiles take at most four row blocks a workgroup (fused16_row_blocks_per_workgroup)
    if constexpr (RBW > 4) {
        if (nchb != 1) return fail(BITNET_HIP_UNSUPPORTED, "fused GEMV: %d row blocks a workgroup for %d k-tiles", RBW, p.kt_count);
        BITNET_F16_LAUNCH(1);
    } else {
        if (nchb == 1) BITNET_F16_LAUNCH(1);
        else if (nchb == 2) BITNET_F16_LAUNCH(2);
        else if constexpr (RBW <= 2) {  // what gemv_fused_supported lets through: no norm
            if (norm) return fail(BITNET_HIP_UNSUPPORTED, "fused GEMV: %d k-tiles with a norm", p.kt_count);
            launch_kernel((gemv_fused16_kernel<MODE, false, 4, RBW>), grid, block, 0, stream, BITNET_HOT_ARGS, p);
        } else return fail(BITNET_HIP_UNSUPPORTED, "fused GEMV: %d row blocks a workgroup for %d k-tiles", RBW, p.kt_count);
    }
#undef BITNET_F16_LAUNCH
#undef BITNET_HOT_ARGS
    BITNET_HIP_CHECK_LAUNCH("gemv_fused16_kernel");
    return BITNET_HIP_OK;
}

// rbw: row blocks per workgroup (rb_end then counts groups of rbw row blocks, per projection)
// Params: GemvParams or Fused16Params
template <typename Params>
int fill_projs(Params &p, const GemvProj *projs, int nproj, size_t t0, size_t k, int rbw = 1)
{
    int rb_end = 0;
    for (int j = 0; j < nproj; ++j) {
        const GemvProj &s = projs[j];
        auto &d = p.proj[j];
        d.w = s.tiled; d.w_scale = s.w_scale; d.bias = s.bias; d.n = (int)s.n;
        d.residual = s.residual ? s.residual + t0 * s.n : nullptr;
        d.out = s.out ? s.out + t0 * s.n : nullptr;
        d.acc = s.acc ? s.acc + t0 * s.n : nullptr;
        rb_end += (int)((row_blocks(s.n) + rbw - 1) / rbw);
        d.rb_end = rb_end;
    }
    for (int j = nproj; j < GEMV_MAX_PROJ; ++j) p.proj[j] = p.proj[nproj - 1];
    p.kt_count = (int)k_tiles(k);
    return rb_end;
}

template <int RB, int NT, bool LOOP>
int launch_rows(const RowsParams &p, int nproj, const int8_t *a, const float *a_scale, size_t m, int nw, hipStream_t stream)
{
    const dim3 grid(8u * (unsigned)((m + 15) / 16), ((unsigned)p.proj[nproj - 1].rb_end + 7u) / 8u);
    const unsigned end0 = nproj > 1 ? (unsigned)p.proj[0].rb_end : 0xffffu, end1 = nproj > 2 ? (unsigned)p.proj[1].rb_end : 0xffffu;
    auto blocks = [&](int j) { return (unsigned)row_blocks((size_t)p.proj[j].n); };
    launch_kernel((gemv_rows_kernel<RB, NT, LOOP>), grid, dim3(64u * (unsigned)nw), (size_t)nw * RB * 1024, stream, a, p.proj[0].w, p.proj[1].w,
                       p.proj[2].w, (unsigned)m | ((unsigned)p.kt_count << 16), end0 | (end1 << 16), blocks(0) | (blocks(1) << 16),
                       blocks(2) | ((unsigned)nw << 16), a_scale, p);
    BITNET_HIP_CHECK_LAUNCH("gemv_rows_kernel");
    return BITNET_HIP_OK;
}

template <int RB, int MT>
int launch_mfma_rb(const GemvProj *projs, int nproj, const int8_t *a, const float *a_scale, size_t m, size_t k,
                   hipStream_t stream)
{
    GemvMfmaParams p = {};
    int end = 0;
    for (int j = 0; j < nproj; ++j) {
        const GemvProj &s = projs[j];
        GemvProjDev &d = p.proj[j];
        d.w = s.tiled; d.w_scale = s.w_scale; d.bias = s.bias; d.residual = s.residual; d.out = s.out; d.acc = s.acc;
        d.n = (int)s.n;
        end += (int)((row_blocks(s.n) + RB - 1) / RB);
        d.rb_end = end;
    }
    for (int j = nproj; j < GEMV_MAX_PROJ; ++j) p.proj[j] = p.proj[nproj - 1];
    p.nproj = nproj; p.a = a; p.a_scale = a_scale; p.m = (int)m; p.k = (int)k; p.kt_count = (int)k_tiles(k);
    if (end == 0) return BITNET_HIP_OK;
    const bool fast = k % TILE_K == 0 && (reinterpret_cast<uintptr_t>(a) & 15) == 0;
    if constexpr (MT == 1) {
        // 5 to 16 tokens whose rows fit LDS: the variant that stages the activations there (with fewer rows the gathers
        // of the other variant are cheap enough, and it is measurably ahead)
        const size_t lds = m * (k + 16);
        if (fast && m >= 5 && lds + 4096 * RB + 512 <= 64 * 1024 && (k <= 3072 || (k <= 8192 && m <= 8))) {  // + the kernel's static LDS
            if (k <= 3072)
                launch_kernel((gemv_mfma_lds_kernel<RB, 0>), dim3((unsigned)end), dim3(256), lds, stream, p.a, p.k, p.m, p.kt_count, p);
            else
                launch_kernel((gemv_mfma_lds_kernel<RB, 1>), dim3((unsigned)end), dim3(256), lds, stream, p.a, p.k, p.m, p.kt_count, p);
            BITNET_HIP_CHECK_LAUNCH("gemv_mfma_lds_kernel");
            return BITNET_HIP_OK;
        }
        // more than one double-buffered batch per wavefront, but few enough k-tiles for one batch without the second buffer
        constexpr int PF2 = RB == 1 ? 4 : (RB == 2 ? 3 : 2), PF1 = RB == 1 ? 8 : (RB == 2 ? 4 : 3);
        if (fast && p.kt_count > 4 * PF2 && p.kt_count <= 4 * PF1) {
            launch_kernel((gemv_mfma_kernel<RB, 1, true, true>), dim3((unsigned)end), dim3(256), 0, stream, p.a, p.k, p.m, p.kt_count, p);
            BITNET_HIP_CHECK_LAUNCH("gemv_mfma_kernel");
            return BITNET_HIP_OK;
        }
    }
    if (fast)
        launch_kernel((gemv_mfma_kernel<RB, MT, true>), dim3((unsigned)end), dim3(256), 0, stream, p.a, p.k, p.m, p.kt_count, p);
    else
        launch_kernel((gemv_mfma_kernel<RB, MT, false>), dim3((unsigned)end), dim3(256), 0, stream, p.a, p.k, p.m, p.kt_count, p);
    BITNET_HIP_CHECK_LAUNCH("gemv_mfma_kernel");
    return BITNET_HIP_OK;
}

// Dynamic LDS of gemv_mfma_tg_kernel: 16 token rows of k + 16 bytes, rounded up to the 1 KiB loads that fill it.
constexpr size_t tg_lds_bytes(size_t k) { return (16 * (k + 16) + 1023) / 1024 * 1024; }

// 17 and more token rows, k a multiple of 256 up to 8192, aligned activations: token groups of 16 (gemv_mfma_tg_kernel)
template <int RB>
int launch_mfma_tg(const GemvProj *projs, int nproj, const int8_t *a, const float *a_scale, size_t m, size_t k, hipStream_t stream)
{
    GemvMfmaParams p = {};
    int end = 0;
    for (int j = 0; j < nproj; ++j) {
        const GemvProj &s = projs[j];
        GemvProjDev &d = p.proj[j];
        d.w = s.tiled; d.w_scale = s.w_scale; d.bias = s.bias; d.residual = s.residual; d.out = s.out; d.acc = s.acc;
        d.n = (int)s.n;
        end += (int)((row_blocks(s.n) + RB - 1) / RB);
        d.rb_end = end;
    }
    for (int j = nproj; j < GEMV_MAX_PROJ; ++j) p.proj[j] = p.proj[nproj - 1];
    p.nproj = nproj; p.a = a; p.a_scale = a_scale; p.m = (int)m; p.k = (int)k; p.kt_count = (int)k_tiles(k);
    if (end == 0) return BITNET_HIP_OK;
    const int tgroups = (int)((m + 15) / 16), total = end * tgroups;
    const unsigned grid = (unsigned)((total + 7) / 8 * 8);
    // The copy fills LDS in whole loads of 1 KiB (64 lanes x 16 bytes); the last one runs past the 16 * (k + 16) bytes
    // of token rows, so the allocation is rounded up to whole loads.
    const size_t lds = tg_lds_bytes(k);
    if ((16 * (k / 16 + 1) + 63) / 64 * 1024 > lds)
        return fail(BITNET_HIP_KERNEL_ERROR, "gemv_mfma_tg: the activation copy would overrun its LDS allocation");
    if (p.kt_count <= 12) {
        static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_mfma_tg_kernel<RB, 3>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)tg_lds_bytes(3072));
        BITNET_HIP_TRY(attr);
        launch_kernel((gemv_mfma_tg_kernel<RB, 3>), dim3(grid), dim3(256), lds, stream, p.a, p.k, p.m, p.kt_count, end, tgroups, p);
    } else {
        static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_mfma_tg_kernel<RB, 8>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)tg_lds_bytes(8192));
        BITNET_HIP_TRY(attr);
        launch_kernel((gemv_mfma_tg_kernel<RB, 8>), dim3(grid), dim3(256), lds, stream, p.a, p.k, p.m, p.kt_count, end, tgroups, p);
    }
    BITNET_HIP_CHECK_LAUNCH("gemv_mfma_tg_kernel");
    return BITNET_HIP_OK;
}

}  // namespace

int launch_gemv_rowmajor(const uint8_t *packed, const int8_t *a, int32_t *out, size_t n, size_t k,
                         hipStream_t stream)
{
    if (n == 0) return BITNET_HIP_OK;
    launch_kernel(gemv_rowmajor_kernel, dim3((unsigned)((n + 3) / 4)), dim3(64, 4), 0, stream, packed, a,
                       out, n, k);
    BITNET_HIP_CHECK_LAUNCH("gemv_rowmajor_kernel");
    return BITNET_HIP_OK;
}

int launch_gemv_tiled(const GemvProj *projs, int nproj, const int8_t *a, const float *a_scale, size_t m, size_t k,
                      hipStream_t stream)
{
    if (m == 0 || nproj <= 0) return BITNET_HIP_OK;
    if (m >= 2) {
        // Several tokens: the MFMA variant, up to 64 token rows per launch (more: in groups of 64).  Workgroups
        // take more row blocks when there are plenty of them, so that fewer workgroups re-read the activations.
        size_t blocks = 0;
        for (int j = 0; j < nproj; ++j) blocks += row_blocks(projs[j].n);
        if (m > 16 && k % TILE_K == 0 && k <= 8192 && (reinterpret_cast<uintptr_t>(a) & 15) == 0 && m * k < ((size_t)1 << 32)) {
            // token groups of 16 with their rows in LDS.  Row blocks per workgroup: the activation copy is what a workgroup
            // spends its time on, so a workgroup takes several row blocks once there are enough workgroups for every
            // compute unit (LDS holds three workgroups up to k = 3072, one above).
            const size_t tgroups = (m + 15) / 16, slots = k <= 3072 ? 768 : 256;
            if (blocks * tgroups > 2 * slots) return launch_mfma_tg<4>(projs, nproj, a, a_scale, m, k, stream);
            if (blocks * tgroups > slots) return launch_mfma_tg<2>(projs, nproj, a, a_scale, m, k, stream);
            return launch_mfma_tg<1>(projs, nproj, a, a_scale, m, k, stream);
        }
        for (size_t t0 = 0; t0 < m; t0 += (size_t)GEMV_MFMA_MAX_M) {
            GemvProj sub[GEMV_MAX_PROJ];
            const size_t rows = m - t0 < (size_t)GEMV_MFMA_MAX_M ? m - t0 : (size_t)GEMV_MFMA_MAX_M;
            for (int j = 0; j < nproj; ++j) {
                sub[j] = projs[j];
                if (sub[j].residual) sub[j].residual += t0 * sub[j].n;
                if (sub[j].out) sub[j].out += t0 * sub[j].n;
                if (sub[j].acc) sub[j].acc += t0 * sub[j].n;
            }
            const int8_t *a0 = a + t0 * k;
            const float *s0 = a_scale ? a_scale + t0 : nullptr;
            int rc;
            if (rows > 32) rc = blocks >= 400 ? launch_mfma_rb<2, 4>(sub, nproj, a0, s0, rows, k, stream)
                                              : launch_mfma_rb<1, 4>(sub, nproj, a0, s0, rows, k, stream);
            else if (rows > 16) rc = blocks >= 400 ? launch_mfma_rb<2, 2>(sub, nproj, a0, s0, rows, k, stream)
                                                   : launch_mfma_rb<1, 2>(sub, nproj, a0, s0, rows, k, stream);
            else if (blocks >= 800) rc = launch_mfma_rb<4, 1>(sub, nproj, a0, s0, rows, k, stream);
            else if (blocks >= 400) rc = launch_mfma_rb<2, 1>(sub, nproj, a0, s0, rows, k, stream);
            else rc = launch_mfma_rb<1, 1>(sub, nproj, a0, s0, rows, k, stream);
            if (rc != BITNET_HIP_OK) return rc;
        }
        return BITNET_HIP_OK;
    }
    if (k_tiles(k) * 16 * sizeof(uint4) > 60 * 1024)
        return fail(BITNET_HIP_UNSUPPORTED, "decode GEMV: k=%zu does not fit the LDS activation buffer", k);
    GemvParams p = {};
    if (fill_projs(p, projs, nproj, 0, k) == 0) return BITNET_HIP_OK;
    p.k = (int)k;
    p.nproj = nproj;
    p.m = 1;
    p.a = a;
    p.a_scale = a_scale;
    return launch_mode<MODE_PREQUANT>(p, stream);
}

int launch_gemv_rows(const GemvProj *projs, int nproj, const int8_t *a, const float *a_scale, size_t m, size_t k, hipStream_t stream)
{
    if (m == 0 || nproj <= 0) return BITNET_HIP_OK;
    size_t blocks = 0;
    for (int j = 0; j < nproj; ++j) blocks += row_blocks(projs[j].n);
    // Row blocks per workgroup: the fewest that keep the launch within one workgroup per compute unit, at most 4 (within two: 36.9
    // against 36.0 us a block of the stack at 42 tokens, 28.7 against 29.1 at 16).
    const size_t tgroups = (m + 15) / 16;
    int rb = 1;
    while (rb < 4 && (blocks + rb - 1) / rb * tgroups > 256) rb *= 2;
    const int kt = (int)k_tiles(k);
    // One k-tile per wavefront up to 16, then two; more go through the loop with 16 wavefronts.
    const int nt = kt <= 16 ? 1 : 2;
    const int nw = kt > 32 ? 16 : ((kt + nt - 1) / nt < 4 ? 4 : (kt + nt - 1) / nt);
    RowsParams p = {};
    if (fill_projs(p, projs, nproj, 0, k, rb) == 0) return BITNET_HIP_OK;
#define BITNET_ROWS(RB, NT, LOOP) return launch_rows<RB, NT, LOOP>(p, nproj, a, a_scale, m, nw, stream)
    if (kt > 32) {
        if (rb == 4) BITNET_ROWS(4, 1, true);
        if (rb == 2) BITNET_ROWS(2, 2, true);
        BITNET_ROWS(1, 2, true);
    }
    if (nt == 2) {
        if (rb == 4) BITNET_ROWS(4, 2, false);
        if (rb == 2) BITNET_ROWS(2, 2, false);
        BITNET_ROWS(1, 2, false);
    }
    if (rb == 4) BITNET_ROWS(4, 1, false);
    if (rb == 2) BITNET_ROWS(2, 1, false);
    BITNET_ROWS(1, 1, false);
#undef BITNET_ROWS
}

// Row blocks per workgroup of gemv_fused16_kernel.  Every workgroup quantises its token's input row for itself: that
// arithmetic is repeated by every workgroup of the launch, and two workgroups on one compute unit take turns on its
// SIMDs, so the launch is sized to about one workgroup per compute unit.
int fused16_row_blocks_per_workgroup(size_t m, size_t k, size_t blocks)
{
    if (m == 1) {
        // one token, gate alone, 432 row blocks: 4.50 us with one row block per workgroup, 3.82 us with two
        if (blocks > 512 && k <= 4096) return 4;
        return (blocks > 256 && k <= 4096) ? 2 : 1;
    }
    // Several tokens, each with its own workgroups: the fewest row blocks per workgroup that keep the launch within one
    // workgroup per compute unit, at most 8 (4 of rows above 4096 columns, whose wavefronts hold two tiles of each, 2 above
    // 8192).  30-block step at 2 / 3 / 4 / 6 tokens: 541 / 593 / 667 / 713 us; with launches of up to 512 workgroups 541 / 606 / 670 / 713.
    int rbw = 1;
    const int most = k_tiles(k) > 32 ? 2 : (k_tiles(k) > 16 ? 4 : 8);
    while (rbw < most && (blocks + rbw - 1) / rbw * m > 256) rbw *= 2;
    return rbw;
}

size_t gemv_fused_tiles(size_t m, size_t k, size_t blocks) { return (size_t)fused16_row_blocks_per_workgroup(m, k, blocks) * k_tiles(k); }

bool gemv_fused_supported(const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode,
                          size_t head_dim, const float *gamma, int sum_order, size_t blocks)
{
    auto al16 = [](const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    // Two to GEMV_FUSED_MAX_ROWS tokens: the 16-wavefront kernel with a set of workgroups per token (half the launches;
    // the weight tiles are fetched once per token, from the caches after the first), where that kernel applies and the
    // workgroups of all tokens stay within GEMV_FUSED_MAX_WGS.  Otherwise: stand-alone quantiser (rows in parallel) + MFMA GEMV.
    if (m == 0 || m > (size_t)GEMV_FUSED_MAX_ROWS) return false;
    if (m > 1) {
        if (!((gamma == nullptr || sum_order == BITNET_HIP_SUM_BLOCK256) && k <= 16384 && ldx < ((size_t)1 << 31))) return false;
        const size_t rbw = (size_t)fused16_row_blocks_per_workgroup(m, k, blocks);
        if ((blocks + rbw - 1) / rbw * m > (size_t)GEMV_FUSED_MAX_WGS) return false;
    }
    // Rows above FUSED_NCH * 1024 columns: only where one round of workgroups serves the launch (each quantises its whole row for
    // itself; one token's may walk several row blocks), and in the declared summation order; above 8192 columns (four chunks per thread) without a norm, whose registers do
    // not fit beside the tiles.  A decoder block with 2560-wide rows, in two launches -> here: 8192-wide FFN at 1 / 2 / 3 tokens
    // 20.3 / 21.5 / 23.4 -> 16.6 / 19.5 / 21.4 us, 13824-wide at 1 / 2 / 3 / 4 tokens 29.4 / 32.8 / 33.2 / 33.9 -> 20.2 / 25.1 /
    // 25.6 / 29.0 (of which the stand-alone quantiser's four chunks per thread give up to 5).
    if (k > (size_t)FUSED_NCH * 1024) {
        if ((m == 1 && blocks > 256 && !gemv_stream_takes(m, k, gamma, sum_order, blocks)) || k > 16384 || ldx >= ((size_t)1 << 31)) return false;
        if (gamma != nullptr && (sum_order != BITNET_HIP_SUM_BLOCK256 || k > 8192)) return false;
    }
    if (k % 4 != 0 || ldx % 4 != 0) return false;
    if (!al16(x) || (x2 && !al16(x2)) || (gamma && !al16(gamma))) return false;
    if (input_mode == BITNET_HIP_INPUT_GQA_BROADCAST && head_dim % 4 != 0) return false;
    return k_tiles(k) * 16 * sizeof(uint4) <= 60 * 1024;
}

int launch_gemv_fused(const GemvProj *projs, int nproj, const float *x, const float *x2, size_t ldx, size_t m,
                      size_t k, int input_mode, size_t gqa_group, size_t head_dim, const float *gamma, float eps,
                      int sum_order, int8_t *q_out, float *a_scale_out, int32_t *a_sum_out, hipStream_t stream)
{
    if (m == 0 || nproj <= 0) return BITNET_HIP_OK;
    // Every workgroup quantises the whole input row for itself, so launches with many row blocks give each
    // workgroup two (short rows only: the tiles of both must fit its registers).
    size_t blocks = 0;
    for (int j = 0; j < nproj; ++j) blocks += row_blocks(projs[j].n);
    // 16 wavefronts per workgroup (the declared summation order only; k <= 16384: up to four chunks per thread, 64 k-tiles)
    if ((gamma == nullptr || sum_order == BITNET_HIP_SUM_BLOCK256) && k <= 16384) {
        // row blocks per workgroup: one round of workgroups on the 256 compute units where the row is short enough for
        // a wavefront to hold the tiles of several row blocks (one token, gate alone, 432 row blocks: 4.50 us with one
        // row block per workgroup, 3.82 us with two)
        const bool streams = gemv_stream_takes(m, k, gamma, sum_order, blocks);
        const int rbw16 = streams ? 1 : fused16_row_blocks_per_workgroup(m, k, blocks);
        Fused16Params p = {};
        if (fill_projs(p, projs, nproj, 0, k, rbw16) == 0) return BITNET_HIP_OK;
        RowSource src = {};
        src.x = x; src.x2 = x2; src.gamma = gamma; src.ldx = ldx; src.k = (int)k;
        src.head_dim = (int)(head_dim ? head_dim : 1); src.gqa_group = (int)(gqa_group ? gqa_group : 1);
        p.eps = eps; p.q_out = q_out; p.a_scale_out = a_scale_out; p.a_sum_out = a_sum_out;
        if (streams) return launch_gemv_stream(p, nproj, src, input_mode, blocks, stream);
#define BITNET_F16_MODES(RBW) \
    switch (input_mode) { \
        case BITNET_HIP_INPUT_PLAIN: return launch_fused16_mode<BITNET_HIP_INPUT_PLAIN, RBW>(p, nproj, src, (int)m, stream); \
        case BITNET_HIP_INPUT_RELU2_MUL: return launch_fused16_mode<BITNET_HIP_INPUT_RELU2_MUL, RBW>(p, nproj, src, (int)m, stream); \
        default: return launch_fused16_mode<BITNET_HIP_INPUT_GQA_BROADCAST, RBW>(p, nproj, src, (int)m, stream); \
    }
        switch (rbw16) {
            case 8: BITNET_F16_MODES(8)
            case 4: BITNET_F16_MODES(4)
            case 2: BITNET_F16_MODES(2)
            default: BITNET_F16_MODES(1)
        }
#undef BITNET_F16_MODES
    }
    const int rbw = (blocks > 512 && k <= 3 * 1024) ? 2 : 1;
    GemvParams p = {};
    if (fill_projs(p, projs, nproj, 0, k, rbw) == 0) return BITNET_HIP_OK;
    p.k = (int)k;
    p.nproj = nproj;
    p.m = (int)m;
    p.src.x = x; p.src.x2 = x2; p.src.gamma = gamma; p.src.ldx = ldx; p.src.k = (int)k;
    p.src.head_dim = (int)(head_dim ? head_dim : 1); p.src.gqa_group = (int)(gqa_group ? gqa_group : 1);
    p.src.sum_order = sum_order; p.src.eps = eps;
    p.q_out = q_out; p.a_scale_out = a_scale_out; p.a_sum_out = a_sum_out;
    if (rbw == 2) {
        switch (input_mode) {
            case BITNET_HIP_INPUT_PLAIN: return launch_fused_mode<BITNET_HIP_INPUT_PLAIN, 2>(p, stream);
            case BITNET_HIP_INPUT_RELU2_MUL: return launch_fused_mode<BITNET_HIP_INPUT_RELU2_MUL, 2>(p, stream);
            default: return launch_fused_mode<BITNET_HIP_INPUT_GQA_BROADCAST, 2>(p, stream);
        }
    }
    switch (input_mode) {
        case BITNET_HIP_INPUT_PLAIN: return launch_fused_mode<BITNET_HIP_INPUT_PLAIN, 1>(p, stream);
        case BITNET_HIP_INPUT_RELU2_MUL: return launch_fused_mode<BITNET_HIP_INPUT_RELU2_MUL, 1>(p, stream);
        default: return launch_fused_mode<BITNET_HIP_INPUT_GQA_BROADCAST, 1>(p, stream);
    }
}

}  // namespace bitnet
