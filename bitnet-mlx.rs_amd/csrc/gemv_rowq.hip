// Several tokens on short rows in one launch: every workgroup quantises the rows of its token group and multiplies them.
//
// The stand-alone quantiser in front of a token GEMV costs a launch (2.3 us of host time; on the GPU 1.7 us for the launch and
// about as much for the way of the row to memory and back).  Where a row is short, doing it again in every workgroup is cheaper: a
// wavefront quantises one of the up to 16 rows, all loads in flight at once and the reductions inside the wavefront, while the
// weight tiles are on their way.  The attention output projection of a decode step always qualifies: its input repeats each
// key/value head for a group of query heads, so only the distinct columns are read and quantised, and the operand is
// read from them repeatedly.
//
// The int8 rows lie in LDS in pieces of 16 columns, [piece][row], the row's place turned by the piece: the 64 dwords a wavefront
// writes for a row and the 16 rows an operand read takes both spread over all banks.  Products, exchange and epilogue are those
// of gemv_rows_kernel: k split over 16 wavefronts, row sums from one more MFMA, partial results through LDS.
// The arithmetic of a row is act_quant_wave_kernel's (rowquant.hpp).
#include "kernels.hpp"
#include "rowquant.hpp"

namespace bitnet {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int WAVES = 16;
constexpr int MAX_KT = 2 * WAVES;  // k-tiles: two per wavefront
constexpr size_t SHORT_WIDTH = 256 * 4, MAX_WIDTH = 256 * 8;  // distinct columns of a row: four or eight chunks of four a lane

struct RowqProj {
    const uint8_t *w;
    const float *w_scale, *bias, *residual;
    float *out;
    int32_t *acc;
    int n;
    int unused[3];
};
static_assert(sizeof(RowqProj) == 64, "one scalar load a projection");
struct RowqParams {
    RowqProj proj[GEMV_MAX_PROJ];
    float eps;
    unsigned head_magic, span_magic;  // multipliers for the pieces of a head and of a group of heads
    unsigned head_pieces;
    unsigned unused[12];
};
static_assert(sizeof(RowqParams) == 64 * (GEMV_MAX_PROJ + 1), "one scalar load more for the rest");
constexpr int ROWQ_ARGS_AT = 64;  // offset of RowqParams in the argument buffer: five pointers and five ints before it

// MODE: PLAIN or GQA_BROADCAST.  RB row blocks, NT k-tiles per wavefront, CPR chunks of four columns a lane holds of its row.
// Counts are packed as for gemv_rows_kernel; hot_blocks_width: row blocks of projection 2, and the distinct columns of a row.
template <int MODE, bool NORM, int RB, int NT, int CPR>
__global__ __launch_bounds__(1024) void gemv_rowq_kernel(const float *hot_x, const float *hot_gamma, const uint8_t *hot_w0, const uint8_t *hot_w1,
                                                         const uint8_t *hot_w2, unsigned hot_m_kt, unsigned hot_ends, unsigned hot_blocks,
                                                         unsigned hot_blocks_width, unsigned hot_groups, [[maybe_unused]] RowqParams args)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // [pieces][16 rows][16 bytes], then [wavefronts][RB][64] partial results
    __shared__ float scale_s[16];
    const int tg = (int)(blockIdx.x >> 3);  // token group; the token groups of a group of row blocks run on one XCD
    const int group = (int)blockIdx.y * 8 + (int)(blockIdx.x & 7);
    if (group >= (int)hot_groups) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = (int)(hot_m_kt & 0xffffu), kt_count = (int)(hot_m_kt >> 16), width = (int)(hot_blocks_width >> 16), chunks = width >> 2;
    const int end0 = (int)(hot_ends & 0xffffu), end1 = (int)(hot_ends >> 16);
    const int pj = group < end0 ? 0 : (group < end1 ? 1 : 2);
    typedef const __attribute__((address_space(4))) v16u *arg_ptr;
    const arg_ptr blocks = (arg_ptr)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + ROWQ_ARGS_AT);
    v16u P = blocks[pj], Q = blocks[GEMV_MAX_PROJ];
    const int rows_here = min(16, m - tg * 16);
    const bool has_row = wave < rows_here;  // uniform over the wavefront

    // the row first, the weight tiles behind it
    auto absent_chunk = [&](int i) { return CPR > 4 && 64 * i >= chunks; };  // of every lane: left out above 1024 columns
    float4 v[CPR], g[NORM ? CPR : 1];
    {
        const global_ptr<const v4f> row = (global_ptr<const v4f>)(uintptr_t)(hot_x + (size_t)(tg * 16 + min(wave, rows_here - 1)) * width);
        const global_ptr<const v4f> gamma = (global_ptr<const v4f>)(uintptr_t)hot_gamma;
#pragma unroll
        for (int i = 0; i < CPR; ++i) {
            if (absent_chunk(i)) continue;
            const int c = min(lane + 64 * i, chunks - 1);
            const v4f e = row[c];
            v[i] = make_float4(e[0], e[1], e[2], e[3]);
            if constexpr (NORM) {
                const v4f w = gamma[c];
                g[i] = make_float4(w[0], w[1], w[2], w[3]);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const int rb0 = (group - (pj == 0 ? 0 : (pj == 1 ? end0 : end1))) * RB;
    const int rb_count = (int)(pj == 0 ? hot_blocks & 0xffffu : (pj == 1 ? hot_blocks >> 16 : hot_blocks_width & 0xffffu));
    const global_ptr<const v4u> tiles = (global_ptr<const v4u>)(uintptr_t)(pj == 0 ? hot_w0 : (pj == 1 ? hot_w1 : hot_w2)) + lane;
    v4u w[NT][RB];
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
        for (int r = 0; r < RB; ++r)
            w[u][r] = __builtin_nontemporal_load(tiles + ((size_t)min(rb0 + r, rb_count - 1) * kt_count + min(wave + WAVES * u, kt_count - 1)) * 64);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" : "+s"(P), "+s"(Q));
    const global_ptr<const float> absent = (global_ptr<const float>)(uintptr_t)hot_x;
    const global_ptr<const float> w_scale = pointer_at<const float>(P, 2), bias = pointer_at<const float>(P, 4), residual = pointer_at<const float>(P, 6);
    const global_ptr<float> out = pointer_at<float>(P, 8);
    const global_ptr<int32_t> acc_out = pointer_at<int32_t>(P, 10);
    const int P_n = (int)P[12];

    // Output e of the workgroup: token e / (16 RB), row block (e / 16) % RB, row e % 16; thread tid finishes tid, tid + 1024, ...
    constexpr int OUTS = (16 * RB * TILE_ROWS + 64 * WAVES - 1) / (64 * WAVES);
    const int outputs = rows_here * RB * TILE_ROWS;
    const float e_ws = (out ? w_scale : absent)[0];
    float e_bias[OUTS], e_res[OUTS];
#pragma unroll
    for (int s = 0; s < OUTS; ++s) {
        const int e = min(tid + s * 64 * WAVES, outputs - 1);
        const int n = min((rb0 + ((e >> 4) & (RB - 1))) * TILE_ROWS + (e & 15), P_n - 1), t = tg * 16 + e / (16 * RB);
        e_bias[s] = (bias ? bias + n : absent)[0];
        e_res[s] = (residual ? residual + ((size_t)t * P_n + n) : absent)[0];
    }
    __builtin_amdgcn_sched_barrier(0);

    if (has_row) {
#pragma unroll
        for (int i = 0; i < CPR; ++i)
            if (lane + 64 * i >= chunks) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (NORM) {
            // chunk c belongs to virtual lane c % 256 of the declared order: four partial sums a lane
            float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < CPR; ++i) {
                if (absent_chunk(i)) continue;
                part[i & 3] = sum_squares4(part[i & 3], v[i]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) part[j] = wave_sum_f32(part[j]);
            const float ss = f32_add(f32_add(f32_add(part[0], part[1]), part[2]), part[3]);
            const Divisor rdiv = make_divisor(rms_from_ss(ss, width, __builtin_bit_cast(float, Q[0])));
#pragma unroll
            for (int i = 0; i < CPR; ++i) {
                if (absent_chunk(i)) continue;
                if (lane + 64 * i < chunks) v[i] = normalize4(v[i], rdiv, g[i]);
            }
        }
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < CPR; ++i) {
            if (absent_chunk(i)) continue;
            amax = absmax4(amax, v[i]);
        }
        const float scale = scale_from_absmax(wave_max_f32(amax));
        int unused = 0;
#pragma unroll
        for (int i = 0; i < CPR; ++i) {
            if (absent_chunk(i)) continue;
            const int c = lane + 64 * i, piece = c >> 2;
            const uint32_t packed = quant4_packed(v[i], scale, &unused);
            if (c < chunks) *reinterpret_cast<uint32_t *>(lds + (piece * 16 + (wave ^ (piece & 15))) * 16 + (c & 3) * 4) = packed;
        }
        if (lane == 0) scale_s[wave] = scale;
    }
    lds_barrier();

    // Rows past the last and columns past the width hold whatever LDS held: such rows are not stored, such columns meet weight 0.
    const int last_piece = (width + 15) / 16 - 1;
    v4i acc[RB], sums = {0, 0, 0, 0};
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[r] = (v4i){0, 0, 0, 0};
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int kt = wave + WAVES * u;
        if (kt >= kt_count) break;  // uniform over the wavefront
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int piece = kt * 16 + t * 4 + (lane >> 4);
            if constexpr (MODE == BITNET_HIP_INPUT_GQA_BROADCAST) {
                const int head = div_by_magic(piece, Q[1]), kv = div_by_magic(piece, Q[2]);
                piece += (kv - head) * (int)Q[3];
            }
            piece = min(piece, last_piece);
            const v4i a = *reinterpret_cast<const v4i *>(lds + (piece * 16 + ((lane & 15) ^ (piece & 15))) * 16);
            sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, ones, sums, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < RB; ++r) {
                const unsigned wd = w[u][r][t];
                const v4i bf = {(int)(wd & 0x03030303u), (int)((wd >> 2) & 0x03030303u), (int)((wd >> 4) & 0x03030303u), (int)((wd >> 6) & 0x03030303u)};
                acc[r] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, bf, acc[r], 0, 0, 0);
            }
        }
    }
    const int parts = min(WAVES, kt_count);  // wavefronts with products
    v4i *part = reinterpret_cast<v4i *>(lds + (size_t)(last_piece + 1) * 256);
    if (wave < parts) {
        // component i is token 4 (lane / 16) + i of row lane % 16, stored at (i + r) % 4: the reads below spread over the banks
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const v4i d = acc[r] - sums;
            part[((size_t)wave * RB + r) * 64 + lane] = (v4i){d[(0 - r) & 3], d[(1 - r) & 3], d[(2 - r) & 3], d[(3 - r) & 3]};
        }
    }
    lds_barrier();
    const int *part_i = reinterpret_cast<const int *>(part);
#pragma unroll
    for (int s = 0; s < OUTS; ++s) {
        const int e = tid + s * 64 * WAVES;
        if (e >= outputs) break;
        const int r = (e >> 4) & (RB - 1), tl = e / (16 * RB), lr = e & 15;
        const int *from = part_i + r * 256 + ((tl >> 2) * 16 + lr) * 4 + ((tl + r) & 3);
        int total = 0;
        for (int p = 0; p < parts; p += 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int got = from[min(p + j, parts - 1) * (RB * 256)];
                total += p + j < parts ? got : 0;
            }
        }
        const int n = (rb0 + r) * TILE_ROWS + lr;
        if (n >= P_n) continue;
        const size_t o = (size_t)(tg * 16 + tl) * P_n + n;
        if (acc_out) acc_out[o] = total;
        if (out) {
            const float scaled = f32_mul((float)total, e_ws), a_scale = scale_s[tl];
            float y = div_by_invariant_unchecked(scaled, a_scale, recip_of_ok_divisor(a_scale));
            if (__builtin_expect(!(invariant_divisor_ok(a_scale) && dividend_ok(scaled)), 0)) y = f32_div(scaled, a_scale);
            if (bias) y = f32_add(y, e_bias[s]);
            if (residual) y = f32_add(y, e_res[s]);
            out[o] = y;
        }
    }
}

struct Launch {
    const float *x, *gamma;
    unsigned m_kt, ends, blocks, blocks_width, groups;
    RowqParams p;
    dim3 grid;
    size_t pieces;
    hipStream_t stream;
};

template <int MODE, bool NORM, int RB, int NT, int CPR>
int launch(const Launch &l)
{
    const int kt = (int)(l.m_kt >> 16);
    const size_t bytes = l.pieces * 256 + (size_t)(kt < WAVES ? kt : WAVES) * RB * 1024;
    constexpr size_t MOST = (size_t)CPR * 64 / 4 * 256 + (size_t)WAVES * RB * 1024;
    static const hipError_t attr = MOST > 64 * 1024 ? hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_rowq_kernel<MODE, NORM, RB, NT, CPR>),
                                                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)MOST)
                                                    : hipSuccess;
    BITNET_HIP_TRY(attr);
    launch_kernel((gemv_rowq_kernel<MODE, NORM, RB, NT, CPR>), l.grid, dim3(64 * WAVES), bytes, l.stream, l.x, l.gamma, l.p.proj[0].w, l.p.proj[1].w,
                       l.p.proj[2].w, l.m_kt, l.ends, l.blocks, l.blocks_width, l.groups, l.p);
    BITNET_HIP_CHECK_LAUNCH("gemv_rowq_kernel");
    return BITNET_HIP_OK;
}
template <int MODE, bool NORM, int NT, int CPR>
int launch_rb(const Launch &l, int rb)
{
    if (rb == 4) return launch<MODE, NORM, 4, NT, CPR>(l);
    if (rb == 2) return launch<MODE, NORM, 2, NT, CPR>(l);
    return launch<MODE, NORM, 1, NT, CPR>(l);
}
// Workgroups that the fullest compute unit runs, of `groups` groups of row blocks and `tgroups` token groups (the kernel's mapping: a
// group of row blocks on one XCD of 32).
size_t rounds_of(size_t groups, size_t tgroups) { return ((groups + 7) / 8 * tgroups + 31) / 32; }
// The fewest row blocks a workgroup that keep the launch within one round, at most 4.  Counted for the fullest XCD: 84 row blocks by 3
// token groups are 252 workgroups, but 11 of one XCD by 3 do not fit its 32 compute units.  One / two / four row blocks a workgroup, us a
// recorded decoder block (this is its attention output projection; 252 to 255 workgroups of one row block): 1344 wide at 33 / 48 tokens
// 25.4 / 25.3 / 26.1, 27.0 / 25.9 / 26.7; 816 at 80 24.4 / 23.5 / 23.9; 672 at 95 26.3 / 23.2 / 23.7.  Where one fits each XCD (2000 wide
// at 32) 27.4 / 27.6 / 28.2.
size_t row_blocks_per_workgroup(size_t blocks, size_t tgroups)
{
    size_t rb = 1;
    while (rb < 4 && rounds_of((blocks + rb - 1) / rb, tgroups) > 1) rb *= 2;
    return rb;
}

}  // namespace

bool gemv_rowq_takes(const float *x, size_t ldx, size_t m, size_t k, int input_mode, size_t gqa_group, size_t head_dim,
                     const float *gamma, int sum_order, size_t blocks, bool alone)
{
    auto al16 = [](const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    const bool gqa = input_mode == BITNET_HIP_INPUT_GQA_BROADCAST;
    if (!gqa && input_mode != BITNET_HIP_INPUT_PLAIN) return false;
    if (gqa && (head_dim % 16 != 0 || gqa_group == 0 || gamma)) return false;
    const size_t width = gqa ? k / gqa_group : k;
    // In one round of workgroups only: a second one quantises again.  What a workgroup pays for it grows with the columns that it
    // quantises, those of its up to 16 rows together; what it saves is the quantiser's launch, 0.5 to 1 us of the GPU's time and, in a call
    // that nothing records, 2.5 us of the host's.  So a call of its own is one launch wherever the kernel takes it, and a recorded one
    // (alone == false: a decoder step, a capture of the caller's) up to lines beyond which the GPU is slower so.  Recorded, two launches -> one, us:
    // plain rows of up to 1024 columns, any number of tokens: 16 x 1024 -> 2560 4.8 -> 4.2, 64 x 1024 -> 2560 5.5 -> 5.0, 512 x 1024 -> 512 6.4 -> 5.3;
    // with norm, up to 12288 columns a workgroup: 9 x 256 -> 2560 5.1 -> 4.7, 9 x 1024 -> 9000 6.2 -> 6.0; beyond them 16 x 1024 -> 2560 5.2 -> 6.0,
    // 64 x 1024 -> 512 5.1 -> 5.8, 128 x 512 -> 512 5.1 -> 5.6 (full groups of 16 rows are behind before the line: 16 x 512 -> 2560 5.05 -> 5.4,
    // 48 x 768 -> 2560 5.4 -> 5.9);
    // plain rows above 1024 columns, up to the same 12288: 5 x 2048 -> 9000 6.5 -> 5.8, 9 x 1280 -> 2560 5.1 -> 4.8; beyond them 16 x 1280 -> 2560
    // 5.1 -> 5.4, 16 x 2048 -> 2560 5.2 -> 6.4, 40 x 2048 -> 5120 6.2 -> 7.4, 256 x 1536 -> 512 5.8 -> 6.0, but above 256 tokens, where the quantiser's
    // launch is longer itself, 512 x 1280 -> 512 7.0 -> 6.3, 512 x 2048 -> 512 8.3 -> 7.5.
    const size_t in_group = m < 16 ? m : 16, tgroups = (m + 15) / 16;
    const bool few_columns = width * in_group <= 12288;
    if (m < 2 || m > (size_t)GEMV_WIDE_MAX_M || (blocks + 3) / 4 * tgroups > 256) return false;
    // More than 95 tokens, and rows above 1024 columns without a norm: as long as no compute unit quantises more than 2048 columns for its
    // 16 tokens (with a norm, in two rounds: not).  In two launches -> here, us a call: 104 x 1024 -> 512 8.0 -> 5.2, 512 x 1024 -> 512 8.0 -> 5.5,
    // 128 x 512 -> 2048 with norm 8.0 -> 6.2, 16 x 1280 -> 2560 8.0 -> 5.4, 64 x 1280 -> 2560 8.0 -> 6.0, 16 x 2048 -> 2560 8.0 -> 6.0, 40 x 2048 -> 5120
    // 7.8 -> 7.3.  Beyond the line: 16 x 1280 -> 2560 with norm 8.1 -> 7.1 and recorded 5.1 -> 7.2, 40 x 2560 -> 5120 9.1 -> 9.1.
    if (m > (size_t)GEMV_MAX_M || width > SHORT_WIDTH) {
        const size_t rb = row_blocks_per_workgroup(blocks, tgroups), rounds = rounds_of((blocks + rb - 1) / rb, tgroups);
        if (gqa || (gamma ? !alone || rounds > 1 || width > SHORT_WIDTH : rounds * width > MAX_WIDTH)) return false;
    }
    if (width % 4 != 0 || ldx != width || width > MAX_WIDTH) return false;
    if (!gqa && !alone && !few_columns && (gamma || (width > SHORT_WIDTH && m <= 256))) return false;
    if (k_tiles(k) > (size_t)MAX_KT || k > 0xffff || blocks > GEMV_ROWS_MAX_BLOCKS) return false;
    // Up to eight tokens gemv_fused16_kernel may be one launch as well, with a set of workgroups for every token.  It has fewer rows to
    // quantise but reads the weight tiles once a token, so it is ahead while its workgroups have few tiles to walk.  A decoder block
    // with the attention output by this kernel instead, where those walk 24 to 40 tiles: 0.5 to 1.0 us slower (1536 to 2560 wide, 2
    // to 8 tokens); 44 and 48: 0.1 to 0.3 slower (2816 and 3072 wide at 3 to 5); 52: 0.4 to 1.0 faster (3200 at 3 to 5), 56 and 64:
    // even (3584 and 4096 at 3, 4), 80 and more: 0.6 to 2.0 faster (2560 at 7 and 8, 4096 at 5 to 8, 5120 to 8192 at 2 to 8).  Where
    // that kernel's workgroups do not fit one round, the other choice is two launches: 6 x 1024 -> 8192 7.5 us a call, 3.7 here.  Above
    // 1024 columns that kernel keeps what it takes.
    if (gemv_fused_supported(x, nullptr, ldx, m, k, input_mode, head_dim, gamma, sum_order, blocks) && (width > SHORT_WIDTH || gemv_fused_tiles(m, k, blocks) <= 48))
        return false;
    return al16(x) && (!gamma || (al16(gamma) && sum_order == BITNET_HIP_SUM_BLOCK256));
}

int launch_gemv_rowq(const GemvProj *projs, int nproj, const float *x, size_t m, size_t k, int input_mode, size_t gqa_group, size_t head_dim,
                     const float *gamma, float eps, hipStream_t stream)
{
    if (m == 0 || nproj <= 0) return BITNET_HIP_OK;
    const bool gqa = input_mode == BITNET_HIP_INPUT_GQA_BROADCAST;
    const size_t width = gqa ? k / gqa_group : k, kt = k_tiles(k), tgroups = (m + 15) / 16;
    size_t blocks = 0;
    for (int j = 0; j < nproj; ++j) blocks += row_blocks(projs[j].n);
    const int rb = (int)row_blocks_per_workgroup(blocks, tgroups);
    Launch l = {};
    size_t groups = 0;
    unsigned ends[GEMV_MAX_PROJ] = {}, counts[GEMV_MAX_PROJ] = {};
    for (int j = 0; j < nproj; ++j) {
        const GemvProj &s = projs[j];
        RowqProj &d = l.p.proj[j];
        d.w = s.tiled; d.w_scale = s.w_scale; d.bias = s.bias; d.residual = s.residual; d.out = s.out; d.acc = s.acc; d.n = (int)s.n;
        counts[j] = (unsigned)row_blocks(s.n);
        groups += (counts[j] + rb - 1) / rb;
        ends[j] = (unsigned)groups;
    }
    if (groups == 0) return BITNET_HIP_OK;
    l.x = x; l.gamma = gamma; l.p.eps = eps; l.stream = stream;
    l.m_kt = (unsigned)m | ((unsigned)kt << 16);
    l.ends = (nproj > 1 ? ends[0] : 0xffffu) | ((nproj > 2 ? ends[1] : 0xffffu) << 16);
    l.blocks = counts[0] | (counts[1] << 16);
    l.blocks_width = counts[2] | ((unsigned)width << 16);
    l.groups = (unsigned)groups;
    l.pieces = (width + 15) / 16;
    l.grid = dim3(8u * (unsigned)tgroups, ((unsigned)groups + 7u) / 8u);
    if (gqa) {
        auto magic = [](size_t d) { return d == 1 ? 0u : (unsigned)((((uint64_t)1 << 32) + d - 1) / d); };
        l.p.head_pieces = (unsigned)(head_dim / 16);
        l.p.head_magic = magic(head_dim / 16); l.p.span_magic = magic(head_dim / 16 * gqa_group);
        return kt > WAVES ? launch_rb<BITNET_HIP_INPUT_GQA_BROADCAST, false, 2, 4>(l, rb) : launch_rb<BITNET_HIP_INPUT_GQA_BROADCAST, false, 1, 4>(l, rb);
    }
    if (gamma) return launch_rb<BITNET_HIP_INPUT_PLAIN, true, 1, 4>(l, rb);
    return width > SHORT_WIDTH ? launch_rb<BITNET_HIP_INPUT_PLAIN, false, 1, 8>(l, rb) : launch_rb<BITNET_HIP_INPUT_PLAIN, false, 1, 4>(l, rb);
}

}  // namespace bitnet
