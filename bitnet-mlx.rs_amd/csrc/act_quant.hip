// Stand-alone fused RMSNorm + per-token absmax int8 activation quantiser for gfx950 (the arithmetic and the
// declared summation order are in rowquant.hpp; the decode GEMV runs the same code inside its prologue).
//
// Three launch shapes, same bits:
//   act_quant_block_kernel    256-thread workgroups that take token rows in turn, a row held in registers between the three
//                             passes (sum of squares, absmax, quantise): 4*K bytes read once, K + 8 bytes written.
//                             The usual shape, for one row or thousands.
//   act_quant_row_kernel      a workgroup of up to 16 wavefronts per token row, one chunk of 4 (two above 4096 columns, four
//                             above 8192) per thread: as many rows as run at once (a decode batch), where the launch is as
//                             long as one row takes.
//   act_quant_wave_kernel     one wavefront per token row: many rows of at most 1024 columns.
#include "kernels.hpp"
#include "rowquant.hpp"

namespace bitnet {

namespace {

struct ActQuantParams {
    RowSource src;
    int8_t *q;
    float *a_scale;
    int32_t *a_sum;
    float *y;
    size_t m;
    size_t ldq;      // row stride of q: k, or more with the bytes from k on (up to the next multiple of 256) cleared
    int tiled;       // layout of q: see RowPlace
    int seq_in_lds;  // the launch carries LDS for the row's squares (literal summation order: sum_sequential_lds)
};

constexpr size_t ROW_QUANT_MAX_ROWS = 512;

// Where the int8 row goes: row-major (stride ldq), or by ActRows::TILES16: the rows of a group of 16 (rows_here of them in the
// last group) interleaved in pieces of 16 bytes, row-fastest, so that a tile of 16 rows by 64 columns is contiguous.
struct RowPlace {
    size_t base;
    unsigned piece;  // from one 16-byte piece of the row to the next
    __device__ __forceinline__ size_t chunk(int c) const { return base + (size_t)((unsigned)(c >> 2) * piece) + (unsigned)(c & 3) * 4u; }
};
__device__ __forceinline__ RowPlace row_place(size_t row, size_t m, size_t ldq, bool tiled)
{
    if (!tiled) return {row * ldq, 16u};
    const size_t group = row >> 4;
    const unsigned rows_here = (unsigned)min((size_t)16, m - group * 16);
    return {group * 16 * ldq + (row & 15) * 16, 16u * rows_here};
}

// One quantised chunk (elements 4c .. 4c + 3 of the row; those from k on are +0 in `e`) to the int8 row, and to y if asked for.
template <bool VEC>
__device__ __forceinline__ void store_chunk(const ActQuantParams &p, const RowPlace &place, size_t row, int c, const float4 &e, float scale, int *isum)
{
    const int k = p.src.k;
    const size_t at = place.chunk(c), base = row * (size_t)k + 4 * (size_t)c;
    if (VEC || p.ldq > (size_t)k) {  // rows start on a dword and have room for a whole last one
        *reinterpret_cast<uint32_t *>(p.q + at) = quant4_packed(e, scale, isum);
        if constexpr (VEC) {
            if (p.y) *reinterpret_cast<float4 *>(p.y + base) = e;
            return;
        }
        if (!p.y) return;
        const float es[4] = {e.x, e.y, e.z, e.w};
        for (int j = 0; j < 4; ++j)
            if (4 * c + j < k) p.y[base + j] = es[j];
        return;
    }
    const float es[4] = {e.x, e.y, e.z, e.w};
    for (int j = 0; j < 4; ++j) {
        if (4 * c + j < k) {
            const int qv = quant1(es[j], scale);
            p.q[at + j] = (int8_t)qv;
            if (p.y) p.y[base + j] = es[j];
            *isum += qv;
        }
    }
}
// Chunk c lies past the row: cleared where the rows are padded.
__device__ __forceinline__ void clear_pad(const ActQuantParams &p, const RowPlace &place, int c)
{
    if (4 * (size_t)c < p.ldq) *reinterpret_cast<uint32_t *>(p.q + place.chunk(c)) = 0u;
}

// The chunks of a thread (first, first + step, ...; zeros from `chunks` on) normalised together: one look at their range in place of one a chunk.
template <int NCH>
__device__ __forceinline__ void normalize_row(float4 (&v)[NCH], const float4 (&gm)[NCH], const Divisor &r, int first, int step, int chunks)
{
    bool ok = r.fast;
#pragma unroll
    for (int i = 0; i < NCH; ++i) ok = ok && (first + step * i >= chunks || chunk_ok(v[i]));
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!ok) == 0, 1)) {
#pragma unroll
        for (int i = 0; i < NCH; ++i)  // no zeros but the padding's
            v[i] = make_float4(f32_mul(div_by_invariant_unchecked<false>(v[i].x, r.d, r.recip), gm[i].x),
                               f32_mul(div_by_invariant_unchecked<false>(v[i].y, r.d, r.recip), gm[i].y),
                               f32_mul(div_by_invariant_unchecked<false>(v[i].z, r.d, r.recip), gm[i].z),
                               f32_mul(div_by_invariant_unchecked<false>(v[i].w, r.d, r.recip), gm[i].w));
    } else {
#pragma unroll
        for (int i = 0; i < NCH; ++i)
            if (first + step * i < chunks) v[i] = normalize4(v[i], r, gm[i]);
    }
}

// One wavefront per row of at most 256 NCH columns: NCH (two or four) chunks a lane, no barriers.  (A workgroup per row leaves most of its
// threads without a chunk there.)  HELD as HELD_NORM below: 65536 x 1024 67.8 -> 59.9 us, 16384 x 1024 18.3 -> 16.1; two chunks where they do: 65536 x
// 512 33.1 -> 29.1 (36.3 with four).
template <int MODE, bool VEC, bool NORM, int NCH, bool HELD>
__global__ __launch_bounds__(256) void act_quant_wave_kernel(ActQuantParams p)
{
    const RowSource &src = p.src;
    const int lane = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * blockDim.y + threadIdx.y;
    if (row >= p.m) return;  // uniform per wavefront: a wavefront is one row
    const int chunks = (src.k + 3) >> 2;

    float4 v[NCH];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        int c = lane + 64 * i;
        v[i] = c < chunks ? load_chunk<MODE, VEC>(src, row, c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if constexpr (NORM) {
        float4 gm[HELD ? NCH : 1];
        if constexpr (HELD) {
#pragma unroll
            for (int i = 0; i < NCH; ++i) gm[i] = lane + 64 * i < chunks ? load_gamma_chunk(src, lane + 64 * i, VEC) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float ss;
        if (src.sum_order == BITNET_HIP_SUM_SEQUENTIAL) {
            ss = sum_squares_sequential<MODE>(src, row);
        } else {
            // chunk lane + 64*i belongs to virtual lane lane + 64*i: four partials per lane
            float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < NCH; ++i) part[i] = wave_sum_f32(sum_squares4(0.0f, v[i]));
            ss = f32_add(f32_add(f32_add(part[0], part[1]), part[2]), part[3]);
        }
        const Divisor rdiv = make_divisor(rms_from_ss(ss, src.k, src.eps));
        if constexpr (HELD) {
            normalize_row(v, gm, rdiv, lane, 64, chunks);
        } else {  // unaligned weights too: behind the sum they overlap other rows (4776 x 691 in front of it: 0.9 us more)
#pragma unroll
            for (int i = 0; i < NCH; ++i)
                if (lane + 64 * i < chunks) v[i] = normalize4(v[i], rdiv, load_gamma_chunk(src, lane + 64 * i, VEC));
        }
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) amax = absmax4(amax, v[i]);
    const float scale = scale_from_absmax(wave_max_f32(amax));

    int isum = 0;
    const RowPlace place = row_place(row, p.m, p.ldq, p.tiled != 0);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = lane + 64 * i;
        if (c < chunks) store_chunk<VEC>(p, place, row, c, v[i], scale, &isum);
        else clear_pad(p, place, c);
    }
    isum = wave_sum_i32(isum);
    if (lane == 0) {
        p.a_scale[row] = scale;
        if (p.a_sum) p.a_sum[row] = isum;
    }
}

// A workgroup per row; NCH chunks per thread in registers (K <= 1024*NCH), NCH == 0: re-read.  A row is three dependent steps
// with barriers between them: the loads of one workgroup overlap the arithmetic of the others on the compute unit.  (1024
// workgroups that take rows in turn and fetch the next one early are slower: 15.8 us against 12.7 us at 2048 x 6912.)
// HELD_NORM: a norm in the declared order, whose weights are asked for with the row and not behind its sum of squares, and whose chunks are divided
// together; NCH is then exactly what a row takes, since every chunk's weights take registers too.  With a norm, before -> now (without one), us:
// (above 14336 columns the registers of a workgroup with held weights leave a compute unit two: 2048 x 16384 37.1 -> 39.4, not taken; fewer rows:
// held_norm_from)
// 6000 x 12288 85 -> 69 (64.5), 2048 x 10240 25.9 -> 21.7 (16.3), 4096 x 5120 21.6 -> 17.9 (17.0), 4096 x 4096 18.5 -> 15.2 (14.0), 8192 x 2560 20.3 -> 18.6 (16.4), 2048 x 6912 16.7 -> 15.2 (12.5).
template <int MODE, int NCH, bool VEC, bool HELD_NORM>
__global__ __launch_bounds__(256) void act_quant_block_kernel(ActQuantParams p)
{
    __shared__ float red_f[2][4];
    __shared__ int red_i[4];
    const RowSource &src = p.src;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int k = src.k;
    const int chunks = (k + 3) >> 2;
    const int nloop = NCH > 0 ? NCH : (chunks + 255) >> 8;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    const bool norm = src.gamma != nullptr;
    const size_t row = blockIdx.x;

    float4 v[NCH > 0 ? NCH : 1];
    if constexpr (NCH > 0) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            int c = tid + 256 * i;
            v[i] = c < chunks ? load_chunk<MODE, VEC>(src, row, c) : zero4;
        }
    }
    float4 gm[HELD_NORM ? NCH : 1];
    if constexpr (HELD_NORM) {
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
            const int c = tid + 256 * i;
            gm[i] = c < chunks ? load_gamma_chunk(src, c, VEC) : zero4;
        }
    }
    auto chunk_at = [&](int i, int c) -> float4 {
        if constexpr (NCH > 0) return v[i];
        else return c < chunks ? load_chunk<MODE, VEC>(src, row, c) : zero4;
    };

    Divisor rdiv = {1.0f, 1.0f, false};
    if (HELD_NORM || norm) {
        float ss;
        if (!HELD_NORM && src.sum_order == BITNET_HIP_SUM_SEQUENTIAL) {
            if (p.seq_in_lds) {
                extern __shared__ float sq_lds[];  // squares_lds_bytes(k)
#pragma unroll
                for (int i = 0; i < nloop; ++i) {
                    const int c = tid + 256 * i;
                    if (c < chunks) store_squares4(sq_lds, c, chunk_at(i, c));
                }
                lds_barrier();
                ss = sum_sequential_lds(sq_lds, k);
            } else {
                ss = sum_squares_sequential<MODE>(src, row);
            }
        } else {
            float part = 0.0f;  // thread tid is virtual lane tid
#pragma unroll
            for (int i = 0; i < nloop; ++i) part = sum_squares4(part, chunk_at(i, tid + 256 * i));
            part = wave_sum_f32(part);
            if (lane == 0) red_f[0][wave] = part;
            lds_barrier();
            ss = f32_add(f32_add(f32_add(red_f[0][0], red_f[0][1]), red_f[0][2]), red_f[0][3]);
        }
        rdiv = make_divisor(rms_from_ss(ss, k, src.eps));
    }

    float amax = 0.0f;
    if constexpr (HELD_NORM) normalize_row(v, gm, rdiv, tid, 256, chunks);
#pragma unroll
    for (int i = 0; i < nloop; ++i) {
        int c = tid + 256 * i;
        float4 e = chunk_at(i, c);
        if (!HELD_NORM && norm && c < chunks) e = normalize4(e, rdiv, load_gamma_chunk(src, c, VEC));
        if constexpr (NCH > 0) v[i] = e;
        amax = absmax4(amax, e);
    }
    amax = wave_max_f32(amax);
    if (lane == 0) red_f[1][wave] = amax;
    lds_barrier();
    amax = fmaxf(fmaxf(red_f[1][0], red_f[1][1]), fmaxf(red_f[1][2], red_f[1][3]));
    const float scale = scale_from_absmax(amax);

    int isum = 0;
    const RowPlace place = row_place(row, p.m, p.ldq, p.tiled != 0);
#pragma unroll
    for (int i = 0; i < nloop; ++i) {
        int c = tid + 256 * i;
        if (c >= chunks) {
            clear_pad(p, place, c);
            continue;
        }
        float4 e;
        if constexpr (NCH > 0) {
            e = v[i];
        } else {
            e = load_chunk<MODE, VEC>(src, row, c);
            if (norm) e = normalize4(e, rdiv, load_gamma_chunk(src, c, VEC));
        }
        store_chunk<VEC>(p, place, row, c, e, scale, &isum);
    }
    isum = wave_sum_i32(isum);
    if (lane == 0) red_i[wave] = isum;
    lds_barrier();
    if (tid == 0) {
        p.a_scale[row] = scale;
        if (p.a_sum) p.a_sum[row] = red_i[0] + red_i[1] + red_i[2] + red_i[3];
    }
}

// A workgroup of up to 16 wavefronts per row (Row16, rowquant.hpp), for the rows of a decode batch: the launch is as long as one
// row takes, which is a chain of dependent steps.  What the first loads need arrives preloaded; the other arguments are one
// scalar load while the row is on its way.  k % 4 == 0 up to 16384, 16-byte aligned rows, the declared summation order.
struct RowQuantArgs {
    int8_t *q;
    float *a_scale;
    int32_t *a_sum;
    float *y;
    int ldq;
    int tiled;
    int unused[6];
};
static_assert(sizeof(RowQuantArgs) == 64, "one scalar load");
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int ROW_QUANT_ARGS_AT = 48;  // its offset in the argument buffer: three pointers and six 4-byte arguments before it

template <int MODE, bool NORM, int NCHB>
__global__ __launch_bounds__(1024) void act_quant_row_kernel(const float *hot_x, const float *hot_x2, const float *hot_gamma, int hot_k, int hot_head_chunks,
                                                            int hot_nw, int hot_ldx, float hot_eps, int hot_m, [[maybe_unused]] RowQuantArgs args)
{
    __shared__ float red_f[2][16];
    __shared__ int sum_s;
    const size_t row = blockIdx.x;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = hot_nw, chunks = hot_k >> 2;
    const float *x = hot_x + row * (size_t)hot_ldx;
    const float *x2 = MODE == BITNET_HIP_INPUT_RELU2_MUL ? hot_x2 + row * (size_t)hot_ldx : nullptr;
    const uint64_t magics = MODE == BITNET_HIP_INPUT_GQA_BROADCAST ? reinterpret_cast<uintptr_t>(hot_x2) : 0;
    Row16<NORM, NCHB> row16;
    row16.template load<MODE>(x, x2, magics, hot_head_chunks, hot_gamma, chunks, nw, wave, tid, tid & 63);
    __builtin_amdgcn_sched_barrier(0);
    typedef const __attribute__((address_space(4))) v16u *arg_ptr;
    v16u block = *(arg_ptr)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + ROW_QUANT_ARGS_AT);
    if (tid < 16 && tid >= nw) red_f[1][tid] = 0.0f;
    if (tid == 0) sum_s = 0;
    float k_f = (float)hot_k, k_recip = recip_of_ok_divisor(k_f);
    asm volatile("" : "+s"(block), "+v"(k_recip));
    const global_ptr<int8_t> q = pointer_at<int8_t>(block, 0);
    const global_ptr<float> a_scale = pointer_at<float>(block, 2), y = pointer_at<float>(block, 6);
    const global_ptr<int32_t> a_sum = pointer_at<int32_t>(block, 4);
    const int ldq = (int)block[8];
    const RowPlace place = row_place(row, (size_t)hot_m, (size_t)ldq, block[9] != 0);

    uint32_t packed[NCHB];
    const float scale = row16.quantise(chunks, k_f, k_recip, hot_eps, wave, tid, red_f, packed);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < NCHB; ++i) {
        const int c = row16.chunk[i];
        if (4 * c < ldq) *(global_ptr<uint32_t>)(q + place.chunk(c)) = packed[i];  // chunks past the row hold zeros
        if (y && c < chunks) *(global_ptr<v4f>)(y + (row * (size_t)hot_k + 4 * (size_t)c)) = (v4f){row16.v[i].x, row16.v[i].y, row16.v[i].z, row16.v[i].w};
        sum = __builtin_amdgcn_sdot4((int)packed[i], 0x01010101, sum, false);
    }
    if (tid == 0) a_scale[row] = scale;
    if (a_sum) {
        sum = wave_sum_i32(sum);
        if ((tid & 63) == 0) atomicAdd(&sum_s, sum);
        lds_barrier();
        if (tid == 0) a_sum[row] = sum_s;
    }
}

size_t row_bytes(const ActQuantParams &p) { return p.m * (size_t)p.src.k * sizeof(float); }

template <int MODE, bool VEC>
void launch_wave(const ActQuantParams &p, hipStream_t s)
{
    const int rows_per_block = 4;
    dim3 block(64, rows_per_block);
    dim3 grid((unsigned)((p.m + rows_per_block - 1) / rows_per_block));
    const bool two = p.src.k <= 512 && p.ldq <= 512;  // the padding is cleared by the same lanes
    // Two chunks and their weights take few registers: held, 1.07 to 1.12 times as fast from 513 rows to 65536.  Four: where the rows come from
    // beyond the L2s (32 MB) a row's chain is what counts, and where all of them run at once (12000 x 1024 14.8 -> 13.2 us, 1024 x 1024 4.14 ->
    // 3.99); between, more wavefronts of fewer registers are the faster (2048 x 640 4.30 held, 3.95 not; 4096 x 1024 5.93 and 5.68; 12000 x 768 11.4
    // and 11.3; 1024 x 516 3.98 and 3.87).
    const bool held = VEC && (two || row_bytes(p) > ((size_t)40 << 20) || (p.m <= 1024 && p.src.k > 768));
    if (p.src.gamma && two && held) launch_kernel((act_quant_wave_kernel<MODE, VEC, true, 2, VEC>), grid, block, 0, s, p);
    else if (p.src.gamma && held) launch_kernel((act_quant_wave_kernel<MODE, VEC, true, 4, VEC>), grid, block, 0, s, p);
    else if (p.src.gamma && two) launch_kernel((act_quant_wave_kernel<MODE, VEC, true, 2, false>), grid, block, 0, s, p);
    else if (p.src.gamma) launch_kernel((act_quant_wave_kernel<MODE, VEC, true, 4, false>), grid, block, 0, s, p);
    else if (two) launch_kernel((act_quant_wave_kernel<MODE, VEC, false, 2, false>), grid, block, 0, s, p);
    else launch_kernel((act_quant_wave_kernel<MODE, VEC, false, 4, false>), grid, block, 0, s, p);
}

// LDS for the row's squares where the literal summation order is asked for and a row fits the default limit
inline size_t launch_squares_lds(const ActQuantParams &p)
{
    if (!p.src.gamma || p.src.sum_order != BITNET_HIP_SUM_SEQUENTIAL) return 0;
    const size_t bytes = squares_lds_bytes(p.src.k);
    return bytes <= 60 * 1024 ? bytes : 0;
}

template <int MODE, int NCH, bool VEC>
void launch_block(ActQuantParams p, hipStream_t s)
{
    const size_t lds = launch_squares_lds(p);
    p.seq_in_lds = lds != 0;
    launch_kernel((act_quant_block_kernel<MODE, NCH, VEC, false>), dim3((unsigned)p.m), dim3(256), lds, s, p);
}

// From how many bytes of rows on the 256-thread kernel holds the norm's weights, by chunks a thread.  Beyond the L2s (32 MB) a row's chain waits for
// memory, and one trip less counts; rows that lie there are the faster the more of them a compute unit holds.  us, not held -> held, around the line:
// 2560 x 2560 7.61 -> 7.67, 4096 x 2560 12.3 -> 11.3; 1280 x 5120 7.30 -> 7.35, 1792 x 5120 10.9 -> 9.8; 1280 x 6912 10.16 -> 10.35, 1536 x 6912 13.2 -> 12.7;
// 1792 x 8192 15.5 (16 wavefronts a row) -> 16.0, 2560 x 8192 20.6 -> 20.0; 1024 x 8448 10.9 -> 11.7; 600 x 12288 9.9 -> 10.9, 768 x 12288 12.8 ->
// 11.7; 1280 x 13824 23.4 -> 23.8, 1536 x 13824 26.5 -> 25.7.  Two and four chunks: at any size, 1.02 to 1.2 times as fast, since the other kernel
// has registers for three, seven and sixteen.
size_t held_norm_from(int per_thread)
{
    constexpr size_t MB = (size_t)1 << 20;
    switch (per_thread) {
        case 3: case 5: case 6: return 29 * MB;
        case 7: return 36 * MB;
        case 8: return 60 * MB;
        case 9: case 10: case 11: return 39 * MB;
        case 12: return 32 * MB;
        case 13: case 14: return 72 * MB;
        default: return 0;
    }
}

template <int MODE, int NCH>
void launch_block_norm(const ActQuantParams &p, hipStream_t s)
{
    launch_kernel((act_quant_block_kernel<MODE, NCH, true, true>), dim3((unsigned)p.m), dim3(256), 0, s, p);
}

template <int MODE>
void launch_mode(const ActQuantParams &p, bool vec, hipStream_t s)
{
    const int chunks = (p.src.k + 3) >> 2;
    // Rows that all run at once: up to 16 wavefronts per row, with four chunks a thread above 8192 columns (213 rows of 13120 columns
    // with norm: 9.8 us in the 256-thread kernel -> 5.6 here; a decoder block with a 13824-wide FFN at 8 tokens: 36.3 -> 31.5).  Rows
    // that come in many rounds are here from 7168 columns on without a norm, and up to 8192 with one as long as the 256-thread kernel does not
    // hold its weights; that is otherwise the faster, since a compute unit holds more of its rows (8192 x 8192 73.0 us here, 62.2 there, 4096 x 7680
    // 33.1 and 27.0, 6000 x 12288 115 and 69).
    const bool ordered = !p.src.gamma || p.src.sum_order == BITNET_HIP_SUM_BLOCK256;
    const bool few = p.m <= ROW_QUANT_MAX_ROWS;
    const int per_thread = (chunks + 255) >> 8;
    const bool held = vec && p.src.gamma && ordered && per_thread <= 14 && row_bytes(p) >= held_norm_from(per_thread);
    if ((few || (chunks > 1792 && (!p.src.gamma || (chunks <= 2048 && !held)))) && vec && ordered && chunks <= 4096 && p.src.ldx < (1u << 31)) {
        const float *x2 = p.src.x2;
        uint64_t magics = 0;
        bool in_range = true;
        if (MODE == BITNET_HIP_INPUT_GQA_BROADCAST) {
            in_range = row16_magics(p.src.head_dim, p.src.gqa_group, &magics);
            x2 = reinterpret_cast<const float *>(static_cast<uintptr_t>(magics));
        }
        if (in_range) {
            const RowQuantArgs args = {p.q, p.a_scale, p.a_sum, p.y, (int)p.ldq, p.tiled, {0, 0, 0, 0, 0, 0}};
            const int kt = (p.src.k + 255) >> 8, nchb = kt > 32 ? 4 : (kt > 16 ? 2 : 1);
            const int nw = nchb == 1 ? row_workgroup_waves(p.src.k) : (kt + nchb - 1) / nchb;
            const dim3 grid((unsigned)p.m), block(64u * (unsigned)nw);
#define BITNET_HOT_ARGS p.src.x, x2, p.src.gamma, p.src.k, p.src.head_dim / 4, nw, (int)p.src.ldx, p.src.eps, (int)p.m, args
            if (p.src.gamma) {
                if (nchb == 1) launch_kernel((act_quant_row_kernel<MODE, true, 1>), grid, block, 0, s, BITNET_HOT_ARGS);
                else if (nchb == 2) launch_kernel((act_quant_row_kernel<MODE, true, 2>), grid, block, 0, s, BITNET_HOT_ARGS);
                else launch_kernel((act_quant_row_kernel<MODE, true, 4>), grid, block, 0, s, BITNET_HOT_ARGS);
            } else {
                if (nchb == 1) launch_kernel((act_quant_row_kernel<MODE, false, 1>), grid, block, 0, s, BITNET_HOT_ARGS);
                else if (nchb == 2) launch_kernel((act_quant_row_kernel<MODE, false, 2>), grid, block, 0, s, BITNET_HOT_ARGS);
                else launch_kernel((act_quant_row_kernel<MODE, false, 4>), grid, block, 0, s, BITNET_HOT_ARGS);
            }
#undef BITNET_HOT_ARGS
            return;
        }
    }
    if (p.m > 32 && chunks <= 256) return vec ? launch_wave<MODE, true>(p, s) : launch_wave<MODE, false>(p, s);
    if (held) {
        switch (per_thread) {
            case 1: return launch_block_norm<MODE, 1>(p, s);
            case 2: return launch_block_norm<MODE, 2>(p, s);
            case 3: return launch_block_norm<MODE, 3>(p, s);
            case 4: return launch_block_norm<MODE, 4>(p, s);
            case 5: return launch_block_norm<MODE, 5>(p, s);
            case 6: return launch_block_norm<MODE, 6>(p, s);
            case 7: return launch_block_norm<MODE, 7>(p, s);
            case 8: return launch_block_norm<MODE, 8>(p, s);
            case 9: case 10: return launch_block_norm<MODE, 10>(p, s);
            case 11: case 12: return launch_block_norm<MODE, 12>(p, s);
            default: return launch_block_norm<MODE, 14>(p, s);
        }
    }
    if (vec) {
        if (per_thread <= 3) return launch_block<MODE, 3, true>(p, s);
        if (per_thread <= 7) return launch_block<MODE, 7, true>(p, s);
        if (per_thread <= 16) return launch_block<MODE, 16, true>(p, s);
        return launch_block<MODE, 0, true>(p, s);
    }
    if (per_thread <= 3) return launch_block<MODE, 3, false>(p, s);
    if (per_thread <= 7) return launch_block<MODE, 7, false>(p, s);
    if (per_thread <= 16) return launch_block<MODE, 16, false>(p, s);
    return launch_block<MODE, 0, false>(p, s);
}

inline bool aligned(const void *ptr, size_t a) { return (reinterpret_cast<uintptr_t>(ptr) % a) == 0; }

// ---- absmax_quantize_activations: one scale for the whole tensor (bitnet-quant/src/quantization/activations.rs:530-641) ----
//
// Pass 1: abs-max / min / max of the tensor (order-free).  Pass 2: q = ternary code or 8-bit value of x / scale and the
// squared error of every element, summed in f64 over "rows" of 4096 consecutive elements (lane l of a wavefront adds
// elements l, l + 64, ... of its row in ascending order, butterfly 32..1; the row sums are combined the same way by
// one wavefront).  Elements past the end count as +0.
struct AbsmaxState {
    float abs_max, lo, hi, scale;
};

__global__ __launch_bounds__(256) void absmax_partial_kernel(const float *x, size_t n, float *part /* [3][gridDim.x] */)
{
    float am = 0.0f, lo = __builtin_inff(), hi = -__builtin_inff();
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float v = x[i];
        am = fmaxf(am, fabsf(v));
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
    }
    __shared__ float sh[3][4];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        am = fmaxf(am, __shfl_xor(am, off, 64));
        lo = fminf(lo, __shfl_xor(lo, off, 64));
        hi = fmaxf(hi, __shfl_xor(hi, off, 64));
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sh[0][wave] = am; sh[1][wave] = lo; sh[2][wave] = hi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[blockIdx.x] = fmaxf(fmaxf(sh[0][0], sh[0][1]), fmaxf(sh[0][2], sh[0][3]));
        part[gridDim.x + blockIdx.x] = fminf(fminf(sh[1][0], sh[1][1]), fminf(sh[1][2], sh[1][3]));
        part[2 * gridDim.x + blockIdx.x] = fmaxf(fmaxf(sh[2][0], sh[2][1]), fmaxf(sh[2][2], sh[2][3]));
    }
}

__global__ __launch_bounds__(64) void absmax_scale_kernel(const float *part, int blocks, int precision, AbsmaxState *state)
{
    float am = 0.0f, lo = __builtin_inff(), hi = -__builtin_inff();
    for (int b = threadIdx.x; b < blocks; b += 64) {
        am = fmaxf(am, part[b]);
        lo = fminf(lo, part[blocks + b]);
        hi = fmaxf(hi, part[2 * blocks + b]);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        am = fmaxf(am, __shfl_xor(am, off, 64));
        lo = fminf(lo, __shfl_xor(lo, off, 64));
        hi = fmaxf(hi, __shfl_xor(hi, off, 64));
    }
    if (threadIdx.x == 0) {
        float scale = 1.0f;  // abs_max below f32::EPSILON: no division by (almost) zero, activations.rs:557-561
        if (!(am < 1.1920929e-07f)) scale = precision == BITNET_HIP_PRECISION_EIGHT_BIT ? f32_div(am, 127.0f) : am;
        state->abs_max = am; state->lo = lo; state->hi = hi; state->scale = scale;
    }
}

// one wavefront per row of 4096 elements
__global__ __launch_bounds__(256) void absmax_quantize_kernel(const float *x, size_t n, size_t rows, int precision,
                                                              const AbsmaxState *state, int8_t *q, double *row_sums)
{
    const int lane = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * blockDim.y + threadIdx.y;
    if (row >= rows) return;
    const float scale = state->scale;
    double s = 0.0;
    for (size_t i = row * 4096 + lane; i < (row + 1) * 4096 && i < n; i += 64) {
        const float v = x[i];
        const float scaled = f32_div(v, scale);
        float qv;
        if (precision == BITNET_HIP_PRECISION_EIGHT_BIT) {
            float c = scaled > 127.0f ? 127.0f : scaled;
            c = c < -127.0f ? -127.0f : c;
            qv = roundf(c);  // halves away from zero, as f32::round
        } else {
            qv = scaled > 0.5f ? 1.0f : (scaled < -0.5f ? -1.0f : 0.0f);
        }
        const int8_t qi = (qv != qv) ? (int8_t)0 : (int8_t)qv;
        q[i] = qi;
        const float d = v - f32_mul((float)qi, scale);
        s = s + (double)f32_mul(d, d);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s = s + __shfl_xor(s, off, 64);
    if (lane == 0) row_sums[row] = s;
}

__global__ __launch_bounds__(64) void absmax_finish_kernel(const double *row_sums, size_t rows, size_t n, const AbsmaxState *state,
                                                           float *stats)
{
    double s = 0.0;
    for (size_t r = threadIdx.x; r < rows; r += 64) s = s + row_sums[r];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s = s + __shfl_xor(s, off, 64);
    if (threadIdx.x == 0) {
        stats[0] = state->scale;
        stats[1] = n ? (float)(s / (double)n) : 0.0f;
        stats[2] = state->lo;
        stats[3] = state->hi;
    }
}

// max |x| for the waiting host: every workgroup stores its maximum and the ticket as one word into pinned memory
// (HostParts).  Bound by the read of the tensor: sixteen wavefronts a compute unit with four 16-byte loads in flight each.
// NaN never enters a maximum.  2048 x 2560: 5.2 + 6.1 us in two kernels, a 4-byte copy and hipMalloc / hipFree around them
// before.
// parts (optional): the maxima for a kernel behind this one.
__global__ __launch_bounds__(1024) void abs_max_kernel(const float *x, size_t n, unsigned long long *answers, unsigned ticket, float *parts)
{
    const size_t stride = (size_t)gridDim.x * 1024;
    float am = 0.0f;
    // whole 16-byte chunks of an aligned tensor; the rest (all of an unaligned one) element by element
    const size_t chunks = (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? n >> 2 : 0;
    const float4 *x4 = reinterpret_cast<const float4 *>(x);
    size_t c = (size_t)blockIdx.x * 1024 + threadIdx.x;
    for (; c + 3 * stride < chunks; c += 4 * stride) {
        float4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = x4[c + i * stride];
#pragma unroll
        for (int i = 0; i < 4; ++i) am = absmax4(am, v[i]);
    }
    for (; c < chunks; c += stride) am = absmax4(am, x4[c]);
    for (size_t i = 4 * chunks + (size_t)blockIdx.x * 1024 + threadIdx.x; i < n; i += stride) am = fmaxf(am, fabsf(x[i]));
    am = wave_max_f32(am);
    __shared__ float sh[16];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = am;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 1; i < 16; ++i) am = fmaxf(am, sh[i]);
        if (parts) parts[blockIdx.x] = am;
        __hip_atomic_store(answers + blockIdx.x, ((unsigned long long)ticket << 32) | __builtin_bit_cast(unsigned, am),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// DynamicActivationQuantizer::quantize with a scale given from outside (activations.rs:269-294, 315-360): y = x * r with
// r = (float)(1.0 / (double)scale), as candle's affine(1.0 / scale as f64, 0.0) computes it on an f32 tensor.
//   ternary: +1 where y > 0.5, -1 where y < -0.5, else 0
//   8-bit:   round(clamp(y, -127, 127)) as int8, or, with reference_u8, the reference's literal clamp(0, 255).round()
//            as the byte of a u8 (every negative activation becomes 0 there)
__device__ __forceinline__ unsigned scaled_quantize_one(float x, int precision, float recip, int reference_u8)
{
    const float y = f32_mul(x, recip);
    int v;
    if (precision == BITNET_HIP_PRECISION_EIGHT_BIT) {
        const float lo = reference_u8 ? 0.0f : -127.0f, hi = reference_u8 ? 255.0f : 127.0f;
        float c = y > hi ? hi : y;
        c = c < lo ? lo : c;
        const float r = roundf(c);  // halves away from zero, as f32::round
        v = (r != r) ? 0 : (int)r;
    } else {
        v = y > 0.5f ? 1 : (y < -0.5f ? -1 : 0);
    }
    return (unsigned)v & 0xffu;  // 0..255 keep their byte in the u8 form
}

// Bound by reading the tensor: a thread takes chunks of four elements (a 16-byte load, a 4-byte store), neighbours in
// neighbouring lanes.  scale_out: one float, or null.
__global__ __launch_bounds__(256) void scaled_quantize_kernel(const float *x, size_t n, int precision, float scale, float recip,
                                                              int reference_u8, int8_t *q, float *scale_out)
{
    const size_t first = (size_t)blockIdx.x * 256 + threadIdx.x, stride = (size_t)gridDim.x * 256;
    if (first == 0 && scale_out) *scale_out = scale;
    const size_t chunks = ((reinterpret_cast<uintptr_t>(x) & 15) | (reinterpret_cast<uintptr_t>(q) & 3)) == 0 ? n >> 2 : 0;
    for (size_t c = first; c < chunks; c += stride) {
        const float4 e = reinterpret_cast<const float4 *>(x)[c];
        reinterpret_cast<uint32_t *>(q)[c] =
            scaled_quantize_one(e.x, precision, recip, reference_u8) | (scaled_quantize_one(e.y, precision, recip, reference_u8) << 8) |
            (scaled_quantize_one(e.z, precision, recip, reference_u8) << 16) | (scaled_quantize_one(e.w, precision, recip, reference_u8) << 24);
    }
    for (size_t i = 4 * chunks + first; i < n; i += stride) q[i] = (int8_t)(uint8_t)scaled_quantize_one(x[i], precision, recip, reference_u8);
}

// The scale of a step from the tensor's largest magnitude and the moving average before it (DynamicActivationQuantizer,
// activations.rs:245-249, 420-433), in the order of the host's state, which computes the same from the same maximum.
__device__ __forceinline__ float dynamic_scale(float am, int precision, DynamicScale d)
{
    const float cur = precision == BITNET_HIP_PRECISION_EIGHT_BIT ? f32_div(am, 127.0f) : am;
    return d.has_average ? f32_add(f32_mul(d.decay, d.average), f32_mul(f32_add(1.0f, -d.decay), cur)) : cur;
}

// The quantiser behind abs_max_kernel on the same stream: every workgroup combines the maxima (count <= 256) and computes the scale
// itself, so that nobody waits for the host between the two; its first chunk of the tensor is on its way meanwhile.  Bound
// by reading the tensor.  Calls, with the scale through the host -> now: 4007 x 6400
// 45.8 -> 37.3 us, 2048 x 2560 22.6 -> 17.4, 389 x 7680 18.9 -> 14.2; of one workgroup (below), 1 x 2056 14.2 -> 12.1.
__global__ __launch_bounds__(256) void dynamic_quantize_kernel(const float *x, size_t n, int precision, DynamicScale d, const float *parts, int count,
                                                               int reference_u8, int8_t *q, float *scale_out)
{
    const size_t first = (size_t)blockIdx.x * 256 + threadIdx.x, stride = (size_t)gridDim.x * 256;
    const size_t chunks = ((reinterpret_cast<uintptr_t>(x) & 15) | (reinterpret_cast<uintptr_t>(q) & 3)) == 0 ? n >> 2 : 0;
    const float4 *x4 = reinterpret_cast<const float4 *>(x);
    float4 e = first < chunks ? x4[first] : make_float4(0.f, 0.f, 0.f, 0.f);
    __shared__ float sh[4];
    float am = wave_max_f32((int)threadIdx.x < count ? parts[threadIdx.x] : 0.0f);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = am;
    __syncthreads();
    const float scale = dynamic_scale(fmaxf(fmaxf(sh[0], sh[1]), fmaxf(sh[2], sh[3])), precision, d), recip = (float)(1.0 / (double)scale);
    if (first == 0) *scale_out = scale;
    for (size_t c = first; c < chunks;) {
        const size_t next = c + stride;
        float4 e_next = e;
        if (next < chunks) e_next = x4[next];
        reinterpret_cast<uint32_t *>(q)[c] =
            scaled_quantize_one(e.x, precision, recip, reference_u8) | (scaled_quantize_one(e.y, precision, recip, reference_u8) << 8) |
            (scaled_quantize_one(e.z, precision, recip, reference_u8) << 16) | (scaled_quantize_one(e.w, precision, recip, reference_u8) << 24);
        e = e_next;
        c = next;
    }
    for (size_t i = 4 * chunks + first; i < n; i += stride) q[i] = (int8_t)(uint8_t)scaled_quantize_one(x[i], precision, recip, reference_u8);
}

// The same for a tensor that one workgroup holds in registers (n <= DYNAMIC_SMALL): one launch.
__global__ __launch_bounds__(1024) void dynamic_quantize_small_kernel(const float *x, int n, int precision, DynamicScale d, int reference_u8, int8_t *q,
                                                                      float *scale_out, unsigned long long *answer, unsigned ticket)
{
    constexpr int NCH = DYNAMIC_SMALL / 4096;
    const int tid = (int)threadIdx.x;
    const int chunks = ((reinterpret_cast<uintptr_t>(x) & 15) | (reinterpret_cast<uintptr_t>(q) & 3)) == 0 ? n >> 2 : 0;
    float4 v[NCH];
    float am = 0.0f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) v[i] = tid + 1024 * i < chunks ? reinterpret_cast<const float4 *>(x)[tid + 1024 * i] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int i = 0; i < NCH; ++i) am = absmax4(am, v[i]);
    for (int i = 4 * chunks + tid; i < n; i += 1024) am = fmaxf(am, fabsf(x[i]));
    __shared__ float sh[16];
    am = wave_max_f32(am);
    if ((tid & 63) == 0) sh[tid >> 6] = am;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) am = fmaxf(am, sh[i]);
    if (tid == 0)
        __hip_atomic_store(answer, ((unsigned long long)ticket << 32) | __builtin_bit_cast(unsigned, am), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const float scale = dynamic_scale(am, precision, d), recip = (float)(1.0 / (double)scale);
    if (tid == 0) *scale_out = scale;
#pragma unroll
    for (int i = 0; i < NCH; ++i)
        if (tid + 1024 * i < chunks)
            reinterpret_cast<uint32_t *>(q)[tid + 1024 * i] =
                scaled_quantize_one(v[i].x, precision, recip, reference_u8) | (scaled_quantize_one(v[i].y, precision, recip, reference_u8) << 8) |
                (scaled_quantize_one(v[i].z, precision, recip, reference_u8) << 16) | (scaled_quantize_one(v[i].w, precision, recip, reference_u8) << 24);
    for (int i = 4 * chunks + tid; i < n; i += 1024) q[i] = (int8_t)(uint8_t)scaled_quantize_one(x[i], precision, recip, reference_u8);
}

}  // namespace

int abs_max_workgroups(size_t n, int most)
{
    const size_t blocks = (n + 16383) / 16384;  // one batch of loads each
    return blocks < 1 ? 1 : (blocks > (size_t)most ? most : (int)blocks);
}

int launch_abs_max(const float *x, size_t n, int workgroups, unsigned long long *answers, unsigned ticket, hipStream_t stream, float *parts)
{
    launch_kernel(abs_max_kernel, dim3((unsigned)workgroups), dim3(1024), 0, stream, x, n, answers, ticket, parts);
    BITNET_HIP_CHECK_LAUNCH("abs_max_kernel");
    return BITNET_HIP_OK;
}

int launch_dynamic_quantize(const float *x, size_t n, int precision, const DynamicScale &d, int reference_u8, int8_t *q, float *scale_out, float *parts,
                            int workgroups, unsigned long long *answers, unsigned ticket, hipStream_t stream)
{
    if (n <= (size_t)DYNAMIC_SMALL) {
        launch_kernel(dynamic_quantize_small_kernel, dim3(1), dim3(1024), 0, stream, x, (int)n, precision, d, reference_u8, q, scale_out, answers, ticket);
        BITNET_HIP_CHECK_LAUNCH("dynamic_quantize_small_kernel");
        return BITNET_HIP_OK;
    }
    const int rc = launch_abs_max(x, n, workgroups, answers, ticket, stream, parts);
    if (rc != BITNET_HIP_OK) return rc;
    const size_t blocks = (n + 1023) / 1024;
    launch_kernel(dynamic_quantize_kernel, dim3((unsigned)(blocks > 2048 ? 2048 : blocks)), dim3(256), 0, stream, x, n, precision, d, parts, workgroups,
                       reference_u8, q, scale_out);
    BITNET_HIP_CHECK_LAUNCH("dynamic_quantize_kernel");
    return BITNET_HIP_OK;
}

int launch_scaled_quantize(const float *x, size_t n, int precision, float scale, int reference_u8, int8_t *q, float *scale_out,
                           hipStream_t stream)
{
    if (n == 0 && !scale_out) return BITNET_HIP_OK;
    const float recip = (float)(1.0 / (double)scale);
    size_t blocks = (n + 1023) / 1024;
    blocks = blocks < 1 ? 1 : (blocks > 2048 ? 2048 : blocks);
    launch_kernel(scaled_quantize_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, n, precision, scale, recip, reference_u8,
                       q, scale_out);
    BITNET_HIP_CHECK_LAUNCH("scaled_quantize_kernel");
    return BITNET_HIP_OK;
}

size_t absmax_quantize_scratch_bytes(size_t n)
{
    const size_t rows = (n + 4095) / 4096;
    return 256 + sizeof(float) * 3 * 1024 + sizeof(double) * (rows ? rows : 1);
}

int launch_absmax_quantize(const float *x, size_t n, int precision, void *scratch, int8_t *q, float *stats, hipStream_t stream)
{
    AbsmaxState *state = static_cast<AbsmaxState *>(scratch);
    float *part = reinterpret_cast<float *>(static_cast<uint8_t *>(scratch) + 256);
    double *row_sums = reinterpret_cast<double *>(static_cast<uint8_t *>(scratch) + 256 + sizeof(float) * 3 * 1024);
    const size_t rows = (n + 4095) / 4096;
    int blocks = (int)((n + 255) / 256);
    blocks = blocks < 1 ? 1 : (blocks > 1024 ? 1024 : blocks);
    launch_kernel(absmax_partial_kernel, dim3(blocks), dim3(256), 0, stream, x, n, part);
    BITNET_HIP_CHECK_LAUNCH("absmax_partial_kernel");
    launch_kernel(absmax_scale_kernel, dim3(1), dim3(64), 0, stream, part, blocks, precision, state);
    BITNET_HIP_CHECK_LAUNCH("absmax_scale_kernel");
    if (rows) {
        launch_kernel(absmax_quantize_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(64, 4), 0, stream, x, n, rows, precision,
                           state, q, row_sums);
        BITNET_HIP_CHECK_LAUNCH("absmax_quantize_kernel");
    }
    launch_kernel(absmax_finish_kernel, dim3(1), dim3(64), 0, stream, row_sums, rows, n, state, stats);
    BITNET_HIP_CHECK_LAUNCH("absmax_finish_kernel");
    return BITNET_HIP_OK;
}

int launch_act_quant(const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode,
                     size_t gqa_group, size_t head_dim, const float *gamma, float eps, int sum_order,
                     int8_t *q, size_t ldq, float *a_scale, int32_t *a_sum, float *y, hipStream_t stream, ActRows rows)
{
    ActQuantParams p;
    p.tiled = rows == ActRows::TILES16;
    p.ldq = ldq;
    p.src.x = x; p.src.x2 = x2; p.src.gamma = gamma; p.src.ldx = ldx; p.src.k = (int)k;
    p.src.head_dim = (int)(head_dim ? head_dim : 1); p.src.gqa_group = (int)(gqa_group ? gqa_group : 1);
    p.src.sum_order = sum_order; p.src.eps = eps;
    p.q = q; p.a_scale = a_scale; p.a_sum = a_sum; p.y = y; p.m = m; p.seq_in_lds = 0;

    if (ldq != k && (ldq % 4 != 0 || !aligned(q, 4) || ldq < k || ldq > (k + 255) / 256 * 256))
        return fail(BITNET_HIP_INVALID_CONFIG, "activation quantiser: int8 row stride %zu for %zu columns", ldq, k);
    if (p.tiled && ldq % 256 != 0) return fail(BITNET_HIP_INVALID_CONFIG, "activation quantiser: tiles of rows of %zu columns", ldq);
    bool vec = (k % 4 == 0) && (ldx % 4 == 0) && aligned(x, 16) && aligned(q, 4) && (!x2 || aligned(x2, 16)) &&
               (!y || aligned(y, 16)) && (!gamma || aligned(gamma, 16));
    if (input_mode == BITNET_HIP_INPUT_GQA_BROADCAST) vec = vec && (head_dim % 4 == 0);

    switch (input_mode) {
        case BITNET_HIP_INPUT_PLAIN: launch_mode<BITNET_HIP_INPUT_PLAIN>(p, vec, stream); break;
        case BITNET_HIP_INPUT_RELU2_MUL: launch_mode<BITNET_HIP_INPUT_RELU2_MUL>(p, vec, stream); break;
        default: launch_mode<BITNET_HIP_INPUT_GQA_BROADCAST>(p, vec, stream); break;
    }
    BITNET_HIP_CHECK_LAUNCH("act_quant kernel");
    return BITNET_HIP_OK;
}

}  // namespace bitnet
