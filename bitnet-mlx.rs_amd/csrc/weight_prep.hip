// Weight-side kernels: ternarisation, 2-bit packing in the reference's byte format, and the re-tiling
// into the layout the contraction kernels stream.  All of them run once per weight update.
//
// Reference byte format (bitnet-quant/src/quantization/packing.rs:353-394 over
// bitnet-quant/src/quantization/utils.rs:434-451): code = w + 1 in {0,1,2}; flat element i lives in
// byte i/4 at bits 2*(i mod 4); missing tail elements leave 0 bits.  Decoding maps 0,1,2,3 to
// -1,0,+1,0 (bitnet-inference/src/engine/weight_conversion.rs:169-184).
//
// Re-tiled layout: the [n, k] matrix is cut into tiles of TILE_ROWS(16) rows x TILE_K(256) columns.  A
// tile is 1 KiB = 64 slots of 16 bytes.  Slot s = kq*16 + r (kq = 0..3, r = 0..15) belongs to row r of the
// tile; its dword t (t = 0..3) holds the 16 columns 64*t + 16*kq .. +15.  Inside a dword the weight with
// column offset 4j + b sits at bits 2j + 8b, so that (dword >> 2j) & 0x03030303 yields the four code
// bytes of columns 4j..4j+3 in activation byte order.  Tiles are stored row-block major: tile (rb, kt)
// starts at byte ((rb * k_tiles) + kt) * 1024.
// Why this order: a wavefront whose lane l loads slot l reads one tile as a single contiguous 1 KiB
// burst, and dword t of every lane is then exactly the B operand of the t-th 16x16x64 int8 MFMA over
// the tile's columns 64t..64t+63 (operand row/column = lane mod 16, 16-column k block = lane / 16).
// Lanes l, l+16, l+32, l+48 share a row, so the decode GEMV combines them with two shuffles.
// Positions outside the matrix hold code 1 (weight 0) and code 3 is rewritten to code 1, so the
// contraction kernels never see code 3.
#include <type_traits>

#include "kernels.hpp"

namespace bitnet {

namespace {

__global__ __launch_bounds__(256) void pack_2bit_kernel(const int8_t *q, size_t count, uint8_t *packed,
                                                        size_t nbytes)
{
    size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbytes) return;
    unsigned byte = 0;
    for (int j = 0; j < 4; ++j) {
        size_t i = 4 * b + j;
        if (i < count) byte |= ((unsigned)(q[i] + 1) & 3u) << (2 * j);
    }
    packed[b] = (uint8_t)byte;
}

__global__ __launch_bounds__(256) void unpack_2bit_kernel(const uint8_t *packed, size_t count, int8_t *q)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    unsigned code = (packed[i >> 2] >> (2 * (i & 3))) & 3u;
    q[i] = code == 0 ? -1 : (code == 2 ? 1 : 0);
}

// Base-3 bytes: value j of byte b is digit j of b in base 3 (bitnet-quant/src/quantization/packing.rs:424-501).
__device__ __forceinline__ unsigned base3_digit(unsigned byte, unsigned j)
{
    const unsigned div = j == 0 ? 1u : (j == 1 ? 3u : (j == 2 ? 9u : (j == 3 ? 27u : 81u)));
    return (byte / div) % 3u;
}

__global__ __launch_bounds__(256) void pack_base3_kernel(const int8_t *q, size_t count, uint8_t *packed, size_t nbytes)
{
    size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbytes) return;
    unsigned byte = 0, mult = 1;
    for (int j = 0; j < 5; ++j) {
        size_t i = 5 * b + j;
        if (i < count) byte += (unsigned)(uint8_t)(q[i] + 1) * mult;
        mult *= 3;
    }
    packed[b] = (uint8_t)byte;
}

__global__ __launch_bounds__(256) void unpack_base3_kernel(const uint8_t *packed, size_t count, int8_t *q)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    q[i] = (int8_t)base3_digit(packed[i / 5], (unsigned)(i % 5)) - 1;
}

// One 2-bit byte (elements 4b .. 4b+3) per thread: both formats use the code w + 1.
__global__ __launch_bounds__(256) void base3_to_2bit_kernel(const uint8_t *base3, size_t count, uint8_t *packed, size_t nbytes)
{
    size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbytes) return;
    unsigned byte = 0;
    for (int j = 0; j < 4; ++j) {
        size_t i = 4 * b + j;
        if (i < count) byte |= base3_digit(base3[i / 5], (unsigned)(i % 5)) << (2 * j);
    }
    packed[b] = (uint8_t)byte;
}

// TernaryLookupKernel / I2SLookupKernel::compute (bitnet-core/src/cpu/kernels/generic.rs:54-75,118-139).
__global__ __launch_bounds__(256) void lookup_compute_kernel(int kind, const int8_t *w, const float *x, float *out, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int v = w[i];
    float l;
    if (kind == BITNET_HIP_LOOKUP_TERNARY) l = v == -1 ? -1.0f : (v == 1 ? 1.0f : 0.0f);
    else l = v == -2 ? -2.0f : (v == -1 ? -1.0f : (v == 1 ? 1.0f : 0.0f));
    out[i] = f32_mul(x[i], l);
}

__device__ __forceinline__ double wave_sum_f64(double p)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) p = p + __shfl_xor(p, off, 64);
    return p;
}

// Element c of a row for c = lane, lane + 64, .. below k, in ascending order, with up to U loads in flight: the f64 chains
// of the row sums fix the order of the additions, not that of the loads.  ready: what is done to the elements of a group, all at once.
template <int U, typename R, typename F>
__device__ __forceinline__ void for_row(const float *row, size_t k, int lane, R &&ready, F &&add)
{
    size_t c = lane;
    for (size_t end = 64 * U; end <= k; end += 64 * U, c += 64 * U) {  // uniform: every lane of the wavefront is in it
        float v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) v[i] = row[c + 64 * i];
        ready(v);
#pragma unroll
        for (int i = 0; i < U; ++i) add(v[i], c + 64 * i);
    }
    for (; c < k; c += 64) {
        float v[1] = {row[c]};
        ready(v);
        add(v[0], c);
    }
}
template <int U, typename F>
__device__ __forceinline__ void for_row(const float *row, size_t k, int lane, F &&add)
{
    for_row<U>(row, k, lane, [](auto &) {}, add);
}

// Sum of |w| of one row in f64: lane l adds columns l, l+64, ... in ascending order, then the
// butterfly.  One wavefront per row.  Bound by the read of the matrix (6912 x 2560: 12 us with ten loads in flight, 16.7 with one).
__global__ __launch_bounds__(256) void absmean_rows_kernel(const float *w, size_t n, size_t k, double *row_sums)
{
    const int lane = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * blockDim.y + threadIdx.y;
    if (row >= n) return;
    double s = 0.0;
    for_row<10>(w + row * k, k, lane, [&](float v, size_t) { s = s + (double)fabsf(v); });
    s = wave_sum_f64(s);
    if (lane == 0) row_sums[row] = s;
}

// The row sums of NACC accumulators (accumulator a at row_sums + a * n), combined in the declared order: lane l takes rows
// l, l+64, ..., then the butterfly.  One workgroup of 1024 threads: all of them bring a round of rows into LDS, loads in
// flight together; the chain of additions belongs to one wavefront per accumulator.  6912 rows: 26 us as one wavefront that
// waits for every load, 5 us with the rows through LDS.  The result is valid in wavefront a for accumulator a.
template <int NACC>
__device__ __forceinline__ double combine_row_sums(const double *row_sums, size_t n)
{
    constexpr int CH = 7168 / NACC / 64 * 64, U = (NACC * CH + 1023) / 1024;  // rows a round: 56 KiB of LDS
    __shared__ double sh[NACC * CH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double s = 0.0;
    for (size_t r0 = 0; r0 < n; r0 += CH) {
        const int rows = n - r0 < (size_t)CH ? (int)(n - r0) : CH;
        double v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int e = tid + 1024 * i, a = min(e / CH, NACC - 1), r = min(e - a * CH, rows - 1);
            v[i] = row_sums[a * n + r0 + r];
        }
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (tid + 1024 * i < NACC * CH) sh[tid + 1024 * i] = v[i];
        __syncthreads();
        if (wave < NACC) {
            const double *mine = sh + wave * CH;
            int r = lane;
            for (; r + 15 * 64 < rows; r += 16 * 64) {
                double t[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) t[i] = mine[r + 64 * i];
#pragma unroll
                for (int i = 0; i < 16; ++i) s = s + t[i];
            }
            for (; r < rows; r += 64) s = s + mine[r];
        }
        __syncthreads();
    }
    return wave_sum_f64(s);
}

// Writes mean|W| as f32.
__global__ __launch_bounds__(1024) void absmean_final_kernel(const double *row_sums, size_t n, size_t k, float *w_scale)
{
    const double s = combine_row_sums<1>(row_sums, n);
    if (threadIdx.x == 0) *w_scale = (n == 0 || k == 0) ? 0.0f : (float)(s / ((double)n * (double)k));
}

// What turns a weight into -1, 0 or +1: +1 where w >= hi (or w > hi if strict), -1 where -w does.
struct TernaryRule {
    float hi;
    bool strict;
};
// RoundClip(w / s, -1, 1) is +1 exactly where the correctly rounded quotient is at least 1/2, that is where w / s is at
// least 1/2 - 2^-26 (halfway to the float below 1/2; the tie goes to 1/2, whose significand is even), so where w is at
// least the smallest float not below s * (1/2 - 2^-26), a product that is exact in f64 (24 + 25 significand bits).  One
// comparison per weight in place of a division and a rounding.  s = 0 and a non-finite s make every weight 0.
__device__ __forceinline__ TernaryRule ternary_rule(int method, float factor, float s)
{
    if (method != BITNET_HIP_TERNARY_ABSMEAN_ROUNDCLIP) return {f32_mul(factor, s), true};  // strict, bitnet-quant/src/simd/ternary.rs:75-83
    if (!(s > 0.0f) || s == __builtin_inff()) return {__builtin_nanf(""), true};  // no comparison holds
    const double bound = (double)s * (0.5 - 0x1p-26);
    float hi = (float)bound;
    if ((double)hi < bound) hi = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, hi) + 1u);  // the next float up (hi >= 0)
    return {hi, false};
}
__device__ __forceinline__ int ternarize_one(float w, const TernaryRule &t)
{
    return t.strict ? (w > t.hi ? 1 : (w < -t.hi ? -1 : 0)) : (w >= t.hi ? 1 : (w <= -t.hi ? -1 : 0));
}

// Four lanes that hold the code bytes of four consecutive groups of four weights each end up with the dword of all four.
__device__ __forceinline__ uint32_t quad_dword(uint32_t byte, int lane)
{
    uint32_t w = byte << (8 * (lane & 3));
    w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0xB1, 0xf, 0xf, true);
    w |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x4E, 0xf, 0xf, true);
    return w;
}

// Byte j of lane i of four becomes byte i of lane j.
__device__ __forceinline__ uint32_t quad_transpose(uint32_t x, int lane)
{
    uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, true);  // lane ^ 1
    x = __builtin_amdgcn_perm(y, x, lane & 1 ? 0x03070105u : 0x06020400u);
    y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, true);  // lane ^ 2
    return __builtin_amdgcn_perm(y, x, lane & 2 ? 0x03020706u : 0x05040100u);
}

// Weights from base (a multiple of 4) up to end by one wavefront, a byte per lane and round.
__device__ __forceinline__ void ternarize_bytes(const float *w, size_t base, size_t end, const TernaryRule &rule, uint8_t *packed, int8_t *q_i8, int lane)
{
    for (size_t e = base + 4 * lane; e < end; e += 256) {
        unsigned byte = 0;
        for (int j = 0; j < 4 && e + j < end; ++j) {
            const int t = ternarize_one(w[e + j], rule);
            if (q_i8) q_i8[e + j] = (int8_t)t;
            byte |= (unsigned)(t + 1) << (2 * j);
        }
        packed[e / 4] = (uint8_t)byte;
    }
}

// A wavefront takes 1024 consecutive weights: load i (of four) is one 16-byte chunk a lane, chunks in lane order, so loads
// are dense; lane l keeps the dword of group i = l mod 4 of its quad and stores it: 256 bytes a wavefront.  Bound by the
// read (6912 x 2560: 24 us as a thread per byte with four scalar loads and a division each, 10 us now).
__global__ __launch_bounds__(256) void ternarize_pack_kernel(const float *w, size_t count, int method,
                                                             float factor, const float *w_scale,
                                                             uint8_t *packed, int8_t *q_i8, bool dense)
{
    const int lane = threadIdx.x & 63;
    const TernaryRule rule = ternary_rule(method, factor, *w_scale);
    size_t base = ((size_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 1024;
    for (; dense && base + 1024 <= count; base += (size_t)gridDim.x * 4096) {
        float4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const float4 *>(w + base + 256 * i + 4 * lane);
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t0 = ternarize_one(v[i].x, rule), t1 = ternarize_one(v[i].y, rule), t2 = ternarize_one(v[i].z, rule),
                      t3 = ternarize_one(v[i].w, rule);
            if (q_i8)
                *reinterpret_cast<uint32_t *>(q_i8 + base + 256 * i + 4 * lane) =
                    (uint32_t)(t0 & 0xff) | ((uint32_t)(t1 & 0xff) << 8) | ((uint32_t)(t2 & 0xff) << 16) | ((uint32_t)(t3 & 0xff) << 24);
            const uint32_t d = quad_dword((uint32_t)((t0 + 1) | ((t1 + 1) << 2) | ((t2 + 1) << 4) | ((t3 + 1) << 6)), lane);
            if ((lane & 3) == i) mine = d;
        }
        *reinterpret_cast<uint32_t *>(packed + base / 4 + 64 * (lane & 3) + (lane & ~3)) = mine;
    }
    // the end of the matrix, and buffers that are not aligned
    for (; base < count; base += (size_t)gridDim.x * 4096) ternarize_bytes(w, base, base + 1024 < count ? base + 1024 : count, rule, packed, q_i8, lane);
}

// absmean_final_kernel and ternarize_pack_kernel in one launch, for row sums that are not where the codes go: the first wavefront of every
// workgroup adds the row sums up (lane l rows l, l+64, ..., then the butterfly, as there) while the first weights of the other 15 are on
// their way.  These have CODES_HELD chunks of 1024 weights each in registers, which is a matrix of 79 MB; of a larger one the next chunk is
// asked for where one has been used.  Bound by the read of the matrix, the second one, and up to 32 MB of weights, which the dies' L2s hold, by the
// sum's way through one wavefront.  A call, with the three launches -> with two:
// 6912 x 2560 27.6 -> 23.8 us, 4096 x 4096 27.2 -> 22.2, 4096 x 2560 18.6 -> 11.9, 4096 x 2048 16.6 -> 9.6, 14336 x 4096 77.6 -> 73.1, 256 x 512 8.1 ->
// 6.9 (the host's launches).  Without the dies' shares, with every chunk on any die: 4096 x 2048 13.6, 6144 x 1024 13.1 (9.5 with, 10.6
// in three launches, whose two passes went over 1024 columns in the same order); beyond 84 MB the shares only spread the reads: 14336 x 4096 72.9
// without, 75.2 with, 6144 x 4096 33.6 and 34.2.  A workgroup has 15 chunks where there are so few: as many workgroups as compute units are no faster
// (1024 x 1024 7.2 and 7.3 us) and keep other launches out (on three streams at once 4.7 and 3.4 us a call).  Beside two more streams of the same
// calls matrices of few columns are still slower than in three launches, whose first two leave room: 14336 x 256 8.5 -> 11.7 (alone 13.9 -> 12.2),
// 8192 x 768 9.4 -> 10.9 (16.3 -> 10.4), 2560 x 2560 and larger even.  With all wavefronts bringing the row sums into LDS ahead of their weights 2 us
// more; the whole quantiser in one launch whose workgroups wait for each other's row sums with the matrix in registers takes 22.1 for 6912 x 2560, but
// two to four such launches on streams of their own keep each other off the compute units: 48 us a call in place of 23.
constexpr int CODES_HELD = 5, CODES_SUMS = 36;  // chunks and rows of 64 row sums on their way to a wavefront
constexpr size_t CODES_MAX_ROWS = 65536;        // beyond, every workgroup reading all row sums is what takes the time
constexpr size_t CODES_SHARED = 21000000;       // weights up to which a die reads its own rows again

// The codes of 1024 consecutive weights, a float4 of each 256 a lane: lane l of a quad ends with the dword of the quad's group l, as above.
__device__ __forceinline__ void codes_of_chunk(const float4 (&v)[4], float t, uint8_t *packed, size_t chunk, int lane)
{
    // A code is 1 where |w| < t, which is the sign of |w| - t, else 0 or 2 by the sign of w: both signs are shifted in, and put right for 16 at a time.
    uint32_t x = 0;
    const auto take = [&](float w) {
        x = __builtin_amdgcn_alignbit(x, __builtin_bit_cast(uint32_t, w), 31);
        x = __builtin_amdgcn_alignbit(x, __builtin_bit_cast(uint32_t, fabsf(w) - t), 31);
    };
#pragma unroll
    for (int i = 3; i >= 0; --i) {
        take(v[i].w);
        take(v[i].z);
        take(v[i].y);
        take(v[i].x);
    }
    x = t == t ? (x & 0x55555555u) | (~(x | (x << 1)) & 0xaaaaaaaau) : 0x55555555u;
    *reinterpret_cast<uint32_t *>(packed + chunk * 256 + 64 * (lane & 3) + (lane & ~3)) = quad_transpose(x, lane);
}

__global__ __launch_bounds__(1024) void absmean_codes_kernel(const float *w, size_t n, size_t k, int method, float factor,
                                                             const double *row_sums, uint8_t *packed, float *w_scale)
{
    __shared__ float scale_s;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const size_t chunks = n * k / 1024, stride = (size_t)gridDim.x * 15;
    size_t first = (size_t)(wave - 1) * gridDim.x + blockIdx.x;  // as many for every workgroup
    // A workgroup runs on the die of its number modulo eight, here and in absmean_rows_kernel, where it has four rows.  Where those are whole
    // chunks, the chunks are dealt out so that a die reads again what it has read, from its own L2: groups of eight times `share` chunks.
    const unsigned share = k % 256 == 0 && n * k <= CODES_SHARED ? (unsigned)(k / 256) : 1, group_chunks = 8 * share;
    const unsigned grouped = share > 1 ? (unsigned)chunks / group_chunks * group_chunks : 0;
    const auto chunk_of = [&](size_t turn) -> size_t {
        if (turn >= grouped) return turn;
        const unsigned group = (unsigned)turn / group_chunks, at = (unsigned)turn - group * group_chunks;
        return group * group_chunks + (at & 7) * share + (at >> 3);
    };
    float4 v[CODES_HELD][4];
    const auto load = [&](float4 (&to)[4], size_t chunk) {  // zeros past the last one: no branch, so that each chunk is waited for by itself
        const __amdgpu_buffer_rsrc_t of = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(w + chunk * 1024), 0, chunk < chunks ? 4096 : 0, 0x00020000);
#pragma unroll
        for (int i = 0; i < 4; ++i) to[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(of, 16 * lane + 1024 * i, 0, 0));
    };
    if (wave == 0) {
        // Zeros past the last row (a sum of absolute values stays what it is), and CODES_SUMS rows of 64 always on their way.
        const __amdgpu_buffer_rsrc_t sums = __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(row_sums), 0, (int)(8 * n), 0x00020000);
        const auto sum = [&](int row) { return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(sums, 8 * row, 0, 0)); };
        double total = 0.0, r[CODES_SUMS];
#pragma unroll
        for (int i = 0; i < CODES_SUMS; ++i) r[i] = sum(lane + 64 * i);
        for (int row = lane; row - lane < (int)n; row += 64 * CODES_SUMS) {
#pragma unroll
            for (int i = 0; i < CODES_SUMS; ++i) {
                total = total + r[i];
                r[i] = sum(row + 64 * (CODES_SUMS + i));
            }
        }
        total = wave_sum_f64(total);
        if (lane == 0) scale_s = (float)(total / ((double)n * (double)k));
        first = chunks;
    } else {
#pragma unroll
        for (int h = 0; h < CODES_HELD; ++h) load(v[h], chunk_of(first + h * stride));
    }
    __syncthreads();
    const float scale = scale_s;
    if (blockIdx.x == 0 && tid == 0) *w_scale = scale;
    // t > 0, or NaN (every code 0): w > hi, for hi >= 0, is w >= the next float up, which is a NaN for an infinite hi.  The next one up of a NaN
    // whose bits are all ones would be -0.
    const TernaryRule rule = ternary_rule(method, factor, scale);
    const float t = rule.strict && rule.hi == rule.hi ? __builtin_bit_cast(float, __builtin_bit_cast(unsigned, fabsf(rule.hi)) + 1u) : rule.hi;
    size_t chunk = first;
    for (; chunk + CODES_HELD * stride < chunks; chunk += CODES_HELD * stride) {
#pragma unroll
        for (int h = 0; h < CODES_HELD; ++h) {
            codes_of_chunk(v[h], t, packed, chunk_of(chunk + h * stride), lane);
            load(v[h], chunk_of(chunk + (h + CODES_HELD) * stride));
        }
    }
#pragma unroll
    for (int h = 0; h < CODES_HELD; ++h)
        if (chunk + h * stride < chunks) codes_of_chunk(v[h], t, packed, chunk_of(chunk + h * stride), lane);
    if (blockIdx.x == gridDim.x - 1 && wave == 15) ternarize_bytes(w, chunks * 1024, n * k, rule, packed, nullptr, lane);
}

// ---- BitNetWeightQuantizer::quantize, the reference's weight pipeline (bitnet-quant/src/quantization/weights.rs:568-611)
//
//   w' = (w - mean) / sqrt(var + 1e-8)                   normalize_before_quantize, :671-686
//   w'' = clamp(w', mean' - t*mad, mean' + t*mad)        handle_outliers, :688-699 (mad = mean|w'|)
//   thr by TernaryMethod from mean|w''| (and max|w''|)   :370-480
//   q = sign(w'') * [|w''| > thr]                        apply_ternary_quantization, :482-496
//   scale = sum(w''*q) / sum(q*q)                        compute_ternary_scale, :546-559
//
// Nothing but the packed codes and the scale is written: w'' is recomputed from w wherever it is needed (the short
// division by the deviation, which is the same for the whole tensor, and a clamp).  Every tensor-wide sum is carried in f64
// in the order of the absmean kernels above (per row: lane l adds columns l, l+64, ..., then the butterfly; the row sums
// the same way), so the f32 scalars have the bits the CPU restatement of the same order has.  The scalars stay on the
// device in WqState.  Who finishes a reduction and derives the next stage's scalars: up to WQ_FOLD_MAX_ROWS rows every workgroup of
// the next pass, for itself (a wavefront adds up to 64 row sums a lane while a launch of its own takes 3.1 us and the gap in front of
// it); above, and where no pass follows, one workgroup in a launch between the passes.  The last pass (the scale's sums) knows the
// threshold, so it writes the codes too where rows start on bytes.
struct WqState {
    float mean, sd;            // normalisation (0, 1 when switched off)
    float clip_mean, clip_mad; // centre and mean |.| of the normalised tensor
    float lo, hi;              // clip bounds (-inf, +inf when switched off)
    float mean_abs, max_abs;   // of the processed tensor
    float thr;
    float num, den, scale;
};
static_assert(sizeof(WqState) == 12 * sizeof(float), "stats are returned as 12 floats");

enum WqPass { WQ_SUM = 0, WQ_SQDIFF, WQ_CLIP_STATS, WQ_ABS_STATS, WQ_OPTIMAL, WQ_SCALE };
constexpr int WQ_MAX_ACC = 10;
constexpr size_t WQ_SCRATCH_SUMS = 4 + WQ_MAX_ACC;  // doubles a row: those of two consecutive passes (two each), and of WQ_OPTIMAL

__device__ __forceinline__ void wq_publish(const WqState &st, int clip, float *w_scale, float *stats)
{
    *w_scale = st.scale;
    if (stats) {
        const float v[12] = {st.mean, st.sd, st.clip_mean, st.clip_mad, clip ? st.lo : 0.0f, clip ? st.hi : 0.0f,
                             st.mean_abs, st.max_abs, st.thr, st.num, st.den, st.scale};
        for (int i = 0; i < 12; ++i) stats[i] = v[i];
    }
}

// The scalars of a pass: the state, and the divisor of the normalisation prepared for div_by_invariant (ieee.hpp).
struct WqView {
    WqState st;
    float recip;
    bool fast, normalize, clip;
};
__device__ __forceinline__ WqView wq_view(const WqState &state, int normalize, int clip)
{
    WqView v;
    v.st = state;
    v.recip = f32_div(1.0f, v.st.sd);
    v.fast = invariant_divisor_ok(v.st.sd);
    v.normalize = normalize != 0;
    v.clip = clip != 0;
    return v;
}
__device__ __forceinline__ float wq_normalised(float w, const WqView &p)
{
    if (!p.normalize) return w;
    const float d = w - p.st.mean;
    // the short division where every lane's dividend allows it: the same bits as the plain one
    if (p.fast && __builtin_amdgcn_ballot_w64(!dividend_ok(d)) == 0) return div_by_invariant_unchecked(d, p.st.sd, p.recip);
    return f32_div(d, p.st.sd);
}
// The same for U elements a lane: one look at the largest and the smallest |dividend| (a zero takes the way above) in place of one at each, and
// U divisions that do not wait for each other.  6912 x 2560, the passes that normalise: 15.3, 16.1 and 22.2 -> 13.8, 14.3 and 19.2 us.
template <int U>
__device__ __forceinline__ void wq_normalise(float (&w)[U], const WqView &p)
{
    if (!p.normalize) return;
    float d[U], lo = __builtin_inff(), hi = 0.0f;
#pragma unroll
    for (int i = 0; i < U; ++i) {
        d[i] = w[i] - p.st.mean;
        lo = fminf(lo, fabsf(d[i]));
        hi = fmaxf(hi, fabsf(d[i]));
    }
    if (p.fast && __builtin_amdgcn_ballot_w64(!(lo >= 0x1p-63f && hi < 0x1p63f)) == 0) {
#pragma unroll
        for (int i = 0; i < U; ++i) w[i] = div_by_invariant_unchecked(d[i], p.st.sd, p.recip);
    } else {
#pragma unroll
        for (int i = 0; i < U; ++i) w[i] = wq_normalised(w[i], p);
    }
}
// x: normalised.
__device__ __forceinline__ float wq_clipped(float x, const WqView &p)
{
    if (p.clip) {
        x = x > p.st.hi ? p.st.hi : x;
        x = x < p.st.lo ? p.st.lo : x;
    }
    return x;
}
__device__ __forceinline__ float wq_processed(float w, const WqView &p) { return wq_clipped(wq_normalised(w, p), p); }
__device__ __forceinline__ float wq_code(float x, float thr) { return x > thr ? 1.0f : (x < -thr ? -1.0f : 0.0f); }

__constant__ float wq_factors[10] = {0.3f, 0.4f, 0.5f, 0.6f, 0.7f, 0.8f, 0.9f, 1.0f, 1.1f, 1.2f};

// Before the first pass (state: none), or what the passes so far have left.
__device__ __forceinline__ WqState wq_state(const WqState *state)
{
    if (state) return *state;
    WqState st;
    st.mean = 0.0f; st.sd = 1.0f; st.clip_mean = 0.0f; st.clip_mad = 0.0f; st.lo = -__builtin_inff(); st.hi = __builtin_inff();
    st.mean_abs = 0.0f; st.max_abs = 0.0f; st.thr = 0.0f; st.num = 0.0f; st.den = 0.0f; st.scale = 1.0f;
    return st;
}

// How thresholds and clip bounds come from the sums.  method: TernaryMethod 0..4; custom <= 0: the method's own factor.
struct WqRule {
    int method;
    float outlier_threshold, custom;
};

// The scalars that the finished sums `tot` (and mx, the largest row_max) of a pass give.
__device__ __forceinline__ void wq_derive(WqState &st, int pass, const double *tot, float mx, double count, const WqRule &rule)
{
    if (pass == WQ_SUM) {
        st.mean = (float)(tot[0] / count);
    } else if (pass == WQ_SQDIFF) {
        const float var = (float)(tot[0] / count);
        st.sd = f32_sqrt(var + 1e-8f);
    } else if (pass == WQ_CLIP_STATS) {
        st.clip_mean = (float)(tot[0] / count);
        st.clip_mad = (float)(tot[1] / count);
        const float spread = f32_mul(rule.outlier_threshold, st.clip_mad);
        st.lo = st.clip_mean - spread;
        st.hi = st.clip_mean + spread;
    } else if (pass == WQ_ABS_STATS) {
        st.mean_abs = (float)(tot[0] / count);
        st.max_abs = mx;
        const bool has_custom = rule.custom > 0.0f;
        float thr;
        if (rule.method == 1) thr = f32_mul(st.mean_abs, has_custom ? rule.custom : 0.8f);
        else if (rule.method == 2)
            thr = has_custom ? f32_mul(st.mean_abs, rule.custom)
                             : (st.max_abs > f32_mul(3.0f, st.mean_abs) ? f32_mul(st.mean_abs, 0.5f) : f32_mul(st.mean_abs, 0.7f));
        else thr = f32_mul(st.mean_abs, has_custom ? rule.custom : 0.7f);  // mean, DetSTE; optimal without its search
        st.thr = thr;
    } else if (pass == WQ_OPTIMAL) {
        float best = __builtin_inff(), thr = f32_mul(st.mean_abs, 0.7f);
#pragma unroll
        for (int f = 0; f < 10; ++f) {
            const float mse = (float)(tot[f] / count);
            if (mse < best) { best = mse; thr = f32_mul(st.mean_abs, wq_factors[f]); }
        }
        st.thr = thr;
    } else {
        st.num = (float)tot[0];
        st.den = (float)tot[1];
        st.scale = fabsf(st.den) < 1.1920929e-07f ? 1.0f : f32_div(st.num, st.den);
    }
}

// What a pass with at most WQ_FOLD_MAX_ROWS rows finishes of the pass before it (pass < 0: nothing is left to finish).
struct WqPrevious {
    int pass;            // of those with one or two accumulators
    const double *sums;  // not those this pass writes
    WqState *state;      // where the state with its scalars goes, for the next pass; not the one this pass reads
    WqRule rule;
};
constexpr size_t WQ_FOLD_MAX_ROWS = 4096;

// By a workgroup of four wavefronts: an accumulator each by the first two (the order of combine_row_sums), the largest row maximum
// by all of them.
__device__ __forceinline__ void wq_finish_previous(WqState &st, const WqPrevious &prev, const float *row_max, size_t n, size_t k)
{
    __shared__ double tot[2];
    __shared__ float maxima[4];
    const int lane = threadIdx.x, wave = threadIdx.y;
    const int nacc = prev.pass == WQ_CLIP_STATS ? 2 : 1, rows = (int)n;
    if (wave < nacc) {
        const double *sums = prev.sums + (size_t)wave * n;
        double s = 0.0;
        int row = lane;
        const auto add = [&](auto batch) {  // so many loads in flight: 32, then 8 (8 throughout: 0.5 us a pass more at 2048 rows)
            constexpr int U = decltype(batch)::value;
            for (; row + 63 - lane + (U - 1) * 64 < rows; row += U * 64) {
                double t[U];
#pragma unroll
                for (int i = 0; i < U; ++i) t[i] = sums[row + 64 * i];
#pragma unroll
                for (int i = 0; i < U; ++i) s = s + t[i];
            }
        };
        add(std::integral_constant<int, 32>());
        add(std::integral_constant<int, 8>());
        for (; row < rows; row += 64) s = s + sums[row];
        s = wave_sum_f64(s);
        if (lane == 0) tot[wave] = s;
    }
    float mx = 0.0f;
    if (prev.pass == WQ_ABS_STATS) {
        for (int row = lane + 64 * wave; row < rows; row += 256) mx = fmaxf(mx, row_max[row]);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        if (lane == 0) maxima[wave] = mx;
    }
    __syncthreads();
    if (prev.pass == WQ_ABS_STATS) mx = fmaxf(fmaxf(maxima[0], maxima[1]), fmaxf(maxima[2], maxima[3]));
    wq_derive(st, prev.pass, tot, mx, (double)n * (double)k, prev.rule);
}

constexpr int wq_accumulators(int pass) { return pass == WQ_OPTIMAL ? 10 : ((pass == WQ_CLIP_STATS || pass == WQ_SCALE) ? 2 : 1); }

// One wavefront per row; accumulator a of row r goes to row_sums[a * n + r] (and the row's max |.| to row_max[r]).
// packed (WQ_SCALE, k a multiple of 4, else null): the codes of the row, four columns a byte, put together by the quad of
// lanes that holds them; q_i8 as ever optional.  Bound by the read of the matrix.
// FOLD: what WqPrevious says comes first, in every workgroup.
template <int PASS, bool FOLD>
__global__ __launch_bounds__(256) void wq_rows_kernel(const float *w, size_t n, size_t k, const WqState *state, int normalize,
                                                      int clip, double *row_sums, float *row_max, uint8_t *packed, int8_t *q_i8,
                                                      WqPrevious prev)
{
    constexpr int NACC = wq_accumulators(PASS);
    const int lane = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * blockDim.y + threadIdx.y;
    WqState st = wq_state(state);
    if constexpr (FOLD) {
        if (prev.pass >= 0) wq_finish_previous(st, prev, row_max, n, k);
        if (blockIdx.x == 0 && threadIdx.x == 0 && threadIdx.y == 0) *prev.state = st;
    }
    if (row >= n) return;
    const WqView p = wq_view(st, normalize, clip);
    double acc[NACC];
#pragma unroll
    for (int a = 0; a < NACC; ++a) acc[a] = 0.0;
    float mx = 0.0f;
    int nonzero = 0;  // of the row
    float cand[PASS == WQ_OPTIMAL ? 10 : 1];
    if constexpr (PASS == WQ_OPTIMAL) {
#pragma unroll
        for (int f = 0; f < 10; ++f) cand[f] = f32_mul(p.st.mean_abs, wq_factors[f]);
    }
    [[maybe_unused]] const auto scale_step = [&](float v) {
        const float x = wq_clipped(v, p);
        const float q = wq_code(x, p.st.thr);
        acc[0] = acc[0] + (double)f32_mul(x, q);
        nonzero += __popcll(__builtin_amdgcn_ballot_w64(q != 0.0f));  // sum of q * q: a count, exact in any order
        return q;
    };
    size_t first = 0;  // column
    if constexpr (PASS == WQ_SCALE) {
        // Four groups of 64 columns at a time: the quads of lanes exchange codes, so that a lane has four consecutive columns of one group
        // and stores them as a dword and a byte, in place of a byte store a column and a byte store a group.  This pass on 6912 x 2560:
        // 25.2 -> 22.2 us, on 14336 x 8192 153 -> 122 (with the normalising above 19.2 and 119; the read alone takes 12 and 85).
        if (packed && (reinterpret_cast<uintptr_t>(q_i8) & 3) == 0) {
            for (const float *p4 = w + row * k + lane; first + 256 <= k;) {
                const int groups = first + 512 <= k ? 8 : 4;  // eight loads in flight
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = p4[first + 64 * min(i, groups - 1)];
                wq_normalise(v, p);
#pragma unroll
                for (int h = 0; h < 8; h += 4) {
                    if (h >= groups) break;
                    uint32_t codes = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) codes |= (uint32_t)((int)scale_step(v[h + i]) + 1) << (8 * i);
                    codes = quad_transpose(codes, lane);
                    const size_t at = row * k + first + 64 * (h + (lane & 3)) + (lane & ~3);
                    if (q_i8) *reinterpret_cast<uint32_t *>(q_i8 + at) = ((codes | 0x80808080u) - 0x01010101u) ^ 0x80808080u;
                    codes |= codes >> 6;
                    packed[at / 4] = (uint8_t)(codes | (codes >> 12));
                }
                first += 64 * groups;
            }
        }
    }
    const auto ready = [&](auto &v) {
        if constexpr (PASS != WQ_SUM && PASS != WQ_SQDIFF) wq_normalise(v, p);
    };
    for_row<PASS == WQ_OPTIMAL ? 4 : 10>(w + row * k + first, k - first, lane, ready, [&](float v, size_t c) {
        if constexpr (PASS == WQ_SUM) {
            acc[0] = acc[0] + (double)v;
        } else if constexpr (PASS == WQ_SQDIFF) {
            const float d = v - p.st.mean;
            acc[0] = acc[0] + (double)f32_mul(d, d);
        } else if constexpr (PASS == WQ_CLIP_STATS) {
            acc[0] = acc[0] + (double)v;
            acc[1] = acc[1] + (double)fabsf(v);
        } else if constexpr (PASS == WQ_ABS_STATS) {
            const float ax = fabsf(wq_clipped(v, p));
            acc[0] = acc[0] + (double)ax;
            mx = fmaxf(mx, ax);
        } else if constexpr (PASS == WQ_OPTIMAL) {
            const float x = wq_clipped(v, p);
#pragma unroll
            for (int f = 0; f < 10; ++f) {
                const float d = x - wq_code(x, cand[f]);
                acc[f] = acc[f] + (double)f32_mul(d, d);
            }
        } else {
            const float q = scale_step(v);
            c += first;
            if (packed) {  // k % 4 == 0: the four columns of a byte are active together
                const int t = (int)q;
                if (q_i8) q_i8[row * k + c] = (int8_t)t;
                uint32_t b = (uint32_t)(t + 1) << (2 * (lane & 3));
                b |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, 0xB1, 0xf, 0xf, true);
                b |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, 0x4E, 0xf, 0xf, true);
                if ((lane & 3) == 0) packed[(row * k + c) / 4] = (uint8_t)b;
            }
        }
    });
#pragma unroll
    for (int a = 0; a < NACC; ++a) {
        const double s = PASS == WQ_SCALE && a == 1 ? (double)nonzero : wave_sum_f64(acc[a]);
        if (lane == 0) row_sums[(size_t)a * n + row] = s;
    }
    if constexpr (PASS == WQ_ABS_STATS) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        if (lane == 0) row_max[row] = mx;
    }
}

// One workgroup: combines the row sums of every accumulator and derives the scalars of the next stage (state: before, next: after,
// may be the same).  WQ_SCALE, the last stage, also publishes the scale and (optionally) the twelve scalars.
template <int PASS>
__global__ __launch_bounds__(1024) void wq_final_kernel(const double *row_sums, const float *row_max, size_t n, size_t k,
                                                        const WqState *state, WqState *next, WqRule rule, int clip, float *w_scale, float *stats)
{
    constexpr int NACC = wq_accumulators(PASS);
    __shared__ double tot[NACC];
    __shared__ float maxima[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if constexpr (PASS == WQ_ABS_STATS) {
        float mx = 0.0f;
        for (size_t r = threadIdx.x; r < n; r += 1024) mx = fmaxf(mx, row_max[r]);
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        if (lane == 0) maxima[wave] = mx;
    }
    const double s = combine_row_sums<NACC>(row_sums, n);
    if (lane == 0 && wave < NACC) tot[wave] = s;
    __syncthreads();
    if (threadIdx.x != 0) return;
    float mx = 0.0f;
    if constexpr (PASS == WQ_ABS_STATS)
        for (int i = 0; i < 16; ++i) mx = fmaxf(mx, maxima[i]);
    WqState st = wq_state(state);
    wq_derive(st, PASS, tot, mx, (double)n * (double)k, rule);
    if constexpr (PASS == WQ_SCALE) wq_publish(st, clip, w_scale, stats);
    *next = st;
}

__global__ void wq_empty_kernel(int clip, float *w_scale, float *stats) { wq_publish(wq_state(nullptr), clip, w_scale, stats); }

// Ternarise the processed tensor with the threshold found, pack; thread b builds byte b (widths that are no multiple of 4,
// where a byte holds columns of two rows).
__global__ __launch_bounds__(256) void wq_ternarize_pack_kernel(const float *w, size_t count, const WqState *state, int normalize,
                                                                int clip, uint8_t *packed, int8_t *q_i8, size_t nbytes)
{
    size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbytes) return;
    const WqView p = wq_view(*state, normalize, clip);
    unsigned byte = 0;
    for (int j = 0; j < 4; ++j) {
        size_t i = 4 * b + j;
        if (i < count) {
            const int t = (int)wq_code(wq_processed(w[i], p), p.st.thr);
            if (q_i8) q_i8[i] = (int8_t)t;
            byte |= ((unsigned)(t + 1) & 3u) << (2 * j);
        }
    }
    packed[b] = (uint8_t)byte;
}

// Codes of 16 consecutive elements e0 .. e0 + 15 (element j at bits 2j), code 3 as code 1; elements from `valid` on hold
// code 1.  Reads the bytes that hold valid elements and no others.
__device__ __forceinline__ uint32_t load_codes16(const uint8_t *packed, size_t e0, int valid, bool dwords)
{
    uint32_t s = 0x55555555u;
    if (valid > 0) {
        if (dwords && valid >= 16) {  // e0 a multiple of 16, packed aligned to 4 bytes
            s = reinterpret_cast<const uint32_t *>(packed)[e0 >> 4];
        } else {
            const int n = valid < 16 ? valid : 16;
            const unsigned first = 2 * (unsigned)(e0 & 3);  // bit of element e0 in its byte
            const size_t b0 = e0 >> 2, bytes = (first + 2 * n + 7) >> 3;
            unsigned long long v = 0;
#pragma unroll
            for (int i = 0; i < 5; ++i)
                if ((size_t)i < bytes) v |= (unsigned long long)packed[b0 + i] << (8 * i);
            s = (uint32_t)(v >> first);
            if (n < 16) s = (s & ((1u << (2 * n)) - 1u)) | (0x55555555u & ~((1u << (2 * n)) - 1u));
        }
    }
    const uint32_t three = s & (s >> 1) & 0x55555555u;
    return s & ~(three << 1);
}

// 4 x 4 transposition of the 2-bit fields of a dword: field 4q + b (flat order) <-> bits 2q + 8b (tile order).  Its own inverse.
__device__ __forceinline__ uint32_t interleave16(uint32_t s)
{
    uint32_t t = ((s >> 6) ^ s) & 0x00cc00ccu;
    s ^= t ^ (t << 6);
    t = ((s >> 12) ^ s) & 0x0000f0f0u;
    return s ^ t ^ (t << 12);
}

// [out, in] source: one thread builds one dword (16 weights of one row) of the tiled layout.  A workgroup reads whole
// 64-byte pieces of 16 rows and writes 1 KiB, for RETILE_KT k-tiles of a row block (a workgroup per tile is bound by the
// dispatch of workgroups).  canonical (optional; rows of whole dwords only): the same codes back in flat order.  w_scale_out
// (optional): receives w_scale.  (6912 x 2560: 37 us element by element.)
constexpr unsigned RETILE_KT = 5;
__global__ __launch_bounds__(256) void retile_kernel(const uint8_t *packed, size_t n, size_t k, uint32_t *tiled, unsigned kt_count,
                                                     bool dwords, uint32_t *canonical, float w_scale, float *w_scale_out)
{
    const unsigned kt0 = blockIdx.x * RETILE_KT, rb = blockIdx.y + gridDim.y * blockIdx.z;
    if (kt0 == 0 && rb == 0 && threadIdx.x == 0 && w_scale_out) *w_scale_out = w_scale;
    if ((size_t)rb * TILE_ROWS >= n) return;
    const unsigned slot = threadIdx.x >> 2, t = threadIdx.x & 3;
    const size_t row = (size_t)rb * TILE_ROWS + (slot & 15);
    uint32_t s[RETILE_KT];
    int valid[RETILE_KT];
#pragma unroll
    for (unsigned i = 0; i < RETILE_KT; ++i) {
        const size_t col = (size_t)(kt0 + i) * TILE_K + 64 * t + 16 * (slot >> 4);
        valid[i] = row < n && col < k ? (int)(k - col < 16 ? k - col : 16) : 0;
        s[i] = load_codes16(packed, row * k + col, valid[i], dwords);
    }
#pragma unroll
    for (unsigned i = 0; i < RETILE_KT; ++i) {
        if (kt0 + i >= kt_count) break;  // uniform
        const size_t col = (size_t)(kt0 + i) * TILE_K + 64 * t + 16 * (slot >> 4);
        if (canonical && valid[i]) canonical[(row * k + col) >> 4] = s[i];
        tiled[((size_t)rb * kt_count + kt0 + i) * 256 + threadIdx.x] = interleave16(s[i]);
    }
}

// [in, out] source: one thread takes the 16 columns of one dword position for all 16 rows of a row block (16 codes of 16
// source rows each), transposes them in registers and stores 16 dwords.  Consecutive lanes take consecutive row blocks, so
// they read consecutive dwords of a source row.
__global__ __launch_bounds__(64) void retile_in_out_kernel(const uint8_t *packed, size_t n, size_t k, uint32_t *tiled, unsigned kt_count,
                                                           bool dwords, float w_scale, float *w_scale_out)
{
    const size_t rb = (size_t)blockIdx.x * 64 + threadIdx.x;
    const unsigned piece = blockIdx.y + gridDim.y * blockIdx.z;
    const unsigned g = piece & 15, kt = piece >> 4;  // column group: columns 64 * (g >> 2) + 16 * (g & 3) of the tile
    if (rb == 0 && piece == 0 && w_scale_out) *w_scale_out = w_scale;
    if (rb * TILE_ROWS >= n || kt >= kt_count) return;
    const unsigned t = g >> 2, kq = g & 3;
    const size_t row0 = rb * TILE_ROWS, col0 = (size_t)kt * TILE_K + 64 * t + 16 * kq;
    const int rows = (int)(n - row0 < 16 ? n - row0 : 16);
    uint32_t src[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) src[j] = load_codes16(packed, (col0 + j) * n + row0, col0 + j < k ? rows : 0, dwords);
    uint32_t *out = tiled + (rb * kt_count + kt) * 256 + 64 * kq + t;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < 16; ++j) word |= ((src[j] >> (2 * r)) & 3u) << (2 * (j >> 2) + 8 * (j & 3));
        out[4 * r] = word;
    }
}

// Inverse, rows of whole dwords (k a multiple of 16): one thread rebuilds the 16 elements of one dword of the flat packing.
__global__ __launch_bounds__(256) void untile_rows_kernel(const uint32_t *tiled, unsigned dwords_per_row, size_t n, uint32_t *packed,
                                                          unsigned kt_count)
{
    const unsigned d = blockIdx.x * 256 + threadIdx.x;
    const size_t row = blockIdx.y + (size_t)gridDim.y * blockIdx.z;
    if (d >= dwords_per_row || row >= n) return;
    const unsigned kt = d >> 4, g = d & 15;
    const size_t tile = (row / TILE_ROWS) * kt_count + kt;
    packed[row * dwords_per_row + d] = interleave16(tiled[tile * 256 + 64 * (g & 3) + 4 * (row % TILE_ROWS) + (g >> 2)]);
}

// Inverse, any width: one thread rebuilds one byte of the flat [n, k] packing.
__global__ __launch_bounds__(256) void untile_kernel(const uint32_t *tiled, size_t n, size_t k, uint8_t *packed,
                                                     size_t kt_count, size_t nbytes)
{
    size_t b = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nbytes) return;
    const size_t count = n * k;
    size_t row = 4 * b / k, kk = 4 * b - row * k;
    unsigned byte = 0;
    for (int j = 0; j < 4; ++j) {
        if (4 * b + j >= count) break;
        size_t tile = (row / TILE_ROWS) * kt_count + kk / TILE_K;
        unsigned g = (unsigned)((kk % TILE_K) / 16), c = (unsigned)(kk % 16);
        unsigned wd = (((g & 3) * 16 + (unsigned)(row % TILE_ROWS)) << 2) + (g >> 2);
        uint32_t word = tiled[tile * 256 + wd];
        byte |= ((word >> (2 * (c >> 2) + 8 * (c & 3))) & 3u) << (2 * j);
        if (++kk == k) { kk = 0; ++row; }
    }
    packed[b] = (uint8_t)byte;
}

// Grid dimensions y and z that together cover `items` (y is limited to 65535).
inline dim3 rows_grid(unsigned x, size_t items)
{
    const unsigned y = items < 32768 ? (unsigned)items : 32768u;
    return dim3(x, y, (unsigned)((items + y - 1) / y));
}
inline bool aligned(const void *ptr, size_t a) { return (reinterpret_cast<uintptr_t>(ptr) % a) == 0; }
inline unsigned blocks_for(size_t items, unsigned per_block) { return (unsigned)((items + per_block - 1) / per_block); }

}  // namespace

int launch_pack_2bit(const int8_t *q, size_t count, uint8_t *packed, hipStream_t stream)
{
    size_t nbytes = (count + 3) / 4;
    if (nbytes == 0) return BITNET_HIP_OK;
    launch_kernel(pack_2bit_kernel, dim3(blocks_for(nbytes, 256)), dim3(256), 0, stream, q, count, packed, nbytes);
    BITNET_HIP_CHECK_LAUNCH("pack_2bit_kernel");
    return BITNET_HIP_OK;
}

int launch_unpack_2bit(const uint8_t *packed, size_t count, int8_t *q, hipStream_t stream)
{
    if (count == 0) return BITNET_HIP_OK;
    launch_kernel(unpack_2bit_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, stream, packed, count, q);
    BITNET_HIP_CHECK_LAUNCH("unpack_2bit_kernel");
    return BITNET_HIP_OK;
}

int launch_lookup_compute(int kind, const int8_t *w, const float *x, float *out, size_t n, hipStream_t stream)
{
    if (n == 0) return BITNET_HIP_OK;
    launch_kernel(lookup_compute_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, stream, kind, w, x, out, n);
    BITNET_HIP_CHECK_LAUNCH("lookup_compute_kernel");
    return BITNET_HIP_OK;
}

int launch_pack_base3(const int8_t *q, size_t count, uint8_t *packed, hipStream_t stream)
{
    size_t nbytes = (count + 4) / 5;
    if (nbytes == 0) return BITNET_HIP_OK;
    launch_kernel(pack_base3_kernel, dim3(blocks_for(nbytes, 256)), dim3(256), 0, stream, q, count, packed, nbytes);
    BITNET_HIP_CHECK_LAUNCH("pack_base3_kernel");
    return BITNET_HIP_OK;
}

int launch_unpack_base3(const uint8_t *packed, size_t count, int8_t *q, hipStream_t stream)
{
    if (count == 0) return BITNET_HIP_OK;
    launch_kernel(unpack_base3_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, stream, packed, count, q);
    BITNET_HIP_CHECK_LAUNCH("unpack_base3_kernel");
    return BITNET_HIP_OK;
}

int launch_base3_to_2bit(const uint8_t *base3, size_t count, uint8_t *packed, hipStream_t stream)
{
    size_t nbytes = (count + 3) / 4;
    if (nbytes == 0) return BITNET_HIP_OK;
    launch_kernel(base3_to_2bit_kernel, dim3(blocks_for(nbytes, 256)), dim3(256), 0, stream, base3, count, packed, nbytes);
    BITNET_HIP_CHECK_LAUNCH("base3_to_2bit_kernel");
    return BITNET_HIP_OK;
}

int launch_quantize_weights(const float *w, size_t n, size_t k, int method, float threshold_factor,
                            double *row_sums, bool apart, uint8_t *packed, float *w_scale, int8_t *q_i8, hipStream_t stream)
{
    const size_t count = n * k;
    if (count != 0) {
        launch_kernel(absmean_rows_kernel, dim3(blocks_for(n, 4)), dim3(64, 4), 0, stream, w, n, k, row_sums);
        BITNET_HIP_CHECK_LAUNCH("absmean_rows_kernel");
    }
    const bool dense = aligned(w, 16) && aligned(packed, 4) && (!q_i8 || aligned(q_i8, 4));
    // No int8 codes, and a threshold that is not negative (what the sign of a difference can tell).
    if (apart && count != 0 && n <= CODES_MAX_ROWS && dense && !q_i8 && (method == BITNET_HIP_TERNARY_ABSMEAN_ROUNDCLIP || threshold_factor >= 0.0f)) {
        const unsigned blocks = (blocks_for(count, 15 * 1024) + 7) / 8 * 8;  // a chunk a wavefront, up to a workgroup a compute unit
        launch_kernel(absmean_codes_kernel, dim3(blocks < 256 ? blocks : 256), dim3(1024), 0, stream, w, n, k, method, threshold_factor,
                      const_cast<const double *>(row_sums), packed, w_scale);
        BITNET_HIP_CHECK_LAUNCH("absmean_codes_kernel");
        return BITNET_HIP_OK;
    }
    launch_kernel(absmean_final_kernel, dim3(1), dim3(1024), 0, stream, row_sums, n, k, w_scale);
    BITNET_HIP_CHECK_LAUNCH("absmean_final_kernel");
    if (count == 0) return BITNET_HIP_OK;
    // at most eight workgroups a compute unit: one round, and no more dispatches than that
    const unsigned blocks = blocks_for(count, 4096);
    launch_kernel(ternarize_pack_kernel, dim3(blocks < 2048 ? blocks : 2048), dim3(256), 0, stream, w, count,
                       method, threshold_factor, w_scale, packed, q_i8, dense);
    BITNET_HIP_CHECK_LAUNCH("ternarize_pack_kernel");
    return BITNET_HIP_OK;
}

size_t quantize_weights_reference_scratch_bytes(size_t n)
{
    return sizeof(double) * WQ_SCRATCH_SUMS * (n ? n : 1) + sizeof(float) * (n ? n : 1) + 256;
}

int launch_quantize_weights_reference(const float *w, size_t n, size_t k, int method, int normalize, float outlier_threshold,
                                      float custom_factor, void *scratch, uint8_t *packed, float *w_scale, int8_t *q_i8,
                                      float *stats, hipStream_t stream)
{
    // scratch: two WqStates (256 bytes reserved), then WQ_SCRATCH_SUMS * n doubles, then n floats
    WqState *states = static_cast<WqState *>(scratch);
    double *row_sums = reinterpret_cast<double *>(static_cast<uint8_t *>(scratch) + 256);
    float *row_max = reinterpret_cast<float *>(row_sums + WQ_SCRATCH_SUMS * (n ? n : 1));
    const int clip = outlier_threshold > 0.0f ? 1 : 0;
    const size_t count = n * k, nbytes = (count + 3) / 4;
    if (count == 0) {
        launch_kernel(wq_empty_kernel, dim3(1), dim3(1), 0, stream, clip, w_scale, stats);
        BITNET_HIP_CHECK_LAUNCH("wq_empty_kernel");
        return BITNET_HIP_OK;
    }
    const dim3 rgrid(blocks_for(n, 4)), rblock(64, 4);
    uint8_t *packed_rows = k % 4 == 0 ? packed : nullptr;  // rows of whole bytes: the last pass writes the codes
    // A call with the default configuration and the wait for it, with a launch for every reduction -> with those that the next pass finishes:
    // 256 x 256 92 -> 74 us, 1280 x 2112 95 -> 84, 2048 x 2048 94 -> 84, 2560 x 2560 105 -> 92, 4096 x 4096 149 -> 145; every workgroup
    // adds all row sums again, so beyond the line it is the other way round: 6912 x 2560 143 and 155, 14045 x 456 133 and 250.
    const bool fold = n <= WQ_FOLD_MAX_ROWS;
    const WqState *state = nullptr;  // of the passes so far
    WqPrevious prev = {-1, nullptr, nullptr, {method, outlier_threshold, custom_factor}};
    int at = 0;
    // FINISH: no pass follows that could finish it, or it has more accumulators than a pass finishes
#define BITNET_WQ_PASS(PASS, FINISH)                                                                                      \
    do {                                                                                                                  \
        double *sums = row_sums + (PASS == WQ_OPTIMAL ? 4 : 2 * at) * n;                                                  \
        prev.state = states + at;                                                                                         \
        if (fold) launch_kernel((wq_rows_kernel<PASS, true>), rgrid, rblock, 0, stream, w, n, k, state, normalize,   \
                                     clip, sums, row_max, packed_rows, q_i8, prev);                                       \
        else launch_kernel((wq_rows_kernel<PASS, false>), rgrid, rblock, 0, stream, w, n, k, state, normalize, clip, \
                                sums, row_max, packed_rows, q_i8, prev);                                                  \
        BITNET_HIP_CHECK_LAUNCH("wq_rows_kernel");                                                                        \
        if (fold) state = states + at;                                                                                    \
        prev.pass = PASS; prev.sums = sums;                                                                               \
        if (!fold || FINISH) {                                                                                            \
            launch_kernel((wq_final_kernel<PASS>), dim3(1), dim3(1024), 0, stream, sums, row_max, n, k, state,       \
                               states + at, prev.rule, clip, w_scale, stats);                                             \
            BITNET_HIP_CHECK_LAUNCH("wq_final_kernel");                                                                   \
            state = states + at;                                                                                          \
            prev.pass = -1;                                                                                               \
        }                                                                                                                 \
        at ^= 1;                                                                                                          \
    } while (0)
    if (normalize) {
        BITNET_WQ_PASS(WQ_SUM, false);
        BITNET_WQ_PASS(WQ_SQDIFF, false);
    }
    if (clip) BITNET_WQ_PASS(WQ_CLIP_STATS, false);
    BITNET_WQ_PASS(WQ_ABS_STATS, false);
    if (method == 3 && !(custom_factor > 0.0f)) BITNET_WQ_PASS(WQ_OPTIMAL, true);
    BITNET_WQ_PASS(WQ_SCALE, true);
#undef BITNET_WQ_PASS
    if (!packed_rows) {
        launch_kernel(wq_ternarize_pack_kernel, dim3(blocks_for(nbytes, 256)), dim3(256), 0, stream, w, count, state,
                           normalize, clip, packed, q_i8, nbytes);
        BITNET_HIP_CHECK_LAUNCH("wq_ternarize_pack_kernel");
    }
    return BITNET_HIP_OK;
}

int launch_retile(const uint8_t *packed, size_t n, size_t k, int layout, uint8_t *tiled, hipStream_t stream, uint8_t *canonical,
                  float w_scale, float *w_scale_out)
{
    if (tiled_bytes(n, k) == 0) return BITNET_HIP_OK;
    uint32_t *out = reinterpret_cast<uint32_t *>(tiled);
    const unsigned kt_count = (unsigned)k_tiles(k);
    if (layout == BITNET_HIP_LAYOUT_OUT_IN) {
        const bool dwords = k % 16 == 0 && aligned(packed, 4);
        uint32_t *back = canonical && k % 16 == 0 && aligned(canonical, 4) ? reinterpret_cast<uint32_t *>(canonical) : nullptr;
        launch_kernel(retile_kernel, rows_grid((kt_count + RETILE_KT - 1) / RETILE_KT, row_blocks(n)), dim3(256), 0, stream, packed, n, k, out, kt_count, dwords,
                           back, w_scale, w_scale_out);
        BITNET_HIP_CHECK_LAUNCH("retile_kernel");
        if (back || !canonical) return BITNET_HIP_OK;
    } else {
        launch_kernel(retile_in_out_kernel, rows_grid(blocks_for(row_blocks(n), 64), 16 * (size_t)kt_count), dim3(64), 0, stream,
                           packed, n, k, out, kt_count, n % 16 == 0 && aligned(packed, 4), w_scale, w_scale_out);
        BITNET_HIP_CHECK_LAUNCH("retile_in_out_kernel");
        if (!canonical) return BITNET_HIP_OK;
    }
    return launch_untile(tiled, n, k, canonical, stream);
}

int launch_untile(const uint8_t *tiled, size_t n, size_t k, uint8_t *packed, hipStream_t stream)
{
    size_t nbytes = (n * k + 3) / 4;
    if (nbytes == 0) return BITNET_HIP_OK;
    const uint32_t *src = reinterpret_cast<const uint32_t *>(tiled);
    if (k % 16 == 0 && aligned(packed, 4)) {
        launch_kernel(untile_rows_kernel, rows_grid(blocks_for(k / 16, 256), n), dim3(256), 0, stream, src, (unsigned)(k / 16), n,
                           reinterpret_cast<uint32_t *>(packed), (unsigned)k_tiles(k));
        BITNET_HIP_CHECK_LAUNCH("untile_rows_kernel");
        return BITNET_HIP_OK;
    }
    launch_kernel(untile_kernel, dim3(blocks_for(nbytes, 256)), dim3(256), 0, stream, src, n, k, packed, k_tiles(k), nbytes);
    BITNET_HIP_CHECK_LAUNCH("untile_kernel");
    return BITNET_HIP_OK;
}

}  // namespace bitnet
