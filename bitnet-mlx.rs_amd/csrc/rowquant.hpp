// Device-side pieces of the fused RMSNorm + per-token absmax int8 quantiser, shared by the stand-alone
// quantiser kernels (act_quant.hip) and by the decode GEMV, which quantises its input row itself
// (gemv_w2a8.hip).  Every caller produces the same bits for the same row.
//
// Arithmetic (each f32 step one IEEE operation):
//   ss      = sum_k x[k]*x[k]                      bitnet-inference/src/engine/inference_integration.rs:476
//   rms     = sqrt(ss / K + eps)                   :477
//   y[k]    = (x[k] / rms) * gamma[k]              :481
//   absmax  = max_k |y[k]|                         bitnet-inference/src/engine/ternary_operations.rs:143-145
//   a_scale = absmax > 0 ? 127 / absmax : 1        :147-151
//   q[k]    = clamp(round(y[k] * a_scale),-128,127) :158-161  (round = half away from zero)
//
// Order of the f32 sum of squares, the only order-dependent step (BITNET_HIP_SUM_BLOCK256):
//   the row is cut into chunks of 4 consecutive elements; chunk c belongs to virtual lane c mod 256; a lane
//   adds the squares of its chunks in ascending chunk order and, inside a chunk, ascending element order,
//   starting from +0; the 256 partials form 4 groups of 64 consecutive lanes, each combined by the butterfly
//   p[l] += p[l ^ off], off = 1,2,4,8,16,32; the four group sums are added as ((s0 + s1) + s2) + s3.
//   (After the step with offset `off` all lanes of an aligned group of 2*off lanes hold the same value, so a
//   step may fetch its operand from ANY lane of the partner group: the kernels use DPP quad permutes and row
//   mirrors for offsets 1..8 and the row / half swap instructions for 16 and 32.)
//   A 256-thread workgroup maps thread = virtual lane; a single wavefront keeps 4 partials per lane
//   (virtual lanes l, l+64, l+128, l+192).  Elements past K count as 0.
// BITNET_HIP_SUM_SEQUENTIAL is the reference's literal running sum over k ascending.
#pragma once
#include <type_traits>

#include "common.hpp"
#include "ieee.hpp"

namespace bitnet {

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also waits for every global load in flight,
// which would stall a kernel that requests its weight tiles ahead of the code that needs them.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Wavefronts per workgroup of gemv_fused16_kernel for a row of k columns: one per 256 columns, at least the four of
// the declared summation order, at most 16.  (The stand-alone quantiser with a workgroup per row gains nothing from
// the same rule: measured on the 8- to 16-token decoder stack.)
__host__ __device__ inline int row_workgroup_waves(int k)
{
    const int kt = (k + 255) >> 8;
    return kt > 16 ? 16 : (kt < 4 ? 4 : kt);
}

struct RowSource {
    const float *x;      // [m, ldx]
    const float *x2;     // second operand of RELU2_MUL
    const float *gamma;  // RMSNorm weight or nullptr
    size_t ldx;
    int k;
    int head_dim;
    int gqa_group;
    int sum_order;
    float eps;
};

// Lane exchanges of the butterfly.  CTRL is a DPP control word: 0xB1 = quad_perm[1,0,3,2] (l ^ 1),
// 0x4E = quad_perm[2,3,0,1] (l ^ 2), 0x141 = row_half_mirror (a lane of the other quad of the same 8),
// 0x140 = row_mirror (a lane of the other half of the same 16).
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
// Offsets 16 and 32 without a trip through LDS: gfx950's row and half swaps.  With both operands holding p,
// v_permlane16_swap leaves (rows 0,0,2,2 of p) in the first and (rows 1,1,3,3) in the second, v_permlane32_swap
// (lower half twice) and (upper half twice): every lane then holds its own value in one of them and its partner's
// in the other, and the combining operations here are commutative.  (Inline asm: the compiler's builtin for these
// instructions folds the two results into one.  The s_nop covers the wait states between a VALU write of the
// operands and the swap.)
template <typename T>
__device__ __forceinline__ void swap_rows16(T &a, T &b)
{
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
template <typename T>
__device__ __forceinline__ void swap_halves32(T &a, T &b)
{
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}

// 4-element sum over lanes l, l ^ 16, l ^ 32, l ^ 48 (the four column groups of a weight-tile row) in every lane.
__device__ __forceinline__ int sum_over_lane_groups(int v)
{
    int a = v, b = v;
    swap_rows16(a, b);
    a += b;
    b = a;
    swap_halves32(a, b);
    return a + b;
}

#define BITNET_WAVE_REDUCE(TYPE, NAME, COMBINE)                                                    \
    __device__ __forceinline__ TYPE NAME(TYPE p)                                                   \
    {                                                                                              \
        auto step = [](TYPE a, int other_bits) { TYPE b = __builtin_bit_cast(TYPE, other_bits); return COMBINE; }; \
        p = step(p, dpp_i32<0xB1>(__builtin_bit_cast(int, p)));                                    \
        p = step(p, dpp_i32<0x4E>(__builtin_bit_cast(int, p)));                                    \
        p = step(p, dpp_i32<0x141>(__builtin_bit_cast(int, p)));                                   \
        p = step(p, dpp_i32<0x140>(__builtin_bit_cast(int, p)));                                   \
        {                                                                                          \
            TYPE a = p, b = p;                                                                     \
            swap_rows16(a, b);                                                                     \
            p = COMBINE;                                                                           \
        }                                                                                          \
        {                                                                                          \
            TYPE a = p, b = p;                                                                     \
            swap_halves32(a, b);                                                                   \
            p = COMBINE;                                                                           \
        }                                                                                          \
        return p;                                                                                  \
    }
BITNET_WAVE_REDUCE(float, wave_sum_f32, f32_add(a, b))
BITNET_WAVE_REDUCE(float, wave_max_f32, fmaxf(a, b))
BITNET_WAVE_REDUCE(int, wave_sum_i32, a + b)
#undef BITNET_WAVE_REDUCE

__device__ __forceinline__ float relu2_mul(float gate, float up)
{
    float r = gate > 0.0f ? gate : 0.0f;
    return f32_mul(up, f32_mul(r, r));
}

// Element i of the (virtual) input row after the fused input transform.
template <int MODE>
__device__ __forceinline__ float load_elem(const RowSource &p, size_t row, int i)
{
    if constexpr (MODE == BITNET_HIP_INPUT_PLAIN) {
        return p.x[row * p.ldx + i];
    } else if constexpr (MODE == BITNET_HIP_INPUT_RELU2_MUL) {
        return relu2_mul(p.x[row * p.ldx + i], p.x2[row * p.ldx + i]);
    } else {
        int h = i / p.head_dim, d = i - h * p.head_dim;
        return p.x[row * p.ldx + (size_t)(h / p.gqa_group) * p.head_dim + d];
    }
}

// Elements i .. i + 3 of a row of k, zeros from k on, at any alignment of four bytes: one 16-byte load, in the row's last chunk that of its last
// four elements, shifted.  The quantiser of rows that are no multiple of four columns, as four loads -> as one, us: 8192 x 1023 13.1 -> 11.7 (the
// host), with a norm 20.3 -> 13.2; 4096 x 5121 26.1 -> 24.1, 43.7 -> 30.4; 2048 x 17001 77.6 -> 49.8, 164 -> 77.
__device__ __forceinline__ float4 load4_any(const float *row, int i, int k)
{
    typedef float v4 __attribute__((ext_vector_type(4), aligned(4)));
    if (k < 4) return make_float4(row[i], i + 1 < k ? row[i + 1] : 0.0f, i + 2 < k ? row[i + 2] : 0.0f, 0.0f);
    const int from = min(i, k - 4), shift = i - from;
    v4 e = *reinterpret_cast<const v4 *>(row + from);
    if (shift & 1) e = (v4){e[1], e[2], e[3], 0.0f};  // two selects: the compiler's code for a branch a shift lost the shift by three
    if (shift & 2) e = (v4){e[2], e[3], 0.0f, 0.0f};
    return make_float4(e[0], e[1], e[2], e[3]);
}

// Chunk c (elements 4c .. 4c+3).  VEC: 16-byte loads, all four elements inside the row.
template <int MODE, bool VEC>
__device__ __forceinline__ float4 load_chunk(const RowSource &p, size_t row, int c)
{
    if constexpr (VEC) {
        if constexpr (MODE == BITNET_HIP_INPUT_PLAIN) {
            return *reinterpret_cast<const float4 *>(p.x + row * p.ldx + 4 * (size_t)c);
        } else if constexpr (MODE == BITNET_HIP_INPUT_RELU2_MUL) {
            float4 g = *reinterpret_cast<const float4 *>(p.x + row * p.ldx + 4 * (size_t)c);
            float4 u = *reinterpret_cast<const float4 *>(p.x2 + row * p.ldx + 4 * (size_t)c);
            return make_float4(relu2_mul(g.x, u.x), relu2_mul(g.y, u.y), relu2_mul(g.z, u.z),
                               relu2_mul(g.w, u.w));
        } else {
            int i = 4 * c;
            int h = i / p.head_dim, d = i - h * p.head_dim;
            return *reinterpret_cast<const float4 *>(p.x + row * p.ldx +
                                                     (size_t)(h / p.gqa_group) * p.head_dim + d);
        }
    } else if constexpr (MODE == BITNET_HIP_INPUT_PLAIN) {
        return load4_any(p.x + row * p.ldx, 4 * c, p.k);
    } else if constexpr (MODE == BITNET_HIP_INPUT_RELU2_MUL) {
        const float4 g = load4_any(p.x + row * p.ldx, 4 * c, p.k), u = load4_any(p.x2 + row * p.ldx, 4 * c, p.k);
        return make_float4(relu2_mul(g.x, u.x), relu2_mul(g.y, u.y), relu2_mul(g.z, u.z), relu2_mul(g.w, u.w));
    } else {
        float4 v;
        int i = 4 * c;
        v.x = i + 0 < p.k ? load_elem<MODE>(p, row, i + 0) : 0.0f;
        v.y = i + 1 < p.k ? load_elem<MODE>(p, row, i + 1) : 0.0f;
        v.z = i + 2 < p.k ? load_elem<MODE>(p, row, i + 2) : 0.0f;
        v.w = i + 3 < p.k ? load_elem<MODE>(p, row, i + 3) : 0.0f;
        return v;
    }
}

__device__ __forceinline__ float4 load_gamma_chunk(const RowSource &p, int c, bool vec)
{
    if (vec) return *reinterpret_cast<const float4 *>(p.gamma + 4 * (size_t)c);
    return load4_any(p.gamma, 4 * c, p.k);
}

__device__ __forceinline__ float sum_squares4(float part, const float4 &e)
{
    part = f32_add(part, f32_mul(e.x, e.x));
    part = f32_add(part, f32_mul(e.y, e.y));
    part = f32_add(part, f32_mul(e.z, e.z));
    part = f32_add(part, f32_mul(e.w, e.w));
    return part;
}

// The reference's literal order: every lane runs the same chain over the whole row.
template <int MODE>
__device__ __forceinline__ float sum_squares_sequential(const RowSource &p, size_t row)
{
    float ss = 0.0f;
    for (int i = 0; i < p.k; ++i) {
        float e = load_elem<MODE>(p, row, i);
        ss = f32_add(ss, f32_mul(e, e));
    }
    return ss;
}

// The same literal order with the squares of the row staged in LDS: sq[i] = x[i] * x[i] in element order, written by
// the workgroup (store_squares4) and made visible by a barrier before the call.  Every lane runs the same chain of k
// additions; its reads are broadcasts (one address for all lanes), 16 bytes at a time.  What is left is the latency of
// a dependent v_add_f32, about 8.5 cycles an element (measured; reading further ahead of the additions gains nothing).
__host__ __device__ inline size_t squares_lds_bytes(int k) { return (size_t)((k + 3) >> 2) * 16; }
__device__ __forceinline__ void store_squares4(float *sq, int c, const float4 &e)  // chunk c: elements 4c .. 4c + 3
{
    *reinterpret_cast<float4 *>(sq + 4 * (size_t)c) =
        make_float4(f32_mul(e.x, e.x), f32_mul(e.y, e.y), f32_mul(e.z, e.z), f32_mul(e.w, e.w));
}
__device__ __forceinline__ float sum_sequential_lds(const float *sq, int k)
{
    float ss = 0.0f;
    const int full = k >> 2;
    const float4 *sq4 = reinterpret_cast<const float4 *>(sq);
#pragma unroll 8
    for (int c = 0; c < full; ++c) {
        const float4 s = sq4[c];
        ss = f32_add(f32_add(f32_add(f32_add(ss, s.x), s.y), s.z), s.w);
    }
    for (int i = full * 4; i < k; ++i) ss = f32_add(ss, sq[i]);
    return ss;
}

__device__ __forceinline__ float rms_from_ss(float ss, int k, float eps)
{
    return sqrt_uniform(f32_add(div_uniform(ss, make_divisor((float)k)), eps));
}

// Whether the largest and the smallest magnitude of a chunk settle that the short division takes all four elements (a chunk
// with a zero in it does not pass; a NaN stays one whichever division runs).
__device__ __forceinline__ bool chunk_ok(const float4 &e)
{
    const float hi = fmaxf(fmaxf(fabsf(e.x), fabsf(e.y)), fmaxf(fabsf(e.z), fabsf(e.w)));
    const float lo = fminf(fminf(fabsf(e.x), fabsf(e.y)), fminf(fabsf(e.z), fabsf(e.w)));
    return lo >= 0x1p-63f && hi < 0x1p63f;
}

// (x / rms) * g for the four elements of a chunk.  The divisor is the same for the whole row, so the division
// uses div_by_invariant (ieee.hpp), which returns the same bits as x / rms.
__device__ __forceinline__ float4 normalize4(const float4 &e, const Divisor &r, const float4 &g)
{
    // the short division when the divisor and, in every lane of the wavefront, all four dividends allow it
    bool lanes_ok = __builtin_amdgcn_ballot_w64(!(r.fast && chunk_ok(e))) == 0;
    if (!lanes_ok)
        lanes_ok = __builtin_amdgcn_ballot_w64(!(r.fast && dividend_ok(e.x) && dividend_ok(e.y) && dividend_ok(e.z) && dividend_ok(e.w))) == 0;
    float4 q;
    if (lanes_ok) {
        q = make_float4(div_by_invariant_unchecked(e.x, r.d, r.recip), div_by_invariant_unchecked(e.y, r.d, r.recip),
                        div_by_invariant_unchecked(e.z, r.d, r.recip), div_by_invariant_unchecked(e.w, r.d, r.recip));
    } else {
        q = make_float4(f32_div(e.x, r.d), f32_div(e.y, r.d), f32_div(e.z, r.d), f32_div(e.w, r.d));
    }
    return make_float4(f32_mul(q.x, g.x), f32_mul(q.y, g.y), f32_mul(q.z, g.z), f32_mul(q.w, g.w));
}

__device__ __forceinline__ float absmax4(float amax, const float4 &e)
{
    return fmaxf(fmaxf(fmaxf(amax, fabsf(e.x)), fabsf(e.y)), fmaxf(fabsf(e.z), fabsf(e.w)));
}

__device__ __forceinline__ float scale_from_absmax(float amax)
{
    return amax > 0.0f ? div_uniform(127.0f, make_divisor(amax)) : 1.0f;
}

// Round half away from zero, then a saturating conversion (NaN converts to 0, as Rust's `as i8` does).  The rounding is one
// addition of +-(1/2 - 2^-25), the largest float below 1/2, and the truncating conversion: with 1/2 itself the sum for
// |t| = 1/2 - 2^-25 would round up to 1; with its predecessor that sum is exact, |t| = 1/2 still rounds up to 1, and every
// other sum is exact or rounds within the gap between two integers (past 2^23, where it may not, the caller's clamp
// decides).  Checked against roundf, cast and clamp over all 2^32 bit patterns of t.  v_cvt_i32_f32 truncates, saturates
// and turns NaN into 0.
__device__ __forceinline__ int round_away(float t)
{
    const float s = f32_add(t, __builtin_copysignf(0x1.fffffep-2f, t));
    int q;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(s));
    return q;
}
__device__ __forceinline__ int quant1(float y, float scale) { return min(max(round_away(f32_mul(y, scale)), -128), 127); }

// Four quantised values of a chunk packed little-endian (byte j = element j).  v_perm_b32: selector 0 and 4 take the low
// byte of the second and the first operand, 12 is a zero byte.
__device__ __forceinline__ uint32_t pack4(int q0, int q1, int q2, int q3)
{
    return __builtin_amdgcn_perm((uint32_t)q1, (uint32_t)q0, 0x0c0c0400u) | __builtin_amdgcn_perm((uint32_t)q3, (uint32_t)q2, 0x04000c0cu);
}
__device__ __forceinline__ uint32_t quant4_clamped(const float4 &e, float scale)
{
    return pack4(quant1(e.x, scale), quant1(e.y, scale), quant1(e.z, scale), quant1(e.w, scale));
}
// While scale, 127 over the row's largest magnitude, is finite no product exceeds 127 (1 + 2^-22), whose rounding is 127:
// the clamp to [-128, 127] has nothing to do.
__device__ __forceinline__ uint32_t quant4_bounded(const float4 &e, float scale)
{
    return pack4(round_away(f32_mul(e.x, scale)), round_away(f32_mul(e.y, scale)), round_away(f32_mul(e.z, scale)), round_away(f32_mul(e.w, scale)));
}
// The same with the choice made on the scale (the row's: the same in every lane); *sum += the four values.
__device__ __forceinline__ uint32_t quant4_packed(const float4 &e, float scale, int *sum)
{
    const uint32_t packed = __builtin_expect(__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, scale)) < 0x7f800000, 1)
                                ? quant4_bounded(e, scale)
                                : quant4_clamped(e, scale);
    *sum = __builtin_amdgcn_sdot4((int)packed, 0x01010101, *sum, false);
    return packed;
}

// ---- a row held by a workgroup of up to 16 wavefronts -----------------------------------------------------------------
//
// The latency-bound form (one decode token, a decode batch): a thread has NCHB chunks of four elements, all loads are issued at
// once, every element-wise step runs once, in parallel, and what is left is the chain of dependent steps.

typedef unsigned v16u __attribute__((ext_vector_type(16)));
template <typename T>
using global_ptr = __attribute__((address_space(1))) T *;
template <typename T>
__device__ __forceinline__ global_ptr<T> pointer_at(const v16u &block, int dword)
{
    return (global_ptr<T>)(uintptr_t)(((uint64_t)block[dword + 1] << 32) | block[dword]);
}

// Combines a value over the wavefront in the order of the butterflies of rowquant.hpp; the result is valid in lane 63.  After the
// row mirrors all lanes of a row hold its value; row_bcast:15 (0x142) adds row 0 to row 1 and row 2 to row 3, row_bcast:31
// (0x143) the first half to the second.
__device__ __forceinline__ float wave_sum_last(float p)
{
    auto other = [](float v, auto ctrl) { return __builtin_bit_cast(float, dpp_i32<decltype(ctrl)::value>(__builtin_bit_cast(int, v))); };
    p = f32_add(p, other(p, std::integral_constant<int, 0xB1>{}));
    p = f32_add(p, other(p, std::integral_constant<int, 0x4E>{}));
    p = f32_add(p, other(p, std::integral_constant<int, 0x141>{}));
    p = f32_add(p, other(p, std::integral_constant<int, 0x140>{}));
    p = f32_add(p, other(p, std::integral_constant<int, 0x142>{}));
    return f32_add(p, other(p, std::integral_constant<int, 0x143>{}));
}
// The largest of 64 non-negative numbers (no NaN): their bits compare as integers.
__device__ __forceinline__ float wave_max_last(float p)
{
    unsigned v = __builtin_bit_cast(unsigned, p);
    auto step = [&](auto ctrl) {
        const unsigned o = (unsigned)dpp_i32<decltype(ctrl)::value>((int)v);
        v = v > o ? v : o;
    };
    step(std::integral_constant<int, 0xB1>{});
    step(std::integral_constant<int, 0x4E>{});
    step(std::integral_constant<int, 0x141>{});
    step(std::integral_constant<int, 0x140>{});
    step(std::integral_constant<int, 0x142>{});
    step(std::integral_constant<int, 0x143>{});
    return __builtin_bit_cast(float, v);
}

// n / d for n < 2^16, d < 2^16 by the host's ceil(2^32 / d) (d = 1: the multiplier does not fit and is given as 0)
__device__ __forceinline__ int div_by_magic(int n, unsigned magic) { return magic ? (int)__umulhi((unsigned)n, magic) : n; }

// One chunk of the (transformed) input row.  GQA: query head h reads value head h / group; hx2 carries the two multipliers
// for the chunks of a head (head_dim / 4) and of a group.
template <int MODE>
__device__ __forceinline__ float4 row16_chunk(const float *row, const float *row2, uint64_t magics, int head_chunks, int c)
{
    if constexpr (MODE == BITNET_HIP_INPUT_PLAIN) {
        return reinterpret_cast<const float4 *>(row)[c];
    } else if constexpr (MODE == BITNET_HIP_INPUT_RELU2_MUL) {
        const float4 g = reinterpret_cast<const float4 *>(row)[c], u = reinterpret_cast<const float4 *>(row2)[c];
        return make_float4(relu2_mul(g.x, u.x), relu2_mul(g.y, u.y), relu2_mul(g.z, u.z), relu2_mul(g.w, u.w));
    } else {
        const int h = div_by_magic(c, (unsigned)magics), g = div_by_magic(c, (unsigned)(magics >> 32));
        return reinterpret_cast<const float4 *>(row)[(g - h) * head_chunks + c];
    }
}

// The multipliers for the chunks of a head and of a GQA group, packed as row16_chunk takes them; false: out of their range.
inline bool row16_magics(int head_dim, int gqa_group, uint64_t *magics)
{
    auto magic = [](uint64_t d) { return d == 1 ? (uint64_t)0 : (((uint64_t)1 << 32) + d - 1) / d; };
    const uint64_t head = (uint64_t)head_dim / 4, span = head * (uint64_t)gqa_group;
    if (head == 0 || span > 0xffff) return false;
    *magics = magic(head) | (magic(span) << 32);
    return true;
}

// NCHB chunks per thread: chunk[i] = 64 (wave + nw i) + in_tile, in_tile a permutation of 0..63 over the lanes.
template <bool NORM, int NCHB>
struct Row16 {
    // The sum of squares keeps the declared order: chunk c belongs to virtual lane c % 256, so threads 0..255 (one per virtual
    // lane) also fetch the chunks of their lane and run its chain.
    static constexpr int NSS = NORM ? 4 * NCHB : 1;  // chunks per virtual lane
    float4 v[NCHB], gm[NORM ? NCHB : 1], vs[NSS];
    int chunk[NCHB];

    // Unconditional loads (clamped indices, values discarded).  ALL: also of the chunks that no virtual lane of a row this short has.  A branch for
    // each costs most kernels more than the loads (the 30-block stack at 4 / 16 / 42 tokens 668 / 808 / 989 us, 666 / 803 / 986 without; 8 x 1024 -> 1024
    // with a norm 2.94 and 2.88), but a fused GEMV whose workgroups have one row block, which is over sooner, less (1 x 1024 -> 1024 2.61 and 2.64,
    // 1 x 2048 -> 4096 2.96 and 3.01).
    template <int MODE, bool ALL = true>
    __device__ __forceinline__ void load(const float *row, const float *row2, uint64_t magics, int head_chunks, const float *gamma, int chunks,
                                         int nw, int wave, int tid, int in_tile)
    {
#pragma unroll
        for (int i = 0; i < NCHB; ++i) {
            chunk[i] = 64 * (wave + nw * i) + in_tile;
            v[i] = row16_chunk<MODE>(row, row2, magics, head_chunks, min(chunk[i], chunks - 1));
        }
        if constexpr (NORM) {
            if (wave < 4) {
#pragma unroll
                for (int i = 0; i < NSS; ++i)
                    if (ALL || 256 * i < chunks) vs[i] = row16_chunk<MODE>(row, row2, magics, head_chunks, min(tid + 256 * i, chunks - 1));
            }
#pragma unroll
            for (int i = 0; i < NCHB; ++i) gm[i] = reinterpret_cast<const float4 *>(gamma)[min(chunk[i], chunks - 1)];
        }
    }

    // v becomes the normalised row (+0 past its end), packed its int8 values; returns the scale.  k_recip: recip_of_ok_divisor(k_f).
    // red_f: two lines of shared memory; the caller has cleared red_f[1][nw ..] (absent wavefronts).
    __device__ __forceinline__ float quantise(int chunks, float k_f, float k_recip, float eps, int wave, int tid, float (&red_f)[2][16],
                                              uint32_t (&packed)[NCHB])
    {
#pragma unroll
        for (int i = 0; i < NCHB; ++i) {
            const bool inside = chunk[i] < chunks;
            v[i].x = inside ? v[i].x : 0.0f; v[i].y = inside ? v[i].y : 0.0f; v[i].z = inside ? v[i].z : 0.0f; v[i].w = inside ? v[i].w : 0.0f;
        }

        if constexpr (NORM) {
            if (wave < 4) {
                float part = 0.0f;
#pragma unroll
                for (int i = 0; i < NSS; ++i) {
                    const float next = sum_squares4(part, vs[i]);
                    part = tid + 256 * i < chunks ? next : part;
                }
                part = wave_sum_last(part);
                if ((tid & 63) == 63) red_f[0][wave] = part;
            }
            lds_barrier();
            const float4 s4 = *reinterpret_cast<const float4 *>(red_f[0]);
            const float ss = f32_add(f32_add(f32_add(s4.x, s4.y), s4.z), s4.w);
            // The short forms of the two divisions and the root, computed without looking; whether every operand was in their
            // range is one question at the end, and where it was not the plain forms run.
            const float mean = f32_add(div_by_invariant_unchecked<false>(ss, k_f, k_recip), eps);
            const float rms = sqrt_in_range(mean);
            const float recip = recip_of_ok_divisor(rms);
            bool ok = ss >= 0x1p-63f && ss < 0x1p63f && mean >= 0x1p-61f && mean < 0x1p61f && significand_ok(rms);
            float4 y[NCHB];
#pragma unroll
            for (int i = 0; i < NCHB; ++i) {
                ok = ok && (chunk_ok(v[i]) || chunk[i] >= chunks);
                y[i] = make_float4(f32_mul(div_by_invariant_unchecked<false>(v[i].x, rms, recip), gm[i].x),
                                   f32_mul(div_by_invariant_unchecked<false>(v[i].y, rms, recip), gm[i].y),
                                   f32_mul(div_by_invariant_unchecked<false>(v[i].z, rms, recip), gm[i].z),
                                   f32_mul(div_by_invariant_unchecked<false>(v[i].w, rms, recip), gm[i].w));
            }
            if (__builtin_expect(!ok, 0)) {
                const float plain_rms = f32_sqrt(f32_add(f32_div(ss, k_f), eps));
#pragma unroll
                for (int i = 0; i < NCHB; ++i)
                    y[i] = make_float4(f32_mul(f32_div(v[i].x, plain_rms), gm[i].x), f32_mul(f32_div(v[i].y, plain_rms), gm[i].y),
                                       f32_mul(f32_div(v[i].z, plain_rms), gm[i].z), f32_mul(f32_div(v[i].w, plain_rms), gm[i].w));
            }
#pragma unroll
            for (int i = 0; i < NCHB; ++i) {
                const bool inside = chunk[i] < chunks;  // a zero of the padding may have met a NaN or an infinity
                v[i].x = inside ? y[i].x : 0.0f; v[i].y = inside ? y[i].y : 0.0f; v[i].z = inside ? y[i].z : 0.0f; v[i].w = inside ? y[i].w : 0.0f;
            }
        }
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < NCHB; ++i) amax = absmax4(amax, v[i]);
        amax = wave_max_last(amax);
        if ((tid & 63) == 63) red_f[1][wave] = amax;
        lds_barrier();
        {
            const float4 *m4 = reinterpret_cast<const float4 *>(red_f[1]);
            const float4 m0 = m4[0], m1 = m4[1], m2 = m4[2], m3 = m4[3];
            // non-negative numbers: their bits compare as integers
            auto hi = [](float x, float y) { return __builtin_bit_cast(float, max(__builtin_bit_cast(int, x), __builtin_bit_cast(int, y))); };
            amax = hi(hi(hi(hi(m0.x, m0.y), hi(m0.z, m0.w)), hi(hi(m1.x, m1.y), hi(m1.z, m1.w))),
                      hi(hi(hi(m2.x, m2.y), hi(m2.z, m2.w)), hi(hi(m3.x, m3.y), hi(m3.z, m3.w))));
        }
        // a_scale = 127 / absmax: again the short form first
        float scale = div_by_invariant_unchecked<false>(127.0f, amax, recip_of_ok_divisor(amax));
        const bool scale_ok = amax >= 0x1p-50f && amax < 0x1p60f && significand_ok(amax);
#pragma unroll
        for (int i = 0; i < NCHB; ++i) packed[i] = quant4_bounded(v[i], scale);
        if (__builtin_expect(!scale_ok, 0)) {
            scale = amax > 0.0f ? f32_div(127.0f, amax) : 1.0f;
#pragma unroll
            for (int i = 0; i < NCHB; ++i) packed[i] = quant4_clamped(v[i], scale);
        }

        return scale;
    }
};

}  // namespace bitnet
