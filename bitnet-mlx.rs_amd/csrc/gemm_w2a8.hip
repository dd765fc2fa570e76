// Prefill GEMM: int8 activations [m, k] x 2-bit ternary weights [n, k] -> int32 [m, n] on the int8 MFMA
// units of gfx950 (v_mfma_i32_16x16x64_i8), with the fp32 scale epilogue fused into the store.
//
//   acc[t, n] = sum_k a[t, k] * w[n, k]      bitnet-quant/src/simd/matrix.rs:256-282 (ternary_gemm_scalar),
//                                            front door bitnet-quant/src/bitlinear/forward.rs:179-214
//   out[t, n] = (float(acc) * w_scale) / a_scale[t] (+ bias[n]) (+ residual[t, n])
//
// Operand mapping of one MFMA (64 lanes): the A operand of lane l is 16 consecutive int8 activations of
// token row l mod 16, k block l / 16; the B operand is 16 weights of output row l mod 16, same k block;
// result register r of lane l is C[4*(l/16) + r][l mod 16].
//
// Weights are never expanded in memory.  A wavefront loads slot l of a 1 KiB weight tile (16 bytes per
// lane, one coalesced burst per 16 rows x 256 columns); dword t of that slot becomes, after four
// shift-and-mask operations, the B operand of the t-th k-step of the tile.  The operand holds the stored
// codes c = w + 1 in {0,1,2}; the epilogue subtracts sum_k a[t, k] per token row (accumulated on the fly
// while the activation tile passes through registers on its way to LDS).
//
// Three kernels share this scheme.
//
// gemm_dma_kernel (k a multiple of 256, 16-byte aligned activations, row sums supplied by the activation
// quantiser): activations AND weight tiles travel global -> LDS with LDS-direct loads
// (global_load_lds_dwordx4), never through registers.  D LDS stages of 128 columns are kept in flight;
// the wait counts are placed by hand (s_waitcnt vmcnt(N)) so that D - 1 stages of loads stay outstanding
// while one is computed (D = 2, a plain double buffer, which leaves LDS and registers for two workgroups of the largest
// tiles and three or four of the others per compute unit; D = 4 for the narrow tiles of short rows).  An
// LDS-direct load writes lane l's 16 bytes at base + 16*l, so the XOR swizzle that keeps the fragment reads free of bank conflicts is applied to the global address each lane fetches.
// The MFMA takes the weight fragment as its first operand, so a lane ends up with four consecutive output
// columns of one token row and the epilogue stores 16 bytes per lane.  The epilogue's per-row operands (a_sum,
// a_scale) arrive by LDS-direct loads in the stage buffer that is free during the last stage; the usual case
// (f32 output only, scales within the short division's range) is straight-line code
// (store_fragments_fast), everything else goes through store_fragments_general: same bits.
//
// gemm_ld8_kernel: the same data path with eight multiplying and two loading wavefronts per workgroup, for launches
// that one round of workgroups holds (see its own comment).
//
// gemm_tiled_kernel (any shape, computes the row sums itself): activations pass through registers.
// Activations are staged through LDS one weight tile (256 columns) at a time, double buffered: the global
// loads of stage s+1 are issued before the 4 k-steps of stage s are computed and written to LDS after them,
// one barrier per stage.  Rows are padded to 272 bytes so that the 16-byte fragment reads of 8 consecutive
// lanes fall in distinct banks.
#include <type_traits>

#include "kernels.hpp"
#include "ldsdma.hpp"

namespace bitnet {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(4)));  // 16-byte accesses need four-byte alignment only
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(4)));

struct GemmProjDev {  // one projection of a launch of the LDS-direct kernels
    const uint8_t *w;
    const float *w_scale;
    const float *bias;
    const float *residual;
    float *out;
    int32_t *acc;
    int n;
    int tn_end;  // column tiles of projections 0..this one, cumulative
};

struct GemmParams {
    GemmProjDev proj[GEMM_MAX_PROJ];  // LDS-direct kernels: projections sharing the activation matrix
    int nproj;
    // single-projection view (the register-staged kernel)
    const uint8_t *w;
    const int8_t *a;
    int32_t *acc;
    const float *w_scale;
    const float *a_scale;
    const float *bias;
    const float *residual;
    const int32_t *a_sum;  // sum_k a[t, k] per token row (required by gemm_dma_kernel)
    float *out;
    int m, n, k;
    int kt_count;   // 256-column weight tiles per row block
    int tiles_m, tiles_n;
    int group_rows; // gemm_dma_kernel: row tiles that consecutive tiles go down before the next column (tile_position), 1 or more
    int rotate;     // gemm_dma_kernel: every workgroup of the launch is resident at once (see there)
};

constexpr int STAGE_K = 256;              // columns per pipeline stage = one weight tile
constexpr int LDS_PITCH = STAGE_K + 16;   // bytes per activation row in LDS

// BM x BN output tile per workgroup of 256 threads (2 x 2 wavefronts).
template <int BM, int BN>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(GemmParams p)
{
    constexpr int WTM = BM / 2, WTN = BN / 2;       // wavefront tile
    constexpr int FM = WTM / 16, FN = WTN / 16;     // MFMA tiles per wavefront
    constexpr int A_LOADS = BM / 16;                // 16-byte chunks each thread moves per stage
    static_assert(WTM % 16 == 0 && WTN % 16 == 0 && A_LOADS >= 1, "tile shape");

    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[];
    uint8_t *lds_a0 = lds_raw, *lds_a1 = lds_raw + BM * LDS_PITCH;
    int *lds_rowsum = reinterpret_cast<int *>(lds_raw + 2 * BM * LDS_PITCH);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 15, lg = lane >> 4;

    // Workgroup -> output tile.  Consecutive workgroup ids land on different XCDs (8 of them, each with
    // its own L2), so ids are regrouped: all workgroups of one XCD walk one band of M tiles, N fastest,
    // and share its activation rows in that XCD's L2.
    int tile_id;
    {
        const int total = p.tiles_m * p.tiles_n;
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        const int per_xcd = (total + 7) >> 3;
        tile_id = xcd * per_xcd + idx;
        if (tile_id >= total) return;  // uniform per workgroup
    }
    const int tm = tile_id / p.tiles_n, tn = tile_id % p.tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;

    // ---- activation tile movement: chunk c = tid + 256*i -> row c / 16, 16-byte column chunk c % 16 ----
    const bool a_vec = (p.k % 16 == 0) && ((reinterpret_cast<uintptr_t>(p.a) & 15) == 0);
    const int a_row = tid >> 4, a_chunk = tid & 15;
    int rowsum[A_LOADS];
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) rowsum[i] = 0;

    auto load_a = [&](int kt, uint4 (&regs)[A_LOADS]) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            const int row = m0 + a_row + 16 * i, col = kt * STAGE_K + a_chunk * 16;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (row < p.m && col < p.k) {
                const int8_t *src = p.a + (size_t)row * p.k + col;
                if (a_vec) {
                    v = *reinterpret_cast<const uint4 *>(src);
                } else {
                    uint32_t d[4] = {0, 0, 0, 0};
                    for (int j = 0; j < 16; ++j)
                        if (col + j < p.k) d[j >> 2] |= (uint32_t)(uint8_t)src[j] << (8 * (j & 3));
                    v = make_uint4(d[0], d[1], d[2], d[3]);
                }
            }
            regs[i] = v;
        }
    };
    auto store_a = [&](uint8_t *buf, const uint4 (&regs)[A_LOADS]) {
#pragma unroll
        for (int i = 0; i < A_LOADS; ++i) {
            *reinterpret_cast<uint4 *>(&buf[(a_row + 16 * i) * LDS_PITCH + a_chunk * 16]) = regs[i];
            int s = rowsum[i];
            s = __builtin_amdgcn_sdot4((int)regs[i].x, 0x01010101, s, false);
            s = __builtin_amdgcn_sdot4((int)regs[i].y, 0x01010101, s, false);
            s = __builtin_amdgcn_sdot4((int)regs[i].z, 0x01010101, s, false);
            s = __builtin_amdgcn_sdot4((int)regs[i].w, 0x01010101, s, false);
            rowsum[i] = s;
        }
    };

    // ---- weight tiles: one uint4 per lane per 16-row block per 256 columns ----
    const int rb0 = (n0 + wn * WTN) / 16;
    const int rb_count = (p.n + 15) / 16;
    const uint4 *wbase = reinterpret_cast<const uint4 *>(p.w) + lane;
    auto load_b = [&](int kt, uint4 (&regs)[FN]) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int rb = rb0 + j;
            regs[j] = rb < rb_count ? wbase[((size_t)rb * p.kt_count + kt) * 64]
                                    : make_uint4(0x55555555u, 0x55555555u, 0x55555555u, 0x55555555u);
        }
    };

    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = (v4i){0, 0, 0, 0};

    uint4 a_regs[A_LOADS];
    uint4 b_cur[FN], b_next[FN];
    load_a(0, a_regs);
    load_b(0, b_cur);
    store_a(lds_a0, a_regs);
    __syncthreads();

    for (int kt = 0; kt < p.kt_count; ++kt) {
        uint8_t *cur = (kt & 1) ? lds_a1 : lds_a0;
        uint8_t *nxt = (kt & 1) ? lds_a0 : lds_a1;
        const bool more = kt + 1 < p.kt_count;
        if (more) {
            load_a(kt + 1, a_regs);
            load_b(kt + 1, b_next);
        }
        const uint8_t *arow = cur + (wm * WTM + lr) * LDS_PITCH + lg * 16;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v4i afrag[FM];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                afrag[i] = *reinterpret_cast<const v4i *>(arow + i * 16 * LDS_PITCH + t * 64);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const uint32_t wd = t == 0 ? b_cur[j].x : (t == 1 ? b_cur[j].y : (t == 2 ? b_cur[j].z : b_cur[j].w));
                v4i bfrag;
                bfrag[0] = (int)(wd & 0x03030303u);
                bfrag[1] = (int)((wd >> 2) & 0x03030303u);
                bfrag[2] = (int)((wd >> 4) & 0x03030303u);
                bfrag[3] = (int)((wd >> 6) & 0x03030303u);
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(afrag[i], bfrag, acc[i][j], 0, 0, 0);
            }
        }
        if (more) {
            store_a(nxt, a_regs);
#pragma unroll
            for (int j = 0; j < FN; ++j) b_cur[j] = b_next[j];
        }
        __syncthreads();
    }

    // ---- row sums of the activations (for the +1 weight code): 16 adjacent threads share a row ----
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i) {
        int s = rowsum[i];
        s += __shfl_xor(s, 1, 64);
        s += __shfl_xor(s, 2, 64);
        s += __shfl_xor(s, 4, 64);
        s += __shfl_xor(s, 8, 64);
        if (a_chunk == 0) lds_rowsum[a_row + 16 * i] = s;
    }
    __syncthreads();

    // ---- epilogue ----
    const float ws = p.out ? *p.w_scale : 0.0f;
    const unsigned ws_expo = (__builtin_bit_cast(unsigned, ws) >> 23) & 0xffu;
    const bool ws_fast = ws > 0.0f && ws_expo > 64u && ws_expo < 160u;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int lrow = wm * WTM + i * 16 + lg * 4 + r;
            const int row = m0 + lrow;
            if (row >= p.m) continue;
            const int rs = lds_rowsum[lrow];
            const float as = p.out ? p.a_scale[row] : 1.0f;
            const float as_recip = f32_div(1.0f, as);
            // the short division needs a well-behaved divisor (per row) and dividends in range: float(total) * ws
            // is zero or has ws's exponent plus at most 24, so one check on ws covers them.  The choice is made
            // per wavefront so that the usual case runs no plain division at all.
            const bool row_fast = ws_fast && invariant_divisor_ok(as);
            const bool wave_fast = __builtin_amdgcn_ballot_w64(!row_fast) == 0;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const int col = n0 + wn * WTN + j * 16 + lr;
                if (col >= p.n) continue;
                const int total = acc[i][j][r] - rs;
                const size_t o = (size_t)row * p.n + col;
                if (p.acc) p.acc[o] = total;
                if (p.out) {
                    const float scaled = f32_mul((float)total, ws);
                    float v = wave_fast ? div_by_invariant_unchecked(scaled, as, as_recip) : f32_div(scaled, as);
                    if (p.bias) v = f32_add(v, p.bias[col]);
                    if (p.residual) v = f32_add(v, p.residual[o]);
                    p.out[o] = v;
                }
            }
        }
    }
}

// ---- LDS-direct pipeline -------------------------------------------------------------------------------

// Per-row epilogue operands of a BM-row tile, fetched into LDS by LDS-direct loads (no registers are held across
// the k loop): a_sum[BM] as int32, then a_scale[BM].  Wavefront w < BM/64 fetches rows 64*w .. of a_sum, the
// next BM/64 wavefronts the same rows of a_scale (skipped when there is no f32 output and hence no a_scale).
// Rows past m re-read row m-1.  The reader waits for vmcnt(0) and a workgroup barrier first.
template <int BM>
constexpr int rowp_bytes() { return BM * 8; }
template <int BM>
__device__ __forceinline__ void fetch_row_operands(const GemmParams &p, int m0, int wave, int lane, uint32_t lds_rowp)
{
    constexpr int CH = BM / 64;
    static_assert(BM % 64 == 0, "row operand chunks");
    if (wave < 2 * CH) {
        const int chunk = wave < CH ? wave : wave - CH;
        int grow = m0 + chunk * 64 + lane;
        if (grow >= p.m) grow = p.m - 1;
        if (wave < CH) dma4(p.a_sum, (uint32_t)grow * 4u, lds_rowp + chunk * 256);
        else if (p.a_scale) dma4(p.a_scale, (uint32_t)grow * 4u, lds_rowp + BM * 4 + chunk * 256);
    }
}

// The epilogue of one wavefront's fragments on the usual path: f32 output only, w_scale and every a_scale of the tile suited to
// the short division (the caller checks).  Straight-line code: per output element a subtraction,
// a conversion, two multiplications, two FMAs and one and a half moves; 16-byte stores, 128 contiguous bytes a row.
// The dividend is float(sum) * w_scale with w_scale > 0: a zero is +0, so the quotient's sign needs no care.
// Fragment i of lane l holds token row rows[i], columns col0 + 16*j + 0..3.  FULL: the tile lies inside the
// matrix, no bounds checks.  EXTRA: bias and / or residual may be present.  LINES: rows of the output begin at whole lines.
// The stores are a quarter of a short-k launch (8192 x 2560 x 6912: 118 us of 153 without them), and the loads of the other
// workgroups of the compute unit wait behind them: so they write whole 128-byte lines, non-temporal.  In 64-byte pieces 1024 x
// 2560 x 6912 took 26.0 us (now 23.9), 2048 x 6912 x 2560 36.5 (34.8), 333 x 3328 x 8640 21.0 (19.5).
// Rows that begin anywhere (n no multiple of 32) are written by the same 16-byte stores, which need four-byte alignment only, through
// the cache, where the halves of a line that two stores share meet.  Such rows took 4-byte stores (n odd) or non-temporal ones:
// 1566 x 256 -> 28790 110 us, now 46, -> 28796 119, now 45; 4000 x 1024 -> 5001 with residual 195, now 62; 439 x 384 -> 23272 27, now 17.
template <int NI, int FN, bool FULL, bool EXTRA, bool LINES>
__device__ __forceinline__ void store_fragments_fast(const v4i (&acc)[NI][FN], const int (&rs)[NI], const float (&as)[NI],
                                                     const float (&rcp)[NI], float ws, const GemmProjDev &PJ, int m,
                                                     const int (&rows)[NI], int col0)
{
    const int lr = threadIdx.x & 15;
    const bool hi = lr >= 8;
    auto scaled4 = [&](const v4i &c, int i) {
        v4f v;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            v[r] = div_by_invariant_unchecked<false>(f32_mul((float)(c[r] - rs[i]), ws), as[i], rcp[i]);
        return v;
    };
    // Store k of fragment row i, FN of them.  Fragments 32 columns apart by pairs (j, j + 1): lanes of rows 8..15 of j change places
    // with lanes of rows 0..7 of j + 1 (a rotation by 8 of the 16 lanes), and each of the two stores then writes eight rows of 128
    // contiguous bytes.  Pairs begin at multiples of 32 columns; a fragment without a partner is stored as it is.
    const bool odd = ((col0 - ((threadIdx.x >> 4) & 3) * 4) >> 4) & 1;  // uniform over the wavefront
    auto place = [&](auto is_odd, int i, int k, int *row, int *col) {
        constexpr int FIRST = decltype(is_odd)::value ? 1 : 0, PAIRED = (FN - FIRST) / 2 * 2;
        const bool single = k < FIRST || k >= FIRST + PAIRED;
        const int second = (k - FIRST) & 1;
        *row = single ? rows[i] : rows[i] - (lr & 8) + 8 * second;
        *col = col0 + (single ? k : k - second + (hi ? 1 : 0)) * 16;
        return FULL || (*row < m && *col < PJ.n);
    };
    // Four values at src + 0..3, of which those past column n are not there.
    auto get = [&](const float *src, int col) {
        if (FULL || col + 4 <= PJ.n) return (v4f)*reinterpret_cast<const v4f_any *>(src);
        v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < 3; ++r)
            if (col + r < PJ.n) v[r] = src[r];
        return v;
    };
    auto run = [&](auto is_odd) {
        constexpr int FIRST = decltype(is_odd)::value ? 1 : 0, PAIRED = (FN - FIRST) / 2 * 2;
        // The residuals of a fragment row are requested together, ahead of its arithmetic; where the registers allow it, while the
        // row before it is finished.  (A lane reads no element that another lane writes: out may be the residual's memory.)
        constexpr bool AHEAD = NI * FN <= 10;
        v4f res[AHEAD ? 2 : 1][FN];
        auto fetch = [&](int i) {
#pragma unroll
            for (int k = 0; k < FN; ++k) {
                int row, col;
                const bool inside = place(is_odd, i, k, &row, &col);
                res[AHEAD ? i & 1 : 0][k] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
                if (inside) res[AHEAD ? i & 1 : 0][k] = get(PJ.residual + (size_t)row * PJ.n + col, col);
            }
        };
        if (AHEAD && EXTRA && PJ.residual) fetch(0);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (EXTRA && PJ.residual && (AHEAD ? i + 1 < NI : true)) fetch(AHEAD ? i + 1 : i);
            v4f v[FN];
#pragma unroll
            for (int j = 0; j < FN; ++j) v[j] = scaled4(acc[i][j], i);
#pragma unroll
            for (int j = FIRST; j < FIRST + PAIRED; j += 2)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    // lanes 8..15 of a row of 16 take the partner's value of j + 1, lanes 0..7 the partner's value of j
                    // (__builtin_bit_cast of a vector's element reads element 0 with this compiler: the elements go through floats)
                    const float fa = v[j][r], fb = v[j + 1][r];
                    const int a = __builtin_bit_cast(int, fa), b = __builtin_bit_cast(int, fb);
                    v[j][r] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false));
                    v[j + 1][r] = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false));
                }
#pragma unroll
            for (int k = 0; k < FN; ++k) {
                int row, col;
                if (!place(is_odd, i, k, &row, &col)) continue;
                v4f y = v[k];
                if (EXTRA && PJ.bias) {
                    const v4f b = get(PJ.bias + col, col);
                    y = (v4f){f32_add(y[0], b[0]), f32_add(y[1], b[1]), f32_add(y[2], b[2]), f32_add(y[3], b[3])};
                }
                if (EXTRA && PJ.residual) {
                    const v4f q = res[AHEAD ? i & 1 : 0][k];
                    y = (v4f){f32_add(y[0], q[0]), f32_add(y[1], q[1]), f32_add(y[2], q[2]), f32_add(y[3], q[3])};
                }
                float *dst = PJ.out + (size_t)row * PJ.n + col;
                if (LINES) __builtin_nontemporal_store(y, reinterpret_cast<v4f *>(dst));
                else if (FULL || col + 4 <= PJ.n) *reinterpret_cast<v4f_any *>(dst) = y;
                else {
#pragma unroll
                    for (int r = 0; r < 3; ++r)
                        if (col + r < PJ.n) dst[r] = y[r];
                }
            }
        }
    };
    if (odd) run(std::true_type{});
    else run(std::false_type{});
}

// The epilogue for every other case (int32 accumulator output, scales outside the short division's
// range): the same arithmetic, choices made per fragment row, a_sum and a_scale read from global memory.
template <int NI, int FN>
__device__ __forceinline__ void store_fragments_general(const v4i (&acc)[NI][FN], const int (&rows)[NI], int col0, float ws,
                                                        bool ws_fast, const GemmProjDev &PJ, const GemmParams &p)
{
    const bool vec_ok = (PJ.n & 3) == 0;  // 16-byte alignment of out[row][4c]
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int row = rows[i];
        const bool row_ok = row < p.m;
        const int rs = row_ok ? p.a_sum[row] : 0;
        const float as = (PJ.out && row_ok) ? p.a_scale[row] : 1.0f;
        const float as_recip = f32_div(1.0f, as);
        // the short division needs a well-behaved divisor (per row) and dividends in range: float(total) * ws
        // is zero or has ws's exponent plus at most 24, so one check on ws covers them.  The choice is made
        // per wavefront so that the usual case runs no plain division at all.
        const bool row_fast = ws_fast && invariant_divisor_ok(as);
        const bool wave_fast = __builtin_amdgcn_ballot_w64(!row_fast) == 0;
        if (!row_ok) continue;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int col = col0 + j * 16;
            if (col >= PJ.n) continue;
            const size_t o = (size_t)row * PJ.n + col;
            int tot[4];
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                tot[r] = acc[i][j][r] - rs;
                const float scaled = f32_mul((float)tot[r], ws);
                v[r] = wave_fast ? div_by_invariant_unchecked(scaled, as, as_recip) : f32_div(scaled, as);
            }
            if (vec_ok) {  // col + 3 < n follows from n % 4 == 0
                if (PJ.acc) *reinterpret_cast<int4 *>(PJ.acc + o) = make_int4(tot[0], tot[1], tot[2], tot[3]);
                if (PJ.out) {
                    if (PJ.bias) {
                        const float4 b = *reinterpret_cast<const float4 *>(PJ.bias + col);
                        v[0] = f32_add(v[0], b.x); v[1] = f32_add(v[1], b.y); v[2] = f32_add(v[2], b.z); v[3] = f32_add(v[3], b.w);
                    }
                    if (PJ.residual) {
                        const float4 q = *reinterpret_cast<const float4 *>(PJ.residual + o);
                        v[0] = f32_add(v[0], q.x); v[1] = f32_add(v[1], q.y); v[2] = f32_add(v[2], q.z); v[3] = f32_add(v[3], q.w);
                    }
                    *reinterpret_cast<float4 *>(PJ.out + o) = make_float4(v[0], v[1], v[2], v[3]);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (col + r >= PJ.n) continue;
                    if (PJ.acc) PJ.acc[o + r] = tot[r];
                    if (PJ.out) {
                        float y = v[r];
                        if (PJ.bias) y = f32_add(y, PJ.bias[col + r]);
                        if (PJ.residual) y = f32_add(y, PJ.residual[o + r]);
                        PJ.out[o + r] = y;
                    }
                }
            }
        }
    }
}

// The whole epilogue of one wavefront.  Fragment i of lane l holds token row m0 + lrows[i] (lrows: row inside the
// BM-row tile), columns col0 + 16*j + 0..3.  rowp is the LDS copy of the tile's a_sum and a_scale
// (fetch_row_operands), complete and visible: the caller has waited for vmcnt(0) and passed a workgroup barrier.
// full: the workgroup's tile lies inside the matrix.
template <int BM, int NI, int FN>
__device__ __forceinline__ void finish_fragments(const v4i (&acc)[NI][FN], const int (&lrows)[NI], int m0, int col0, bool full,
                                                 const uint8_t *rowp, const GemmProjDev &PJ, const GemmParams &p)
{
    const float ws = PJ.out ? *PJ.w_scale : 0.0f;
    const unsigned ws_expo = (__builtin_bit_cast(unsigned, ws) >> 23) & 0xffu;
    const bool ws_fast = ws > 0.0f && ws_expo > 64u && ws_expo < 160u;
    int rows[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) rows[i] = m0 + lrows[i];
    if (PJ.out && !PJ.acc && ws_fast) {
        const int *sum_l = reinterpret_cast<const int *>(rowp);
        const float *scale_l = reinterpret_cast<const float *>(rowp + BM * 4);
        int rs[NI];
        float as[NI], rcp[NI];
        bool ok = true;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            rs[i] = sum_l[lrows[i]];
            as[i] = scale_l[lrows[i]];
            rcp[i] = f32_div(1.0f, as[i]);
            ok = ok && invariant_divisor_ok(as[i]);
        }
        if (__builtin_amdgcn_ballot_w64(!ok) == 0) {
            const bool extra = PJ.bias != nullptr || PJ.residual != nullptr;
            // (a run-time choice in place of this one costs the loop of 128 x 160 tiles spilled registers: 10 % of the kernel)
            auto store = [&](auto lines) {
                constexpr bool LINES = decltype(lines)::value;
                if (full && !extra) store_fragments_fast<NI, FN, true, false, LINES>(acc, rs, as, rcp, ws, PJ, p.m, rows, col0);
                else if (full) store_fragments_fast<NI, FN, true, true, LINES>(acc, rs, as, rcp, ws, PJ, p.m, rows, col0);
                else if (!extra) store_fragments_fast<NI, FN, false, false, LINES>(acc, rs, as, rcp, ws, PJ, p.m, rows, col0);
                else store_fragments_fast<NI, FN, false, true, LINES>(acc, rs, as, rcp, ws, PJ, p.m, rows, col0);
            };
            if ((PJ.n & 31) == 0 && (reinterpret_cast<uintptr_t>(PJ.out) & 15) == 0) store(std::true_type{});
            else store(std::false_type{});
            return;
        }
    }
    store_fragments_general<NI, FN>(acc, rows, col0, ws, ws_fast, PJ, p);
}

// The epilogue by way of LDS, for gemm_ld8_kernel: the workgroup's int32 tile (COPIES partial tiles of different parts of k, added here) is
// laid down row by row and read back in output order, RP rows at a time.  put(pass) writes this wavefront's fragments of rows RP * pass
// .. into the area; rowp is the LDS copy of the tile's a_sum and a_scale (outside the area).  Every thread of the workgroup
// comes here, after a barrier behind the last use of the area; loaders and multipliers store alike.  Against exchanging halves and the
// epilogue in registers (finish_fragments) a few hundred instructions instead of up to ten thousand that a wavefront runs through
// once, whole rows of the tile per store at any n, and the residuals of a pass requested ahead of the barrier: 333 x 3328 -> 8640 with bias,
// 128 x 160 tiles, 24.4 -> 23.6 us.  Non-temporal where a row begins at 16 bytes (128 x 2560 -> 30000: 20.1 us, through the cache 22.1).
// PITCH: ints per row, padded so that the rows a store instruction touches start in different banks.
template <int BN>
constexpr int tile_pitch() { return BN + 4; }
template <int BN, int COPIES, int RP>
constexpr size_t tile_area_bytes() { return (size_t)COPIES * RP * tile_pitch<BN>() * 4; }

template <int BM, int BN, int COPIES, int RP, int THREADS, typename Put>
__device__ __forceinline__ void store_tile(uint8_t *area, const uint8_t *rowp, int m0, int n0, const GemmProjDev &PJ, const GemmParams &p,
                                           Put put)
{
    constexpr int PITCH = tile_pitch<BN>(), QUADS = BN / 4, PER = (RP * QUADS + THREADS - 1) / THREADS;
    const int *tile = reinterpret_cast<const int *>(area);
    const int *sum_l = reinterpret_cast<const int *>(rowp);
    const float *scale_l = reinterpret_cast<const float *>(rowp + BM * 4);
    const float ws = PJ.out ? *PJ.w_scale : 0.0f;
    const unsigned ws_expo = (__builtin_bit_cast(unsigned, ws) >> 23) & 0xffu;
    const bool ws_fast = ws > 0.0f && ws_expo > 64u && ws_expo < 160u;
    const bool stream = (PJ.n & 3) == 0 && (reinterpret_cast<uintptr_t>(PJ.out) & 15) == 0;
    const int tid = threadIdx.x;
#pragma unroll
    for (int pass = 0; pass < (BM + RP - 1) / RP; ++pass) {
        if (pass) __syncthreads();  // the pass before has been read
        put(pass);
        v4f res[PER];
        if (PJ.residual) {
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                const int at = tid + q * THREADS, r = at / QUADS, col = n0 + (at - r * QUADS) * 4, row = m0 + pass * RP + r;
                res[q] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
                if (r >= RP || row >= p.m || col >= PJ.n) continue;
                const float *src = PJ.residual + (size_t)row * PJ.n + col;
                if (col + 4 <= PJ.n) res[q] = *reinterpret_cast<const v4f_any *>(src);
                else
                    for (int c = 0; c < 3; ++c)
                        if (col + c < PJ.n) res[q][c] = src[c];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int at = tid + q * THREADS, r = at / QUADS, quad = at - r * QUADS, col = n0 + quad * 4, lrow = pass * RP + r, row = m0 + lrow;
            if (r >= RP || row >= p.m || col >= PJ.n) continue;
            v4i total = *reinterpret_cast<const v4i *>(tile + r * PITCH + quad * 4);
#pragma unroll
            for (int c = 1; c < COPIES; ++c) total += *reinterpret_cast<const v4i *>(tile + (c * RP + r) * PITCH + quad * 4);
            total -= sum_l[lrow];
            const size_t o = (size_t)row * PJ.n + col;
            const bool whole = col + 4 <= PJ.n;
            if (PJ.acc) {
                if (whole) *reinterpret_cast<v4i_any *>(PJ.acc + o) = total;
                else
                    for (int c = 0; c < 3; ++c)
                        if (col + c < PJ.n) PJ.acc[o + c] = total[c];
            }
            if (!PJ.out) continue;
            const float as = scale_l[lrow];
            v4f y;
            // the short division where w_scale and the rows' scales allow it, chosen per wavefront; float(sum) * w_scale of a zero is +0
            if (ws_fast && __builtin_amdgcn_ballot_w64(!invariant_divisor_ok(as)) == 0) {
                const float rcp = recip_of_ok_divisor(as);
#pragma unroll
                for (int c = 0; c < 4; ++c) y[c] = div_by_invariant_unchecked<false>(f32_mul((float)total[c], ws), as, rcp);
            } else {
                for (int c = 0; c < 4; ++c) y[c] = f32_div(f32_mul((float)total[c], ws), as);
            }
            if (PJ.bias) {
                v4f b = {0.0f, 0.0f, 0.0f, 0.0f};
                if (whole) b = *reinterpret_cast<const v4f_any *>(PJ.bias + col);
                else
                    for (int c = 0; c < 3; ++c)
                        if (col + c < PJ.n) b[c] = PJ.bias[col + c];
#pragma unroll
                for (int c = 0; c < 4; ++c) y[c] = f32_add(y[c], b[c]);
            }
            if (PJ.residual) {
#pragma unroll
                for (int c = 0; c < 4; ++c) y[c] = f32_add(y[c], res[q][c]);
            }
            float *dst = PJ.out + o;
            if (stream) __builtin_nontemporal_store(y, reinterpret_cast<v4f *>(dst));
            else if (whole) *reinterpret_cast<v4f_any *>(dst) = y;
            else
                for (int c = 0; c < 3; ++c)
                    if (col + c < PJ.n) dst[c] = y[c];
        }
    }
}

constexpr int DMA_SK = 128;  // columns per activation stage; a 256-column weight tile serves two stages

// D activation stages and NB weight buffers live in LDS; loads run P = D - 1 stages ahead of the MFMAs.
template <int D>
constexpr int dma_nb() { return (D - 1 + 2 + 1) / 2; }
template <int BM, int BN, int D>
constexpr size_t dma_lds_bytes() { return (size_t)D * BM * DMA_SK + (size_t)dma_nb<D>() * (BN / 16) * 1024; }

// Loads of the groups issued after stage s's own group and before the wait at the top of stage s: the groups
// of stages s+1 .. s+P-1; a group holds A_DMA activation loads, plus B_DMA weight loads when its stage is even.
template <int PHASE, int P, int A_DMA, int B_DMA>
constexpr int dma_in_flight()
{
    int n = 0;
    for (int j = 1; j < P; ++j) n += A_DMA + (((PHASE + j) & 1) == 0 ? B_DMA : 0);
    return n;
}

// Tile -> position.  Consecutive tiles run on one XCD at the same time.  Column by column of a row of tiles, they share one row
// tile's activations in the XCD's L2 and sweep all of the weights for every row of tiles.  With p.group_rows they go down that many
// row tiles before the next column, share those rows' activations and a few columns of weights, and the weights are swept once per group.
// The rule (launch_dma): where the weights do not fit an L2 of 4 MiB, the group's activations do (3 MiB), and an XCD would sweep the weights three
// times or more.  8192 x 2560 -> 6912 + 6912: loads alone 98 -> 75 us, the whole call 276 -> 264; 3402 x 1664 -> 11968 + 11968 151 -> 146.
// Elsewhere it gains nothing or loses up to 3 % (4096 x 4096 -> 8192, 1531 x 2816 -> 27824: output rows in more, shorter pieces).
constexpr int TILE_GROUP = 8;
__device__ __forceinline__ void tile_position(const GemmParams &p, int tile_id, int *tm, int *tn)
{
    const int per = p.group_rows * p.tiles_n, group = tile_id / per, in = tile_id - group * per;
    const int high = min(p.group_rows, p.tiles_m - group * p.group_rows);
    *tn = in / high;
    *tm = group * p.group_rows + in - *tn * high;
}

// WN: of the four wavefronts, how many lie side by side along n (2: 2 x 2, 4: 1 x 4).
template <int BM, int BN, int D, int OCC, int WN = 2>
__global__ __launch_bounds__(256, OCC) void gemm_dma_kernel(GemmParams p)
{
    constexpr int WTM = BM * WN / 4, WTN = BN / WN, FM = WTM / 16, FN = WTN / 16;
    constexpr int P = D - 1, NB = dma_nb<D>();
    constexpr bool GROUPS = BM == 128 && BN == 256;  // 128 x 160 tiles spill registers with it
    constexpr int A_STAGE = BM * DMA_SK;
    constexpr int A_DMA = A_STAGE / 1024 / 4;  // LDS-direct loads per wavefront per activation stage
    constexpr int B_TILES = BN / 16;           // weight tiles per 256 columns
    constexpr int B_DMA = (B_TILES + 3) / 4;   // per wavefront (the last ones may repeat a tile)
    constexpr int B_STAGE = B_TILES * 1024;
    static_assert(A_STAGE % 4096 == 0 && WTM % 16 == 0 && WTN % 16 == 0 && D >= 2, "tile shape");
    static_assert(dma_in_flight<0, P, A_DMA, B_DMA>() < 64 && dma_in_flight<1, P, A_DMA, B_DMA>() < 64, "vmcnt range");

    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];  // [D][A_STAGE] then [NB][B_STAGE]
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = WN == 2 ? wave >> 1 : 0, wn = WN == 2 ? wave & 1 : wave, lr = lane & 15, lg = lane >> 4;

    int tile_id;
    {
        const int total = p.tiles_m * p.tiles_n;
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        const int per_xcd = (total + 7) >> 3;
        tile_id = xcd * per_xcd + idx;
        if (tile_id >= total) return;
    }
    // tiles_n counts the column tiles of all projections of the launch, one after the other
    int tm = tile_id / p.tiles_n, tn_all = tile_id % p.tiles_n;
    if (GROUPS && p.group_rows > 1) tile_position(p, tile_id, &tm, &tn_all);
    int pj = 0;
    if (p.nproj > 1 && tn_all >= p.proj[0].tn_end) pj = 1;
    if (p.nproj > 2 && tn_all >= p.proj[1].tn_end) pj = 2;
    const GemmProjDev PJ = p.proj[pj];  // uniform over the workgroup
    const int tn = tn_all - (pj ? p.proj[pj - 1].tn_end : 0);
    const int m0 = tm * BM, n0 = tn * BN;
    const int nstage = p.kt_count * 2;

    // Activation loads: load q of this wavefront covers tile rows 8*(wave*A_DMA + q) .. +7; lane l lands in
    // row l/8 at physical 16-byte chunk l%8 and therefore fetches logical chunk (l%8) ^ (row & 7).
    // Rows past m re-read row m-1 (their results are never stored).
    uint32_t a_off[A_DMA];  // byte offsets into the activation matrix (below 4 GiB: checked by the launcher)
#pragma unroll
    for (int q = 0; q < A_DMA; ++q) {
        const int row = 8 * (wave * A_DMA + q) + (lane >> 3);
        const int lc = (lane & 7) ^ (row & 7);
        int grow = m0 + row;
        if (grow >= p.m) grow = p.m - 1;
        a_off[q] = (uint32_t)grow * (uint32_t)p.k + lc * 16;
    }
    // Weight tiles: wavefront w fetches tiles w, w+4, ... of the workgroup's BN/16 row blocks; lane l = slot l.
    const int rb0 = n0 / 16;
    const int rb_last = (PJ.n + 15) / 16 - 1;
    uint32_t b_off[B_DMA], b_dst[B_DMA];  // byte offsets into the re-tiled weights, tile positions in a weight stage
#pragma unroll
    for (int q = 0; q < B_DMA; ++q) {
        int tix = wave + 4 * q;
        if (tix >= B_TILES) tix = B_TILES - 1;
        int rb = rb0 + tix;
        if (rb > rb_last) rb = rb_last;
        b_off[q] = ((uint32_t)rb * (uint32_t)p.kt_count * 64 + lane) * 16;
        b_dst[q] = tix * 1024;
    }
    // The load group of stage s: the weight tile of k-tile s/2 when s is even, then the activation stage.
    auto issue = [&](int s) {
        if ((s & 1) == 0) {
            const int kt = s >> 1;
            const uint32_t dst = lds_base + D * A_STAGE + (kt % NB) * B_STAGE;
#pragma unroll
            for (int q = 0; q < B_DMA; ++q) dma16(PJ.w + (size_t)kt * 1024, b_off[q], dst + b_dst[q]);
        }
        const uint32_t dst = lds_base + (s % D) * A_STAGE + wave * A_DMA * 1024;
#pragma unroll
        for (int q = 0; q < A_DMA; ++q) dma16(p.a + (size_t)s * DMA_SK, a_off[q], dst + q * 1024);
    };

    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = (v4i){0, 0, 0, 0};

#pragma unroll
    for (int s = 0; s < P; ++s)
        if (s < nstage) issue(s);

    uint32_t a_rd[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) a_rd[i] = (wm * WTM + i * 16 + lr) * DMA_SK;
    const int sw = lr & 7;

    // The MFMA computes C^T: the weight fragment is the first operand, so that result register r of lane l is
    // out[token row l % 16][output column 4*(l/16) + r]: four consecutive columns, one 16-byte store.
    uint4 bp[FN];  // the wavefront's slots of the current weight tiles: read at an even stage, used by two
    auto compute = [&](int s, bool second_half) {
        const int kt = s >> 1;
        const uint8_t *abuf = lds + (s % D) * A_STAGE;
        if (!second_half) {
            const uint8_t *bbuf = lds + D * A_STAGE + (kt % NB) * B_STAGE + (wn * FN) * 1024 + lane * 16;
#pragma unroll
            for (int j = 0; j < FN; ++j) bp[j] = *reinterpret_cast<const uint4 *>(bbuf + j * 1024);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            v4i afrag[FM];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                afrag[i] = *reinterpret_cast<const v4i *>(abuf + a_rd[i] + (((t * 4 + lg) ^ sw) << 4));
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const uint32_t wd = second_half ? (t == 0 ? bp[j].z : bp[j].w) : (t == 0 ? bp[j].x : bp[j].y);
                v4i bfrag;
                bfrag[0] = (int)(wd & 0x03030303u);
                bfrag[1] = (int)((wd >> 2) & 0x03030303u);
                bfrag[2] = (int)((wd >> 4) & 0x03030303u);
                bfrag[3] = (int)((wd >> 6) & 0x03030303u);
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bfrag, afrag[i], acc[i][j], 0, 0, 0);
            }
        }
    };

    // Loads retire in issue order.  At the top of stage s its own group must have landed; the groups of the
    // P - 1 later stages stay in flight.  The last P - 1 stages, with fewer groups behind them, drain everything.
    // When the whole launch is resident at once (OCC workgroups on every compute unit, all started together), the
    // hardware's oldest-first choice among wavefronts lets the OCC workgroups of a compute unit finish one after the
    // other, the last one running alone at a fraction of the MFMA rate.  Workgroup ids b, b + 256, ... share a
    // compute unit; rotating their wavefront priorities every k-tile keeps them level (measured: 5 % at
    // 2048 x 6912 x 2560).  With several rounds of workgroups the staggered finish is wanted and nothing is done.
    const int rank = blockIdx.x >> 8;
    for (int s = 0; s < nstage; s += 2) {
        if (p.rotate) set_wave_priority((rank + (s >> 1)) % OCC);
        if (s + P <= nstage) wait_vm<dma_in_flight<0, P, A_DMA, B_DMA>()>(); else wait_vm<0>();
        __syncthreads();
        if (s + P < nstage) issue(s + P);
        compute(s, false);

        if (s + 1 + P <= nstage) wait_vm<dma_in_flight<1, P, A_DMA, B_DMA>()>(); else wait_vm<0>();
        __syncthreads();
        if (s + 1 + P < nstage) issue(s + 1 + P);
        // In the last stage the buffer of the stage before it is free: the per-row epilogue operands land there
        // while the last MFMAs run.
        else if (s + 2 == nstage) fetch_row_operands<BM>(p, m0, wave, lane, lds_base + (s % D) * A_STAGE);
        compute(s + 1, true);
    }
    const uint32_t ROWP = ((nstage - 2) % D) * A_STAGE;
    static_assert(rowp_bytes<BM>() <= A_STAGE, "row operands fit an activation stage");
    wait_vm<0>();
    __syncthreads();
    int lrows[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) lrows[i] = wm * WTM + i * 16 + lr;
    finish_fragments<BM, FM, FN>(acc, lrows, m0, n0 + wn * WTN + lg * 4, m0 + BM <= p.m && n0 + BN <= PJ.n, lds + ROWP, PJ, p);
}

// Raising a kernel's dynamic LDS limit is needed once per process; a function-local static makes that once
// thread-safe (forward may be called from many threads).
template <typename Kernel>
hipError_t raise_lds_limit(Kernel kernel, size_t bytes)
{
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

template <int BM, int BN, int D, int OCC, int WN = 2>
int launch_dma(GemmParams p, hipStream_t stream)
{
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = 0;
    for (int j = 0; j < p.nproj; ++j) p.proj[j].tn_end = p.tiles_n += (p.proj[j].n + BN - 1) / BN;
    const int total = p.tiles_m * p.tiles_n;
    const int grid = ((total + 7) / 8) * 8;
    p.rotate = total <= 256 * OCC && total > 256;
    p.group_rows = BM == 128 && BN == 256 && p.tiles_m >= 3 * 8 && (size_t)p.tiles_n * BN * p.k / 4 > (4u << 20) &&
                           (size_t)TILE_GROUP * BM * p.k <= (3u << 20) ? TILE_GROUP : 1;
    constexpr size_t lds = dma_lds_bytes<BM, BN, D>();
    static_assert(lds <= 160 * 1024 && lds * OCC <= 160 * 1024 && OCC <= 4, "LDS budget, priorities 0..3");
    static const hipError_t attr = lds > 64 * 1024 ? raise_lds_limit(&gemm_dma_kernel<BM, BN, D, OCC, WN>, lds) : hipSuccess;
    BITNET_HIP_TRY(attr);
    launch_kernel((gemm_dma_kernel<BM, BN, D, OCC, WN>), dim3(grid), dim3(256), lds, stream, p);
    BITNET_HIP_CHECK_LAUNCH("gemm_dma_kernel");
    return BITNET_HIP_OK;
}

// ---- eight MFMA wavefronts per workgroup fed by two loader wavefronts -------------------------------------------
//
// For launches that one round of workgroups holds.  One wavefront per SIMD cannot keep the MFMA pipe
// busy (its own LDS waits and unpack instructions sit between its MFMAs); two can.  With too few tiles for two
// workgroups per compute unit the second wavefront per SIMD comes from inside the workgroup: wavefronts 0..3 take
// columns 0..127 of every 256-column stage and wavefronts 4..7 columns 128..255, each group accumulating the whole
// BM x BN tile; the two partial tiles are added in the epilogue (int32 sums: exact).  A stage is one 256-column weight
// tile plus BM x 256 activation bytes, NST stages in LDS, loads NST - 1 stages ahead (more than three gain nothing).
// The LDS-direct loads are issued by two further wavefronts (8 and 9) that never multiply.  A wavefront that issues
// a load while the queue of the load path is full waits at that instruction, and while it waits it issues no MFMA;
// with the loads spread over the multiplying wavefronts every one of them paid that wait every stage (measured at
// 2048 x 2560 x 6912: 40.8 us with the loads on the eight wavefronts, 33.6 us with no loads in the loop at all,
// 35.8 us with the two loaders).  The multiplying wavefronts meet the loaders at the stage barrier and otherwise
// only read LDS and run MFMAs.
// Which tile: choose_ld8.  In place of four-wavefront workgroups of 64 x 32 and 64 x 64 with four stages in flight, and of k split across
// workgroups (us, quantiser included): 128 x 6912 -> 2560 15.0 -> 12.6, 213 x 13120 -> 3008 36.6 -> 26.2, 378 x 6656 -> 3264 24.5 -> 19.9, 640 x
// 6912 -> 2560 28.9 -> 23.3, 2100 x 13952 -> 768 65.7 -> 53, 110 x 8192 -> 14336 29 -> 22.6; of 128 x 160 alone 300 x 8192 -> 8192 37.0 -> 33.7.
// Four multiplying wavefronts of 128 x 80 with their fragments read a half step ahead, and the fragments of the next stage read before the
// barrier, were measured and are not faster: per compute unit the loop is bound by LDS reads and MFMAs together.
// Waits until at most `groups` groups of G loads each, MAX at most, are in flight.
template <int G, int MAX>
__device__ __forceinline__ void wait_groups(int groups)
{
    if constexpr (MAX == 0) wait_vm<0>();
    else if (groups >= MAX) wait_vm<MAX * G>();
    else wait_groups<G, MAX - 1>(groups);
}

template <int BM, int BN, int NST>
constexpr size_t ld8_lds_bytes() { return (size_t)NST * (BM * 256 + (BN / 16) * 1024) + rowp_bytes<BM>(); }

template <int BM, int BN, int NST>
__global__ __launch_bounds__(640, 1) void gemm_ld8_kernel(GemmParams p)
{
    constexpr int WTM = BM / 2, WTN = BN / 2, FM = WTM / 16, FN = WTN / 16;
    constexpr int A_STAGE = BM * 256;
    constexpr int A_CHUNKS = A_STAGE / 1024;    // 1 KiB LDS-direct loads per stage
    constexpr int B_TILES = BN / 16;
    constexpr int B_STAGE = B_TILES * 1024;
    constexpr int STAGE = A_STAGE + B_STAGE;
    constexpr int A_PER = A_CHUNKS / 2, B_PER = (B_TILES + 1) / 2;  // per loader wavefront
    constexpr int GROUP = A_PER + B_PER;
    static_assert(A_CHUNKS % 2 == 0 && WTM % 32 == 0 && WTN % 16 == 0 && (NST - 1) * GROUP < 64, "tile shape, vmcnt range");
    static_assert(tile_area_bytes<BN, 2, WTM>() <= (size_t)NST * STAGE, "epilogue area");

    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];  // [NST][A half 0 | A half 1 | B], then the row operands
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    int tile_id;
    {
        const int total = p.tiles_m * p.tiles_n;
        const int xcd = blockIdx.x & 7, idx = blockIdx.x >> 3;
        const int per_xcd = (total + 7) >> 3;
        tile_id = xcd * per_xcd + idx;
        if (tile_id >= total) return;
    }
    const int tm = tile_id / p.tiles_n, tn_all = tile_id % p.tiles_n;
    int pj = 0;
    if (p.nproj > 1 && tn_all >= p.proj[0].tn_end) pj = 1;
    if (p.nproj > 2 && tn_all >= p.proj[1].tn_end) pj = 2;
    const GemmProjDev PJ = p.proj[pj];  // uniform over the workgroup
    const int tn = tn_all - (pj ? p.proj[pj - 1].tn_end : 0);
    const int m0 = tm * BM, n0 = tn * BN;
    constexpr uint32_t ROWP = NST * STAGE;

    if (wave >= 8) {
        // ---- loader wavefront L: activation chunks A_PER*L .. and weight tiles B_PER*L .. of every stage ----
        const int L = wave - 8;
        uint32_t a_off[A_PER], b_off[B_PER], b_dst[B_PER];
#pragma unroll
        for (int q = 0; q < A_PER; ++q) {
            const int c = L * A_PER + q;
            const int half = c / (BM / 8), row = 8 * (c % (BM / 8)) + (lane >> 3);
            const int lc = (lane & 7) ^ (row & 7);
            int grow = m0 + row;
            if (grow >= p.m) grow = p.m - 1;
            a_off[q] = (uint32_t)grow * (uint32_t)p.k + half * 128 + lc * 16;
        }
        const int rb0 = n0 / 16, rb_last = (PJ.n + 15) / 16 - 1;
#pragma unroll
        for (int q = 0; q < B_PER; ++q) {
            int tix = L * B_PER + q;
            if (tix >= B_TILES) tix = B_TILES - 1;
            int rb = rb0 + tix;
            if (rb > rb_last) rb = rb_last;
            b_off[q] = ((uint32_t)rb * (uint32_t)p.kt_count * 64 + lane) * 16;
            b_dst[q] = A_STAGE + tix * 1024;
        }
        auto issue = [&](int kt) {
            const uint32_t stage = lds_base + (kt % NST) * STAGE;
#pragma unroll
            for (int q = 0; q < B_PER; ++q) dma16(PJ.w + (size_t)kt * 1024, b_off[q], stage + b_dst[q]);
#pragma unroll
            for (int q = 0; q < A_PER; ++q) dma16(p.a + (size_t)kt * 256, a_off[q], stage + (L * A_PER + q) * 1024);
        };
        // the per-row epilogue operands: a_sum by loader 0, a_scale by loader 1 (BM / 64 loads of 64 rows each)
#pragma unroll
        for (int ch = 0; ch < BM / 64; ++ch) {
            int grow = m0 + ch * 64 + lane;
            if (grow >= p.m) grow = p.m - 1;
            if (L == 0) dma4(p.a_sum, (uint32_t)grow * 4u, lds_base + ROWP + ch * 256);
            else if (p.a_scale) dma4(p.a_scale, (uint32_t)grow * 4u, lds_base + ROWP + BM * 4 + ch * 256);
        }
#pragma unroll
        for (int kt = 0; kt < NST - 1; ++kt)
            if (kt < p.kt_count) issue(kt);
        for (int kt = 0; kt < p.kt_count; ++kt) {
            wait_groups<GROUP, NST - 2>(p.kt_count - 1 - kt);
            __syncthreads();
            if (kt + NST - 1 < p.kt_count) issue(kt + NST - 1);  // into the buffer of stage kt - 1, which nobody reads any more
        }
        __syncthreads();  // every wavefront is done with the stage buffers
        store_tile<BM, BN, 2, WTM, 640>(lds, lds + ROWP, m0, n0, PJ, p, [](int) {});
        return;
    }

    const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1, lr = lane & 15, lg = lane >> 4;
    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = (v4i){0, 0, 0, 0};
    uint32_t a_rd[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) a_rd[i] = kg * (BM * 128) + (wm * WTM + i * 16 + lr) * 128;
    const int sw = lr & 7;

    auto compute = [&](int kt) {
        const uint8_t *abuf = lds + (kt % NST) * STAGE;
        const uint8_t *bbuf = abuf + A_STAGE + (wn * FN) * 1024 + lane * 16 + kg * 8;
        uint2 bp[FN];  // dwords 2*kg, 2*kg+1 of the slot: this group's two k-steps
#pragma unroll
        for (int j = 0; j < FN; ++j) bp[j] = *reinterpret_cast<const uint2 *>(bbuf + j * 1024);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            v4i afrag[FM];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                afrag[i] = *reinterpret_cast<const v4i *>(abuf + a_rd[i] + (((t * 4 + lg) ^ sw) << 4));
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const uint32_t wd = t == 0 ? bp[j].x : bp[j].y;
                v4i bfrag;
                bfrag[0] = (int)(wd & 0x03030303u);
                bfrag[1] = (int)((wd >> 2) & 0x03030303u);
                bfrag[2] = (int)((wd >> 4) & 0x03030303u);
                bfrag[3] = (int)((wd >> 6) & 0x03030303u);
#pragma unroll
                for (int i = 0; i < FM; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(bfrag, afrag[i], acc[i][j], 0, 0, 0);
            }
        }
    };
    for (int kt = 0; kt < p.kt_count; ++kt) {
        __syncthreads();  // the loaders arrive here once stage kt has landed
        compute(kt);
    }

    __syncthreads();  // every wavefront is done with the stage buffers
    store_tile<BM, BN, 2, WTM, 640>(lds, lds + ROWP, m0, n0, PJ, p, [&](int pass) {
        if (pass != wm) return;
        int *at = reinterpret_cast<int *>(lds) + (kg * WTM + lr) * tile_pitch<BN>() + wn * WTN + lg * 4;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) *reinterpret_cast<v4i *>(at + i * 16 * tile_pitch<BN>() + j * 16) = acc[i][j];
    });
}

template <int BM, int BN, int NST>
int launch_ld8(GemmParams p, hipStream_t stream)
{
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = 0;
    for (int j = 0; j < p.nproj; ++j) p.proj[j].tn_end = p.tiles_n += (p.proj[j].n + BN - 1) / BN;
    const int total = p.tiles_m * p.tiles_n;
    const int grid = ((total + 7) / 8) * 8;
    constexpr size_t lds = ld8_lds_bytes<BM, BN, NST>();
    static_assert(lds <= 160 * 1024, "LDS budget");
    static const hipError_t attr = raise_lds_limit(&gemm_ld8_kernel<BM, BN, NST>, lds);
    BITNET_HIP_TRY(attr);
    launch_kernel((gemm_ld8_kernel<BM, BN, NST>), dim3(grid), dim3(640), lds, stream, p);
    BITNET_HIP_CHECK_LAUNCH("gemm_ld8_kernel");
    return BITNET_HIP_OK;
}

// The tiles of gemm_ld8_kernel, with what a stage of 256 columns costs a compute unit in each (ns: the slope over k at few
// workgroups; the smaller ones are bound by LDS reads per MFMA, the larger ones by unpacking and MFMA).
struct Ld8Tile {
    int bm, bn, stage_ns;
    int per_cu;  // workgroups that a compute unit holds (LDS)
    int (*launch)(GemmParams, hipStream_t);
};
const Ld8Tile LD8_TILES[] = {
    {64, 32, 140, 2, &launch_ld8<64, 32, 4>},     {64, 64, 250, 2, &launch_ld8<64, 64, 3>},    {64, 96, 330, 2, &launch_ld8<64, 96, 3>},
    {128, 64, 400, 1, &launch_ld8<128, 64, 3>},   {64, 128, 430, 2, &launch_ld8<64, 128, 3>},  {128, 96, 560, 1, &launch_ld8<128, 96, 3>},
    {128, 128, 720, 1, &launch_ld8<128, 128, 3>}, {128, 160, 880, 1, &launch_ld8<128, 160, 3>},
};
// The tile with which a stage takes least among those that need one round of workgroups: what the fullest compute unit multiplies, or
// what all of them load at the 24 TB/s that the L2s together give; null: none needs one round.  n: output widths.
const Ld8Tile *choose_ld8(size_t m, const size_t *n, int nproj, size_t *stage_ns)
{
    const Ld8Tile *best = nullptr;
    for (const Ld8Tile &t : LD8_TILES) {
        size_t count = 0;
        for (int j = 0; j < nproj; ++j) count += ((m + t.bm - 1) / t.bm) * ((n[j] + t.bn - 1) / t.bn);
        const size_t here = (count + 255) / 256, bytes = (size_t)t.bm * 256 + t.bn * 64;
        if (here > (size_t)t.per_cu) continue;
        const size_t multiply = here * t.stage_ns, load = count * bytes / 24000, cost = multiply > load ? multiply : load;
        if (!best || cost < *stage_ns) { best = &t; *stage_ns = cost; }
    }
    return best;
}

constexpr size_t LD8_LEAST_K = 1024;      // rows shorter than four stages do not take gemm_ld8_kernel (launch_gemm_multi)
constexpr size_t LARGE_TILES_FROM = 640;  // tiles of 128 x 160 from which gemm_dma_kernel takes its largest ones

template <int BM, int BN>
int launch_tile(GemmParams p, hipStream_t stream)
{
    p.tiles_m = (p.m + BM - 1) / BM;
    p.tiles_n = (p.n + BN - 1) / BN;
    const int total = p.tiles_m * p.tiles_n;
    const int grid = ((total + 7) / 8) * 8;
    constexpr size_t lds = 2 * BM * LDS_PITCH + BM * sizeof(int);
    static const hipError_t attr = lds > 64 * 1024 ? raise_lds_limit(&gemm_tiled_kernel<BM, BN>, lds) : hipSuccess;
    BITNET_HIP_TRY(attr);
    launch_kernel((gemm_tiled_kernel<BM, BN>), dim3(grid), dim3(256), lds, stream, p);
    BITNET_HIP_CHECK_LAUNCH("gemm_tiled_kernel");
    return BITNET_HIP_OK;
}

}  // namespace

// What a launch takes (ns) beyond what the token GEMV takes as well, for the choice between the two (gemm_beats_token_gemv): where one
// round of gemm_ld8_kernel holds it, its start, its stages (the cost of choose_ld8 is that of a stage alone; with what both kernels do taken
// off, five eighths of it) and an epilogue by the outputs of whole tiles; elsewhere its start and, per output of a row of tiles (64
// tokens; 128 from LARGE_TILES_FROM on), the k-tiles.
size_t gemm_beyond_ns(size_t m, size_t k, size_t n)
{
    const size_t kt = k / TILE_K, rows64 = (m + 63) / 64, rows128 = (m + 127) / 128;
    size_t stage_ns = 0;
    if (k >= LD8_LEAST_K && choose_ld8(m, &n, 1, &stage_ns)) return 2800 + stage_ns * kt * 5 / 8 + rows64 * n / 40;
    const bool large = rows128 * ((n + 159) / 160) >= LARGE_TILES_FROM;
    return 2300 + (large ? 2 * rows128 : rows64) * n * kt / 85;
}

// Up to GEMM_MAX_PROJ projections of the same activation matrix in one launch of the LDS-direct kernels (q, k, v
// or gate, up at prefill: small projections alone would leave most compute units idle).  Returns
// BITNET_HIP_UNSUPPORTED (without a message) when the shapes do not fit those kernels.
int launch_gemm_multi(const GemvProj *projs, int nproj, const int8_t *a, const int32_t *a_sum, const float *a_scale,
                      size_t m, size_t k, hipStream_t stream)
{
    if (m == 0 || nproj <= 0) return BITNET_HIP_OK;
    if (nproj > GEMM_MAX_PROJ) return BITNET_HIP_UNSUPPORTED;
    // One k-tile is enough for the LDS-direct kernels (two load stages: their prologue issues what there is); the eight-wavefront
    // one wants two.  Through the register-staged kernel 1151 x 256 -> 1024 + 1024 took 37.9 us, now 10.5; 334 x 256 -> 2700
    // with residual 24.7, now 9.6.
    bool dma_ok = a_sum != nullptr && m > 16 && k % 256 == 0 && k > 0 && (reinterpret_cast<uintptr_t>(a) & 15) == 0 &&
                  m * k < (1ull << 32);  // 32-bit lane offsets
    size_t tiles = 0, tiles64 = 0, tiles32 = 0;  // 128 x 160, 64 x 64 and 64 x 32 tiles of the launch
    GemmParams p = {};
    for (int j = 0; j < nproj && dma_ok; ++j) {
        const GemvProj &s = projs[j];
        dma_ok = s.n > 0 && s.n <= 0x7fffffffu && tiled_bytes(s.n, k) < (1ull << 32);
        tiles += ((m + 127) / 128) * ((s.n + 159) / 160);
        tiles64 += ((m + 63) / 64) * ((s.n + 63) / 64);
        tiles32 += ((m + 63) / 64) * ((s.n + 31) / 32);
        GemmProjDev &d = p.proj[j];
        d.w = s.tiled; d.w_scale = s.w_scale; d.bias = s.bias; d.residual = s.residual; d.out = s.out; d.acc = s.acc;
        d.n = (int)s.n; d.tn_end = 0;
    }
    if (!dma_ok) return BITNET_HIP_UNSUPPORTED;
    for (int j = nproj; j < GEMM_MAX_PROJ; ++j) p.proj[j] = p.proj[nproj - 1];
    p.nproj = nproj; p.a = a; p.a_sum = a_sum; p.a_scale = a_scale; p.m = (int)m; p.k = (int)k; p.kt_count = (int)k_tiles(k);
    // gemm_ld8_kernel where one round of its workgroups holds the launch (256 compute units); with less than four stages its start and
    // epilogue cost more than the shorter loop saves (1000 x 512 -> 2560: 11.0 us, 9.6 with the kernels below).
    if (k >= LD8_LEAST_K) {
        size_t widths[GEMM_MAX_PROJ], stage_ns = 0;
        for (int j = 0; j < nproj; ++j) widths[j] = projs[j].n;
        const Ld8Tile *tile = choose_ld8(m, widths, nproj, &stage_ns);
        if (tile) return tile->launch(p, stream);
    }
    if (tiles >= LARGE_TILES_FROM) {
        // 128 x 256 tiles as four wavefronts of 128 x 64 side by side, two workgroups per compute unit: half the unpacking per MFMA
        // (a weight fragment serves eight token fragments instead of four) and a tenth fewer bytes loaded per output.  Per unit of work it takes
        // 0.95 of the time of 128 x 160, so it is chosen where the outputs of the fullest compute unit leave that gain:
        // 8192 x 2560 -> 6912 + 6912 280 -> 264 us, 4096 x 4096 -> 8192 132 -> 122, 3402 x 1664 -> 11968 + 11968 155 -> 146; not
        // 8192 x 6912 -> 2560 (three tiles of 256 columns where four of 160 come out even: 190 against 180).
        auto fullest = [&](size_t bn) {
            size_t count = 0;
            for (int j = 0; j < nproj; ++j) count += ((m + 127) / 128) * ((projs[j].n + bn - 1) / bn);
            return (count + 255) / 256 * bn;
        };
        if (fullest(256) * 95 <= fullest(160) * 100) return launch_dma<128, 256, 2, 2, 4>(p, stream);
        return launch_dma<128, 160, 2, 3>(p, stream);
    }
    // Short rows with few tiles: narrow tiles (more workgroups, all resident at once), four stages of loads in flight, four or three
    // workgroups per compute unit.
    if (tiles < 100 && tiles32 <= 704) return launch_dma<64, 32, 4, 4>(p, stream);
    if (tiles <= 140 && tiles64 <= 768) return launch_dma<64, 64, 4, 3>(p, stream);
    // Between one round of loader-fed tiles and 2.5 tiles of 128 x 160 per compute unit: whatever leaves the fullest compute unit least, in
    // outputs, weighted by what an output costs (64 x 160, two by two wavefronts, unpacks once for two token fragments instead of four and
    // takes a fifth longer; launches beyond one round of workgroups start over).  In place of 64 x 160 and 128 x 128 (us, quantiser included):
    // 1024 x 4096 -> 8192 44.1 -> 38.7, 1500 x 8192 -> 4096 62.5 -> 54.5, 1566 x 2560 -> 5000 32.2 -> 28.8, 512 x 4096 -> 14336 38.0 -> 35.1, 6000 x
    // 1024 -> 1024 21.4 -> 20.0, 1200 x 4096 -> 4096 31.9 -> 30.2, 2600 x 6912 -> 2560 61.0 -> 58.4.
    struct Shape { size_t bm, bn, slots, cost; int (*launch)(GemmParams, hipStream_t); };
    static const Shape shapes[] = {{64, 128, 1024, 100, &launch_dma<64, 128, 2, 4, 4>}, {64, 256, 768, 100, &launch_dma<64, 256, 2, 3, 4>},
                                   {128, 128, 768, 100, &launch_dma<128, 128, 2, 3>},   {64, 160, 1024, 121, &launch_dma<64, 160, 2, 4>}};
    const Shape *best = nullptr;
    size_t least = 0;
    for (const Shape &t : shapes) {
        size_t count = 0;
        for (int j = 0; j < nproj; ++j) count += ((m + t.bm - 1) / t.bm) * ((projs[j].n + t.bn - 1) / t.bn);
        const size_t cost = (count + 255) / 256 * t.bm * t.bn * t.cost * (count > t.slots ? 5 : 4);
        if (!best || cost < least) { best = &t; least = cost; }
    }
    return best->launch(p, stream);
}

int launch_gemm_tiled(const uint8_t *tiled, const int8_t *a, const int32_t *a_sum, size_t m, size_t n, size_t k,
                      int32_t *acc, const float *w_scale, const float *a_scale, const float *bias,
                      const float *residual, float *out, hipStream_t stream)
{
    if (m == 0 || n == 0) return BITNET_HIP_OK;
    {
        const GemvProj one = {tiled, w_scale, bias, residual, out, acc, n};
        const int rc = launch_gemm_multi(&one, 1, a, a_sum, a_scale, m, k, stream);
        if (rc != BITNET_HIP_UNSUPPORTED) return rc;
    }
    GemmParams p = {};
    p.w = tiled; p.a = a; p.acc = acc; p.w_scale = w_scale; p.a_scale = a_scale; p.bias = bias;
    p.residual = residual; p.a_sum = a_sum; p.out = out; p.m = (int)m; p.n = (int)n; p.k = (int)k; p.kt_count = (int)k_tiles(k);
    p.tiles_m = p.tiles_n = 0;
    if (m < 96) return launch_tile<64, 128>(p, stream);
    auto waste = [&](size_t bn) {
        const size_t tiles = ((m + 127) / 128) * ((n + bn - 1) / bn), slots = 256;
        const size_t rounds = (tiles + slots - 1) / slots;
        return (double)(rounds * slots) / (double)tiles;
    };
    const double w256 = waste(256), w160 = waste(160), w128 = waste(128);
    if (w256 <= w160 && w256 <= w128) return launch_tile<128, 256>(p, stream);
    if (w160 <= w128) return launch_tile<128, 160>(p, stream);
    return launch_tile<128, 128>(p, stream);
}

// ---- matrix-unit rate (diagnostic) -----------------------------------------------------------------------------
// A loop of nothing but v_mfma_i32_16x16x64_i8 with its operands in registers: eight independent accumulators per
// wavefront, two wavefronts per SIMD on every compute unit.  What it sustains is the ceiling of the GEMM above on the
// device at hand (clock under a matrix load included); RANDOM gives every lane different int8 activations and 2-bit
// codes 0..2 as weights, as the GEMM's operands are, otherwise every byte of both operands is 1.
namespace {
template <bool RANDOM>
__global__ __launch_bounds__(512, 1) void mfma_rate_kernel(int iters, int *sink, unsigned seed)
{
    v4i acc[8], a[4], b[4];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = (v4i){0, 0, 0, 0};
    unsigned w = seed * (threadIdx.x + 1) * 2654435761u + blockIdx.x * 97u + 12345u;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            w = w * 1664525u + 1013904223u;
            a[i][c] = RANDOM ? (int)w : 0x01010101;
            w = w * 1664525u + 1013904223u;
            const unsigned two = (w >> 8) & 0x03030303u;  // bytes 0..3; 3 becomes 2 (no carry between bytes)
            b[i][c] = RANDOM ? (int)(two - ((two >> 1) & two & 0x01010101u)) : 0x01010101;
        }
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[i & 3], a[(i + (i >> 2)) & 3], acc[i], 0, 0, 0);
    }
    int s = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
    sink[blockIdx.x * blockDim.x + threadIdx.x] = s;
}
}  // namespace

int launch_mfma_rate(bool random_operands, int iters, int compute_units, int *sink, hipStream_t stream)
{
    const dim3 grid((unsigned)compute_units), block(MFMA_RATE_THREADS);
    if (random_operands) launch_kernel((mfma_rate_kernel<true>), grid, block, 0, stream, iters, sink, 7u);
    else launch_kernel((mfma_rate_kernel<false>), grid, block, 0, stream, iters, sink, 7u);
    BITNET_HIP_CHECK_LAUNCH("mfma_rate_kernel");
    return BITNET_HIP_OK;
}

}  // namespace bitnet
