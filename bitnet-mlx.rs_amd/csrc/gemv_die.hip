// Several tokens in one launch, their rows quantised once on every die (XCD): the workgroups of a die share the work through its L2.
//
// A token GEMV on rows that a launch before it quantised pays for that launch: 1.3 us from its last workgroup to the first of the next,
// about 1 us until the rows are back from memory, and nothing of the weights' way overlaps either; a call that nothing records pays the
// host's 4 us for the second launch.  A workgroup that quantises all of its rows for itself (gemv_rowq_kernel) is bound by vector
// instructions from a few thousand columns on.  Between the two: workgroups whose number modulo eight is the same run on one die.  The
// first m of each die quantise a row each, into a buffer that all dies write (the same bytes from each), and end; the others ask for their
// weight tiles at once and multiply when the rows of their token group have reached the die's L2.  What a launch takes is a row's way
// through the quantiser (2.9 us with a norm, 2.2 without), the hand-over (0.7) and the products, exchange and epilogue of
// gemv_rows_kernel (2.5).  gate + up of 2560 -> 2 x 6912 at 8 tokens: 6.0 us from its first workgroup to its last, where quantiser and GEMV
// took 7.4 with the gap between them.  The 30-block stack of 2560 columns, recorded, at 2 / 3 / 4 / 8 / 12 / 16 / 24 / 32 / 42 / 64 tokens: 548 /
// 605 / 665 / 743 / 787 / 815 / 879 / 910 / 995 / 1108 us before, 543 / 550 / 580 / 629 / 668 / 702 / 790 / 819 / 945 / 1089 with it.  Calls of their own, us:
// 16 x 6912 -> 2560 7.9 -> 5.6, 32 x 4096 -> 5120 7.8 -> 5.8, 64 x 2560 -> 2560 with norm 8.1 -> 6.2.  (A first form, in which workgroups with
// products took the rows beside them, was 0.5 to 2 us slower a launch: their tiles came late, and a row's registers beside the tiles' left
// room for fewer workgroups.)
//
// The hand-over inside the die.  A row's workgroup waits until its stores have reached L2, which the vector memory counter says, and then
// stores the launch's tag into the flag of (die, row).  Readers poll the flags, and load the rows, with device-scope loads (sc1), which
// are not answered from the compute unit's L1.  Each die has flags of its own, found by the die's hardware number and not by the
// workgroup's, so a flag always speaks for the reader's L2.  (Device-scope release and acquire fences write back and invalidate the whole
// L2: 16 us more a launch as measured here; polling with atomics holds up the flags' line: 40 us.  Words that carry their own tag through
// memory that all dies share take 2 to 10 us, see diag_hop_kernel.)
//
// Every wait ends.  The workgroups that quantise wait for nobody; they come first in a die's order, so they are running or done when one
// that waits for them is started; and a reader that has looked `looks` times (about 0.5 ms) quantises the rows of its token group itself:
// the bytes are the same whoever writes them.  The results depend neither on how workgroups are dealt to the dies nor on their order,
// only the time does.
//
// Flags hold 64-bit tags.  Before a launch none of the flags that it looks at may hold its tag: a call of its own takes a tag that no other
// launch has; a decoder, whose steps are replayed with the same arguments, passes sets of flags in turn and tag 1, and a launch clears the set
// of the launch before it (enqueue_step says which).
#include "rowsgemv.hpp"

namespace bitnet {

namespace {

// Arguments behind the preloaded ones, in blocks of 64 bytes: each is one scalar load.
struct DieParams {
    Fused16Proj proj[GEMV_MAX_PROJ];  // rb_end counts groups of RB row blocks
    uint8_t *q;                       // rows in ActRows::TILES16 order
    float *a_scale;
    uint64_t *flags, *clear;
    uint64_t tag;
    unsigned stride;                  // flags of a die
    int looks;
    float eps;
    unsigned blocks01, blocks2;          // row blocks of projections 0 and 1 (16 bits each), and of 2
    unsigned clear_halves;               // eights of dies whose flags start at clear
};
static_assert(sizeof(DieParams) == 64 * (1 + GEMV_MAX_PROJ), "one scalar load a block");
constexpr int DIE_ARGS_AT = 56;  // its offset in the argument buffer: three pointers and seven 4-byte arguments before it, aligned to eight
// The last block, taken apart.
struct DieArgs {
    global_ptr<uint8_t> q;
    global_ptr<float> a_scale;
    global_ptr<uint64_t> flags, clear;
    uint64_t tag;
    unsigned stride;
    int looks;
    float eps;
    __device__ __forceinline__ explicit DieArgs(const v16u &C)
    {
        q = pointer_at<uint8_t>(C, 0); a_scale = pointer_at<float>(C, 2);
        flags = pointer_at<uint64_t>(C, 4); clear = pointer_at<uint64_t>(C, 6);
        tag = ((uint64_t)C[9] << 32) | C[8];
        stride = C[10]; looks = (int)C[11];
        eps = __builtin_bit_cast(float, (unsigned)C[12]);
    }
};

__device__ __forceinline__ unsigned die_number()
{
    unsigned id;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID, 0, 4)" : "=s"(id));
    return id;
}
// A look past this compute unit's L1.
__device__ __forceinline__ uint64_t look(const uint64_t *flag)
{
    uint64_t v;
    asm volatile("global_load_dwordx2 %0, %1, off sc1\n\ts_waitcnt vmcnt(0)" : "=v"(v) : "v"(flag) : "memory");
    return v;
}

// Where a row of the launch lies (ActRows::TILES16).
struct DieRow {
    global_ptr<uint8_t> base;
    unsigned piece;
    __device__ __forceinline__ DieRow(global_ptr<uint8_t> q, int row, int m, int kt_count)
    {
        const int group = row >> 4;
        piece = 16u * (unsigned)min(16, m - group * 16);
        base = q + (size_t)group * 16 * TILE_K * kt_count + (row & 15) * 16;
    }
    __device__ __forceinline__ global_ptr<uint32_t> chunk(int c) const { return (global_ptr<uint32_t>)(base + ((unsigned)(c >> 2) * piece + (unsigned)(c & 3) * 4u)); }
};

// A row by one wavefront that holds none of it: for a workgroup that has waited too long, beside the tiles it already has.  The same bits
// (the order of the sum: a lane stands for the virtual lanes l, l + 64, l + 128, l + 192).
template <int MODE, bool NORM>
__device__ __forceinline__ void quantise_row_alone(const float *x, const float *x2, const float *gamma, int k, float eps, int lane,
                                                    const DieRow &place, int kt_count, global_ptr<float> a_scale)
{
    const int chunks = k >> 2;
    float rms = 1.0f;
    if constexpr (NORM) {
        float ss = 0.0f;
#pragma unroll 1
        for (int j = 0; j < 4; ++j) {
            float part = 0.0f;
#pragma unroll 1
            for (int c = 64 * j + lane; c < chunks; c += 256) part = sum_squares4(part, row16_chunk<MODE>(x, x2, 0, 0, c));
            part = wave_sum_f32(part);
            ss = j == 0 ? part : f32_add(ss, part);
        }
        rms = f32_sqrt(f32_add(f32_div(ss, (float)k), eps));
    }
    auto value = [&](int c) {
        float4 v = row16_chunk<MODE>(x, x2, 0, 0, c);
        if constexpr (NORM) {
            const float4 g = reinterpret_cast<const float4 *>(gamma)[c];
            v = make_float4(f32_mul(f32_div(v.x, rms), g.x), f32_mul(f32_div(v.y, rms), g.y), f32_mul(f32_div(v.z, rms), g.z), f32_mul(f32_div(v.w, rms), g.w));
        }
        return v;
    };
    float amax = 0.0f;
#pragma unroll 1
    for (int c = lane; c < chunks; c += 64) amax = absmax4(amax, value(c));
    amax = wave_max_f32(amax);
    const float scale = amax > 0.0f ? f32_div(127.0f, amax) : 1.0f;
#pragma unroll 1
    for (int c = lane; c < kt_count * (TILE_K / 4); c += 64) *place.chunk(c) = c < chunks ? quant4_clamped(value(c), scale) : 0u;
    if (lane == 0) *a_scale = scale;
}

// MODE: the input transform of Row16.  NT: k-tiles a wavefront (and chunks a thread of the row that it quantises).
template <int MODE, bool NORM, int RB, int NT>
__global__ __launch_bounds__(1024) void gemv_die_kernel(const float *hot_x, const float *hot_x2, const float *hot_gamma, int hot_k, int hot_nw,
                                                        int hot_ldx, unsigned hot_m_kt, unsigned hot_ends, unsigned hot_quantisers_tgroups, unsigned hot_tg_magic,
                                                        [[maybe_unused]] DieParams args)
{
    extern __shared__ v4i part[];  // [nw][RB][64]
    __shared__ float red_f[2][16];
    __shared__ int late_s;
    const int slot = (int)(blockIdx.x & 7), local = (int)(blockIdx.x >> 3);  // the workgroup's number among those of its die
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = hot_nw, chunks = hot_k >> 2, m = (int)(hot_m_kt & 0xffffu), kt_count = (int)(hot_m_kt >> 16);
    const int quantisers = (int)(hot_quantisers_tgroups & 0xffffu), tgroups = (int)(hot_quantisers_tgroups >> 16);
    typedef const __attribute__((address_space(4))) v16u *arg_ptr;
    const arg_ptr arg_blocks = (arg_ptr)((uintptr_t)__builtin_amdgcn_kernarg_segment_ptr() + DIE_ARGS_AT);

    if (local < quantisers) {
        Row16<NORM, NT> row16;
        const int row = local;
        row16.template load<MODE>(hot_x + row * (size_t)hot_ldx, MODE == BITNET_HIP_INPUT_RELU2_MUL ? hot_x2 + row * (size_t)hot_ldx : nullptr, 0, 0, hot_gamma,
                                  chunks, nw, wave, tid, lane);
        __builtin_amdgcn_sched_barrier(0);
        v16u C = arg_blocks[GEMV_MAX_PROJ];
        if (tid < 16 && tid >= nw) red_f[1][tid] = 0.0f;
        float k_f = (float)hot_k, k_recip = recip_of_ok_divisor(k_f);
        asm volatile("" : "+s"(C), "+v"(k_recip));
        const DieArgs d(C);
        const unsigned die = die_number();
        uint32_t packed[NT];
        const float scale = row16.quantise(chunks, k_f, k_recip, d.eps, wave, tid, red_f, packed);
        const DieRow place(d.q, row, m, kt_count);
#pragma unroll
        for (int i = 0; i < NT; ++i)
            if (row16.chunk[i] < kt_count * (TILE_K / 4)) *place.chunk(row16.chunk[i]) = packed[i];  // chunks past the row hold zeros
        if (tid == 0) d.a_scale[row] = scale;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // in L2
        lds_barrier();
        if (tid == 0) d.flags[die * d.stride + row] = d.tag;
        if (local == 0)
            for (unsigned half = 0; half < C[15]; ++half)
                for (int i = tid; i < m; i += 64 * nw) d.clear[(slot + 8 * half) * d.stride + i] = 0;
        return;
    }

    // the token groups of a group of row blocks are neighbours on the die
    const int at = local - quantisers, part_of = tgroups == 1 ? at : (int)__umulhi((unsigned)at, hot_tg_magic), tg = at - part_of * tgroups;
    const int group = part_of * 8 + slot;  // may lie past the last group: such workgroups store no outputs
    const int end0 = (int)(hot_ends & 0xffffu), end1 = (int)(hot_ends >> 16);
    const int pj = group < end0 ? 0 : (group < end1 ? 1 : 2);
    v16u P = arg_blocks[pj], C = arg_blocks[GEMV_MAX_PROJ];
    asm volatile("" : "+s"(P), "+s"(C));
    const DieArgs d(C);
    const unsigned die = die_number();
    const int rows_here = min(16, m - tg * 16);
    const int rb0 = (group - (pj == 0 ? 0 : (pj == 1 ? end0 : end1))) * RB;
    const int rb_count = (int)(pj == 0 ? C[13] & 0xffffu : (pj == 1 ? C[13] >> 16 : C[14]));
    v4u_t w[NT][RB];
    rows_load_w<RB, NT>(w, pointer_at<const v4u_t>(P, 0) + lane, rb0, rb_count, wave, nw, kt_count);
    __builtin_amdgcn_sched_barrier(0);
    RowsFinish end(P, reinterpret_cast<const float *>((uintptr_t)d.a_scale), rb0, RB, wave, lane, tg, rows_here);
    if constexpr (RB < 4) end.request_operands();
    if (wave == 0) {
        const uint64_t *mine = reinterpret_cast<const uint64_t *>((uintptr_t)d.flags) + (die * d.stride + tg * 16 + min(lane, rows_here - 1));
        bool here = false;
        for (int i = 0; i < d.looks && !here; ++i) here = __builtin_amdgcn_ballot_w64(look(mine) != d.tag) == 0;
        if (lane == 0) late_s = !here;
    }
    lds_barrier();
    if (__builtin_expect(late_s != 0, 0)) {
        for (int r = wave; r < rows_here; r += nw) {  // uniform over the wavefront
            const size_t row = (size_t)(tg * 16 + r);
            quantise_row_alone<MODE, NORM>(hot_x + row * (size_t)hot_ldx, MODE == BITNET_HIP_INPUT_RELU2_MUL ? hot_x2 + row * (size_t)hot_ldx : nullptr,
                                           hot_gamma, hot_k, d.eps, lane, DieRow(d.q, (int)row, m, kt_count), kt_count, d.a_scale + row);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
    }
    v4i af[NT][4];
    const size_t group_at = (size_t)tg * 16 * TILE_K * kt_count;
    const __amdgpu_buffer_rsrc_t group_rows =
        __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((uintptr_t)(d.q + group_at)), 0, rows_here * TILE_K * kt_count, 0x00020000);
    rows_load_a_l2<NT>(af, group_rows, lane, rows_here, wave, nw, kt_count);
    if constexpr (RB < 4) end.request_scales_l2();
    __builtin_amdgcn_sched_barrier(0);

    v4i acc[RB], sums = {0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[r] = (v4i){0, 0, 0, 0};
    rows_multiply<RB, NT>(af, w, wave, nw, kt_count, acc, sums);
    if constexpr (RB >= 4) {
        __builtin_amdgcn_sched_barrier(0);
        end.request_scales_l2();
        end.request_operands();
        __builtin_amdgcn_sched_barrier(0);
    }
    end.template finish<RB>(acc, sums, part, wave, lane, nw);
}

__global__ __launch_bounds__(128) void clear_die_flags_kernel(uint64_t *flags, int stride, int m)
{
    for (int i = (int)threadIdx.x; i < m; i += 128) flags[(int)blockIdx.x * stride + i] = 0;
}

struct Launch {
    const float *x, *x2, *gamma;
    int k, nw, ldx;
    unsigned m_kt, ends, quantisers_tgroups, tg_magic;
    DieParams p;
    dim3 grid;
    hipStream_t stream;
};

template <int MODE, bool NORM, int RB, int NT>
int launch(const Launch &l)
{
    constexpr size_t MOST = (size_t)16 * RB * 1024;
    static const hipError_t attr = MOST >= 64 * 1024 ? hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_die_kernel<MODE, NORM, RB, NT>),
                                                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)MOST)
                                                     : hipSuccess;
    BITNET_HIP_TRY(attr);
    launch_kernel((gemv_die_kernel<MODE, NORM, RB, NT>), l.grid, dim3(64u * (unsigned)l.nw), (size_t)l.nw * RB * 1024, l.stream, l.x, l.x2, l.gamma, l.k,
                       l.nw, l.ldx, l.m_kt, l.ends, l.quantisers_tgroups, l.tg_magic, l.p);
    BITNET_HIP_CHECK_LAUNCH("gemv_die_kernel");
    return BITNET_HIP_OK;
}
template <int MODE, bool NORM>
int launch_shape(const Launch &l, int rb, int nt)
{
    if (nt == 1) return rb == 4 ? launch<MODE, NORM, 4, 1>(l) : (rb == 2 ? launch<MODE, NORM, 2, 1>(l) : launch<MODE, NORM, 1, 1>(l));
    return rb == 4 ? launch<MODE, NORM, 4, 2>(l) : (rb == 2 ? launch<MODE, NORM, 2, 2>(l) : launch<MODE, NORM, 1, 2>(l));
}

}  // namespace

namespace {

constexpr size_t DIE_CUS = 32;  // compute units of a die

// Row blocks and k-tiles as in launch_gemv_rows, and the workgroups of a die.
struct Shape {
    int rb, nt, nw;
    size_t quantisers, multipliers;  // workgroups of a die
    size_t slots;                    // of them that run at once
};
Shape shape_of(size_t m, size_t k, size_t blocks)
{
    const size_t kt = k_tiles(k), tgroups = (m + 15) / 16;
    Shape s = {};
    s.rb = 1;
    while (s.rb < 4 && (blocks + s.rb - 1) / s.rb * tgroups > 256) s.rb *= 2;
    s.nt = kt <= 16 ? 1 : 2;
    s.nw = s.nt == 1 ? row_workgroup_waves((int)k) : (int)((kt + 1) / 2);
    s.quantisers = m;
    s.multipliers = ((blocks + s.rb - 1) / s.rb + 7) / 8 * tgroups;
    // wavefronts of a compute unit by the kernel's registers: up to 64 with one tile a wavefront; 70, and 90 to 92, with two
    const size_t waves = s.nt == 1 ? 32 : (s.rb == 1 ? 28 : 20);
    s.slots = DIE_CUS * (waves / (size_t)s.nw);
    return s;
}

}  // namespace

bool gemv_die_takes(const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode, const float *gamma, int sum_order, size_t blocks,
                    bool alone)
{
    auto al16 = [](const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    if (m < 2 || m > (size_t)GEMV_DIE_MAX_M || blocks == 0 || blocks > GEMV_ROWS_MAX_BLOCKS) return false;
    const bool gated = input_mode == BITNET_HIP_INPUT_RELU2_MUL;
    if (!(input_mode == BITNET_HIP_INPUT_PLAIN || (gated && !gamma))) return false;
    if (k % 4 != 0 || ldx % 4 != 0 || ldx >= ((size_t)1 << 31) || k_tiles(k) > 32) return false;
    if (gamma && sum_order != BITNET_HIP_SUM_BLOCK256) return false;
    if (!al16(x) || (x2 && !al16(x2)) || (gamma && !al16(gamma))) return false;
    // Up to eight tokens gemv_fused16_kernel may be one launch as well, which pays while its workgroups have few tiles to walk, and in a call of
    // its own, which takes as long as the host's launch, always (4.4 us against 4.8).  A decoder block with this kernel where that one's
    // workgroups walk 24 to 44 tiles: 0.1 to 1.1 us slower; 48: 0.6 faster to 0.1 slower; 64: 0.2 to 0.7 faster, but at two tokens 0.1 faster to
    // 0.4 slower; 80 and more: 0.2 to 2.4 faster.  At two tokens there is little to gain, and it is lost where that kernel has a workgroup for
    // every compute unit and the two that quantise are one too many: blocks of 2560 to 4096 columns with gate + up of 30 multiplying workgroups a
    // die 0.0 to 0.6 us faster, of 31 and 32 0.4 faster to 0.8 slower, of 33 0.1 to 1.3 faster.
    if (gemv_fused_supported(x, x2, ldx, m, k, input_mode, 1, gamma, sum_order, blocks)) {
        const size_t tiles = gemv_fused_tiles(m, k, blocks);
        if (alone || tiles < (m > 2 ? 64 : 80)) return false;
        const Shape s = shape_of(m, k, blocks);
        return m > 2 || s.multipliers > DIE_CUS || s.quantisers + s.multipliers <= DIE_CUS;
    }
    // Otherwise the other choice is two launches, and what decides is whether the workgroups of a die run at once: those that multiply
    // are to be there when the rows are, and a second round of them waits for the first.  Decoder blocks of 512 to 4096 columns at 9 to 64
    // tokens, one launch group by this kernel, by workgroups over slots: up to 0.8 0.3 to 2.4 us faster, to 1.1 even to 1.2 faster, beyond up to
    // 11 slower; rows with a gate before them (wider, two tiles a wavefront) up to 0.8 even to 1.5 faster, at 0.9 to 1.0 even to 0.2 slower (but
    // 0.3 to 0.9 faster at up to 12 tokens), beyond up to 4 slower.
    const Shape s = shape_of(m, k, blocks);
    const size_t total = s.quantisers + s.multipliers;
    if (!alone) return 20 * total <= (gated ? 17 : 22) * s.slots;
    // A call of its own saves the host's second launch, 2 us, and may take that much longer.  us in two launches -> here, without and with
    // norm: 2560 -> 5120 at 64 tokens (1.1 times the slots) 8.0 -> 6.7, 8.2 -> 8.3; 4096 -> 13824 at 32 (1.3) 8.9 -> 8.1, 9.3 -> 9.8; 2560 -> 5120 at 95
    // (1.6) 8.0 -> 8.3, 8.3 -> 9.2; with one workgroup a compute unit 6912 -> 5120 at 32 (1.6) 8.7 -> 8.3, 9.4 -> 9.2, 6912 -> 13824 at 24 (2.4)
    // 12.7 -> 13.1, 13.6 -> 14.0; long rows of many tokens, whose quantisers fill the die: 8192 -> 640 at 48 7.8 -> 7.3, 8.0 -> 9.2, at 64
    // 7.8 -> 8.2, 8.2 -> 10.1.  With calls on a second stream beside it, both queued behind long work, the rows' eight copies take the other's compute
    // units: 48 x 2560 -> 5120 3.7 -> 4.5 us a call, 32 x 6912 -> 5120 5.6 -> 6.2, 24 x 4096 -> 4096 3.75 -> 3.7, 16 x 6912 -> 2560 3.8 -> 3.5; as the host's calls
    // come from one thread, on one to four streams, 14 -> 11 for each.
    if (s.nt == 2 && m > (gamma ? 32u : 48u)) return false;
    return 20 * total <= (s.slots == DIE_CUS ? 33 : (gamma ? 23 : 28)) * s.slots;
}

int launch_gemv_die(const GemvProj *projs, int nproj, const float *x, const float *x2, size_t ldx, size_t m, size_t k, int input_mode, const float *gamma,
                    float eps, int8_t *q, float *a_scale, const DieFlags &f, hipStream_t stream)
{
    if (m == 0 || nproj <= 0) return BITNET_HIP_OK;
    const size_t kt = k_tiles(k), tgroups = (m + 15) / 16;
    size_t blocks = 0;
    for (int j = 0; j < nproj; ++j) blocks += row_blocks(projs[j].n);
    const Shape shape = shape_of(m, k, blocks);
    Launch l = {};
    size_t groups = 0;
    unsigned ends[GEMV_MAX_PROJ] = {}, counts[GEMV_MAX_PROJ] = {};
    for (int j = 0; j < nproj; ++j) {
        const GemvProj &s = projs[j];
        Fused16Proj &d = l.p.proj[j];
        d.w = s.tiled; d.w_scale = s.w_scale; d.bias = s.bias; d.residual = s.residual; d.out = s.out; d.acc = s.acc; d.n = (int)s.n;
        counts[j] = (unsigned)row_blocks(s.n);
        groups += (counts[j] + shape.rb - 1) / shape.rb;
        ends[j] = (unsigned)groups;
        d.rb_end = (int)groups;
    }
    for (int j = nproj; j < GEMV_MAX_PROJ; ++j) l.p.proj[j] = l.p.proj[nproj - 1];
    if (groups == 0) return BITNET_HIP_OK;
    l.x = x; l.x2 = x2; l.gamma = gamma; l.k = (int)k; l.ldx = (int)ldx; l.nw = shape.nw; l.stream = stream;
    l.m_kt = (unsigned)m | ((unsigned)kt << 16);
    l.ends = (nproj > 1 ? ends[0] : 0xffffu) | ((nproj > 2 ? ends[1] : 0xffffu) << 16);
    l.grid = dim3(8u * (unsigned)(m + (groups + 7) / 8 * tgroups));
    l.quantisers_tgroups = (unsigned)m | ((unsigned)tgroups << 16);
    l.tg_magic = (unsigned)((((uint64_t)1 << 32) + tgroups - 1) / tgroups);  // not used for one group
    l.p.q = reinterpret_cast<uint8_t *>(q); l.p.a_scale = a_scale; l.p.eps = eps;
    l.p.flags = f.flags; l.p.clear = f.clear; l.p.clear_halves = f.clear ? (unsigned)(f.clear_sets * GEMV_DIE_SETS / 8) : 0; l.p.tag = f.tag; l.p.stride = f.stride; l.p.looks = f.looks;
    l.p.blocks01 = counts[0] | (counts[1] << 16);
    l.p.blocks2 = counts[2];
    if (input_mode == BITNET_HIP_INPUT_RELU2_MUL) return launch_shape<BITNET_HIP_INPUT_RELU2_MUL, false>(l, shape.rb, shape.nt);
    return gamma ? launch_shape<BITNET_HIP_INPUT_PLAIN, true>(l, shape.rb, shape.nt) : launch_shape<BITNET_HIP_INPUT_PLAIN, false>(l, shape.rb, shape.nt);
}

int launch_clear_die_flags(uint64_t *flags, size_t stride, size_t m, hipStream_t stream)
{
    launch_kernel(clear_die_flags_kernel, dim3((unsigned)GEMV_DIE_SETS), dim3(128), 0, stream, flags, (int)stride, (int)m);
    BITNET_HIP_CHECK_LAUNCH("clear_die_flags_kernel");
    return BITNET_HIP_OK;
}

}  // namespace bitnet
