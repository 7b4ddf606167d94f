// EXL3 linear for many rows: trellis decode fused into an fp16 MFMA GEMM
// (v_mfma_f32_32x32x16_f16, fp32 accumulate).  Covers the row counts the
// reference spreads over a cooperative GEMM (<= 144 rows) and reconstruct +
// dense GEMM (> 144 rows), crates/berth-kernels/csrc/prefill_lin/linear.cu:184-344;
// the weight is never written back to memory.
//
//   launch 1: a_had = Hh(a * suh)                        (had_r_128, pre-scale)
//   launch 2: c = Hh(a_had @ W) * svh                    (this file)
//
// Work split: a workgroup of 4 waves owns BM = 32*MB rows x 256 columns; each
// wave owns 64 of the columns for all BM rows, so decoded weights stay in the
// registers of the wave that decoded them.  Per 32 rows of K a wave decodes 2
// tile rows x 4 tile columns: lanes 0..31 take tile row kt, lanes 32..63 tile row
// kt+1, eight lanes per tile (octet layout).  The four register quads a lane ends
// up with ((column u or u+8) x (k 0..7 or 8..15 of its tile row)) are exactly four
// MFMA B operands: B[k-slot][col-slot] with col-slot = lane % 32 and k-slot =
// 8*(lane/32) + i.  The A operand for the same slots is a_had[row][16*(kt +
// lane/32) + 8h + i], one 16-byte LDS read.  Column slots map to columns
// 16*(slot/8) + slot%8 + 8f; the epilogue undoes that when it stages the fp32
// tile in LDS for the output Hadamard.
//
// K can be split over S workgroups (few rows, or few columns: not enough tiles to
// fill the chip).  The last workgroup to arrive at a tile (self-resetting counters)
// finishes it: the others leave their partial accumulators in the library workspace
// in register layout, and the finisher adds all parts in k order, so the result does
// not depend on timing.
#pragma once

#include "exl3_gemv_kernel.cuh"
#include "silu.cuh"

namespace berth {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// one linear of a bundle whose lists the host knows
struct GemmSlice {
    const uint32_t* trellis;
    const _Float16* svh;
    void* c;
    int width;                  // columns of this linear (a multiple of 128, at most N)
    int n_stride;               // columns of the whole weight the slice is cut from: elements between
                                // output rows and, in tiles of 16, between the tile rows of its trellis
    const _Float16* a_had;      // the rotated copy of the input it multiplies, [M][K]
};
constexpr int kGemmMaxSlices = 16;

struct GemmParams {
    const _Float16* a_had[2];   // [rows][K], already rotated (one per linear of the launch)
    ExpertLin lin;              // dense mode
    void* c[2];
    int M, K, N, out_fp32;
    // grouped mode (problems != nullptr): group_tile says which problem (<= BM rows), linear of the
    // launch and column block a workgroup takes
    const ExpertLin* experts;
    const GroupProblem* problems;
    const int* num_problems;
    int lins_per_expert, lin_base;
    ExpertLin shared[3];        // an always-on expert passed by value (problem.expert == shared_expert)
    int shared_expert;
    // mixed grouped launches (exl3_gemm_mixed_kernel): problems of up to 128 rows, whose units
    // of work come first; those of `problems` follow (max_big: the list's capacity)
    const GroupProblem* big_problems;
    const int* num_big;
    int max_big;
    int tiles_y;                // dense: row blocks; grouped: capacity of the problem list
    int tile0;                  // dense: first (row block, column block) tile of this launch, row-major
    // split-K
    int S;
    float* partials;            // [unit][S][4 waves][MB][2][16][64]
    unsigned* counters;         // [unit], cstride words apart ("arrived"; "written" kGemmWrittenBase further on)
    int cstride;
    // balanced dense launches (exl3_gemm_balanced_kernel): the launch's (tile, k-block) units,
    // tile-major, are dealt out evenly to gridDim.x workgroups
    int units;                  // tiles * K/128; 0: not a balanced launch
    int unit_q, unit_r;         // units = unit_q * gridDim.x + unit_r
    // A tile's finisher waits for the other sharers' partial sums with a bound: after
    // spin_limit polls it gives up, zeroes the tile's counters, stores 1 + the tile's counter
    // index to *fault (host-visible memory; may be null) and leaves the tile unwritten.
    unsigned* fault;
    unsigned spin_limit;
    // Bundles (crates/berth-kernels/src/ops.rs:264-293 with more than 8 rows): num_slices
    // linears that share K and the row count run as one dense launch.  Every slice owns
    // ceil(N / 256) column blocks of the launch (N = the widest slice); a block past the end of
    // a narrower slice is empty.  The slice's tensors come from the device lists when b_list is
    // set (uniform mode: c_ptrs null, outputs [slice][M][N] behind c[0], rotated input = slab
    // `slice`; sliced mode: all seven lists; a_had[0] holds the rotated inputs, slab_stride
    // elements apart), else from `slice` by value.
    int num_slices;             // 0: one linear (lin, c[0], a_had[0])
    size_t slab_stride;
    const uint64_t* b_list;
    const uint64_t* svh_list;
    const uint64_t* c_ptrs;
    const int* size_n_list;
    const int* n_stride_list;
    const int* had_src_list;
    // few-row launches (exl3_gemm_rows_kernel): unit_q / unit_r deal out units of 64 x 128 weights;
    // or, with S > 0, cut every column block into S parts; floor(2^32 / d) + 1 (0 for d = 1) for d = K / 64,
    // N / 128, unit_q, unit_q + 1, S (exact for the operands used)
    // The row-block launches (exl3_gemm_block_kernel) deal out steps of 256 x 128 weights of tiles
    // of rows_per_tile rows, tiles_y row blocks per column block: m_tr for the steps of a tile,
    // m_rt for tiles_y.
    unsigned m_tr, m_nb, m_q, m_q1, m_s, m_rt;
    int rows_per_tile;
    int group_blocks;           // grouped few-row launches: column blocks of 128 per problem, all linears (m_rt divides by it)
    unsigned lds_bytes;         // dynamic LDS of the launch
    const float* out_add;       // optional fp32 [M][N] (one linear, fp32 output): added to the output
    GemmSlice slice[kGemmMaxSlices];
    // grouped: where row r of the sorted order lies in a_had (optional; rows of the always-on expert: at r)
    const int32_t* a_rows;
    int group_lins;             // linears of a problem that are units of their own (1 or 2)
    int places;                 // exl3_gemm_mixed_kernel: workgroups that run at a time; tiles run as halves of 128 columns up to this many
    int ramp_problems;          // grouped 32-row tiles: PriorityRamp up to this many problems
    _Float16* act_had;          // exl3_gemm_pair_kernel: the down projection's rotated input, in sorted order
};

// Few-row launches that rotate the input themselves: where it comes from and where the rotated rows go, for
// one linear and lists in device memory, or per slice.  (Arguments of their own: every launch copies its
// arguments, and these are half a kilobyte.)
struct GemmRotation {
    const _Float16* suh;
    const _Float16* in;
    _Float16* had_out;          // null: another slice leaves them
};
struct GemmRotateParams : GemmParams {
    const _Float16* rot_in;
    _Float16* rot_out;          // [slab][M][K]
    const uint64_t* suh_list;
    size_t rot_in_stride;       // elements between the slabs' inputs (0: one for all)
    unsigned m_rows;            // divides by M
    GemmRotation rotation[kGemmMaxSlices];
};

// the tensors of the column block `nblk` of a dense launch
struct TileView {
    ExpertLin lin;
    const _Float16* a_had;
    void* cout;
    int N;                      // columns of the linear
    int ldc;                    // elements between output rows
    int nblk;                   // column block inside the linear
    bool empty;                 // the block lies past the end of its (narrower) slice
};
__device__ __forceinline__ TileView dense_tile_view(const GemmParams& p, const int nblk)
{
    TileView v;
    v.lin = p.lin;
    v.a_had = p.a_had[0];
    v.cout = p.c[0];
    v.N = p.N;
    v.ldc = p.N;
    v.nblk = nblk;
    v.empty = false;
    if (p.num_slices > 0) {
        const int per = (p.N + 255) >> 8;
        const int sl = nblk / per;
        v.nblk = nblk - sl * per;
        if (p.b_list) {
            int slab = sl;
            v.lin.trellis = (const uint32_t*)p.b_list[sl];
            v.lin.svh = (const _Float16*)p.svh_list[sl];
            if (p.c_ptrs) {
                v.N = p.size_n_list[sl];
                v.ldc = p.n_stride_list[sl];
                slab = p.had_src_list[sl];
                v.cout = (void*)p.c_ptrs[sl];
            } else {
                v.cout = (char*)p.c[0] + (size_t)sl * p.M * p.N * (p.out_fp32 ? 4 : 2);
            }
            v.a_had = p.a_had[0] + (size_t)slab * p.slab_stride;
        } else {
            const GemmSlice& g = p.slice[sl];
            v.lin.trellis = g.trellis;
            v.lin.svh = g.svh;
            v.cout = g.c;
            v.N = g.width;
            v.ldc = g.n_stride;
            v.a_had = g.a_had;
        }
        v.empty = v.nblk * 256 >= v.N;
    }
    return v;
}

// The finisher's wait for `counter` to reach `want`, bounded.  Called by one thread.  A
// workgroup that has arrived is running and depends on nothing, so the counter gets there
// within microseconds unless the counters were left inconsistent (two launches sharing the
// workspace at once, a launch that was aborted); then this ends the wait instead of hanging.
__device__ __forceinline__ bool wait_counter_bounded(unsigned* counter, unsigned want, unsigned limit)
{
    for (unsigned polls = 0; __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != want; ++polls) {
        if (polls >= limit) return false;
        __builtin_amdgcn_s_sleep(2);
    }
    return true;
}

// the k-blocks of one tile that a workgroup accumulates, and its place among the
// workgroups that share the tile
struct KRange {
    int kb0, kb1, step;         // k-blocks kb0, kb0 + step, ... < kb1
    int part, parts;            // this workgroup's position (k order) and the number of sharers
    size_t slot0;               // partial-sum slot of part 0; part j > 0 has slot_rest + j * slot_step
    size_t slot_rest;
    int slot_step;
    __device__ size_t slot(int j) const { return j == 0 ? slot0 : slot_rest + (size_t)j * slot_step; }
    size_t counter;             // arrival counter of the tile
};

constexpr int kGemmWrittenBase = 32768;   // second half of the counter table: "partial sums written" per tile

// a pointer that every lane of the wave agrees on, in scalar registers
template <typename T>
__device__ __forceinline__ const T* rows_uniform(const T* q)
{
    const uint64_t v = (uint64_t)q;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return (const T*)(((uint64_t)hi << 32) | lo);
}

constexpr int kAStride = 128 + 8;   // halves per LDS row of the A tile (272 B: conflict-free b128 reads)

// The waves of a SIMD run nearly oldest first, so that the last ones end alone, with nobody to fill the cycles that they
// wait.  A wave gives up its priority in three steps over its second half, which lets the ones behind it catch up.
// Grouped launches of 32-row problems, layers of 2048 x 768: 64 tokens x 128 experts 104.8 -> 102.7 us, with popular
// ones 80.2 -> 77.3, 20 tokens 96.0 -> 92.8, 100 tokens x 64 experts 77.2 -> 74.9.  Only where the workgroups there are come
// in one round of four a compute unit, of gate and up together in one and a half, and in fewer with many bits
// (ramp_workgroups): those of a later round start ahead
// of the ones that give way, which end the later (down, traced: 128 tokens x 512 experts of 768x2048, 3760 workgroups, 122 ->
// 133 us, 64 tokens x 160 of 1664x4096, 2500, 195 -> 207, 40 tokens x 64 of 2048x7168, 1790, 148 -> 155; gate and up of
// 128 tokens x 512 experts, 2820, 245 -> 257, but 64 tokens x 512 experts x 512, 1470, 130 -> 122, 40 tokens x 64 of 7168x2048,
// 1020, 295 -> 281).  Not in mixed launches, whose long tiles have to end first (256
// tokens x 512 experts 113.8 -> 115.8), nor dense, which have few waves a SIMD (76 rows of 1152x3584 14.7 -> 14.8).
template <bool ON>
struct PriorityRamp {
    int k2, k1, k0, step;
    __device__ __forceinline__ PriorityRamp(const int kb0, const int kb1, const int step_, const bool on) : step(step_)
    {
        const int n = kb1 - kb0;
        k2 = on ? kb0 + (n >> 1) : kb1;                 // (never reached)
        k1 = on ? kb0 + (n * 3 >> 2) : kb1;
        k0 = on ? kb0 + (n * 7 >> 3) : kb1;
        if constexpr (ON) {
            if (on) __builtin_amdgcn_s_setprio(3);
        }
    }
    // ahead of the k-block kb of kb0, kb0 + step, ...
    __device__ __forceinline__ void at(const int kb) const
    {
        if constexpr (ON) {
            if ((unsigned)(kb - k2) < (unsigned)step) __builtin_amdgcn_s_setprio(2);
            if ((unsigned)(kb - k1) < (unsigned)step) __builtin_amdgcn_s_setprio(1);
            if ((unsigned)(kb - k0) < (unsigned)step) __builtin_amdgcn_s_setprio(0);
        }
    }
    __device__ __forceinline__ void end() const
    {
        if constexpr (ON) __builtin_amdgcn_s_setprio(0);
    }
};

// The k-loop of a 32-row tile, 64 columns from nw on: every wave is on its own.  The A operand of a lane (row
// `slot`, 8 k values) is one 16-byte load straight from the rotated rows, so
// there is no LDS tile and no barrier in the loop.  Trellis and A registers are
// reloaded for the wave's next k-block as soon as a step has consumed them
// (rolling prefetch, one k-block ahead; the activation behind the products that read it: asked for ahead of
// them it lands in other registers and is moved, 16 of the 513 vector instructions of a k-block.  Layers of 64
// and 20 tokens x 128 experts 120.7 -> 118.3 and 106.4 -> 104.3 us); on the last k-block the reload reads
// the same addresses again and is ignored, which keeps the loop free of branches.
// `requested` is called when the first loads are on their way; RAMP: PriorityRamp, where `ramp_on`.
template <int BITS, int CB, bool RAMP, typename F>
__device__ __forceinline__ void accumulate_32_rows(const uint32_t* trellis, const size_t row_dw, const int nw, const _Float16* a_had,
                                                   const int arow, const int K, const int kb0, const int kb1, const int step,
                                                   const int lane, float16_t (&acc)[2], F requested, const bool ramp_on = false)
{
    constexpr int tile_dw = 8 * BITS;
    const int half_id = lane >> 5, slot = lane & 31;
    const global_ptr<const uint32_t> tb = as_global(trellis) + (size_t)half_id * row_dw +
                                         (size_t)((nw >> 4) + (slot >> 3)) * tile_dw + (slot & 7) * BITS;
    const global_ptr<const half8_t> ab =
        (global_ptr<const half8_t>)(as_global(a_had) + (size_t)arow * K + 16 * half_id);
    uint32_t cur[4][BITS];
    half8_t av[4][2];
    {
        const global_ptr<const uint32_t> t0 = tb + (size_t)(kb0 * 8) * row_dw;
        const global_ptr<const half8_t> a0 = ab + kb0 * 16;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            load_tile_dwords<BITS>(t0 + (size_t)(2 * st) * row_dw, cur[st]);
            av[st][0] = a0[4 * st];
            av[st][1] = a0[4 * st + 1];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    requested();
    const PriorityRamp<RAMP> ramp(kb0, kb1, step, ramp_on);
    for (int kb = kb0; kb < kb1; kb += step) {
        ramp.at(kb);
        const int nkb = kb + step < kb1 ? kb + step : kb;
        const global_ptr<const uint32_t> tnx = tb + (size_t)(nkb * 8) * row_dw;
        const global_ptr<const half8_t> anx = ab + nkb * 16;
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            uint32_t prev = fetch_prev(lane, cur[st][BITS - 1]);
            uint32_t w2[16];
            decode_lane<BITS, CB>(cur[st], prev, w2);
            load_tile_dwords<BITS>(tnx + (size_t)(2 * st) * row_dw, cur[st]);
            half8_t b[2][2];
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint4 q = {w2[2 * f + h], w2[4 + 2 * f + h], w2[8 + 2 * f + h], w2[12 + 2 * f + h]};
                    b[f][h] = __builtin_bit_cast(half8_t, q);
                }
            settle<CB>(b[0][0], b[1][0], b[0][1], b[1][1]);
            __builtin_amdgcn_sched_barrier(0);
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[st][0], b[0][0], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[st][0], b[1][0], acc[1], 0, 0, 0);
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[st][1], b[0][1], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[st][1], b[1][1], acc[1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            av[st][0] = anx[4 * st];
            av[st][1] = anx[4 * st + 1];
        }
    }
    ramp.end();
}

// The same for an expert whose rows all fit into sixteen: v_mfma_f32_16x16x32_f16, half the matrix work of the
// products above.  A step is 64 rows of K x 32 columns: lanes l and l + 8 of a sixteen take two neighbouring tiles,
// the four sixteens four tile rows (as in the few-row kernel), and both halves of a wave's columns multiply the
// same activation.  What the matrix units take there the decode does not get, on a pipe of its own or not: a layer of
// 64 tokens x 128 experts, four rows an expert, 126 -> 110 us.  The sums of sixteen rows form in another order
// than those of 32, so that the choice must not depend on how a call cuts its rows into problems: `lone` says that
// the expert has no more rows, in whichever list it is.  Whole K only: launches that cut K (gemm_split) keep the 32-row
// products, whose partial sums they exchange.
// Rows past the problem repeat its last row: zeros there, with the loads of their lanes switched off, cost the
// loop more than the zeros save (that layer 104.2 -> 107.4, of 256 tokens x 512 experts 109.9 -> 112.9).
template <int BITS, int CB, int CG, bool RAMP, typename F>            // CG: column groups of 32 a wave
__device__ __forceinline__ void accumulate_16_rows(const uint32_t* trellis, const size_t row_dw, const int nw, const _Float16* a_had,
                                                   const int arow, const int K, const int lane, float4_t (&acc)[CG][2], F requested,
                                                   const bool ramp_on = false)
{
    constexpr int tile_dw = 8 * BITS;
    const int l16 = lane & 15, lg = lane >> 4;
    const global_ptr<const uint32_t> tb = as_global(trellis) + (size_t)lg * row_dw +
                                         (size_t)((nw >> 4) + (l16 >> 3)) * tile_dw + (l16 & 7) * BITS;
    const global_ptr<const half8_t> ab = (global_ptr<const half8_t>)(as_global(a_had) + (size_t)arow * K + 16 * lg);
    uint32_t cur[2 * CG][BITS];
    half8_t av[2][2];
#pragma unroll
    for (int st = 0; st < 2 * CG; ++st) {
        const int ks = st / CG, cg = st % CG;
        load_tile_dwords<BITS>(tb + (size_t)(4 * ks) * row_dw + cg * 2 * tile_dw, cur[st]);
        if (cg == 0) {
            av[ks][0] = ab[8 * ks];
            av[ks][1] = ab[8 * ks + 1];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    requested();
    const int KB = K >> 7;
    const PriorityRamp<RAMP> ramp(0, KB, 1, ramp_on);
    for (int kb = 0; kb < KB; ++kb) {
        ramp.at(kb);
        const int nkb = min(kb + 1, KB - 1);
        const global_ptr<const uint32_t> tnx = tb + (size_t)(nkb * 8) * row_dw;
        const global_ptr<const half8_t> anx = ab + nkb * 16;
#pragma unroll
        for (int st = 0; st < 2 * CG; ++st) {
            const int ks = st / CG, cg = st % CG;
            uint32_t prev = fetch_prev(lane, cur[st][BITS - 1]);
            uint32_t w2[16];
            decode_lane<BITS, CB>(cur[st], prev, w2);
            load_tile_dwords<BITS>(tnx + (size_t)(4 * ks) * row_dw + cg * 2 * tile_dw, cur[st]);
            half8_t b[2][2];
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint4 q = {w2[2 * f + h], w2[4 + 2 * f + h], w2[8 + 2 * f + h], w2[12 + 2 * f + h]};
                    b[f][h] = __builtin_bit_cast(half8_t, q);
                }
            settle<CB>(b[0][0], b[1][0], b[0][1], b[1][1]);
            __builtin_amdgcn_sched_barrier(0);
            acc[cg][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[ks][0], b[0][0], acc[cg][0], 0, 0, 0);
            acc[cg][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[ks][0], b[1][0], acc[cg][1], 0, 0, 0);
            acc[cg][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[ks][1], b[0][1], acc[cg][0], 0, 0, 0);
            acc[cg][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[ks][1], b[1][1], acc[cg][1], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (cg == CG - 1) {
                av[ks][0] = anx[8 * ks];
                av[ks][1] = anx[8 * ks + 1];
            }
        }
    }
    ramp.end();
}
// its sums to the fp32 tile, 32 * CG columns from z on
template <int STRIDE, int CG>
__device__ __forceinline__ void stage_16_rows(float* z, const float4_t (&acc)[CG][2], const int lane)
{
    float* const at = z + 4 * (lane >> 4) * STRIDE + ((lane >> 3) & 1) * 16 + (lane & 7);
#pragma unroll
    for (int cg = 0; cg < CG; ++cg)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 4; ++r) at[r * STRIDE + 32 * cg + 8 * f] = acc[cg][f][r];
}

// one output tile: rows of problem / row block `tile_y`, 256 columns
// MB = 32-row blocks per workgroup; DENSE: never a problem list; SCALAR: the weights' pointer in scalar registers;
// RAMP: PriorityRamp in tiles of up to 32 rows
template <int BITS, int CB, int MB, bool DENSE, bool SCALAR = false, bool RAMP = false>
__device__ __forceinline__ void gemm_tile(const GemmParams& p, const int tile_y, const int nblk, const KRange kr,
                                          const int which, unsigned char* smem, const GroupProblem* problems = nullptr,
                                          const bool ramp_on = false)
{
    constexpr int BM = MB * 32;
    _Float16* a_tile = (_Float16*)smem;                 // [2][BM][kAStride]
    float* z_tile = (float*)smem;                       // epilogue: [32][256 + 4]
    constexpr int kZStride = 256 + 4;
    __shared__ unsigned s_last;

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int half_id = lane >> 5;                      // which of the two tile rows
    const int slot = lane & 31;                         // MFMA row / column slot
    int m0 = tile_y * BM;
    int m_end = p.M;
    ExpertLin lin = p.lin;
    const _Float16* a_had = p.a_had[0];
    void* cout = p.c[0];
    int N = p.N, ldc = p.N, nblk_lin = nblk;
    const int32_t* a_rows = nullptr;
    bool lone = false;                                  // accumulate_16_rows (whole K)
    if constexpr (DENSE) {
        const TileView v = dense_tile_view(p, nblk);
        if (v.empty) return;                            // the same for every workgroup that shares the tile
        lin = v.lin;
        a_had = v.a_had;
        cout = v.cout;
        N = v.N;
        ldc = v.ldc;
        nblk_lin = v.nblk;
    }
    const int n0 = nblk_lin * 256;
    if constexpr (!DENSE) {
        // (dynamic indexing of the parameter block: kept out of the dense instantiations, where
        // it would force the whole block into private memory)
        const GroupProblem gp = problems[tile_y];
        lin = gp.expert == p.shared_expert ? p.shared[p.lin_base + which]
                                           : p.experts[gp.expert * p.lins_per_expert + p.lin_base + which];
        m0 = gp.row0;
        m_end = gp.row0 + gp.nrows;
        a_had = p.a_had[which];
        cout = p.c[which];
        if (gp.expert != p.shared_expert) a_rows = p.a_rows;
        lone = MB == 1 && gp.lone && kr.parts == 1;
    }
    // row r of the tile in a_had
    auto a_row_at = [&](int r) { return !DENSE && a_rows ? as_global(a_rows)[m0 + r] : m0 + r; };
    const int rows_here = min(BM, m_end - m0);          // >= 1
    const int nw = n0 + wave * 64;                      // first column of this wave
    const bool active = nw < N;
    const int tn = ldc >> 4;                            // tiles per tile row of the weight (of the whole weight, for a slice)
    constexpr int tile_dw = 8 * BITS;
    const size_t row_dw = (size_t)tn * tile_dw;
    const int KB = p.K >> 7;
    // The output scales of a problem's tile, eight columns a thread: asked for ahead of the operands and kept in
    // LDS.  They come from memory, and the end of the tile waited for them: layer of 64 tokens x 128 experts
    // 121.4 -> 119.5 us, whose workgroups all end together.  (Dense tiles ask for them at the end: with
    // few tiles a head that waits costs more, 76 rows of 1152x3584 15.0 -> 15.4 us, 317 of 2944x8320 47.5 -> 48.5.)
    __shared__ __align__(16) half8_t s_scale[32];
    half8_t scale_mine = {0, 0, 0, 0, 0, 0, 0, 0};
    if (!DENSE && threadIdx.x < 32 && n0 + 8 * (int)threadIdx.x < N)
        scale_mine = ((global_ptr<const half8_t>)as_global(lin.svh + n0))[threadIdx.x];
    auto keep_scale = [&]() {
        if (!DENSE && threadIdx.x < 32) s_scale[threadIdx.x] = scale_mine;
    };

    float16_t acc[MB][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][f][r] = 0.0f;

    // (the list of linears is read as vectors: the pointer would be two of a lane's registers through the loop)
    const uint32_t* const trellis = SCALAR ? rows_uniform(lin.trellis) : lin.trellis;
    float4_t acc16[2][2] = {};
    if (lone) {
        if (active)
            accumulate_16_rows<BITS, CB, 2, RAMP>(trellis, row_dw, nw, a_had, a_row_at(min(lane & 15, rows_here - 1)), p.K, lane, acc16, keep_scale, ramp_on);
        else keep_scale();
    } else if constexpr (MB == 1) {
        if (active && kr.kb0 < kr.kb1)
            accumulate_32_rows<BITS, CB, RAMP>(trellis, row_dw, nw, a_had, a_row_at(min(slot, rows_here - 1)), p.K, kr.kb0, kr.kb1,
                                         kr.step, lane, acc[0], keep_scale, ramp_on);      // (rows past the problem repeat its last row)
        else keep_scale();
    } else {
        // lane's trellis position inside a k-block: tile row 2*step + half_id, tile (nw/16 + slot/8)
        const uint32_t* tbase = lin.trellis + (size_t)half_id * row_dw +
                                (size_t)((nw >> 4) + (slot >> 3)) * tile_dw + (slot & 7) * BITS;

        // Operands run ahead in registers: this thread's share of the next k-block's A tile
        // (a_nxt, 32 bytes per 256-thread pass; the tile is double-buffered in LDS, so a
        // k-block costs one barrier) and the trellis dwords of the wave's four steps (ring),
        // each reloaded for the next k-block as soon as its step is decoded.
        //
        // A step's 32 weights per lane are 16 pairs; the even pairs are the B operands for
        // k 0..7 of each lane's 16 (A operand a0), the odd pairs those for k 8..15 (a1).  The
        // loop runs in half-steps: the eight MFMAs of one half are issued two at a time, and
        // behind every two a quarter of the decode of the NEXT half (the odd pairs of the same
        // step, or the even pairs of the next step, which across the barrier is step 0 of the
        // next k-block), so the vector pipe decodes while the matrix pipe multiplies.  Row
        // blocks past the end of the rows are multiplied too (their A rows are zero): the loop
        // has no branch.  The order is given to the scheduler as groups after each half-step.
        constexpr int kAPasses = BM * 8 / 256;
        uint32_t ring[4][BITS];
        u32x4_t a_nxt[kAPasses][2];
        const int a_row = threadIdx.x >> 3, a_ch = threadIdx.x & 7;       // + 32 rows per pass
        int a_at[kAPasses];
        if constexpr (!DENSE) {
    #pragma unroll
            for (int ps = 0; ps < kAPasses; ++ps) a_at[ps] = a_row_at(min(a_row + 32 * ps, rows_here - 1));
        }
        auto load_a = [&](int kb) {
    #pragma unroll
            for (int ps = 0; ps < kAPasses; ++ps) {
                const int r = a_row + 32 * ps;
                u32x4_t v0 = {0, 0, 0, 0}, v1 = {0, 0, 0, 0};
                if (m0 + r < m_end) {
                    const global_ptr<const u32x4_t> src = (global_ptr<const u32x4_t>)(
                        as_global(a_had) + (size_t)(DENSE ? m0 + r : a_at[ps]) * p.K + kb * 128 + a_ch * 16);
                    v0 = src[0];
                    v1 = src[1];
                }
                a_nxt[ps][0] = v0;
                a_nxt[ps][1] = v1;
            }
        };
        auto load_b_step = [&](int kb, int st) {
            const global_ptr<const uint32_t> nb = as_global(tbase) + (size_t)(kb * 8 + 2 * st) * row_dw;
    #pragma unroll
            for (int j = 0; j < BITS; ++j) ring[st][j] = nb[j];
        };
        // the eight pairs of one half, numbered j = 4f + q: out[f][q] = pair 4q + 2f + h
        auto decode_pairs = [&](const LaneWindows<BITS>& w, int h, int j0, int n, uint32_t (&out)[2][4]) {
    #pragma unroll
            for (int j = j0; j < j0 + n; ++j) {
                const int f = j >> 2, q = j & 3;
                const int pr = 4 * q + 2 * f + h;
                out[f][q] = decode_pair<CB>(w.state(2 * pr), w.state(2 * pr + 1));
            }
        };
        uint32_t b_half[2][2][4];                       // [which half-step buffer][f][q]
        LaneWindows<BITS> win;
        if (kr.kb0 < kr.kb1) {
            load_a(kr.kb0);
            if (active) {
    #pragma unroll
                for (int st = 0; st < 4; ++st) load_b_step(kr.kb0, st);
                win = LaneWindows<BITS>(ring[0], fetch_prev(lane, ring[0][BITS - 1]));
                decode_pairs(win, 0, 0, 8, b_half[0]);
                settle<CB>(b_half[0][0]);
            }
        }
        keep_scale();

        int buf = 0;
        for (int kb = kr.kb0; kb < kr.kb1; kb += kr.step, buf ^= 1) {
            // publish this k-block's A tile; the other buffer may still be read by slower waves
            _Float16* a_buf = a_tile + (size_t)buf * BM * kAStride;
    #pragma unroll
            for (int ps = 0; ps < kAPasses; ++ps) {
                u32x4_t* dst = (u32x4_t*)(a_buf + (a_row + 32 * ps) * kAStride + a_ch * 16);
                dst[0] = a_nxt[ps][0];
                dst[1] = a_nxt[ps][1];
            }
            // the next k-block (on the last one the same again: read and ignored, no branch)
            const int nkb = kb + kr.step < kr.kb1 ? kb + kr.step : kb;
            load_a(nkb);
            __syncthreads();

            if (active) {
                const _Float16* a_lane = a_buf + slot * kAStride + 16 * half_id;
                // A operand of half-step hs = 2 * st + h, row block mb: k = 32 * st + 16 * half_id + 8 * h .. + 7 of the k-block
                auto a_operand = [&](int hs, int mb) {
                    return *(const half8_t*)(a_lane + mb * 32 * kAStride + 32 * (hs >> 1) + 8 * (hs & 1));
                };
                half8_t a_op = a_operand(0, 0);
    #pragma unroll
                for (int hs = 0; hs < 8; ++hs) {
                    const int st = hs >> 1, h = hs & 1;
                    __builtin_amdgcn_sched_barrier(0);
                    uint32_t (&b_cur)[2][4] = b_half[h];
                    uint32_t (&b_nx)[2][4] = b_half[h ^ 1];
                    half8_t b0 = __builtin_bit_cast(half8_t, uint4{b_cur[0][0], b_cur[0][1], b_cur[0][2], b_cur[0][3]});
                    half8_t b1 = __builtin_bit_cast(half8_t, uint4{b_cur[1][0], b_cur[1][1], b_cur[1][2], b_cur[1][3]});
                    if (h == 1) {
                        // the step after this one: its windows, then (below) its even pairs
                        const int ns = (st + 1) & 3;
                        win = LaneWindows<BITS>(ring[ns], fetch_prev(lane, ring[ns][BITS - 1]));
                    }
    #pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        const half8_t a_now = a_op;
                        if (mb + 1 < MB) a_op = a_operand(hs, mb + 1);
                        else if (hs < 7) a_op = a_operand(hs + 1, 0);
                        acc[mb][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_now, b0, acc[mb][0], 0, 0, 0);
                        if (mb == 0) settle<CB>(b1);
                        acc[mb][1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_now, b1, acc[mb][1], 0, 0, 0);
                        decode_pairs(win, h ^ 1, mb * 8 / MB, (mb + 1) * 8 / MB - mb * 8 / MB, b_nx);
                        if ((mb + 1) * 8 / MB >= 4 && mb * 8 / MB < 4) settle<CB>(b_nx[0]);
                    }
                    // the step's dwords are decoded once its odd pairs exist: request the next k-block's
                    if (h == 0) load_b_step(nkb, st);
    #define BERTH_GEMM_CHUNK(valu0, valu1)                                              \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                              \
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                              \
        __builtin_amdgcn_sched_group_barrier(0x002, valu0, 0);                          \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                              \
        __builtin_amdgcn_sched_group_barrier(0x002, valu1, 0);
                    // (the decode of a half-step spread over its 2 * MB MFMAs)
                    static_assert(MB >= 2 && MB <= 4, "the groups below describe four to eight MFMAs per half-step");
                    if constexpr (MB == 4) {
                        BERTH_GEMM_CHUNK(9, 9) BERTH_GEMM_CHUNK(9, 9) BERTH_GEMM_CHUNK(9, 9) BERTH_GEMM_CHUNK(9, 9)
                    } else if constexpr (MB == 3) {
                        BERTH_GEMM_CHUNK(12, 12) BERTH_GEMM_CHUNK(12, 12) BERTH_GEMM_CHUNK(12, 12)
                    } else {
                        BERTH_GEMM_CHUNK(18, 18) BERTH_GEMM_CHUNK(18, 18)
                    }
    #undef BERTH_GEMM_CHUNK
                }
            }
        }

    }

    // ---- split-K handoff.  Register r of a lane holds tile row 8*(r/4) + 4*half_id + r%4,
    // so only registers with 8*(r/4) < rows matter.
    if (kr.parts > 1) {
        // Arrive first.  The last workgroup to arrive finishes the tile: it waits until the
        // others have written their partial sums (they bump the tile's second counter after
        // their stores; a workgroup that has arrived is running and depends on nothing, so
        // the wait is short and cannot block) and adds the parts in k order.  If it holds
        // part 0 itself it starts from its registers and never writes them out.
        constexpr size_t kPerWg = (size_t)4 * MB * 2 * 16 * 64;
        unsigned* arrived = p.counters + kr.counter * p.cstride;
        unsigned* written = arrived + kGemmWrittenBase;
        if (threadIdx.x == 0) {
            unsigned old = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_last = (old == (unsigned)(kr.parts - 1)) ? 1u : 0u;
        }
        __syncthreads();
        const bool finisher = s_last != 0;
        const float* all = p.partials + (size_t)wave * MB * 2 * 16 * 64;
        if (!(finisher && kr.part == 0)) {
            float* mine = p.partials + kr.slot(kr.part) * kPerWg + (size_t)wave * MB * 2 * 16 * 64;
            if (active) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int f = 0; f < 2; ++f)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (mb * 32 + 8 * (r >> 2) < rows_here)
                                __hip_atomic_store(mine + ((mb * 2 + f) * 16 + r) * 64 + lane, acc[mb][f][r],
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (!finisher) {
            wait_own_stores();
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            __syncthreads();
            if (threadIdx.x == 0) __hip_atomic_fetch_add(written, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        if (threadIdx.x == 0) {
            const bool complete = wait_counter_bounded(written, (unsigned)(kr.parts - 1), p.spin_limit);
            __hip_atomic_store(written, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(arrived, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (!complete && p.fault)
                __hip_atomic_store(p.fault, 1u + (unsigned)kr.counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            s_last = complete ? 1u : 2u;
        }
        __syncthreads();
        if (s_last == 2u) return;       // gave up: the tile stays unwritten, the host is told
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (active) {
            // part 0 first (from memory unless it is this workgroup's own), then parts 1, 2, ...
            // added in order.  64 (128-row tiles), 128 (32-row tiles) or, for problems, 64 loads a lane are in
            // flight at a time: half of a part's register blocks, or four or two whole parts.
            constexpr int kGroup = MB & 1 ? 2 : 4;              // (mb, f) register blocks per batch
            constexpr int kParts = MB > 1 ? 1 : DENSE ? 4 : 2;  // parts per batch
            const int first = kr.part == 0 ? 1 : 0;
            for (int j0 = first; j0 < kr.parts; j0 += kParts) {
#pragma unroll
                for (int g0 = 0; g0 < MB * 2; g0 += kGroup) {
                    float tmp[kParts][kGroup][16];
#pragma unroll
                    for (int jj = 0; jj < kParts; ++jj) {
                        const int j = j0 + jj < kr.parts ? j0 + jj : kr.parts - 1;      // past the end: ignored
                        const float* src = all + kr.slot(j) * kPerWg;
#pragma unroll
                        for (int b = 0; b < kGroup; ++b) {
                            const int blk = g0 + b;             // = mb * 2 + f
                            if ((blk >> 1) * 32 >= rows_here) continue;                 // workgroup-uniform
#pragma unroll
                            for (int r = 0; r < 16; ++r)
                                tmp[jj][b][r] = __hip_atomic_load(src + (blk * 16 + r) * 64 + lane, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
#pragma unroll
                    for (int jj = 0; jj < kParts; ++jj) {
                        if (j0 + jj >= kr.parts) break;
#pragma unroll
                        for (int b = 0; b < kGroup; ++b) {
                            const int blk = g0 + b;
                            if ((blk >> 1) * 32 >= rows_here) continue;
#pragma unroll
                            for (int r = 0; r < 16; ++r)
                                acc[blk >> 1][blk & 1][r] =
                                    j0 + jj == 0 ? tmp[jj][b][r] : acc[blk >> 1][blk & 1][r] + tmp[jj][b][r];
                        }
                    }
                }
            }
        }
    }

    // ---- epilogue, 32 rows at a time: stage fp32 tile, output Hadamard, svh, store
    const int col_in_wave = (slot >> 3) * 16 + (slot & 7);     // + 8f
    // output scales: a lane of the epilogue owns columns 8 * had_chunk(lane) .. + 7 of a block
    const int chunk = had_chunk(lane);
    half8_t sv_blk[2];
    if constexpr (DENSE) {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const int gn = n0 + blk * 128;
            sv_blk[blk] = gn < N ? ((global_ptr<const half8_t>)as_global(lin.svh + gn))[chunk] : half8_t{0, 0, 0, 0, 0, 0, 0, 0};
        }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb * 32 >= rows_here) break;                        // workgroup-uniform
        __syncthreads();
        if (lone) {
            if (active) stage_16_rows<kZStride>(z_tile + wave * 64, acc16, lane);
        } else if (active) {
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = 8 * (r >> 2) + 4 * half_id + (r & 3);
                    z_tile[row * kZStride + wave * 64 + col_in_wave + 8 * f] = acc[mb][f][r];
                }
        }
        __syncthreads();
        const int rows_blk = min(32, rows_here - mb * 32);
        // 64 vectors (32 rows x 2 column blocks); a wave rotates four per pass, sixteen lanes each.  Grouped tiles of
        // several blocks take two passes at a time: exl3_gemm_mixed_kernel, which holds every kind of them, was 138 KB
        // long with four (4 bits, 3INST) and needed indirect branches, which reach further than 128 KB
        constexpr int kPasses = DENSE || MB == 1 ? 4 : 2;
#pragma unroll kPasses
        for (int pass = 0; pass < 4; ++pass) {
            const int vec = pass * 16 + wave * 4 + (lane >> 4);
            const int row = vec >> 1, blk = vec & 1;
            const int gn = n0 + blk * 128;
            if (row < rows_blk && gn < N) {
                float v[8];
                const float4_t* zp = (const float4_t*)&z_tile[row * kZStride + blk * 128 + 8 * chunk];
                const float4_t z0 = zp[0], z1 = zp[1];
#pragma unroll
                for (int i = 0; i < 4; ++i) { v[i] = z0[i]; v[4 + i] = z1[i]; }
                const float unit = had128_row16(v, lane) * kRsqrt128;
                const half8_t sv = !DENSE ? s_scale[blk * 16 + chunk] : blk ? sv_blk[1] : sv_blk[0];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = had_scale(v[i], unit) * (float)sv[i];
                const size_t at = (size_t)(m0 + mb * 32 + row) * ldc + gn + 8 * chunk;
                if (p.out_fp32) {
                    if (p.out_add) {
                        const global_ptr<const float4_t> add = (global_ptr<const float4_t>)(as_global(p.out_add) + at);
                        const float4_t a0 = add[0], a1 = add[1];
#pragma unroll
                        for (int i = 0; i < 4; ++i) { v[i] += a0[i]; v[4 + i] += a1[i]; }
                    }
                    global_ptr<float4_t> dst = (global_ptr<float4_t>)(as_global((float*)cout) + at);
                    dst[0] = float4_t{v[0], v[1], v[2], v[3]};
                    dst[1] = float4_t{v[4], v[5], v[6], v[7]};
                } else {
                    half8_t o;
#pragma unroll
                    for (int i = 0; i < 8; ++i) o[i] = (_Float16)v[i];
                    *(global_ptr<half8_t>)(as_global((_Float16*)cout) + at) = o;
                }
            }
        }
    }
}

// Grouped launches.  Workgroup i runs on die i % 8, and every die has its own L2: the column blocks of one
// problem and linear, which read the same rows, go to one die, one after the other.  Of the grid
// (8 * column blocks, groups / 8) blockIdx.x % 8 and blockIdx.y name the group (problem-major, then the
// launch's one or two linears, so that the few real problems come ahead of the empty tail of the list)
// and blockIdx.x / 8 the column block.  1500 tokens through 128 experts of 2048 x 768: 283 -> 275 us against column
// blocks spread over the dies, whose rows every L2 then read for itself.
struct GroupTile {
    int col, which, problem;
};
__device__ __forceinline__ GroupTile group_tile(const GemmParams& p)
{
    const int g = (int)blockIdx.y * 8 + ((int)blockIdx.x & 7);
    const int two = p.group_lins - 1;                   // 0 or 1
    return {(int)blockIdx.x >> 3, g & two, g >> two};
}
inline dim3 group_grid(int cols, int lins, int problems)
{
    return dim3((unsigned)(8 * cols), (unsigned)((lins * problems + 7) / 8));
}

// Dense launches: blockIdx.x = (tile - tile0) * S + split with tiles numbered row
// block by row block, so that one linear can be issued as several launches with
// different split factors.  Grouped launches: group_tile, a "column block" being one of S parts of it.
//
// 32-row problems: up to four workgroups on a compute unit (with four parts in flight at the end of a
// split tile it was 173 registers a lane and two of them, so that the 756 workgroups of 64 tokens x 128
// experts ran in two rounds: layer 125.6 -> 122.6 us).  The launch bound keeps 3INST and MCG there as well, whose
// kernels of 3 and 4 bits had 130..132 registers with both row forms in them: the same time with three workgroups as with
// four (64 tokens x 128 experts MCG 110.8 -> 109.1 and 111.0 -> 107.8 us at 4 and 3 bits, runs of one side 4 and 8 % apart,
// 3INST 122.4 -> 122.6 and 120.0 -> 120.5).  8 bits take three, four would need scratch.  MUL1 is below 128 up to 6 bits
// without the bound, and the schedule that the bound gives costs it 0.4 to 0.7 % (150 and 300 tokens x 128 experts 120.5 ->
// 121.4 and 141.7 -> 142.6).
template <int BITS, int CB, int MB, bool DENSE = true>
__global__ __launch_bounds__(256, MB > 1 || DENSE ? 2 : CB != 2 && BITS < 8 ? 4 : 3) void exl3_gemm_kernel(GemmParams p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const GroupTile gt = DENSE ? GroupTile{(int)blockIdx.x, 0, 0} : group_tile(p);
    const int unit = gt.col / p.S;
    const int split = gt.col - unit * p.S;
    const int nblocks = ((p.N + 255) >> 8) * (p.num_slices > 0 ? p.num_slices : 1);
    KRange kr;
    kr.kb0 = split;
    kr.kb1 = p.K >> 7;
    kr.step = p.S;
    kr.slot_step = 1;
    kr.part = split;
    kr.parts = p.S;
    if constexpr (DENSE) {
        const int tile = p.tile0 + unit;
        kr.counter = (size_t)unit;
        kr.slot0 = kr.slot_rest = kr.counter * p.S;
        gemm_tile<BITS, CB, MB, true>(p, tile / nblocks, tile % nblocks, kr, 0, smem);
    } else {
        const int problems = *p.num_problems;
        if (gt.problem >= problems) return;
        // grouped: (linear, problem, column block)
        kr.counter = ((size_t)gt.which * p.tiles_y + gt.problem) * nblocks + unit;
        kr.slot0 = kr.slot_rest = kr.counter * p.S;
        gemm_tile<BITS, CB, MB, false, CB != 2, true>(p, gt.problem, unit, kr, gt.which, smem, p.problems, problems <= p.ramp_problems);
    }
}

// Gate and up of a list of problems of up to 32 rows, and the input of their down projections: waves 0
// and 1 take 128 columns of gate, waves 2 and 3 the same columns of up, so that the workgroup holds both
// factors of silu(g) * u and a whole block of the next rotation when its k-loops end.  The grid is
// group_tile's of one linear; linears lin_base, lin_base + 1 and, for its input scales,
// lin_base + 2 of an expert.  Gate and up are written too (fp16, c[0] and c[1]).
// The values are those of the 32-row tiles and of moe_had_rows_kernel behind them.
// What bounds it: the decode, as there (experts of up to sixteen rows: accumulate_16_rows); the end of a row is three rotations (of 128 values by sixteen
// lanes) instead of two, against a launch that reads both factors back: layer of 64 tokens x 128 experts
// x 768 122.6 -> 121.4 us, of 20 tokens x 128 experts x 896 (seven column blocks, which 256-column tiles
// cover as eight) 107 -> 94.  The launch bound: exl3_gemm_kernel's.
template <int BITS, int CB>
__global__ __launch_bounds__(256, CB != 2 ? 4 : 3) void exl3_gemm_pair_kernel(GemmParams p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const GroupTile gt = group_tile(p);
    const int problems = *p.num_problems;
    if (gt.problem >= problems) return;
    const bool ramp_on = problems <= p.ramp_problems;
    constexpr int kZStride = 256 + 4;
    float* const z_tile = (float*)smem;                 // [32][kZStride]: gate's 128 columns, up's
    const int lane = threadIdx.x & 63, slot = lane & 31, half_id = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int which = wave >> 1;
    const int n0 = gt.col * 128;
    const GroupProblem gp = p.problems[gt.problem];
    const bool shared = gp.expert == p.shared_expert;
    auto linear = [&](int l) { return shared ? p.shared[p.lin_base + l] : p.experts[gp.expert * p.lins_per_expert + p.lin_base + l]; };
    const ExpertLin lin = linear(which);
    const int rows = gp.nrows;
    int arow = gp.row0 + min(gp.lone ? slot & 15 : slot, rows - 1);   // rows past the problem repeat its last row
    if (p.a_rows && !shared) arow = as_global(p.a_rows)[arow];

    // the output scales of gate and up, the input scales of down: asked for first, as in gemm_tile
    __shared__ __align__(16) half8_t s_scale[3][16];
    half8_t scale_mine = {0, 0, 0, 0, 0, 0, 0, 0};
    if (threadIdx.x < 48) {
        const ExpertLin l = linear((int)threadIdx.x >> 4);
        scale_mine = ((global_ptr<const half8_t>)as_global((threadIdx.x < 32 ? l.svh : l.suh) + n0))[threadIdx.x & 15];
    }
    const size_t row_dw = (size_t)(p.N >> 4) * (8 * BITS);
    const int nw = n0 + (wave & 1) * 64;
    auto keep_scale = [&]() {
        if (threadIdx.x < 48) s_scale[threadIdx.x >> 4][threadIdx.x & 15] = scale_mine;
    };
    // sixteen lanes a row, eight columns of both factors each
    const int chunk = had_chunk(lane);
    const int at = n0 + 8 * chunk;
    if (gp.lone) {
        float4_t acc[2][2] = {};
        accumulate_16_rows<BITS, CB, 2, true>(lin.trellis, row_dw, nw, p.a_had[which], arow, p.K, lane, acc, keep_scale, ramp_on);
        stage_16_rows<kZStride>(z_tile + wave * 64, acc, lane);
    } else {
        float16_t acc[2];
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[f][r] = 0.0f;
        accumulate_32_rows<BITS, CB, true>(lin.trellis, row_dw, nw, p.a_had[which], arow, p.K, 0, p.K >> 7, 1, lane, acc, keep_scale, ramp_on);
        const int col = wave * 64 + (slot >> 3) * 16 + (slot & 7);
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) z_tile[(8 * (r >> 2) + 4 * half_id + (r & 3)) * kZStride + col + 8 * f] = acc[f][r];
    }
    __syncthreads();
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const int row = pass * 16 + wave * 4 + (lane >> 4);
        if (row >= rows) break;
        const size_t out = (size_t)(gp.row0 + row) * p.N + at;
        half8_t gu[2];
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            const float4_t* const zp = (const float4_t*)&z_tile[row * kZStride + l * 128 + (at - n0)];
            const float4_t z0 = zp[0], z1 = zp[1];
            float v[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
            const float unit = had128_row16(v, lane) * kRsqrt128;
#pragma unroll
            for (int i = 0; i < 8; ++i) gu[l][i] = (_Float16)rounded(had_scale(v[i], unit) * (float)s_scale[l][chunk][i]);
            *(global_ptr<half8_t>)(as_global((_Float16*)p.c[l]) + out) = gu[l];
        }
        half8_t x;
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = silu_mul_h(gu[0][i], gu[1][i]);
        float v[8];
        mul_half8(x, s_scale[2][chunk], v);
        const float unit = had128_row16(v, lane) * kRsqrt128;
        half8_t o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = (_Float16)had_scale(v[i], unit);
        *(global_ptr<half8_t>)(as_global(p.act_had) + out) = o;
    }
}

// Rows 32 * mb .. + 31 of a problem, 128 columns from n0 on: from the fp32 tile through the output rotation to the output.
constexpr int kHalfZStride = 128 + 4;
__device__ __forceinline__ void finish_half_rows(const GemmParams& p, const GroupProblem gp, const int which, const int n0, const int mb,
                                                 const float* z_tile, const half8_t* s_scale)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, chunk = had_chunk(lane);
    // 32 vectors; a wave rotates four per pass, sixteen lanes each
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const int row = pass * 16 + wave * 4 + (lane >> 4);
        if (mb * 32 + row >= gp.nrows) continue;
        const float4_t* zp = (const float4_t*)&z_tile[row * kHalfZStride + 8 * chunk];
        const float4_t z0 = zp[0], z1 = zp[1];
        float v[8] = {z0.x, z0.y, z0.z, z0.w, z1.x, z1.y, z1.z, z1.w};
        const float unit = had128_row16(v, lane) * kRsqrt128;
        const half8_t sv = s_scale[chunk];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = had_scale(v[i], unit) * (float)sv[i];
        const size_t at = (size_t)(gp.row0 + mb * 32 + row) * p.N + n0 + 8 * chunk;
        if (p.out_fp32) {
            global_ptr<float4_t> dst = (global_ptr<float4_t>)(as_global((float*)p.c[which]) + at);
            dst[0] = float4_t{v[0], v[1], v[2], v[3]};
            dst[1] = float4_t{v[4], v[5], v[6], v[7]};
        } else {
            half8_t o;
#pragma unroll
            for (int i = 0; i < 8; ++i) o[i] = (_Float16)v[i];
            *(global_ptr<half8_t>)(as_global((_Float16*)p.c[which]) + at) = o;
        }
    }
}

// One tile of a problem, 128 columns from n0 on, whole K: half of what gemm_tile's workgroup does, for launches of
// few tiles.  A wave owns 32 columns instead of 64, so
// that its 64 lanes decode four tile rows of a k-block at a time instead of two: lane bits 4 and 5 name the
// tile row (bit 5: which of the step's two, as in gemm_tile; bit 4: which step), and v_permlane16_swap_b32 trades
// the columns u + 8 of the first step's lanes for the columns u of the second's.  The matrix instructions get
// the same k values in the same order as gemm_tile's, so the sums are the same bits; column slots map to columns
// 16 * (slot / 8 % 2) + slot % 8 + 8 * (slot / 16).
// Bound by the decode and the multiplications, which a wave that is alone on its SIMD does one after the other.  The
// trades are 16 of the 270 vector instructions of a k-block, and every A operand is read from LDS
// for one multiplication instead of two.
template <int BITS, int CB, int MB>
__device__ __forceinline__ void gemm_half_tile(const GemmParams& p, const GroupProblem gp, const int which, const int n0, unsigned char* smem)
{
    constexpr int BM = MB * 32;
    _Float16* a_tile = (_Float16*)smem;                 // [2][BM][kAStride]
    float* z_tile = (float*)smem;                       // epilogue: [32][kHalfZStride]
    if (n0 >= p.N) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int half_id = lane >> 5, slot = lane & 31;
    const bool shared = gp.expert == p.shared_expert;
    const ExpertLin lin = shared ? p.shared[p.lin_base + which] : p.experts[gp.expert * p.lins_per_expert + p.lin_base + which];
    const int rows_here = gp.nrows;
    constexpr int tile_dw = 8 * BITS;
    const size_t row_dw = (size_t)(p.N >> 4) * tile_dw;
    const int KB = p.K >> 7;

    __shared__ __align__(16) half8_t s_scale[16];
    half8_t scale_mine = {0, 0, 0, 0, 0, 0, 0, 0};
    if (threadIdx.x < 16) scale_mine = ((global_ptr<const half8_t>)as_global(lin.svh + n0))[threadIdx.x];

    float16_t acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][r] = 0.0f;

    const global_ptr<const uint32_t> tbase = as_global(lin.trellis) + (size_t)(half_id + 2 * ((lane >> 4) & 1)) * row_dw +
                                             (size_t)((n0 >> 4) + 2 * wave + ((lane >> 3) & 1)) * tile_dw + (lane & 7) * BITS;
    uint32_t ring[2][BITS];                             // tile rows 0..3 and 4..7 of a k-block
    u32x4_t a_nxt[MB][2];
    const int a_row = threadIdx.x >> 3, a_ch = threadIdx.x & 7;           // + 32 rows per pass
    global_ptr<const u32x4_t> a_src[MB];
#pragma unroll
    for (int ps = 0; ps < MB; ++ps) {
        int r = gp.row0 + min(a_row + 32 * ps, rows_here - 1);            // rows past the problem repeat its last row
        if (p.a_rows && !shared) r = as_global(p.a_rows)[r];
        a_src[ps] = (global_ptr<const u32x4_t>)(as_global(p.a_had[which]) + (size_t)r * p.K + a_ch * 16);
    }
    auto load_a = [&](int kb) {
#pragma unroll
        for (int ps = 0; ps < MB; ++ps) {
            a_nxt[ps][0] = a_src[ps][kb * 16];
            a_nxt[ps][1] = a_src[ps][kb * 16 + 1];
        }
    };
    auto load_b = [&](int kb, int d) { load_tile_dwords<BITS>(tbase + (size_t)(kb * 8 + 4 * d) * row_dw, ring[d]); };
    // pairs j0 .. j0 + n - 1 of half h, numbered j = 4f + q: out[f][q] = pair 4q + 2f + h
    auto decode_pairs = [&](const LaneWindows<BITS>& w, int h, int j0, int n, uint32_t (&out)[2][4]) {
#pragma unroll
        for (int j = j0; j < j0 + n; ++j) {
            const int f = j >> 2, q = j & 3;
            const int pr = 4 * q + 2 * f + h;
            out[f][q] = decode_pair<CB>(w.state(2 * pr), w.state(2 * pr + 1));
        }
    };
    // [column half][q] of a lane's own step -> [step][q] of its own column half
    auto trade = [&](uint32_t (&b)[2][4]) {
        asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %4\n\tv_permlane16_swap_b32 %1, %5\n\t"
            "v_permlane16_swap_b32 %2, %6\n\tv_permlane16_swap_b32 %3, %7\n\ts_nop 1"
            : "+v"(b[0][0]), "+v"(b[0][1]), "+v"(b[0][2]), "+v"(b[0][3]), "+v"(b[1][0]), "+v"(b[1][1]), "+v"(b[1][2]), "+v"(b[1][3]));
    };
    uint32_t b[2][2][2][4];                             // [two steps' buffer][h][step][q]
    load_a(0);
    load_b(0, 0);
    load_b(0, 1);
    LaneWindows<BITS> win(ring[0], fetch_prev(lane, ring[0][BITS - 1]));
    load_b(min(1, KB - 1), 0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        decode_pairs(win, h, 0, 8, b[0][h]);
        trade(b[0][h]);
    }
    if (threadIdx.x < 16) s_scale[threadIdx.x] = scale_mine;

    int buf = 0;
    for (int kb = 0; kb < KB; ++kb, buf ^= 1) {
        _Float16* a_buf = a_tile + (size_t)buf * BM * kAStride;
#pragma unroll
        for (int ps = 0; ps < MB; ++ps) {
            u32x4_t* dst = (u32x4_t*)(a_buf + (a_row + 32 * ps) * kAStride + a_ch * 16);
            dst[0] = a_nxt[ps][0];
            dst[1] = a_nxt[ps][1];
        }
        load_a(min(kb + 1, KB - 1));                    // on the last one the same again: read and ignored
        __syncthreads();
        const _Float16* a_lane = a_buf + slot * kAStride + 16 * half_id;
        // A operand of half-step hs = 2 * st + h, row block mb: k = 32 * st + 16 * half_id + 8 * h .. + 7 of the k-block
        auto a_operand = [&](int hs, int mb) {
            return *(const half8_t*)(a_lane + mb * 32 * kAStride + 32 * (hs >> 1) + 8 * (hs & 1));
        };
        half8_t a_op = a_operand(0, 0);
#pragma unroll
        for (int hs = 0; hs < 8; ++hs) {
            const int d = hs >> 2, s = (hs >> 1) & 1, h = hs & 1;
            __builtin_amdgcn_sched_barrier(0);
            uint32_t (&b_nx)[2][4] = b[d ^ 1][s];       // the half of the next two steps decoded in this one and its neighbour
            const half8_t b_op = __builtin_bit_cast(half8_t, uint4{b[d][h][s][0], b[d][h][s][1], b[d][h][s][2], b[d][h][s][3]});
            if (s == 0 && h == 0) {
                win = LaneWindows<BITS>(ring[d ^ 1], fetch_prev(lane, ring[d ^ 1][BITS - 1]));
                load_b(min(kb + 1 + d, KB - 1), d ^ 1);
            }
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const half8_t a_now = a_op;
                if (mb + 1 < MB) a_op = a_operand(hs, mb + 1);
                else if (hs < 7) a_op = a_operand(hs + 1, 0);
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a_now, b_op, acc[mb], 0, 0, 0);
                decode_pairs(win, s, 4 * h + mb * 4 / MB, (mb + 1) * 4 / MB - mb * 4 / MB, b_nx);
            }
            if (h == 1) trade(b_nx);
            // (the decode of a half-step spread over its MB matrix instructions)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 36 / MB, 0);
            }
        }
    }

    const int col = wave * 32 + ((slot >> 3) & 1) * 16 + (slot >> 4) * 8 + (slot & 7);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (mb * 32 >= rows_here) break;                        // workgroup-uniform
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) z_tile[(8 * (r >> 2) + 4 * half_id + (r & 3)) * kHalfZStride + col] = acc[mb][r];
        __syncthreads();
        finish_half_rows(p, gp, which, n0, mb, z_tile, s_scale);
    }
}

// The same for an expert of up to sixteen rows (accumulate_16_rows, 32 columns a wave; the bits of a whole tile).  Bound
// by the decode of a wave that has its SIMD nearly to itself: 60 experts of 1024 x 512 (180 tokens) 44.8 us a layer as halves
// of 32-row products, 48.2 whole, 42.9 so.
template <int BITS, int CB>
__device__ __forceinline__ void gemm_half_tile_16(const GemmParams& p, const GroupProblem gp, const int which, const int n0, unsigned char* smem)
{
    float* z_tile = (float*)smem;                       // [16][kHalfZStride]
    if (n0 >= p.N) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool shared = gp.expert == p.shared_expert;
    const ExpertLin lin = shared ? p.shared[p.lin_base + which] : p.experts[gp.expert * p.lins_per_expert + p.lin_base + which];
    __shared__ __align__(16) half8_t s_scale[16];
    half8_t scale_mine = {0, 0, 0, 0, 0, 0, 0, 0};
    if (threadIdx.x < 16) scale_mine = ((global_ptr<const half8_t>)as_global(lin.svh + n0))[threadIdx.x];
    int arow = gp.row0 + min(lane & 15, gp.nrows - 1);  // rows past the problem repeat its last row
    if (p.a_rows && !shared) arow = as_global(p.a_rows)[arow];
    float4_t acc[1][2] = {};
    accumulate_16_rows<BITS, CB, 1, false>(lin.trellis, (size_t)(p.N >> 4) * (8 * BITS), n0 + 32 * wave, p.a_had[which], arow, p.K, lane, acc, [&]() {
        if (threadIdx.x < 16) s_scale[threadIdx.x] = scale_mine;
    });
    stage_16_rows<kHalfZStride>(z_tile + 32 * wave, acc, lane);
    __syncthreads();
    finish_half_rows(p, gp, which, n0, 0, z_tile, s_scale);
}

// What problem number `problem` of a mixed launch is: the first list, its second halves, the second list, its second
// halves.  `tiles` of 256 columns a problem; halves where all of the launch then runs at once, in `places`.
struct MixedPlace {
    bool first_list, halves, second, empty;     // second: columns 128.. of the tiles
    int at;                                     // in its list
};
constexpr MixedPlace mixed_place(const int problem, const int big, const int small, const int tiles, const int places)
{
    const bool big_halves = (2 * big + small) * tiles <= places, small_halves = 2 * (big + small) * tiles <= places;
    const int first_small = big_halves ? 2 * big : big;
    const bool first_list = problem < first_small;
    const bool second = problem >= (first_list ? big : first_small + small);
    const bool empty = second && !first_list && (!small_halves || problem >= first_small + 2 * small);
    return {first_list, first_list ? big_halves : small_halves, second, empty,
            first_list ? problem - (second ? big : 0) : problem - first_small - (second ? small : 0)};
}
// problems that may have second halves: the room that a launch needs behind its lists
constexpr int mixed_extra(const int tiles, const int places) { return places / (2 * tiles); }

// Grouped launch over two problem lists at once: the first problems of group_tile are those of up
// to 128 rows (weights decoded once for all of them, so an expert with many rows costs one
// decode per 128 rows instead of one per 32), the ones after them the problems of up to 32
// rows.  Both kinds sit in one launch, the long tiles first, so the short ones fill in around
// them (as two launches the 128-row tiles would run alone on a fraction of the compute units).
// Whole K per workgroup: no hand-over.
// A problem of up to 64 or 96 rows runs as two or three 32-row blocks (the loop multiplies all the blocks
// it has, needed or not): gate + up and down of 800 tokens that choose 8 of 128 experts 137 + 82 -> 119 +
// 70 us, of 1500 tokens (94 rows an expert) 133 + 89 -> 131 + 85.
// Tiles run as halves of 128 columns (gemm_half_tile; bits the same) where every workgroup of the launch then has a
// place at once, two on a compute unit: the problems of the first list, or those of both lists.  A launch of one round
// is as long as its longest workgroup, and a half is the shorter one.
// Layers of 2048 x 768: 200 tokens that choose 4 of 16 experts 69.7 -> 54.4 us (64 and 128 tiles), of
// 1024 x 512, 300 tokens 58.2 -> 47.0, of 2048 x 1024, 150 tokens that choose 8 of 32 (256 tiles) 84.9 -> 80.8;
// 400 tokens that choose 6 of 16 (256 tiles, half of them of 128 rows) 104.4 -> 105.  The first list alone, popular
// experts: 512 of 2048 x 512 at 129 / 200 / 256 tokens 102.6 -> 95.5, 111.7 -> 104.2, 116.4 -> 111.2, 128 of 2048 x 768
// at 150 101.8 -> 94.0, 256 of 1024 x 512 at 600 80.5 -> 70.9.  Experts of up to sixteen rows too (gemm_half_tile_16):
// 60 experts of 2048 x 512 at 150 and 180 tokens 66.2 -> 61.7 and 70.9 -> 64.7 against whole ones, of 1024 x 512 at 180
// 48.2 -> 42.9.
// Beyond that whole tiles, which are the cheaper ones: the first list up to 576 and 640 workgroups 110 -> 118 (128
// experts, 256 tokens) and 139 -> 148 (512, 400), both up to 768 (1000 tokens that choose 4 of 16) 119 -> 126, and
// with the tiles of a last, half empty round as halves 1500 tokens of 128 experts 278 -> 289 (the rounds are not in
// step).  Operands asked for two multiplications ahead of their use change nothing there.
// Measured and dropped: cutting K in two with the split-K hand-over, for every tile or for the
// 128-row tiles only (the shorter units pack better, the hand-over of 128 KB of partial sums per
// tile costs far more than that gains: 150 -> 183 us per layer), 128-column units whose four waves
// cut K in two and add through LDS (gate + up of 256 tokens x 512 experts 61.3 -> 54.9 us, but its
// down projection 32.0 -> 39.6 and both launches of 64 tokens x 128 experts 5 - 6 us slower: twice
// the units pay twice the problem -> expert -> pointer chain), and resident workgroups that take units
// from a counter (the same schedule as the hardware's, with slower code).
template <int BITS, int CB>
__global__ __launch_bounds__(256, 2) void exl3_gemm_mixed_kernel(GemmParams p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    KRange kr;
    kr.kb0 = 0;
    kr.kb1 = p.K >> 7;
    kr.step = 1;
    kr.part = 0;
    kr.parts = 1;
    kr.counter = 0;
    kr.slot0 = kr.slot_rest = 0;
    kr.slot_step = 0;
    const GroupTile gt = group_tile(p);
    const MixedPlace place = mixed_place(gt.problem, *p.num_big, *p.num_problems, p.group_lins * ((int)gridDim.x >> 3), p.places);
    if (place.empty) return;
    const GroupProblem* const list = place.first_list ? p.big_problems : p.problems;
    const int at = place.at;
    const GroupProblem gp = list[at];
    if (place.halves) {
        const int n0 = gt.col * 256 + 128 * place.second;
        if (gp.lone) gemm_half_tile_16<BITS, CB>(p, gp, gt.which, n0, smem);
        else if (gp.nrows > 96) gemm_half_tile<BITS, CB, 4>(p, gp, gt.which, n0, smem);
        else if (gp.nrows > 64) gemm_half_tile<BITS, CB, 3>(p, gp, gt.which, n0, smem);
        else if (gp.nrows > 32) gemm_half_tile<BITS, CB, 2>(p, gp, gt.which, n0, smem);
        else gemm_half_tile<BITS, CB, 1>(p, gp, gt.which, n0, smem);
        return;
    }
    // as many 32-row blocks as the problem has
    if (gp.nrows > 96) gemm_tile<BITS, CB, 4, false>(p, at, gt.col, kr, gt.which, smem, list);
    else if (gp.nrows > 64) gemm_tile<BITS, CB, 3, false>(p, at, gt.col, kr, gt.which, smem, list);
    else if (gp.nrows > 32) gemm_tile<BITS, CB, 2, false>(p, at, gt.col, kr, gt.which, smem, list);
    else gemm_tile<BITS, CB, 1, false>(p, at, gt.col, kr, gt.which, smem, list);
}

// Dense launches whose tile count does not divide over the compute units: the
// (tile, k-block) units of the launch, tile-major, are cut into gridDim.x equal
// contiguous ranges, one per workgroup (two workgroups per compute unit), so every
// workgroup does the same amount of decode and MFMA work.  A range covers the end
// of one tile, possibly whole tiles, and the start of another; a tile shared by
// several workgroups is finished by the last of them to arrive, which adds the
// partial sums in k order, so the result does not depend on timing.
// Workgroup w owns unit_q + 1 units if w < unit_r, else unit_q (units = unit_q * G + unit_r),
// starting at w * unit_q + min(w, unit_r).  32-bit arithmetic on workgroup-uniform values
// only, so the k loop and its addresses stay in scalar registers as in the plain kernel.
__device__ __forceinline__ int range_start(const GemmParams& p, int w) { return w * p.unit_q + min(w, p.unit_r); }
__device__ __forceinline__ int range_owner(const GemmParams& p, int x)
{
    const int big = p.unit_r * (p.unit_q + 1);      // units held by the workgroups with one extra
    return x < big ? x / (p.unit_q + 1) : p.unit_r + (x - big) / p.unit_q;
}

// Workgroups are handed to the eight compute dies round-robin (workgroup i runs on die
// i % 8), and every die has its own L2.  Renumbering them so that a die gets a contiguous
// eighth of the ranges makes the tiles of one die share their rows of the activation
// (one 128-row block, 1.3 MB at K = 5120, instead of all of them): a quarter less traffic
// behind the L2 on the 27B gate projection at 512 rows.
__device__ __forceinline__ int die_major_index(int i, int n)
{
    return (n & 7) == 0 ? (i & 7) * (n >> 3) + (i >> 3) : i;
}

// the k-blocks of the tile that unit u lies in, up to `stop`, for workgroup w.  Every workgroup has two
// partial-sum slots, one for the tile its range starts in and one for the tile it ends in (no other is
// shared), so that any number of tiles can be dealt out.
__device__ __forceinline__ KRange range_segment(const GemmParams& p, const int w, const int u, const int stop, int& tile)
{
    const int KB = p.K >> 7;
    tile = u / KB;
    const int t0 = tile * KB;                                   // the tile's first unit
    const int w_first = range_owner(p, t0);
    const int w_last = range_owner(p, t0 + KB - 1);
    KRange kr;
    kr.kb0 = u - t0;
    kr.kb1 = stop - t0;
    kr.step = 1;
    kr.part = w - w_first;
    kr.parts = w_last - w_first + 1;
    kr.counter = (size_t)tile;
    kr.slot_rest = 2 * (size_t)w_first;
    kr.slot0 = kr.slot_rest + (range_start(p, w_first) < t0 ? 1 : 0);
    kr.slot_step = 2;
    return kr;
}

template <int BITS, int CB, int MB>
__device__ __forceinline__ void gemm_segment(const GemmParams& p, const int w, const int u, const int stop,
                                             unsigned char* smem)
{
    const int nblocks = ((p.N + 255) >> 8) * (p.num_slices > 0 ? p.num_slices : 1);
    int tile;
    const KRange kr = range_segment(p, w, u, stop, tile);
    const int t = p.tile0 + tile;
    gemm_tile<BITS, CB, MB, true>(p, t / nblocks, t % nblocks, kr, 0, smem);
}

// A range runs through the end of one tile, any whole tiles after it and the start of another.
template <int BITS, int CB, int MB>
__global__ __launch_bounds__(256, 2) void exl3_gemm_balanced_kernel(GemmParams p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int KB = p.K >> 7;
    const int w = die_major_index((int)blockIdx.x, (int)gridDim.x);
    const int u_end = range_start(p, w + 1);
    int u = range_start(p, w);
    // the first two segments are written out (as the body of a loop the compiler's scheduler does
    // not reliably keep the interleaved order of the main loop); the loop takes the rest
    {
        const int stop = min(u_end, (u / KB + 1) * KB);
        gemm_segment<BITS, CB, MB>(p, w, u, stop, smem);
        u = stop;
    }
    if (u < u_end) {
        __syncthreads();                                        // the epilogue's LDS tile is the next A tile
        const int stop = min(u_end, (u / KB + 1) * KB);
        gemm_segment<BITS, CB, MB>(p, w, u, stop, smem);
        u = stop;
    }
    while (u < u_end) {
        __syncthreads();
        const int stop = min(u_end, (u / KB + 1) * KB);
        gemm_segment<BITS, CB, MB>(p, w, u, stop, smem);
        u = stop;
    }
}

}  // namespace berth
