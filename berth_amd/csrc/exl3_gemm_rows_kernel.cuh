// EXL3 linear for a few rows (2..32): every weight is decoded once and multiplied on the matrix
// units, as a single resident round of sixteen-wave workgroups.
//
//   c = Hh(a_had @ W) * svh (+ out_add),   a_had = Hh(a * suh) rotated by an earlier launch, or by this one (ROT)
//
// What bounds it: the decode (about 4.0 vector instructions per weight, 124 for the 32 weights a
// lane takes per step); the four v_mfma_f32_16x16x32_f16 of a step and 16 rows need 64 of the
// 496 cycles that the decode takes, so rows up to 32 cost little more than one.
//
//   * A unit of work is 64 rows of K x 128 columns, column block major.  The launch's units are
//     dealt out evenly to the workgroups (one per compute unit), whatever the shape is: no
//     second round, no tail.  Few column blocks: each is cut into S parts of its own instead,
//     so that no workgroup hands over two of them.
//   * Of a workgroup's sixteen waves four share a unit (32 columns each) and four such groups
//     take a contiguous quarter of the units each.  A wave walks its quarter alone: no barrier
//     in the loop, two units of trellis and activation in registers, and the walk crosses
//     column blocks without draining them.
//   * Operands: 16 lanes cover 2 tiles (32 columns) of one tile row in the octet layout, the
//     four lane groups four tile rows.  The four register quads a lane decodes (column u or u + 8,
//     k 0..7 or 8..15 of its tile row) are four B operands of the 16x16x32 form, with k slot
//     8 * group + i standing for k = 16 * group + 8h + i.  The A operand of the same slots is 16
//     bytes of a rotated row.  The rotation leaves a second copy of its result in operand order
//     (rows_operand_offset), so a wave reads an operand as 1 KB in a row; from the row-major copy
//     the same loads touch a line per lane and cost the launch a third of its time.  All column
//     groups of a compute unit read the same operands at about the same time, from its L1.
//   * A wave leaves its part of a column block in LDS, in fp32; the parts are added in k order.
//     A column block that lies inside one workgroup's units is finished there.  Otherwise the
//     sharers leave their sums in the workspace and the last to arrive adds them in k order, so
//     results repeat bit for bit.
//   * GROUPED: the column blocks are those of a list of problems (up to 16 expert-sorted rows each,
//     problem-major, then the launch's one or two linears).  The list's length is only known on the
//     device, so the deal is worked out there.  A workgroup looks its few blocks up once, into LDS.
//     A operands come straight from the row-major rotated rows: a problem has few of them, and the
//     lanes past the last repeat it, so that a load touches as many lines as there are rows.
//     Gate and up, 2048 x 768 at 4 bits, 2 / 8 / 16 tokens that choose 8 of 128 experts: 15 / 30 / 45 us.
//
//   * PAIR: gate and up of an MLP, their blocks of the same columns next to each other.  What is handed over is a
//     pair of them, and its finisher goes on to silu(g) * u and the rotated input of the down projection, for which a
//     launch of its own would read both back: decoder layers of 5120 x 17408 at 5 / 8 / 12 / 24 / 32 rows 89.1 -> 86.1,
//     91.4 -> 87.9, 92.4 -> 89.4, 111.6 -> 108.4, 121.3 -> 118.5 us, of 2048 x 5632 at 5 and 32 rows 57.7 -> 54.5,
//     72.2 -> 66.8.  The grouped form gained nothing (8 tokens 67.4 -> 66.7, 16 85.4 -> 85.3): its tail grew by what the
//     launch took.  The tail of gate + up at 24 rows takes a quarter of the launch (the last wave ends its walk at 29 us, the
//     finishers at 38): sums in LDS 2 us, stores until they are there 1, the counter 0.7, parts read and finished 2
//     for each row of a wave, so that a wave asks for both of its rows together.  (The same at the end of the other
//     launches, which have more sharers: 20 rows of 2048x8192 12.2 -> 12.8.)
//
// Measured (27B layer, traced): gate + up at 5 rows and 3 bits 62.6 -> 32.5 us against the VALU
// kernel, at 24 rows and 4 bits 49.0 -> 40.6 against 32-row tiles (whose 544 workgroups also
// ran in one and a bit rounds), down 47.4 -> 19.1 and 38 -> 23.0.  Of the 41 us at 24 rows the
// vector pipes issue for 65 %, the MFMAs take 13 %, 4 us are launch, head and hand-over.
#pragma once

#include "exl3_gemm_kernel.cuh"
#include "rows_operand.cuh"

#include <type_traits>

namespace berth {

constexpr int kRowsWaves = 16;
constexpr int kRowsStride = 132;            // floats per row of a partial column block in LDS

// Launches that rotate the input themselves (ROT): the most (row, 128 block) items a workgroup takes, sixteen
// lanes each, and the LDS of their result, `units` units of 64 k behind everything else.  Where a column
// block is cut into parts of its own, a workgroup needs a part of K only, so all workgroups of a part of
// K rotating it cost less than the launch that did it once, as long as it is a few items a lane group.  us, two
// launches -> one, weights from memory:
//   linears   4096x4096 at 5 / 16 / 32 rows (20 / 64 / 128 items)     11.7 / 13.4 / 17.2 -> 10.1 / 11.6 / 16.0
//             6144x5120 at 5 / 24 / 28 / 32 (40 / 192 / 224 / 256)    14.3 / 17.7 / 18.7 / 19.6 -> 12.6 / 16.7 / 17.8 / 19.1
//             10240x5120 at 8 / 14 / 17 (112 / 196 / 238)             17.8 / 18.9 / 20.8 -> 16.5 / 18.3 / 19.6
//             17408x5120 at 8 / 11 (184 / 253)                        22.7 / 23.0 -> 21.9 / 22.7
//   q, k, v   5120 -> 6144 + 2 x 1024 at 9 / 24 (90 / 240)            17.1 / 20.4 -> 15.6 / 19.3
//             4096 -> 4096 + 2 x 1024 at 16 / 32 (112 / 224)          15.6 / 20.0 -> 13.8 / 18.4
// Of 100 linears and 47 bundles of up to 256 items, four a lane group, none lost more than 0.1; the gain is 1.6 to 2.2 up to
// 64 items and 0.2 to 1.6 above 192.
constexpr int kRowsRotItems = 256;
__host__ __device__ constexpr size_t rows_rot_lds_bytes(int units, int mt) { return (size_t)units * mt * 2048; }

// dynamic LDS of a launch: the pieces, the output scales of the column blocks, two flags
__host__ __device__ constexpr size_t rows_lds_bytes(int rows, int ncb)
{
    return (size_t)(ncb + 3) * rows * kRowsStride * 4 + (size_t)ncb * 256 + 16;
}
// of a GROUPED launch, behind that: the column blocks' tensors
struct RowsGroupBlock {
    const uint32_t* trellis;
    const _Float16* svh;
    const _Float16* a_had;
    void* c;
    int rows;
    uint32_t row_at[16];        // byte offset of each of its rows (past the last: the last) in a_had
};
__host__ __device__ constexpr size_t rows_group_lds_bytes(int rows, int ncb)
{
    return rows_lds_bytes(rows, ncb) + (size_t)ncb * sizeof(RowsGroupBlock);
}

// PAIR: what follows gate and up
struct RowsPairParams : GemmParams {
    const _Float16* suh;        // input scales of the down projection
    _Float16* operand;          // a second copy of its rotated rows in operand order (may be null)
    int operand_mt;
    int keep_up;                // 1: up goes to its output; 0: the activation does
};

// x / d for the launch's exact divisors, m = floor(2^32 / d) + 1 (0 for d = 1)
__device__ __forceinline__ unsigned div_exact(unsigned x, unsigned m) { return m ? __umulhi(x, m) : x; }

// the tensors of one 128-column block of the launch
struct RowsBlock {
    const uint32_t* trellis;    // of the linear (of the whole weight's slice)
    const _Float16* svh;
    const _Float16* a_had;      // the rotated input in operand order
    void* c;
    int n0;                     // first column inside the linear
    int ldc;                    // elements between output rows, and columns of the weight
    bool empty;                 // past the end of a narrower slice: nothing to compute
    int rows;                   // of the block (GROUPED only)
};
template <bool PAIR = false>
__device__ __forceinline__ RowsBlock rows_block(const GemmParams& p, const unsigned cb)
{
    RowsBlock b;
    b.trellis = p.lin.trellis;
    b.svh = p.lin.svh;
    b.a_had = p.a_had[0];
    b.c = p.c[0];
    b.n0 = (int)cb * 128;
    b.ldc = p.N;
    b.empty = false;
    b.rows = p.M;
    if (PAIR) {
        const GemmSlice& g = p.slice[cb & 1];
        b.trellis = g.trellis;
        b.svh = g.svh;
        b.a_had = g.a_had;
        b.c = g.c;
        b.n0 = (int)(cb >> 1) * 128;
    } else if (p.num_slices > 0) {
        const unsigned nb = (unsigned)p.N >> 7;
        const unsigned sl = div_exact(cb, p.m_nb);
        b.n0 = (int)(cb - sl * nb) * 128;
        int width = p.N;
        if (p.b_list) {
            unsigned slab = sl;
            b.trellis = (const uint32_t*)p.b_list[sl];
            b.svh = (const _Float16*)p.svh_list[sl];
            if (p.c_ptrs) {
                width = p.size_n_list[sl];
                b.ldc = p.n_stride_list[sl];
                slab = (unsigned)p.had_src_list[sl];
                b.c = (void*)p.c_ptrs[sl];
            } else {
                b.c = (char*)p.c[0] + (size_t)sl * p.M * p.N * (p.out_fp32 ? 4 : 2);
            }
            b.a_had = p.a_had[0] + (size_t)slab * p.slab_stride;
        } else {
            const GemmSlice& g = p.slice[sl];
            b.trellis = g.trellis;
            b.svh = g.svh;
            b.c = g.c;
            width = g.width;
            b.ldc = g.n_stride;
            b.a_had = g.a_had;
        }
        b.empty = b.n0 >= width;
    }
    return b;
}

// the input of the column block `cb`, its scales and, for one column block per input, where its rotated rows go
// (lists in device memory: of linears with an input each)
__device__ __forceinline__ GemmRotation rows_rotation(const GemmRotateParams& p, const unsigned cb)
{
    if (p.num_slices == 0) return {p.lin.suh, p.rot_in, cb == 0 ? p.rot_out : nullptr};
    const unsigned sl = div_exact(cb, p.m_nb);
    const bool first = cb == sl * ((unsigned)p.N >> 7);
    if (!p.b_list) {
        const GemmRotation& r = p.rotation[sl];
        return {r.suh, r.in, first ? r.had_out : nullptr};
    }
    return {(const _Float16*)p.suh_list[sl], p.rot_in + (size_t)sl * p.rot_in_stride,
            first ? p.rot_out + (size_t)sl * p.M * p.K : nullptr};
}

template <int BITS, int CB, int MT, bool GROUPED, bool ROT = false, bool PAIR = false>      // MT: tiles of 16 rows
__global__ __launch_bounds__(1024, 1) void exl3_gemm_rows_kernel(
    std::conditional_t<ROT, GemmRotateParams, std::conditional_t<PAIR, RowsPairParams, GemmParams>> p)
{
    static_assert(GROUPED + ROT + PAIR <= 1, "a problem list and a pair bring their rows rotated");
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int tile_dw = 8 * BITS;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cg = wave & 3, kg = wave >> 2;
    const int l16 = lane & 15, lg = lane >> 4;
    const unsigned TR4 = (unsigned)p.K >> 6;            // units per column block
    const int M = p.M;                                  // rows of the input; GROUPED: most rows of a problem

    // ---- this workgroup's units [u0, u1), this wave's quarter [w0, w1)
    const unsigned w = blockIdx.x;
    unsigned q = (unsigned)p.unit_q, rem = (unsigned)p.unit_r;
    const unsigned S = GROUPED ? 0u : (unsigned)p.S;
    if constexpr (GROUPED) {
        const unsigned U = (unsigned)*p.num_problems * (unsigned)p.group_blocks * TR4;
        const unsigned G = min((unsigned)gridDim.x, U >> 2);            // a unit for each k group at least
        if (w >= G) return;
        q = U / G;
        rem = U - q * G;
    }
    unsigned u0 = w * q + min(w, rem), u1 = (w + 1) * q + min(w + 1, rem);
    if (S) {
        const unsigned blk = div_exact(w, p.m_s), part = w - blk * S;
        u0 = blk * TR4 + div_exact(part * TR4, p.m_s);
        u1 = blk * TR4 + div_exact((part + 1) * TR4, p.m_s);
    }
    const unsigned L = u1 - u0;
    const unsigned cb_first = div_exact(u0, p.m_tr), cb_last = div_exact(u1 - 1, p.m_tr);
    const unsigned ncb = cb_last - cb_first + 1;
    const unsigned w0 = u0 + (L * (unsigned)kg >> 2), w1 = u0 + (L * (unsigned)(kg + 1) >> 2);

    float* const red = (float*)smem;
    uint32_t* const sv_lds = (uint32_t*)(red + (size_t)(ncb + 3) * M * kRowsStride);
    unsigned* const flags = sv_lds + ncb * 64;
    RowsGroupBlock* const table = (RowsGroupBlock*)(flags + 4);
    if constexpr (GROUPED) {
        if (threadIdx.x < ncb) {
            const unsigned cb = cb_first + threadIdx.x;
            const unsigned prob = div_exact(cb, p.m_rt), in_prob = cb - prob * (unsigned)p.group_blocks;
            const int which = (int)div_exact(in_prob, p.m_nb);
            const GroupProblem gp = p.problems[prob];
            const ExpertLin lin = gp.expert == p.shared_expert ? p.shared[p.lin_base + which]
                                                               : p.experts[gp.expert * p.lins_per_expert + p.lin_base + which];
            RowsGroupBlock& g = table[threadIdx.x];
            g.trellis = lin.trellis;
            g.svh = lin.svh;
            g.a_had = p.a_had[which];
            g.c = (char*)p.c[which] + (size_t)gp.row0 * p.N * (p.out_fp32 ? 4 : 2);
            g.rows = gp.nrows;
        }
        if (threadIdx.x < 16 * ncb) {
            const GroupProblem gp = p.problems[div_exact(cb_first + (threadIdx.x >> 4), p.m_rt)];
            const int r = gp.row0 + min((int)threadIdx.x & 15, gp.nrows - 1);
            const int at = p.a_rows && gp.expert != p.shared_expert ? p.a_rows[r] : r;
            table[threadIdx.x >> 4].row_at[threadIdx.x & 15] = (uint32_t)at * (uint32_t)p.K * 2;
        }
        __syncthreads();
    }
    auto block = [&](const unsigned cb) -> RowsBlock {
        if constexpr (GROUPED) {
            const RowsGroupBlock& g = table[cb - cb_first];
            const unsigned nb = (unsigned)p.N >> 7;
            RowsBlock b;
            b.trellis = rows_uniform(g.trellis);
            b.svh = rows_uniform(g.svh);
            b.a_had = rows_uniform(g.a_had);
            b.c = (void*)rows_uniform((const char*)g.c);
            b.n0 = (int)(cb - div_exact(cb, p.m_nb) * nb) * 128;
            b.ldc = p.N;
            b.empty = false;
            b.rows = __builtin_amdgcn_readfirstlane(g.rows);
            return b;
        } else {
            return rows_block<PAIR>(p, cb);
        }
    };

    // ---- the walk's operands: a pointer pair that runs two units ahead of the decode
    unsigned f_cb = div_exact(w0, p.m_tr);
    unsigned f_k = w0 - f_cb * TR4, f_left = w1 - w0;
    const char* f_t;
    const char* f_a;
    long f_step;
    uint32_t t_off;                                     // bytes, per lane
    uint32_t a_off = (uint32_t)lane * 16;
    constexpr int kUnitA = GROUPED ? 128 : MT * 2 * 1024;   // bytes of A operands per unit (GROUPED: of one row)
    // ROT: a workgroup's units lie in one column block; the 128 blocks of its rows' input that they need
    const unsigned rot0 = (u0 - cb_first * TR4) & ~1u;          // first unit in LDS
    unsigned char* const rot_lds = (unsigned char*)(flags + 4);
    uint32_t f_lds = 0;                                         // this wave's next unit in it
    constexpr int kNextA = GROUPED ? 1 : 64;            // from a lane's operand to its next, in 16 bytes
    auto seek = [&](unsigned cb, unsigned k) {
        const RowsBlock b = block(cb);
        if constexpr (GROUPED) a_off = table[cb - cb_first].row_at[l16] + (uint32_t)lg * 32;
        if (b.empty) {                                  // read anything valid, use nothing
            if constexpr (ROT) f_t = (const char*)rows_uniform(rows_rotation(p, cb).in);
            else f_t = (const char*)rows_uniform(b.a_had);
            f_step = 0;
            t_off = 0;
        } else {
            const uint32_t row_bytes = (uint32_t)(b.ldc >> 4) * (tile_dw * 4);
            f_step = 4 * (long)row_bytes;
            f_t = (const char*)rows_uniform(b.trellis) + (size_t)(b.n0 >> 4) * (tile_dw * 4) + (size_t)(4 * k) * row_bytes;
            t_off = (uint32_t)lg * row_bytes + (uint32_t)(cg * 16 + l16) * (BITS * 4);
        }
        if constexpr (ROT) f_lds = (k - rot0) * (uint32_t)kUnitA;
        else f_a = (const char*)rows_uniform(b.a_had) + (size_t)k * kUnitA;
    };
    seek(f_cb, f_k);

    uint32_t own[2][BITS];
    half8_t av[2][MT][2];
    auto fetch_t = [&](int j) { load_tile_dwords<BITS>((global_ptr<const uint32_t>)(as_global(f_t) + t_off), own[j]); };
    auto fetch_a = [&](int j) {
        if constexpr (ROT) {
            const half8_t* const src = (const half8_t*)(rot_lds + f_lds + a_off);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                av[j][mt][0] = src[(2 * mt) * kNextA];
                av[j][mt][1] = src[(2 * mt + 1) * kNextA];
            }
        } else {
            const global_ptr<const half8_t> src = (global_ptr<const half8_t>)(as_global(f_a) + a_off);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                av[j][mt][0] = src[(2 * mt) * kNextA];
                av[j][mt][1] = src[(2 * mt + 1) * kNextA];
            }
        }
    };
    auto advance = [&]() {                              // on the last unit it stays: read again, not used
        if (f_left > 1) {
            --f_left;
            f_t += f_step;
            if constexpr (ROT) {                        // (all units in one column block)
                f_lds += kUnitA;
                return;
            }
            f_a += kUnitA;
            if (++f_k == TR4) {
                f_k = 0;
                ++f_cb;
                seek(f_cb, 0);
            }
        }
    };
    if constexpr (ROT) {
        // The rows' part of the input, rotated into LDS in operand order: all of its loads at once, behind
        // the first weights of the wave.
        const GemmRotation r = rows_rotation(p, cb_first);
        const unsigned nb = ((u1 - cb_first * TR4 + 1) >> 1) - (rot0 >> 1);
        const unsigned items = nb * (unsigned)M;
        const int chunk = had_chunk(lane);
        const uint32_t col0 = rot0 * 64 + 8 * (uint32_t)chunk;
        half8_t x[kRowsRotItems / 64], sc[kRowsRotItems / 64];
        unsigned row[kRowsRotItems / 64], blk[kRowsRotItems / 64];
        const global_ptr<const _Float16> in = as_global(rows_uniform(r.in)), suh = as_global(rows_uniform(r.suh));
        fetch_t(0);
#pragma unroll
        for (int i = 0; i < kRowsRotItems / 64; ++i) {
            const unsigned it = min(threadIdx.x / 16 + 64u * i, items - 1);     // (past the end: the last one, stored again)
            blk[i] = div_exact(it, p.m_rows);
            row[i] = it - blk[i] * (unsigned)M;
            if (64u * i < items) {                                              // workgroup-uniform
                x[i] = *(global_ptr<const half8_t>)(in + (size_t)row[i] * p.K + col0 + 128 * blk[i]);
                sc[i] = *(global_ptr<const half8_t>)(suh + col0 + 128 * blk[i]);
            }
        }
        const unsigned left = f_left;
        advance();
        fetch_t(1);
#pragma unroll
        for (int i = 0; i < kRowsRotItems / 64; ++i) {
            if (64u * i >= items) break;
            float v[8];
            mul_half8(x[i], sc[i], v);
            const float unit = had128_row16(v, lane) * kRsqrt128;
            half8_t o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (_Float16)had_scale(v[e], unit);
            const uint32_t unit_at = 2 * blk[i] + ((uint32_t)chunk >> 3);
            *(half8_t*)(rot_lds + unit_at * (uint32_t)kUnitA + 2 * rows_operand_offset((int)row[i], 8 * (chunk & 7), MT)) = o;
            if (r.had_out) *(global_ptr<half8_t>)(as_global(r.had_out) + (size_t)row[i] * p.K + col0 + 128 * blk[i]) = o;
        }
        __syncthreads();
        f_lds -= left > 1 ? kUnitA : 0;
        fetch_a(0);
        f_lds += left > 1 ? kUnitA : 0;
        fetch_a(1);
        advance();
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            fetch_t(j);
            fetch_a(j);
            advance();
        }
    }
    // the output scales, asked for now: the finish does not wait for them
    uint32_t sv_mine = 0;
    if (!PAIR && (unsigned)wave < ncb) {
        const RowsBlock b = block(cb_first + (unsigned)wave);
        if (!b.empty) sv_mine = as_global((const uint32_t*)(b.svh + b.n0))[lane];
    }

    float4_t acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    unsigned cb = div_exact(w0, p.m_tr);
    unsigned k = w0 - cb * TR4;
    // piece of (quarter, column block): the quarters are consecutive runs, so kg + (cb - cb_first)
    // names each of them once
    auto flush = [&]() {
        float* const piece = red + (size_t)((unsigned)kg + cb - cb_first) * M * kRowsStride;
        const int col = cg * 32 + (l16 >> 3) * 16 + (l16 & 7);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = mt * 16 + 4 * lg + r;
                if (row < M) {
                    piece[row * kRowsStride + col] = acc[mt][0][r];
                    piece[row * kRowsStride + col + 8] = acc[mt][1][r];
                }
            }
    };
    // The registers of a step are reloaded as soon as they have been used, the trellis behind the
    // decode and the A operands behind the MFMAs; the barriers keep the compiler from issuing the
    // loads ahead of that into other registers, which costs a move per register and step.
    auto stage = [&](int j) {
        const uint32_t prev = fetch_prev(lane, own[j][BITS - 1]);
        uint32_t w2[16];
        decode_lane<BITS, CB>(own[j], prev, w2);
        __builtin_amdgcn_sched_barrier(0);
        fetch_t(j);
        half8_t b[2][2];                                // [k half][column half]
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const uint4 bq = {w2[2 * f + h], w2[4 + 2 * f + h], w2[8 + 2 * f + h], w2[12 + 2 * f + h]};
                b[h][f] = __builtin_bit_cast(half8_t, bq);
            }
        settle<CB>(b[0][0], b[0][1], b[1][0], b[1][1]);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[mt][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[j][mt][h], b[h][f], acc[mt][f], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_a(j);
        advance();
        if constexpr (ROT) return;
        if (++k == TR4) {
            flush();
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
            ++cb;
            k = 0;
        }
    };
    const unsigned pairs = (w1 - w0) >> 1;
    // Waves give up their priority over their second half (PriorityRamp's reason: of the four on a SIMD the last ones
    // ended alone).  Decoder layers of 5 rows at 3 bits (MCG) 91.8 -> 87.7 us, of 8 and 24 at 4 bits 97.5 -> 93.9 and 114.1 ->
    // 111.8, MoE layers of 4 and 12 tokens 53.9 -> 52.1 and 82.4 -> 78.9.  Launches that rotate have few units a wave:
    // 12 rows of 4096x4096 10.2 -> 10.4.
    const unsigned p2 = ROT ? ~0u : pairs >> 1, p1 = ROT ? ~0u : pairs * 3 >> 2, p0 = ROT ? ~0u : pairs * 7 >> 3;
    if constexpr (!ROT) __builtin_amdgcn_s_setprio(3);
    for (unsigned g = 0; g < pairs; ++g) {
        if (g == p2) __builtin_amdgcn_s_setprio(2);
        if (g == p1) __builtin_amdgcn_s_setprio(1);
        if (g == p0) __builtin_amdgcn_s_setprio(0);
        stage(0);
        stage(1);
    }
    if constexpr (!ROT) __builtin_amdgcn_s_setprio(0);
    if ((w1 - w0) & 1) stage(0);
    if (ROT || k != 0) flush();
    if (!PAIR && (unsigned)wave < ncb) sv_lds[wave * 64 + lane] = sv_mine;
    __syncthreads();

    const unsigned qs1 = u0 + (L >> 2), qs2 = u0 + (L * 2 >> 2), qs3 = u0 + (L * 3 >> 2);
    // this workgroup's sum of a row of column block cb_first + cbi, two columns a lane
    auto own_sum = [&](const unsigned cbi, const int row, float& z0, float& z1) {
        const unsigned c0 = (cb_first + cbi) * TR4, c1 = c0 + TR4;
        const float* const base = red + (size_t)cbi * M * kRowsStride + row * kRowsStride + 2 * lane;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const unsigned a0 = g == 0 ? u0 : g == 1 ? qs1 : g == 2 ? qs2 : qs3;
            const unsigned a1 = g == 0 ? qs1 : g == 1 ? qs2 : g == 2 ? qs3 : u1;
            if (a0 < c1 && a1 > c0) {
                const float2_t part = *(const float2_t*)(base + (size_t)g * M * kRowsStride);
                z0 += part.x;
                z1 += part.y;
            }
        }
    };
    // the workgroup that unit x of the launch belongs to
    auto owner = [&](unsigned x) {
        const unsigned big = rem * (q + 1);
        if constexpr (GROUPED) return x < big ? x / (q + 1) : rem + (x - big) / q;
        if (S) return div_exact(x, p.m_tr) * S + (x % TR4 ? S - 1 : 0u);     // asked for a block's first or last unit
        return x < big ? div_exact(x, p.m_q1) : rem + div_exact(x - big, p.m_q);
    };

    if constexpr (PAIR) {
        // ---- finish: a wave takes (pair, row) vectors, two columns a lane of gate, of up and of what follows them
        const unsigned P0 = cb_first >> 1, P1 = cb_last >> 1, PU = 2 * TR4;
        const bool first_shared = !(u0 == P0 * PU && u1 >= (P0 + 1) * PU), last_shared = P1 > P0 && u1 < (P1 + 1) * PU;
        struct Scales {
            half2_t sv[2], su;
        };
        auto scales = [&](const unsigned pair) -> Scales {
            const int n0 = (int)pair * 128;
            return {{((global_ptr<const half2_t>)as_global(p.slice[0].svh + n0))[lane], ((global_ptr<const half2_t>)as_global(p.slice[1].svh + n0))[lane]},
                    ((global_ptr<const half2_t>)as_global(p.suh + n0))[lane]};
        };
        auto finish_row = [&](const unsigned pair, const int row, float (&z)[2][2], const Scales& sc) {
            half2_t gu[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                had128_wave(z[h][0], z[h][1], lane);
                gu[h].x = (_Float16)rounded((z[h][0] * kRsqrt128) * (float)sc.sv[h].x);
                gu[h].y = (_Float16)rounded((z[h][1] * kRsqrt128) * (float)sc.sv[h].y);
            }
            half2_t x;
            x.x = silu_mul_h(gu[0].x, gu[1].x);
            x.y = silu_mul_h(gu[0].y, gu[1].y);
            float v0 = __builtin_fmaf((float)x.x, (float)sc.su.x, 0.0f), v1 = __builtin_fmaf((float)x.y, (float)sc.su.y, 0.0f);
            had128_wave(v0, v1, lane);
            half2_t o;
            o.x = (_Float16)had_scale(v0, kRsqrt128);
            o.y = (_Float16)had_scale(v1, kRsqrt128);
            const int col = (int)pair * 128 + 2 * lane;
            const size_t at = (size_t)row * p.N + col;
            *(global_ptr<half2_t>)(as_global((_Float16*)p.slice[0].c) + at) = gu[0];
            *(global_ptr<half2_t>)(as_global((_Float16*)p.slice[1].c) + at) = p.keep_up ? gu[1] : x;
            *(global_ptr<half2_t>)(as_global(p.act_had) + at) = o;
            if (p.operand) *(global_ptr<half2_t>)(as_global(p.operand) + rows_operand_offset(row, col & ~7, p.operand_mt) + (col & 7)) = o;
        };
        // the partial sums: [workgroup][first or last pair][gate, up][M][128]
        auto slot = [&](unsigned x, unsigned which) { return p.partials + ((size_t)x * 4 + which) * M * 128; };
        for (unsigned pair = P0; pair <= P1; ++pair) {
            const bool shared = (pair == P0 && first_shared) || (pair == P1 && last_shared);
            for (int row = wave; row < M; row += kRowsWaves) {
                float z[2][2] = {};
#pragma unroll
                for (unsigned h = 0; h < 2; ++h) {
                    const unsigned cbx = 2 * pair + h;
                    if (cbx < cb_first || cbx > cb_last) continue;
                    own_sum(cbx - cb_first, row, z[h][0], z[h][1]);
                    if (!shared) continue;
                    unsigned long long* const dst = (unsigned long long*)(slot(w, (pair == P0 ? 0u : 2u) + h) + row * 128) + lane;
                    __hip_atomic_store(dst, __builtin_bit_cast(unsigned long long, float2_t{z[h][0], z[h][1]}), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                }
                if (!shared) finish_row(pair, row, z, scales(pair));
            }
        }
        if (!first_shared && !last_shared) return;
        wait_own_stores();
        __syncthreads();
        if (threadIdx.x < 2) {
            unsigned done = 0;
            if (threadIdx.x == 0 ? first_shared : last_shared) {
                const unsigned pair = threadIdx.x == 0 ? P0 : P1;
                const unsigned parts = owner(pair * PU + PU - 1) - owner(pair * PU) + 1;
                unsigned* const counter = p.counters + (size_t)pair * p.cstride;
                const unsigned old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (old == parts - 1) {
                    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    done = 1;
                }
            }
            flags[threadIdx.x] = done;
        }
        __syncthreads();
        // The wave's one or two rows of a pair together, four parts of gate and of up at a time (there are seldom more).
        constexpr int kRowsEach = MT;
#pragma unroll 1
        for (int t = 0; t < 2; ++t) {
            if (!__builtin_amdgcn_readfirstlane((int)flags[t])) continue;
            const unsigned pair = t == 0 ? P0 : P1;
            const Scales sc = scales(pair);
            const unsigned wp = owner(pair * PU);       // only the pair's first sharer may have begun ahead of it
            const unsigned base_p = S || wp * q + min(wp, rem) >= pair * PU ? 0u : 2u;
            unsigned wa[2], wb[2];
#pragma unroll
            for (unsigned h = 0; h < 2; ++h) {
                wa[h] = owner((2 * pair + h) * TR4);
                wb[h] = owner((2 * pair + h) * TR4 + TR4 - 1);
            }
            float z[kRowsEach][2][2] = {};
            for (unsigned x = 0; x <= max(wb[0] - wa[0], wb[1] - wa[1]); x += 4) {
                float2_t part[kRowsEach][2][4];
#pragma unroll
                for (int j = 0; j < kRowsEach; ++j)
#pragma unroll
                    for (unsigned h = 0; h < 2; ++h)
#pragma unroll
                        for (unsigned i = 0; i < 4; ++i) {
                            const unsigned xi = min(wa[h] + x + i, wb[h]);
                            const unsigned long long* const src =
                                (const unsigned long long*)(slot(xi, (xi == wp ? base_p : 0u) + h) + min(wave + 16 * j, M - 1) * 128) + lane;
                            part[j][h][i] = __builtin_bit_cast(float2_t, __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                        }
#pragma unroll
                for (int j = 0; j < kRowsEach; ++j)
#pragma unroll
                    for (unsigned h = 0; h < 2; ++h)
#pragma unroll
                        for (unsigned i = 0; i < 4; ++i)
                            if (wa[h] + x + i <= wb[h]) {
                                z[j][h][0] += part[j][h][i].x;
                                z[j][h][1] += part[j][h][i].y;
                            }
            }
#pragma unroll
            for (int j = 0; j < kRowsEach; ++j)
                if (wave + 16 * j < M) finish_row(pair, wave + 16 * j, z[j], sc);
        }
        return;
    }

    // ---- finish: a wave takes (column block, row) vectors, two columns a lane
    auto store_row = [&](const RowsBlock& b, unsigned cbi, int row, float z0, float z1) {
        had128_wave(z0, z1, lane);
        const half2_t sv = as_half2(sv_lds[cbi * 64 + lane]);
        z0 = (z0 * kRsqrt128) * (float)sv.x;
        z1 = (z1 * kRsqrt128) * (float)sv.y;
        const size_t at = (size_t)row * b.ldc + b.n0 + 2 * lane;
        if (p.out_fp32) {
            if (p.out_add) {
                const float2_t add = *(global_ptr<const float2_t>)(as_global(p.out_add) + at);
                z0 += add.x;
                z1 += add.y;
            }
            *(global_ptr<float2_t>)(as_global((float*)b.c) + at) = float2_t{z0, z1};
        } else {
            half2_t o;
            o.x = (_Float16)z0;
            o.y = (_Float16)z1;
            *(global_ptr<half2_t>)(as_global((_Float16*)b.c) + at) = o;
        }
    };
    const bool first_shared = !(u0 == cb_first * TR4 && u1 >= (cb_first + 1) * TR4);
    const bool last_shared = ncb > 1 && u1 < (cb_last + 1) * TR4;
    int row = wave;
    unsigned cbi = 0;
    while (true) {
        if constexpr (GROUPED) {
            for (int n; cbi < ncb && row >= (n = __builtin_amdgcn_readfirstlane(table[cbi].rows)); ++cbi) row -= n;
        } else {
            while (row >= M) {
                row -= M;
                ++cbi;
            }
        }
        if (cbi >= ncb) break;
        const unsigned cbx = cb_first + cbi;
        const RowsBlock b = block(cbx);
        if (!b.empty) {
            float z0 = 0.0f, z1 = 0.0f;
            own_sum(cbi, row, z0, z1);
            if ((cbi == 0 && first_shared) || (cbi == ncb - 1 && last_shared)) {
                unsigned long long* const slot =
                    (unsigned long long*)(p.partials + ((size_t)w * 2 + (cbi == 0 ? 0 : 1)) * M * 128 + row * 128) + lane;
                __hip_atomic_store(slot, __builtin_bit_cast(unsigned long long, float2_t{z0, z1}), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            } else {
                store_row(b, cbi, row, z0, z1);
            }
        }
        row += kRowsWaves;
    }
    if (!first_shared && !last_shared) return;

    // ---- shared column blocks (the first and the last of the range at most): count this
    // workgroup in; the last sharer to arrive adds the parts in k order and finishes the block
    wait_own_stores();
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned done = 0;
        if (threadIdx.x == 0 ? first_shared : last_shared) {
            const unsigned cbx = threadIdx.x == 0 ? cb_first : cb_last;
            const unsigned parts = owner(cbx * TR4 + TR4 - 1) - owner(cbx * TR4) + 1;
            unsigned* const counter = p.counters + (size_t)cbx * p.cstride;
            const unsigned old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (old == parts - 1) {
                __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                done = 1;
            }
        }
        flags[threadIdx.x] = done;
    }
    __syncthreads();
#pragma unroll 1
    for (int t = 0; t < 2; ++t) {
        if (!__builtin_amdgcn_readfirstlane((int)flags[t])) continue;
        const unsigned cbx = t == 0 ? cb_first : cb_last;
        const RowsBlock b = block(cbx);
        if (b.empty) continue;
        const unsigned wa = owner(cbx * TR4), wb = owner(cbx * TR4 + TR4 - 1);
        // the block is the first of every sharer's range but, unless that starts with it, the first sharer's
        const unsigned slot_a = S || wa * q + min(wa, rem) >= cbx * TR4 ? 0u : 1u;
        for (int r = wave; r < (GROUPED ? b.rows : M); r += kRowsWaves) {
            float z0 = 0.0f, z1 = 0.0f;
            for (unsigned x = wa; x <= wb; x += 8) {
                float2_t part[8];
#pragma unroll
                for (unsigned i = 0; i < 8; ++i) {
                    const unsigned xi = min(x + i, wb);
                    const unsigned long long* const src =
                        (const unsigned long long*)(p.partials + ((size_t)xi * 2 + (xi == wa ? slot_a : 0u)) * M * 128 +
                                                    r * 128) + lane;
                    part[i] = __builtin_bit_cast(float2_t, __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                }
#pragma unroll
                for (unsigned i = 0; i < 8; ++i)
                    if (x + i <= wb) {
                        z0 += part[i].x;
                        z1 += part[i].y;
                    }
            }
            store_row(b, cbx - cb_first, r, z0, z1);
        }
    }
}

}  // namespace berth
