// EXL3 linear for more than 32 rows: row blocks of up to 128 rows, every weight decoded once per
// block and multiplied on the matrix units while other waves decode.
//
//   c = Hh(a_had @ W) * svh (+ out_add),   a_had = Hh(a * suh) rotated by an earlier launch
//
// What bounds it: issue and power.  Per step a wave decodes 32 weights a lane (about 140 vector
// instructions) and issues 4 * MT v_mfma_f32_16x16x32_f16.  In loops of nothing else the decode of a
// step takes 1.15 us (at 2.16 GHz, what the card holds under it) and the MFMAs of 128 rows 1.36 us
// (1.66 GHz); both, interleaved in their proportion, 1.65 us; the kernel 1.9.  (Eight waves of
// 32x32x16 MFMAs, decode interleaved by the instruction, loads three half steps ahead: 2.05.)
//
//   * Tile: rows_per_tile = 16 * MT rows x 128 columns, MT 3 to 8: a block of 112 rows as one of 128, with a
//     row tile of nothing, cost a layer of 100 rows 4 % (one of 72 rows as 96: 5 %).  Tiles of one
//     column block are neighbours, so their weights are in the caches for the next row block.
//   * Sixteen waves: four column groups of 32 columns x four k groups.  A step is 256 rows of K,
//     64 per k group (octet layout and operand assignment as in the few-row kernel).
//   * The k groups 0, 1 and 2, 3 run half a step apart, a barrier between the halves: while one
//     pair decodes, the other multiplies.  A SIMD holds one wave of each k group, so both of its
//     pipes always have two waves to choose from; left to themselves, waves that meet at one
//     barrier per step decode together and then queue for the matrix pipe.
//   * A tile, double-buffered: 256 k of every row, from the copy of the rotated rows in operand
//     order (rows_operand_offset) by direct global-to-LDS loads of 1 KB.  In memory a step is one
//     contiguous run, so the workgroups of a die draw on all channels of its L2, and operand
//     reads from LDS are lane-linear.
//   * The steps of the launch, tile-major, are dealt out evenly to one workgroup per compute unit
//     (or, with few tiles, each tile is cut into S parts).  At the end of a tile the k groups' sums
//     meet in LDS, in two exchanges of which every wave takes its part: a step each of half of the row
//     tiles and of a quarter, so that all sixteen waves add, and leave a quarter of the tile in rows.
//     (Half of the waves adding, then a quarter, which left the rows: layers of 64 and 120 rows 141.8 ->
//     139.3 and 194.3 -> 184.9 us, the latter also for nine registers that went to scratch memory.)  A tile inside one workgroup's steps is finished there; of a shared one every
//     sharer leaves its sums in the workspace, and a second launch adds them in k order and
//     finishes it (exl3_gemm_finish_kernel: inside the first launch the same work falls to the
//     last sharer alone, which reads half a megabyte per tile through one compute unit: 28 us
//     instead of 13 outside the steps).
//
// Measured (27B layer, 4 bits, whole layer on the host clock, against 32-row and 128-row tiles): 33
// rows 181 -> 135 us, 64 rows 196 -> 151, 100 rows 245 -> 190, 256 rows 420 -> 311, 384 rows 548 -> 441.  With
// odd heights and the exchanges as they are now (another box) 40 rows 131.0 -> 125.4, 72 158 -> 149, 100 185 -> 171, 136 235 -> 222.
#pragma once

#include "exl3_gemm_rows_kernel.cuh"

namespace berth {

__host__ __device__ constexpr size_t block_lds_bytes(int mt)
{
    // A buffers / the k groups' sums on their way (16 KB per 16 rows); then the output scales
    return (size_t)mt * 16384 + 256;
}

// Sixteen bytes a lane from base + offset to LDS at lds_at + 16 * lane.  m0 is an output, so that the
// compiler knows it is written; the s_nop is the wait state between that and the load.  (As an input,
// set by the compiler, the loads move behind the last MFMA of their sixteen rows: 64 rows 5120x17408
// 37.0 -> 37.3 us.)  The compiler sees neither a load here nor what it writes: whoever reads or
// overwrites the bytes waits first.  (__builtin_amdgcn_global_load_lds from an LDS offset gets no waits
// either, and takes its address in a pair of vector registers instead of the scalar base.)
__device__ __forceinline__ void load_to_lds(const char* base, uint32_t offset, uint32_t lds_at)
{
    uint32_t m0;
    asm volatile("s_mov_b32 %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
                 : "={m0}"(m0) : "s"(lds_at), "v"(offset), "s"(base) : "memory");
}

// The end of one output row of a 128-column block, sixteen lanes with eight sums each: Hadamard, svh,
// the optional addend, the store (`live` false: a lane group past the last row, which only takes part
// in the exchanges).
__device__ __forceinline__ void block_finish_row(const GemmParams& p, const RowsBlock& b, float (&v)[8], const half8_t sv,
                                                 const int row, const bool live, const int lane)
{
    const float unit = had128_row16(v, lane) * kRsqrt128;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = had_scale(v[e], unit) * (float)sv[e];
    if (!live) return;
    const size_t at = (size_t)row * b.ldc + b.n0 + 8 * had_chunk(lane);
    if (p.out_fp32) {
        if (p.out_add) {
            const global_ptr<const float4_t> add = (global_ptr<const float4_t>)(as_global(p.out_add) + at);
            const float4_t a0 = add[0], a1 = add[1];
#pragma unroll
            for (int e = 0; e < 4; ++e) { v[e] += a0[e]; v[4 + e] += a1[e]; }
        }
        const global_ptr<float4_t> dst = (global_ptr<float4_t>)(as_global((float*)b.c) + at);
        dst[0] = float4_t{v[0], v[1], v[2], v[3]};
        dst[1] = float4_t{v[4], v[5], v[6], v[7]};
    } else {
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (_Float16)v[e];
        *(global_ptr<half8_t>)(as_global((_Float16*)b.c) + at) = o;
    }
}

template <int BITS, int CB, int MT>         // MT: tiles of 16 rows of a block
__global__ __launch_bounds__(1024, 1) void exl3_gemm_block_kernel(GemmParams p)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int tile_dw = 8 * BITS;
    constexpr int kBuf = MT * 8192;                     // bytes of one A buffer: [k group][row tile][k half][lane][16]
    constexpr int kLoads = (MT + 1) / 2;                // A loads of a wave per step
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cg = wave & 3, kg = wave >> 2;
    const int l16 = lane & 15, lg = lane >> 4;
    const unsigned TR4 = (unsigned)p.K >> 6;
    const unsigned SPT = (TR4 + 3) >> 2;                // steps per tile
    const unsigned RT = (unsigned)p.tiles_y;            // row blocks
    constexpr int BM = 16 * MT;

    // ---- this workgroup's steps [u0, u1)
    const unsigned w = blockIdx.x;
    const unsigned q = (unsigned)p.unit_q, rem = (unsigned)p.unit_r;
    const unsigned S = (unsigned)p.S;
    unsigned u0 = w * q + min(w, rem), u1 = (w + 1) * q + min(w + 1, rem);
    if (S) {
        const unsigned tile = div_exact(w, p.m_s), part = w - tile * S;
        u0 = tile * SPT + div_exact(part * SPT, p.m_s);
        u1 = tile * SPT + div_exact((part + 1) * SPT, p.m_s);
    }
    const unsigned t_first = div_exact(u0, p.m_tr), t_last = div_exact(u1 - 1, p.m_tr);

    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    uint32_t* const sv_lds = (uint32_t*)(smem + MT * 16384);

    // ---- operands
    uint32_t own[2][BITS];
    const char* t_base = nullptr;                       // trellis of the segment's tile, this wave's k group, step 0
    long t_step = 0;                                    // bytes per step
    uint32_t t_off = 0, t_kg = 0;                       // per lane; bytes from k group 0 to this one
    const char* a_base = nullptr;                       // rotated rows of the tile
    constexpr uint32_t a_unit = (uint32_t)BM * 128;     // bytes of 64 k of the block
    auto seek = [&](unsigned tile) {
        const unsigned cb = div_exact(tile, p.m_rt);
        const RowsBlock b = rows_block(p, cb);
        a_base = (const char*)rows_uniform(b.a_had + (size_t)((tile - cb * RT) * (unsigned)BM) * p.K);
        if (b.empty) {                                  // read anything valid, use nothing
            t_base = a_base;
            t_step = 0;
            t_off = t_kg = 0;
        } else {
            const uint32_t row_bytes = (uint32_t)(b.ldc >> 4) * (tile_dw * 4);
            t_step = 16 * (long)row_bytes;
            t_kg = (uint32_t)kg * 4 * row_bytes;
            t_base = (const char*)rows_uniform(b.trellis) + (size_t)(b.n0 >> 4) * (tile_dw * 4) + t_kg;
            t_off = (uint32_t)lg * row_bytes + (uint32_t)(cg * 16 + l16) * (BITS * 4);
        }
    };
    auto fetch_t = [&](int j, unsigned s) {
        // (in the last step of a K that is no multiple of 256 a k group may have no rows: it reads those of group 0)
        const char* src = t_base + (size_t)s * t_step - (s * 4 + (unsigned)kg < TR4 ? 0u : t_kg);
        load_tile_dwords<BITS>((global_ptr<const uint32_t>)(as_global(src) + t_off), own[j]);
    };
    auto a_source = [&](unsigned s) {
        return a_base + (size_t)(s * 4 + (s * 4 + (unsigned)kg < TR4 ? (unsigned)kg : 0u)) * a_unit;
    };
    auto fetch_a = [&](const char* src, int buf, int j) {       // (MT odd: the last piece again)
        const uint32_t at = min((uint32_t)(cg * kLoads + j) * 1024u, a_unit - 1024u);
        load_to_lds(src + at, (uint32_t)lane * 16, lds0 + (uint32_t)(buf * kBuf + kg * 2048 * MT) + at);
    };
    const uint32_t ra = (uint32_t)(kg * 2048 * MT + lane * 16);     // this lane's part of its k group's first operand

    float4_t acc[MT][2];
    auto stage = [&](int j, unsigned s, unsigned last) {
        const uint32_t prev = fetch_prev(lane, own[j][BITS - 1]);
        uint32_t w2[16];
        decode_lane<BITS, CB>(own[j], prev, w2);
        if (s * 4 + (unsigned)kg >= TR4) {              // a k group past the end of K multiplies zeros
#pragma unroll
            for (int i = 0; i < 16; ++i) w2[i] = 0;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(w2[i]));       // decoded here, not behind the barrier
        // (the wait and the barrier are also the two wait states that `settle` puts before an MFMA)
        // this step's A loads of this wave are older than the next step's trellis loads (one or
        // more), so they have landed when at most one load is outstanding; behind the barrier the
        // other three waves' have, too, and everybody has left the other buffer
        asm volatile("s_waitcnt vmcnt(1)\n\ts_barrier" ::: "memory");
        // (on the segment's last step the loads bring in the same step again, unused: no branch)
        const char* const next = a_source(min(s + 1, last));
        half8_t b[2][2];                                // [k half][column half]
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                const uint4 v = {w2[2 * f + h], w2[4 + 2 * f + h], w2[8 + 2 * f + h], w2[12 + 2 * f + h]};
                b[h][f] = __builtin_bit_cast(half8_t, v);
            }
        // the operands of the next sixteen rows are read behind the MFMAs of these
        const unsigned char* const a0 = smem + j * kBuf + ra;
        const unsigned char* const a1 = a0 + 1024;
        half8_t x[2][2];
        x[0][0] = *(const half8_t*)a0;
        x[0][1] = *(const half8_t*)a1;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            if (mt + 1 < MT) {
                x[(mt + 1) & 1][0] = *(const half8_t*)(a0 + (mt + 1) * 2048);
                x[(mt + 1) & 1][1] = *(const half8_t*)(a1 + (mt + 1) * 2048);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int f = 0; f < 2; ++f)
                    acc[mt][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[mt & 1][h], b[h][f], acc[mt][f], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // the next step's loads go out one at a time behind MFMAs: issued together ahead of
            // them they hold every wave of the group up at the memory pipe
            if (mt < kLoads) fetch_a(next, j ^ 1, mt);
            else if (mt == kLoads) fetch_t(j, min(s + 2, last));
        }
        asm volatile("s_barrier" ::: "memory");
    };

    seek(t_first);
    {
        const unsigned s0 = u0 - t_first * SPT, s1 = min(SPT, s0 + (u1 - u0));
        fetch_t(0, s0);
        fetch_t(1, min(s0 + 1, s1 - 1));
    }
    for (unsigned tile = t_first; tile <= t_last; ++tile) {
        const unsigned base = tile * SPT;
        const unsigned s0 = u0 > base ? u0 - base : 0u, s1 = min(SPT, u1 - base);
        const unsigned cb = div_exact(tile, p.m_rt);
        const RowsBlock b = rows_block(p, cb);
        const int m0 = (int)(tile - cb * RT) * BM;
        const int rows = min(BM, p.M - m0);
        uint32_t sv_mine = 0;
        if (wave == 0 && !b.empty) sv_mine = as_global((const uint32_t*)(b.svh + b.n0))[lane];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt][0] = acc[mt][1] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < kLoads; ++j) fetch_a(a_source(s0), 0, j);
        // (the segment's first trellis loads are older than these: its first step waits for everything)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (kg >= 2) asm volatile("s_barrier" ::: "memory");       // half a step behind
        unsigned s = s0;
        for (; s + 1 < s1; s += 2) {
            stage(0, s, s1 - 1);
            stage(1, s + 1, s1 - 1);
        }
        if (s < s1) stage(0, s, s1 - 1);
        // The last step's A loads bring nothing that is used, but they land in the buffers that the register
        // dumps lie over, some of them in another wave's dump: every wave has its own behind it before
        // the first barrier of the finish.  Ahead of the next tile's trellis loads, which go on.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (kg < 2) asm volatile("s_barrier" ::: "memory");
        if (tile < t_last) {                            // the next tile's first steps, behind the finish of this one
            seek(tile + 1);
            fetch_t(0, 0);
            fetch_t(1, min(1u, min(SPT, u1 - base - SPT) - 1));
        }
        // ---- the k groups' sums, (0 + 2) + (1 + 3): groups kg and kg ^ 2 exchange every other row tile, kg and
        // kg ^ 1 every other one of those that they kept.  A row tile has a place for either parity of the
        // group that reads it first; what a wave has read there is its own to write.
        int at = lane;                                  // (what follows from it is worked out here, not kept over the steps)
        asm volatile("" : "+v"(at));
        const int par = kg & 1, hi = kg >> 1;
        unsigned char* const mine = smem + par * 8192 + cg * 2048 + at * 16;
        __syncthreads();
        constexpr int kHalf = (MT + 1) / 2, kQuarter = (MT + 3) / 4;
        float4_t half[kHalf][2], sum[kQuarter][2];
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
            const bool both = 2 * i + 1 < MT;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                if (hi) {
                    *(float4_t*)(mine + 2 * i * 16384 + f * 1024) = acc[2 * i][f];
                    if (both) half[i][f] = acc[both ? 2 * i + 1 : 0][f];
                } else {
                    if (both) *(float4_t*)(mine + (2 * i + 1) * 16384 + f * 1024) = acc[both ? 2 * i + 1 : 0][f];
                    half[i][f] = acc[2 * i][f];
                }
            }
        }
        if (wave == 0) sv_lds[at] = sv_mine;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kHalf; ++i) {
            if (2 * i + 1 < MT || !hi) {
#pragma unroll
                for (int f = 0; f < 2; ++f) half[i][f] += *(const float4_t*)(mine + (2 * i + hi) * 16384 + f * 1024);
            }
        }
#pragma unroll
        for (int j = 0; j < kQuarter; ++j) {
            const bool both = 2 * j + 1 < kHalf;
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                if (par) {
                    if (4 * j + 1 < MT || !hi) *(float4_t*)(mine + (4 * j + hi) * 16384 + f * 1024) = half[2 * j][f];
                    if (both) sum[j][f] = half[both ? 2 * j + 1 : 0][f];
                } else {
                    if (both && (4 * j + 3 < MT || !hi)) *(float4_t*)(mine + (4 * j + 2 + hi) * 16384 + f * 1024) = half[both ? 2 * j + 1 : 0][f];
                    sum[j][f] = half[2 * j][f];
                }
            }
        }
        __syncthreads();
        // Row-major, 16 x 32 of a column group together; four columns at a time change places so that neither side
        // meets more than two lanes of a bank.
        const int l16e = at & 15, lge = at >> 4;
        const uint32_t z_lane = (uint32_t)lge * 512 + (uint32_t)((((l16e >> 3) * 4 + ((l16e >> 2) & 1)) ^ (cg & 1) ^ (2 * (lge & 1))) * 16 + (l16e & 3) * 4);
#pragma unroll
        for (int j = 0; j < kQuarter; ++j) {
            const int mt = 4 * j + 2 * par + hi;
            if (mt < MT) {
                const unsigned char* const other = smem + (2 * mt + 1 - par) * 8192 + cg * 2048 + at * 16;
                unsigned char* const row = smem + (2 * mt + par) * 8192 + cg * 2048;
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    const float4_t v = sum[j][f] + *(const float4_t*)(other + f * 1024);
#pragma unroll
                    for (int r = 0; r < 4; ++r) *(float*)(row + (z_lane ^ (uint32_t)(f * 32)) + r * 128) = v[r];
                }
            }
        }
        __syncthreads();
        if (!b.empty) {
            // sixteen lanes a row, eight columns each: a wave takes four rows at a time
            const int chunk = had_chunk(at);
            const bool whole = s0 == 0 && s1 == SPT;
            float* const part = p.partials + ((size_t)w * 2 + (tile == t_first ? 0 : 1)) * BM * 128;
            const uint32_t z_read = (uint32_t)((wave >> 2) * 2 + (wave >> 3)) * 8192 + (uint32_t)(chunk >> 2) * 2048 +
                                    (uint32_t)((wave & 3) * 4 + lge) * 128 +
                                    (uint32_t)(((chunk & 3) * 2) ^ ((chunk >> 2) & 1) ^ (2 * (wave & 1))) * 16;
#pragma unroll
            for (int pass = 0; pass < kQuarter; ++pass) {
                const int r = pass * 64 + wave * 4 + lge;
                if (pass * 64 + wave * 4 >= rows) break;
                const float4_t v0 = *(const float4_t*)(smem + pass * 65536 + z_read);
                const float4_t v1 = *(const float4_t*)(smem + pass * 65536 + (z_read ^ 16u));
                if (whole) {
                    float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
                    block_finish_row(p, b, v, ((const half8_t*)sv_lds)[chunk], m0 + r, r < rows, at);
                } else if (r < rows) {
                    const global_ptr<float4_t> dst = (global_ptr<float4_t>)as_global(part + r * 128 + 8 * chunk);
                    dst[0] = v0;
                    dst[1] = v1;
                }
            }
        }
        __syncthreads();                                // the next tile's A loads land here
    }
}

// The workgroups that share a tile of the row-block launch, and the partial-sum slot of the first of them
// (the tile is the first of every other sharer's range).
struct TileSharers {
    unsigned first, last, slot_first;
};
__device__ __forceinline__ TileSharers tile_sharers(const GemmParams& p, const unsigned tile)
{
    const unsigned SPT = (((unsigned)p.K >> 6) + 3) >> 2;
    const unsigned q = (unsigned)p.unit_q, rem = (unsigned)p.unit_r, S = (unsigned)p.S;
    auto owner = [&](unsigned x) {
        const unsigned big = rem * (q + 1);
        return x < big ? div_exact(x, p.m_q1) : rem + div_exact(x - big, p.m_q);
    };
    TileSharers t;
    t.first = S ? tile * S : owner(tile * SPT);
    t.last = S ? tile * S + S - 1 : owner(tile * SPT + SPT - 1);
    t.slot_first = S || t.first * q + min(t.first, rem) >= tile * SPT ? 0u : 1u;
    return t;
}
// The sums of row r of the tile, columns 8 * chunk .. + 7: those of four sharers from x on (past the last: the last
// again), added in k order.
struct SharerSums {
    float4_t part[4][2];
};
__device__ __forceinline__ SharerSums load_sharers(const GemmParams& p, const TileSharers t, const unsigned x, const int r, const int chunk)
{
    SharerSums s;
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
        const unsigned xi = min(x + i, t.last);
        const global_ptr<const float4_t> src = (global_ptr<const float4_t>)as_global(
            p.partials + ((size_t)xi * 2 + (xi == t.first ? t.slot_first : 0u)) * p.rows_per_tile * 128 + r * 128 + 8 * chunk);
        s.part[i][0] = src[0];
        s.part[i][1] = src[1];
    }
    return s;
}
__device__ __forceinline__ void add_sharers(const TileSharers t, const unsigned x, const SharerSums& s, float (&v)[8])
{
#pragma unroll
    for (unsigned i = 0; i < 4; ++i)
        if (x + i <= t.last) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += s.part[i][e >> 2][e & 3];
        }
}

// Finishes the tiles that several workgroups of the launch before share: adds their sums in k order,
// then output Hadamard, svh, the optional addend and the store.  blockIdx.x = tile, blockIdx.y =
// sixteen rows of it; sixteen lanes a row, eight columns each.  Bound by the bytes of the sums,
// which are still in the caches.
static __global__ __launch_bounds__(256) void exl3_gemm_finish_kernel(GemmParams p)
{
    const unsigned RT = (unsigned)p.tiles_y;
    const unsigned tile = blockIdx.x;
    const TileSharers t = tile_sharers(p, tile);
    if (t.first == t.last) return;                      // finished by its only workgroup
    const unsigned cb = div_exact(tile, p.m_rt);
    const RowsBlock b = rows_block(p, cb);
    if (b.empty) return;
    const int lane = threadIdx.x & 63, chunk = had_chunk(lane);
    const int BM = p.rows_per_tile, m0 = (int)(tile - cb * RT) * BM;
    const int row = (int)blockIdx.y * 16 + (int)(threadIdx.x >> 4);
    const int rows = min(BM, p.M - m0);
    if ((int)blockIdx.y * 16 + (int)(threadIdx.x >> 6) * 4 >= rows) return;
    const int r = min(row, rows - 1);
    const half8_t sv = ((global_ptr<const half8_t>)as_global(b.svh + b.n0))[chunk];
    float v[8] = {};
    for (unsigned x = t.first; x <= t.last; x += 4) add_sharers(t, x, load_sharers(p, t, x, r, chunk), v);
    block_finish_row(p, b, v, sv, m0 + row, row < rows, lane);
}

// Finishes gate and up of an MLP (the two slices of the launch before) and forms the input of the down
// projection: a workgroup takes the same sixteen rows and 128 columns of both, so that silu(g) * u and its
// rotation need no launch of their own behind this one that reads both back.  Gate goes to its output,
// the activation where up would have gone, the rotated rows to act_had and, in operand order, to `operand`
// (may be null).  blockIdx.x = row block and column block of gate as the tiles are numbered, blockIdx.y = sixteen
// rows of it.  The values are those of exl3_gemm_finish_kernel and silu_mul_had_r_128_kernel.
// Bound by latency and the bytes of the sums, 16 to 32 bytes per value of gate and up: everything a row needs is asked
// for at once (with the loads of gate waited for before those of up a layer of 40 rows took 1 us more).  Decoder
// layers with an MLP of 5120 x 17408, instead of a finish, silu_mul_had_r_128_kernel and a second entry of the host:
// 40 rows 132.8 -> 128.5 us, 100 rows 182.8 -> 178.4, 130 rows 232.1 -> 227.3; MLP widths 2048 x 5632, 100 rows
// 101.6 -> 98.5; where gate and up take another kernel (250 and 400 rows) the same.
struct FinishActivation {
    const _Float16* suh;        // input scales of the down projection
    _Float16* act_had;
    _Float16* operand;
    int mt;                     // tiles of 16 rows of a block of the operand copy
};
static __global__ __launch_bounds__(256) void exl3_gemm_silu_mul_finish_kernel(GemmParams p, FinishActivation f)
{
    const unsigned RT = (unsigned)p.tiles_y, tiles = gridDim.x;
    const unsigned cb = div_exact(blockIdx.x, p.m_rt);
    const int lane = threadIdx.x & 63, chunk = had_chunk(lane);
    const int m0 = (int)(blockIdx.x - cb * RT) * p.rows_per_tile;
    const int rows = min(p.rows_per_tile, p.M - m0);
    if ((int)blockIdx.y * 16 + (int)(threadIdx.x >> 6) * 4 >= rows) return;
    const int row = (int)blockIdx.y * 16 + (int)(threadIdx.x >> 4);
    const int r = min(row, rows - 1);                   // (lane groups past the last row redo it, and store nothing)
    const bool live = row < rows;
    const size_t at = (size_t)(m0 + r) * p.N + cb * 128 + 8 * chunk;
    const half8_t su = ((global_ptr<const half8_t>)as_global(f.suh + cb * 128))[chunk];
    half8_t gu[2], sv[2];
    TileSharers t[2];
    SharerSums sums[2];
    float v2[2][8] = {};
    // everything that is read is asked for together: four sharers of either tile (there are seldom more), or, of a
    // tile that its only workgroup has finished, the result
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        t[s] = tile_sharers(p, blockIdx.x + (unsigned)s * tiles);
        sv[s] = ((global_ptr<const half8_t>)as_global(p.slice[s].svh + cb * 128))[chunk];
        if (t[s].first == t[s].last) gu[s] = *(global_ptr<const half8_t>)(as_global((const _Float16*)p.slice[s].c) + at);
        else sums[s] = load_sharers(p, t[s], t[s].first, r, chunk);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (t[s].first == t[s].last) continue;
        add_sharers(t[s], t[s].first, sums[s], v2[s]);
        for (unsigned x = t[s].first + 4; x <= t[s].last; x += 4) add_sharers(t[s], x, load_sharers(p, t[s], x, r, chunk), v2[s]);
        const float unit = had128_row16(v2[s], lane) * kRsqrt128;
#pragma unroll
        for (int e = 0; e < 8; ++e) gu[s][e] = (_Float16)rounded(had_scale(v2[s][e], unit) * (float)sv[s][e]);
        if (s == 0 && live) *(global_ptr<half8_t>)(as_global((_Float16*)p.slice[0].c) + at) = gu[0];
    }
    half8_t x;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = silu_mul_h(gu[0][e], gu[1][e]);
    float v[8];
    mul_half8(x, su, v);
    const float unit = had128_row16(v, lane) * kRsqrt128;
    half8_t o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (_Float16)had_scale(v[e], unit);
    if (!live) return;
    *(global_ptr<half8_t>)(as_global((_Float16*)p.slice[1].c) + at) = x;
    *(global_ptr<half8_t>)(as_global(f.act_had) + at) = o;
    if (f.operand) {
        const int R = m0 + row, block = R / (16 * f.mt);
        *(global_ptr<half8_t>)(as_global(f.operand) + (size_t)block * rows_operand_elements(p.N, f.mt) +
                               rows_operand_offset(R - block * 16 * f.mt, (int)cb * 128 + 8 * chunk, f.mt)) = o;
    }
}

}  // namespace berth
