// Launchers of the EXL3 MFMA GEMM (exl3_gemm_kernel.cuh): dense rows through
// berth_prefill_exl3_linear / berth_exl3_linear, grouped MoE problems, and the
// plain fp16 GEMM of crates/berth-kernels/csrc/prefill_lin/linear.cu:387-418.
#include "exl3_gemm_block_kernel.cuh"
#include "launch.h"
#include "rows_operand.cuh"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <optional>

namespace berth {

static_assert(kGemmWrittenBase * 2 == kCounters, "the GEMM keeps two counters per tile");
static_assert(kGemmMaxSlices == kBundleMaxSlices, "one limit for the by-value slices of a bundle");

// one translation unit per codebook (exl3_gemm_cb{0,1,2}.hip) keeps the build parallel
void launch_gemm_cb0(const GemmParams& p, int bits, int mb, hipStream_t stream, std::string& desc, dim3 grid);
void launch_gemm_cb1(const GemmParams& p, int bits, int mb, hipStream_t stream, std::string& desc, dim3 grid);
void launch_gemm_cb2(const GemmParams& p, int bits, int mb, hipStream_t stream, std::string& desc, dim3 grid);

static void gemm_bits(const GemmParams& p, int bits, int cb, int mb, hipStream_t stream, std::string& desc, dim3 grid)
{
    switch (cb) {
    case 0: launch_gemm_cb0(p, bits, mb, stream, desc, grid); break;
    case 1: launch_gemm_cb1(p, bits, mb, stream, desc, grid); break;
    default: launch_gemm_cb2(p, bits, mb, stream, desc, grid); break;
    }
}

// split-K factor for `tiles` output tiles of MB*32 x 256: one workgroup per compute unit
// (fewer workgroups share a tile); two for a dense launch of at most 32 rows with at least a
// quarter as many tiles as compute units (a workgroup of four waves leaves a compute unit's
// vector pipes half idle, and each workgroup still keeps several k-blocks: the 27B gate + up
// bundle at 16 rows 63 -> 54 us; with few tiles the extra hand-overs cost more than that, q/k/v
// 24 -> 30 us, and with several row tiles nothing is gained: k at 512 rows 34.9 -> 36.0 us),
// at least two k-blocks per workgroup, inside the workspace
static int gemm_split(const Workspace& ws, long tiles, int KB, int mb, bool one_row_tile = false)
{
    const int per_cu = knobs().gemm_wg_per_cu > 0 ? knobs().gemm_wg_per_cu
                                                  : (mb == 1 && one_row_tile && tiles * 4 >= ws.cu_count ? 2 : 1);
    long S = ((long)ws.cu_count * per_cu + tiles - 1) / tiles;
    if (S > KB / 2) S = KB / 2;
    if (S < 1) S = 1;
    const size_t per_wg = (size_t)4 * mb * 2 * 16 * 64 * sizeof(float);
    while (S > 1 && (size_t)tiles * S * per_wg > kPartialBytes) --S;
    if (tiles > kCounters / 2) S = 1;          // two counters per tile
    return (int)S;
}

// words between the counters of neighbouring tiles (see counter_stride); `tiles` bounds the
// tile count of every launch the call makes
static int gemm_counter_stride(long tiles)
{
    const int cap = knobs().counter_stride;
    int stride = 1;
    while (stride * 2 <= cap && tiles * stride * 2 <= kCounters / 2) stride *= 2;
    return stride;
}

// ---- few rows (exl3_gemm_rows_kernel): how the launch's units are dealt out, and when it applies
struct RowsPlan {
    bool ok = false;
    int mt = 1;                 // tiles of 16 rows
    long units = 0;             // 64 x 128 weights each
    unsigned grid = 0, q = 0, rem = 0, S = 0;
    size_t lds = 0, lds_rotate = 0;
    size_t operand_at = 0;      // bytes into the partial-sum workspace
    bool rotate = false;        // the launch can rotate its input itself
};

static unsigned magic(unsigned d) { return d == 1 ? 0u : (unsigned)((1ull << 32) / d) + 1u; }

// Fewest units for which a launch can take the few-row kernel.  Above 8 rows the alternative is the 32-row MFMA
// kernel, whose hand-over and half-empty rounds cost more from the start (2048 x 1024, 256 units: 14.1 -> 10.6 us at
// 12 rows, 16.0 -> 13.9 at 32).  Up to 8 rows it is the VALU kernel of exl3_gemv.hip, and gemm_rows_applies chooses.
// BERTH_GEMM_ROWS_UNITS replaces both rules (0: never).
static int rows_min_units(int size_m)
{
    const int forced = knobs().gemm_rows_units;
    if (forced >= 0) return forced;
    return size_m <= 8 ? 32 : 192;
}

static RowsPlan plan_rows(const Workspace& ws, int slices, int slabs, int size_m, int size_k, int size_n)
{
    RowsPlan pl;
    const int min_units = rows_min_units(size_m);
    if (min_units <= 0 || size_m < 2 || size_m > 32 || size_k % 64 != 0 || size_n % 128 != 0) return pl;
    const unsigned TR4 = (unsigned)size_k / 64;
    const long blocks = (long)slices * (size_n / 128);
    const unsigned long long U = (unsigned long long)blocks * TR4;
    if (U < (unsigned long long)min_units || U >= (1ull << 30) || blocks > kCounters / 2) return pl;
    if ((unsigned long long)size_m * size_k >= (1ull << 31)) return pl;
    // one workgroup per compute unit with at least a unit per wave group; several rounds of them
    // where the column blocks that a range touches would not fit the LDS together
    for (int rounds = 1; rounds <= 64; rounds *= 2) {
        unsigned long long G = (unsigned long long)ws.cu_count * rounds;
        if (G > U / 4) G = U / 4;
        if (G < 1) return pl;
        unsigned q = (unsigned)(U / G), rem = (unsigned)(U % G), S = 0;
        const unsigned most = q + (rem ? 1 : 0);
        unsigned ncb = (most + TR4 - 2) / TR4 + 1;                  // column blocks a range can touch
        // At least two workgroups per column block: parts of its own for each block where the longest part is no more than
        // an eighth or six units above the even share.  A range across two blocks hands both over (2688 x 4096 at 8 / 32
        // rows: 12.8 / 22.1 -> 11.1 / 16.1 us with parts of its own), and needs the whole input, which a launch ahead of it
        // rotates then: 4096x3072, 7 units instead of 6, at 4 / 8 / 16 / 32 rows 13.2 / 14.5 / 17.7 / 23.5 -> 9.8 / 10.2 / 12.2 /
        // 17.4; 2048x11264, 16 instead of 11, 14.1 / 14.5 / 16.1 / 20.8 -> 11.2 / 11.6 / 12.9 / 17.4; 17408x5632, 55 instead of
        // 47, even (23.3 -> 23.8 at 8 rows, 31.1 -> 28.4 at 32); 5120x11520, 40 instead of 29, 19.2 -> 19.8; 8192x11264, 64
        // instead of 44, 23.2 -> 26.1.  Gate and up whose input the norm's launch rotates, 16 units instead of 11: layers of
        // hidden 2048 at 8 rows 51.0 -> 47.6.
        if (G >= 2 * (unsigned long long)blocks) {
            const unsigned s = (unsigned)(G / blocks), longest = (TR4 + s - 1) / s;
            if (TR4 / s >= 4 && (longest * 8ull <= most * 9ull || longest <= most + 6)) {
                S = s;
                G = (unsigned long long)blocks * s;
                q = rem = 0;
                ncb = 1;
            }
        }
        const size_t lds = rows_lds_bytes(size_m, (int)ncb);
        if (ncb > (unsigned)kRowsWaves || lds > 160 * 1024) continue;
        // exact division by multiply-high needs dividend * divisor < 2^32
        if (U * (q + 2) >= (1ull << 32) || U * TR4 >= (1ull << 32)) return pl;
        // the workspace holds two partial column blocks per workgroup, then the operand copies
        const int mt = size_m <= 16 ? 1 : 2;
        pl.operand_at = (size_t)G * 2 * size_m * 512;
        if (pl.operand_at + slabs * rows_operand_elements(size_k, mt) * 2 > ws.partial_bytes) return pl;
        pl.ok = true;
        pl.mt = mt;
        pl.units = (long)U;
        pl.grid = (unsigned)G;
        pl.q = q;
        pl.rem = rem;
        pl.S = S;
        pl.lds = lds;
        if (S) {
            unsigned nb = 0;                                        // most 128 blocks that a part touches
            for (unsigned s = 0; s < S; ++s) nb = std::max(nb, ((s + 1) * TR4 / S + 1) / 2 - s * TR4 / S / 2);
            pl.lds_rotate = lds + rows_rot_lds_bytes((int)(2 * nb), mt);
            pl.rotate = nb * (unsigned)size_m <= (unsigned)kRowsRotItems && pl.lds_rotate <= 160 * 1024;
        }
        return pl;
    }
    return pl;
}

// Up to 8 rows: units from which the few-row kernel is the quicker one whichever launches stand ahead (4096x8192, 4096
// units, at two rows 13.4 -> 12.8; 4096x2048 with a rotation launch at 2 / 5 / 8 rows 9.8 / 13.4 / 16.8 -> 10.3 / 10.9 / 11.3).
static long rows_large_units(int size_m) { return size_m <= 3 ? 3072 : 1024; }

// Up to 8 rows the VALU kernel of exl3_gemv.hip rotates the input itself, cuts size_k into parts of two k-blocks at
// the least (four waves have a k-block of 512 each), and pays half an instruction per weight and row: 4 bits, K x N,
// us, VALU -> here.
bool gemm_rows_applies(const Workspace& ws, int slices, int size_m, int size_k, int size_n, RowsInput input)
{
    const RowsPlan pl = plan_rows(ws, slices, slices, size_m, size_k, size_n);
    if (!pl.ok || size_m > 8 || knobs().gemm_rows_units >= 0) return pl.ok;
    if (pl.units >= rows_large_units(size_m)) return true;
    if (size_k < 512) return false;         // (256x512 at 2 / 4 / 8 rows 7.2 / 8.5 / 12.6 -> 8.2 / 10.4 / 10.4)
    switch (input) {
    case RowsInput::kSelf:
        // The launch rotates its input itself: one launch either way.  1024x1024 at 2 / 3 / 5 / 8 rows 9.2 / 9.6 / 11.4 /
        // 14.3 -> 8.4 / 8.3 / 8.5 / 8.5, 3072x2048 9.7 / 10.8 / 12.9 / 16.1 -> 8.8 / 9.0 / 9.2 / 9.7; four k-blocks, which
        // the VALU kernel takes in one part without partial sums, 512x2048 at 2 / 3 / 4 / 8 rows 7.3 / 8.1 / 8.9 / 12.8 ->
        // 7.8 / 8.2 / 8.5 / 8.5.
        if (pl.rotate) return size_m >= (size_k < 768 ? 4 : 2);
        break;
    case RowsInput::kNorm:
        // The launch that forms the norm rotates, gate and up leave down's input, the residual is added where down writes:
        // three launches beside five.  Blocks of 512x1024 at 2 / 4 / 8 rows 23.4 / 26.6 / 36.4 -> 20.4 / 20.7 / 20.9,
        // 1024x2048 25.1 / 28.6 / 38.5 -> 23.7 / 24.3 / 24.9, 2048x6144 at two 28.7 -> 25.2, 4096x4096 28.2 -> 28.0.
        return true;
    case RowsInput::kMlp:
        // Three launches beside two: MLPs of 2048x4096 at 2 / 3 rows 19.9 / 21.9 -> 24.1 / 24.4, of 1536x3072 at 4 / 5 / 8
        // rows 23.6 / 25.1 / 29.8 -> 23.9 / 24.6 / 24.7; down alone, 1024 x 2048 at 4 / 5 / 8 rows, saves 0 / 3 / 7.  Up to
        // 1024 of hidden the two launches stay, which the entry states for small weights, although three would be quicker
        // (512x1024 at 2 / 4 / 5 / 8 rows 15.9 / 19.3 / 21.7 / 29.3 beside 15.9 / 16.1 / 16.5 / 16.7, 1024x2048 18.3 / 21.7 / 24.3 /
        // 32.1 beside 19.6 / 19.3 / 19.1 / 20.4).
        return size_m >= 5 && size_k >= 1024 && (slices == 2 ? size_k : size_n) > 1024;
    case RowsInput::kLaunch:
        break;
    }
    // Two launches beside one: q / k / v of 1024 x (2048, 256, 256) at 4 / 5 / 8 rows 10.8 / 12.0 / 15.5 -> 11.9 / 11.8 /
    // 11.8, of 512 x (512, 128, 128) at five 10.6 -> 11.9.
    return size_m >= 5 && size_k >= 1024;
}

// rotate: p is a GemmRotateParams; pair: a RowsPairParams
static void run_rows(const RowsPlan& pl, GemmParams& p, bool rotate, int k_bits, int codebook, hipStream_t stream, std::string& desc,
                     bool pair = false)
{
    p.cstride = gemm_counter_stride((long)(p.num_slices > 0 ? p.num_slices : 1) * (p.N / 128));
    p.units = (int)pl.units;
    p.unit_q = (int)pl.q;
    p.unit_r = (int)pl.rem;
    p.m_tr = magic((unsigned)p.K / 64);
    p.m_nb = magic((unsigned)p.N / 128);
    p.S = (int)pl.S;
    p.m_s = pl.S ? magic(pl.S) : 0;
    p.m_q = pl.S ? 0u : magic(pl.q);
    p.m_q1 = magic(pl.q + 1);
    p.lds_bytes = (unsigned)(rotate ? pl.lds_rotate : pl.lds);
    if (rotate) static_cast<GemmRotateParams&>(p).m_rows = magic((unsigned)p.M);
    gemm_bits(p, k_bits, codebook, (pair ? -6 : rotate ? -4 : 0) - pl.mt, stream, desc, dim3(pl.grid));
    hip_ok(hipGetLastError(), "exl3_gemm_rows_kernel launch");
}

// ---- row blocks (exl3_gemm_block_kernel)
struct BlockPlan {
    bool ok = false;
    int rows_per_tile = 0, mt = 0, row_blocks = 0;     // mt: tiles of 16 rows of a block
    long units = 0;             // steps of 256 x 128 weights
    unsigned grid = 0, q = 0, rem = 0, S = 0, spt = 0;
    size_t operand_at = 0;      // bytes into the partial-sum workspace
    size_t operand_stride = 0;  // elements of one slab's copy
};

// 128-row tiles of 256 columns enough to spread over the chip (dispatch_dense)
static bool fills_128_row_tiles(const Workspace& ws, long nblocks, int size_m)
{
    return nblocks * ((size_m + 127) / 128) * 4 >= ws.cu_count;
}

// How a dense launch of 128-row tiles or larger is cut up.  Whole tiles: a workgroup of four waves per
// 128 x 256 tile, two of them on a compute unit.  Dealt out: one workgroup per compute unit with an even
// share of the (tile, k-block) units, the workgroups of a shared tile adding their parts in k order;
// of 128-row tiles, or of 256-row tiles (eight waves, every weight decoded once per 256 rows).
enum class DenseTiles { kWhole128, kDealt128, kDealt256 };

// The cheapest by what a compute unit spends, in 10 ns: k-blocks, the epilogue of every tile, and the
// hand-over of shared ones, which takes longer the more workgroups share a tile.
//   * Whole tiles hide part of an epilogue behind the other workgroup's k-loop, but come in rounds; a
//     round with r of its tiles takes about (1 + r) / 2 of a full one, the first a whole one.
//   * Dealt-out tiles have no partial round; their epilogue and hand-over are in nobody's shadow.  So a
//     short K, where those weigh against few k-blocks, takes whole tiles, and a long one is dealt out.
//   * The decode of 128-row tiles does not quite fit behind their MFMAs, so a k-block costs more with the
//     codebooks of longer decode; with 256-row tiles it does fit (6144 columns of 4096 at 1500 rows, dealt 128 /
//     dealt 256 us: MUL1 108/105, MCG 112/103, 3INST 123/105; the bit rate matters less).
// Fitted to 499 launches at 4 bits (K 128 .. 10240, 2048 .. 32768 columns, 460 .. 1500 rows): the choice costs
// 0.7 % over the fastest of the three on average, 14 % at most.  Examples, K x N at rows: whole / dealt
// 128 / dealt 256 us: 256x8192 at 512 16/26/31, 512x16384 at 1500 46/59/59, 1024x4096 at 512 27/31/50,
// 1024x16384 at 1500 72/88/81, 2048x4096 at 512 43/36/54, 2048x16384 at 1024 87/96/83, 5120x12288 at 600
// 99/106/121, 4096x16384 at 600 128/111/122 and at 1500 231/254/225.
struct TilesCost {
    DenseTiles tiles;
    long cost;          // in 10 ns, without what every form has in common
};
static TilesCost cheapest_tiles(long cus, int codebook, long KB, long tiles128, long tiles256, bool whole_allowed, bool wide_allowed)
{
    const long whole_kb = codebook == 0 ? 250 : codebook == 1 ? 236 : 230;
    const long dealt_kb = codebook == 0 ? 260 : codebook == 1 ? 243 : 235;
    const long n = tiles128 / cus, r = tiles128 % cus;          // full rounds, tiles of the last one
    const long m = tiles256 / cus, s = tiles256 % cus;
    // (one workgroup on a compute unit has no other to hide its epilogue behind)
    const long whole = n == 0 || tiles128 == cus ? KB * whole_kb + 500 + 400 * tiles128 / cus
                                                 : (2 * n * cus + (r ? cus + r : 0)) * (KB * whole_kb + 500) / (2 * cus);
    const long dealt128 = tiles128 * KB * dealt_kb / cus + 800 * n + (r == 0 ? 0 : n ? 800 : 2500 - 1600 * r / cus);
    const long dealt256 = tiles256 * KB * 415 / cus + 900 * m + (s == 0 ? 0 : m ? 1900 : 3700 - 2200 * s / cus);
    if (whole_allowed && whole < dealt128 && (!wide_allowed || whole <= dealt256)) return {DenseTiles::kWhole128, whole};
    return wide_allowed && dealt256 < dealt128 ? TilesCost{DenseTiles::kDealt256, dealt256} : TilesCost{DenseTiles::kDealt128, dealt128};
}

// When row blocks are taken (more than 32 rows).  Measured against the tiles of exl3_gemm_kernel.cuh at 4 bits,
// 40..511 rows (K x N, us, tiles -> row blocks):
//   * enough steps that the second launch and the hand-over pay: one per compute unit up to 64 rows (512x4096 14.0 ->
//     14.7, 512x16384 20.4 -> 19.1, 4096x4096 23.5 -> 21.0), 2.25 of them above (4096x4096 at 100 rows 24.8 -> 27.0,
//     7296x2688 33.8 -> 28.4);
//     Fewer are enough of deep weights, whose 32-row tiles share a tile between many workgroups, for up to two blocks of
//     96 rows (not for the last few rows of a third tile of sixteen): 48 steps at 36 / 64 / 96 rows of 3072x512 16.8 / 17.5 /
//     18.4 -> 14.4 / 15.1 / 16.5, 4096x1024 20.6 / 21.9 / 22.9 -> 15.5 / 16.9 / 19.1, 8192x512 26.6 / 28.3 / 28.6 -> 18.8 / 20.4 /
//     23.6, at 160 rows 29.9 -> 26.6; but 3072x256 at 80 rows 17.2 -> 18.1, 2048x2048 at 36 / 96 rows 17.3 / 19.6 -> 16.6 /
//     19.8, 1024x2048 13.0 / 14.8 -> 15.6 / 17.7, 4864x1536 at 112 rows 24.3 -> 26.4.  Bundles of several inputs, whose
//     copies in operand order are several as well, want 300 of two blocks (174 rows of 5120 x (384, 128, 128), 200 steps:
//     23.4 -> 26.5; 155 rows of 4096 x (1536, 256, 256), 512: 28.9 -> 25.9).
//   * narrow outputs, which would run as 32-row tiles and decode every weight once per 32 rows: always (17408x5120 at
//     64, 128, 256 and 384 rows 59, 88, 162, 167 -> 32, 46, 72, 100), of 449 rows and more where they cost less
//     (narrow_blocks_cost), up to gemm_block_rows;
//   * wide outputs: one row block (5120x34816 at 64 rows 62 -> 51, at 128 rows even) and several of up to 96 rows (160
//     rows 112 -> 104); several of more where they cost less than 128-row or 256-row tiles, a launch of which costs the
//     same for any rows up to a multiple of those (blocks_beside_wide_tiles, wide_blocks_cost).

// what a step costs beyond MUL1's, whose decode is the shortest
static long block_decode(int codebook, long mcg, long inst3) { return codebook == 1 ? mcg : codebook == 0 ? inst3 : 0; }
// whether some tile is shared by ranges of steps that are no parts of it
static bool uneven_ranges(const BlockPlan& pl) { return !pl.S && (pl.rem || pl.q % pl.spt); }
static long longest_range(const BlockPlan& pl) { return pl.S ? (pl.spt + pl.S - 1) / pl.S : pl.q + (pl.rem ? 1 : 0); }

// Several row blocks of more than 96 rows, in cheapest_tiles' unit: a step goes by the block's rows, the copies of the
// input by their elements (in millions), a finished tile 3.4 us; the launch that finishes shared tiles, with the stores and
// the uneven end that come with it, 13 us.  Fitted to 1700 linears and bundles (129..511 rows, 2..6 bits, K 256 .. 17408, up
// to 32768 columns) for the choice beside cheapest_tiles.
static long wide_blocks_cost(const Workspace& ws, int codebook, int slabs, int size_m, int size_k, const BlockPlan& pl, long tiles)
{
    return 240 + 110 * slabs * ((long)size_m * size_k >> 10) / 1024 + longest_range(pl) * (28 * pl.mt - 16 + block_decode(codebook, 24, 35)) +
           (pl.S || uneven_ranges(pl) ? 1340 : 0) + 338 * tiles / ws.cu_count;
}

// Four row blocks beside 32-row tiles, likewise: 650 launches of 449..511 rows.  32-row tiles cost by the k-blocks of a
// workgroup, nearly twice as much where more than one of them comes to a compute unit, and by the rows of the output;
// row blocks also by the partial tiles that they leave.  511 rows of 3072x2048, 256 tiles on 256 compute units, 29.2 -> 31.0,
// 450 rows, 360 tiles, 33.0 -> 29.6; 505 rows of 2304 x (1536, 256, 256) 28.2 -> 35.8; 468 rows of 8192x1024 51.9 -> 37.0.
// Of 187 launches 14 were slower as row blocks; from 3 % below none of the 146 that are left.
static long narrow_blocks_cost(int codebook, int slabs, int size_m, int size_k, const BlockPlan& pl, long tiles)
{
    const long parts = pl.S ? tiles * pl.S : uneven_ranges(pl) ? std::min<long>(pl.grid + tiles, 2l * pl.grid) : 0;
    return 430 + 144 * slabs * ((long)size_m * size_k >> 10) / 1024 + longest_range(pl) * (16 * pl.mt + block_decode(codebook, 25, 32)) +
           parts * pl.mt * 537 / 1000;
}
static long tiles_of_32_rows_cost(const Workspace& ws, int codebook, long nblocks, int size_m, int size_k, long columns)
{
    const long KB = size_k / 128, tiles = nblocks * ((size_m + 31) / 32), S = gemm_split(ws, tiles, (int)KB, 1);
    return (KB + S - 1) / S * (126 + (tiles * S > ws.cu_count ? 110 : 0) + block_decode(codebook, 12, 43)) + 62 * S +
           247 * (size_m * columns >> 10) / 1024;
}

static bool blocks_beside_wide_tiles(const Workspace& ws, int codebook, long nblocks, int size_m, const BlockPlan& pl)
{
    const long tiles128 = nblocks * ((size_m + 127) / 128), cus = ws.cu_count, steps = pl.units;
    // (1024x6144 at 300 and 448 rows, 2.25 and 3 steps a compute unit: 26.2 -> 28.4, 27.2 -> 31.0)
    if (steps < 4 * cus) return false;
    // 3INST and MCG decode a weight in 4.4 instead of 3.6 instructions, and row blocks decode it more often: where
    // tiles are few (MCG, K 5120: 200, 256, 336 and 448 rows x 8192 50.6 -> 40.7, 49.5 -> 42.4, 58.2 -> 55.3, 68.8 -> 55.5,
    // but 336 x 17408 94 -> 97, 200 x 34816 110 -> 119; 3INST 256 rows 2048x12288 39.0 -> 39.7)
    if (codebook != 2) return tiles128 <= (pl.rows_per_tile > 112 ? cus / 4 : cus / 2);
    // Blocks of 128 rows where whole 128-row tiles would fill half of the chip at most and the second launch pays
    // (256 rows, K 5120 x 8192, 64 tiles: 47.4 -> 41.2; 2048x16384, 128 tiles and eight steps a compute unit: 39.1 -> 28.2;
    // 2048x12288, 96 tiles and six steps: 36.5 -> 37.7; 384 rows of 5120x12288, 144 tiles: 74.8 -> 80).
    // Four of them (449..511 rows) where a workgroup has one tile or a part of one: 8192x4096 61.5 -> 55.0, 3072x8192 48.3 ->
    // 37.6, but 6144x5120, ranges across tiles, 58.2 -> 58.8.
    if (pl.rows_per_tile > 112)
        return tiles128 <= cus / 2 && steps >= 8 * cus && steps <= 32 * cus &&
               (pl.row_blocks <= 3 || !uneven_ranges(pl));
    // Of 112: two blocks (200 rows, K 5120 x 8192, 17408, 34816: 47.5 -> 37.3, 69.7 -> 63.1, 114 -> 113); three beside less than
    // half a chip or more than a whole of tiles (336 rows x 8192, 17408, 25600, 34816: 57.3 -> 53.5, 91.3 -> 92.0, 134 ->
    // 128, 175 -> 166); four, which leave little of the second 256 rows empty, beside up to a whole one and up to 32 steps a
    // compute unit (448 rows x 8192, 12288, 25600: 67 -> 53.5, 86.4 -> 81.7, 155 -> 164; 17408x5120, 42.5 steps: 123 -> 133).
    return pl.row_blocks == 2 || (pl.row_blocks == 3 ? tiles128 <= cus / 2 || tiles128 > cus : tiles128 <= cus && steps <= 32 * cus);
}

// activation: the launch that finishes gate's and up's tiles forms an MLP's activation too, which tiles leave to one more
static bool blocks_beside_tiles(const Workspace& ws, int codebook, int slices, int slabs, int size_m, int size_k, int size_n,
                                const BlockPlan& pl, bool activation)
{
    const long nblocks = (long)slices * ((size_n + 255) / 256), tiles = (long)slices * (size_n / 128) * pl.row_blocks;
    if (!fills_128_row_tiles(ws, nblocks, size_m))
        return activation || pl.row_blocks < 4 || pl.mt < 8 ||
               narrow_blocks_cost(codebook, slabs, size_m, size_k, pl, tiles) * 33 <=
                   tiles_of_32_rows_cost(ws, codebook, nblocks, size_m, size_k, (long)slices * size_n) * 32;
    // One row block (5120x34816 at 64 rows 62 -> 51, at 128 rows even) and several of up to 96 rows (160 rows 112 -> 104).
    if (pl.row_blocks == 1 || pl.rows_per_tile <= 96) return true;
    if (!blocks_beside_wide_tiles(ws, codebook, nblocks, size_m, pl)) return false;
    if (activation) return true;
    // Of these the ones whose ranges across tiles are no longer than 32 steps, where the row blocks of a column block come at
    // different times and each brings its weights in again (13568x6016 at 410 rows, MCG, 128 -> 134; 17408x8064 at 450, 172 ->
    // 227), and that cost 2 % less than tiles: of 470 launches 56 were slower than tiles, 4 of the 320 that are left, by 6 % at most:
    // 640x12288 at 385 rows 21.9 -> 35.8, 1024x29312 at 224 29.9 -> 41.4, 1152x15872 at 435 33.9 -> 42.7, 2304 x ten slices of
    // 1024 at 418 47.2 -> 52.1.
    if (uneven_ranges(pl) && longest_range(pl) > 32) return false;
    const Knobs& kn = knobs();
    const long best = cheapest_tiles(ws.cu_count, codebook, size_k / 128, nblocks * ((size_m + 127) / 128), nblocks * ((size_m + 255) / 256),
                                     kn.gemm_balanced == 1, kn.gemm_rows256 > 0).cost;
    return wide_blocks_cost(ws, codebook, slabs, size_m, size_k, pl, tiles) * 50 <= best * 49;
}

static BlockPlan plan_block(const Workspace& ws, int codebook, int slices, int slabs, int size_m, int size_k, int size_n, bool activation)
{
    BlockPlan pl;
    if (!knobs().gemm_balanced || size_m <= 32 || size_m > knobs().gemm_block_rows || size_n % 128 != 0) return pl;
    // row blocks of equal height, as few as 128 rows each allow
    const int blocks_min = (size_m + 127) / 128;
    pl.rows_per_tile = ((size_m + blocks_min - 1) / blocks_min + 15) / 16 * 16;
    pl.row_blocks = (size_m + pl.rows_per_tile - 1) / pl.rows_per_tile;
    pl.mt = pl.rows_per_tile / 16;
    const unsigned spt = (unsigned)(size_k / 64 + 3) / 4;
    const unsigned long long tiles = (unsigned long long)slices * (size_n / 128) * pl.row_blocks;
    const unsigned long long U = tiles * spt;
    if (U >= (1ull << 30)) return pl;
    const int least = knobs().gemm_block_steps;
    const bool deep = size_m >= 36 && pl.rows_per_tile <= 96 && (pl.row_blocks == 1 ? size_k >= 3072 : pl.row_blocks == 2 && size_k >= 3584);
    const int deep_least = slabs > 1 && pl.row_blocks > 1 && !activation ? 300 : 48;
    if (U < (unsigned long long)(least >= 0 ? least : deep ? deep_least : size_m <= 64 ? 256 : 576)) return pl;
    unsigned long long G = (unsigned long long)ws.cu_count;
    if (G > U) G = U;
    unsigned q = (unsigned)(U / G), rem = (unsigned)(U % G), S = 0;
    const unsigned most = q + (rem ? 1 : 0);
    if (G >= 2 * tiles) {       // parts of its own for each tile, as for few rows
        const unsigned s = (unsigned)(G / tiles);
        if (((spt + s - 1) / s) * 8ull <= most * 9ull) {
            S = s;
            G = tiles * s;
            q = rem = 0;
        }
    }
    if (U * (q + 2) >= (1ull << 32) || U * spt >= (1ull << 32)) return pl;
    // the workspace holds two partial tiles per workgroup, then the operand copies
    pl.operand_at = (size_t)G * 2 * pl.rows_per_tile * 512;
    pl.operand_stride = (size_t)pl.row_blocks * rows_operand_elements(size_k, pl.rows_per_tile / 16);
    if (pl.operand_at + slabs * pl.operand_stride * 2 > ws.partial_bytes) return pl;
    pl.units = (long)U;
    pl.grid = (unsigned)G;
    pl.q = q;
    pl.rem = rem;
    pl.S = S;
    pl.spt = spt;
    if (least < 0 && !blocks_beside_tiles(ws, codebook, slices, slabs, size_m, size_k, size_n, pl, activation)) return BlockPlan{};
    pl.ok = true;
    return pl;
}

// next: the two slices are gate and up, finished with what follows them
static void run_block(const BlockPlan& pl, GemmParams& p, int k_bits, int codebook, hipStream_t stream, std::string& desc,
                      const FinishActivation* next = nullptr)
{
    const long tiles = (long)(p.num_slices > 0 ? p.num_slices : 1) * (p.N / 128) * pl.row_blocks;
    p.units = (int)pl.units;
    p.unit_q = (int)pl.q;
    p.unit_r = (int)pl.rem;
    p.S = (int)pl.S;
    p.tiles_y = pl.row_blocks;
    p.rows_per_tile = pl.rows_per_tile;
    p.m_tr = magic(pl.spt);
    p.m_rt = magic((unsigned)pl.row_blocks);
    p.m_nb = magic((unsigned)p.N / 128);
    p.m_s = pl.S ? magic(pl.S) : 0;
    p.m_q = pl.S ? 0u : magic(pl.q);
    p.m_q1 = magic(pl.q + 1);
    p.lds_bytes = (unsigned)block_lds_bytes(pl.mt);
    gemm_bits(p, k_bits, codebook, -8 - pl.mt, stream, desc, dim3(pl.grid));
    hip_ok(hipGetLastError(), "exl3_gemm_block_kernel launch");
    if (next) {
        const dim3 grid((unsigned)(tiles / 2), (unsigned)(pl.rows_per_tile / 16));
        hipLaunchKernelGGL(exl3_gemm_silu_mul_finish_kernel, grid, dim3(256), 0, stream, p, *next);
        hip_ok(hipGetLastError(), "exl3_gemm_silu_mul_finish_kernel launch");
        desc += " + exl3_gemm_silu_mul_finish_kernel grid=" + std::to_string(grid.x) + "x" + std::to_string(grid.y);
    } else if (pl.S || pl.rem || pl.q % pl.spt) {       // some tile is shared
        const dim3 grid((unsigned)tiles, (unsigned)(pl.rows_per_tile / 16));
        hipLaunchKernelGGL(exl3_gemm_finish_kernel, grid, dim3(256), 0, stream, p);
        hip_ok(hipGetLastError(), "exl3_gemm_finish_kernel launch");
        desc += " + exl3_gemm_finish_kernel grid=" + std::to_string(grid.x) + "x" + std::to_string(grid.y);
    }
}

// Which of the two kernels that read operand-ordered copies a dense launch takes, if any.
struct OperandPlan {
    RowsPlan rows;
    BlockPlan block;
    OperandPlan(const Workspace& ws, int codebook, int slices, int slabs, int size_m, int size_k, int size_n, bool activation = false,
                bool few_rows_if_large = false)
        : rows(plan_rows(ws, slices, slabs, size_m, size_k, size_n)),
          block(rows.ok ? BlockPlan{} : plan_block(ws, codebook, slices, slabs, size_m, size_k, size_n, activation))
    {
        if (few_rows_if_large && rows.ok && knobs().gemm_rows_units < 0 && rows.units < rows_large_units(size_m)) rows = RowsPlan{};
        stride = rows.ok ? rows_operand_elements(size_k, rows.mt) : block.operand_stride;
        at = (_Float16*)((char*)ws.partials + (rows.ok ? rows.operand_at : block.operand_at));
    }
    bool ok() const { return rows.ok || block.ok; }
    int mt() const { return rows.ok ? rows.mt : block.rows_per_tile / 16; }
    void run(GemmParams& p, bool rotate, int k_bits, int codebook, hipStream_t stream, std::string& desc) const
    {
        if (rows.ok) run_rows(rows, p, rotate, k_bits, codebook, stream, desc);
        else run_block(block, p, k_bits, codebook, stream, desc);
    }
    _Float16* at = nullptr;     // the first slab's copy
    size_t stride = 0;          // elements between slabs
};

// Tile shape and work split of a dense launch: `nblocks` column blocks of 256 (all slices of
// a bundle together), size_m rows.  Fills the split fields of p and launches.
static void dispatch_dense(const Workspace& ws, GemmParams& p, int k_bits, int codebook, int size_m, int size_k,
                           int nblocks, hipStream_t stream, std::string& desc)
{
    // 128-row tiles decode a weight once per 128 rows, but need enough tiles to spread
    // over the chip; narrow outputs (few column tiles) run as 32-row tiles instead
    p.cstride = gemm_counter_stride((long)nblocks * ((size_m + 31) / 32));
    const int mb_plain = (size_m <= 32 || !fills_128_row_tiles(ws, nblocks, size_m)) ? 1 : 4;
    const int KB = size_k / 128;
    p.tile0 = 0;
    // 0: whole tiles, K split by gemm_split; 1 (default): by cost; more: dealt out to this many workgroups
    const int balance = knobs().gemm_balanced;
    // 0: never 256-row tiles; 1 (default): where they are faster; 2: wherever they are possible
    const int rows256 = knobs().gemm_rows256;
    // over more workgroups than compute units the dealt-out 128-row tiles lose (the 27B down projection at
    // 512 rows takes 147 us with 256 workgroups, 160 with 512): a wave interleaves its own decode with
    // its MFMAs, and more workgroups share a tile
    auto balanced = [&](int mb) {
        const int mtiles = (size_m + mb * 32 - 1) / (mb * 32);
        const long tiles = (long)nblocks * mtiles;
        const long units = tiles * KB;
        long slots = ws.cu_count;
        if (balance > 1) slots = balance;
        const long G = units < slots ? units : slots;
        const size_t part_bytes = (size_t)4 * mb * 2 * 16 * 64 * sizeof(float);
        if (!(tiles <= kCounters / 2 && units < (1L << 30) && (size_t)G * 2 * part_bytes <= ws.partial_bytes))
            return false;
        p.tiles_y = mtiles;
        p.S = 1;
        p.units = (int)units;
        p.unit_q = (int)(units / G);
        p.unit_r = (int)(units % G);
        gemm_bits(p, k_bits, codebook, mb, stream, desc, dim3((unsigned)G, 1, 1));
        hip_ok(hipGetLastError(), "exl3_gemm_kernel launch");
        return true;
    };
    bool whole = false;
    if (mb_plain == 4 && balance) {
        const long tiles128 = (long)nblocks * ((size_m + 127) / 128), tiles256 = (long)nblocks * ((size_m + 255) / 256);
        const DenseTiles cheapest = cheapest_tiles(ws.cu_count, codebook, KB, tiles128, tiles256, balance == 1, rows256 > 0 && size_m > 128).tiles;
        const bool wide = size_m > 128 && (rows256 >= 2 || cheapest == DenseTiles::kDealt256);
        if (wide && balanced(8)) return;
        whole = cheapest == DenseTiles::kWhole128;
        if (!whole && balanced(4)) return;
    }
    const int mtiles = (size_m + mb_plain * 32 - 1) / (mb_plain * 32);
    const long tiles = (long)nblocks * mtiles;
    p.tiles_y = mtiles;
    p.units = 0;
    p.S = whole ? 1 : gemm_split(ws, tiles, KB, mb_plain, size_m <= 32);
    gemm_bits(p, k_bits, codebook, mb_plain, stream, desc, dim3((unsigned)(tiles * p.S), 1, 1));
    hip_ok(hipGetLastError(), "exl3_gemm_kernel launch");
}

// whether two buffers do not overlap
static bool apart(const void* a, size_t a_bytes, const void* b, size_t b_bytes)
{
    return (uintptr_t)a + a_bytes <= (uintptr_t)b || (uintptr_t)b + b_bytes <= (uintptr_t)a;
}

std::string launch_gemm(const LinearArgs& a, const Workspace* scratch)
{
    if (a.size_k % 128 != 0) throw std::runtime_error("exl3 linear: size_k must be a multiple of 128");
    std::optional<LaunchScope> scope;
    if (!scratch) scope.emplace(a.stream);
    const Workspace& ws = scratch ? *scratch : scope->ws;
    throw_pending_device_fault(ws);
    const OperandPlan plan(ws, a.codebook, 1, 1, a.size_m, a.size_k, a.size_n, false, a.few_rows_if_large);
    RotateArgs rot;
    rot.in = a.a;
    rot.up = a.a_up;
    rot.act_out = a.act_out;
    rot.out = a.a_had;
    rot.suh_host = &a.suh;
    rot.rows = a.size_m;
    rot.cols = a.size_k;
    rot.stream = a.stream;
    if (plan.ok()) {
        rot.operand = plan.at;
        rot.mt = plan.mt();
    }
    // (the rotation overlaps the reads of other workgroups then, the output their reads of the input and their rotated rows)
    const size_t in_bytes = (size_t)a.size_m * a.size_k * 2, out_bytes = (size_t)a.size_m * a.size_n * (a.out_fp32 ? 4 : 2);
    const bool rotate = plan.rows.ok && plan.rows.rotate && !a.a_up && !a.act_out && !a.rotated &&
                        apart(a.a, in_bytes, a.a_had, in_bytes) && apart(a.a, in_bytes, a.c, out_bytes) &&
                        apart(a.a_had, in_bytes, a.c, out_bytes);
    std::string d0 = rotate || a.rotated ? "" : launch_rotate(rot) + " + ";
    GemmRotateParams p{};
    if (rotate) {
        p.rot_in = (const _Float16*)a.a;
        p.rot_out = (_Float16*)a.a_had;
        p.lin.suh = (const _Float16*)a.suh;
    }
    p.fault = ws.fault_dev;
    p.spin_limit = spin_limit();
    p.a_had[0] = (const _Float16*)(!plan.ok() ? a.a_had : a.rotated ? a.rotated_operand : plan.at);
    p.lin.trellis = (const uint32_t*)a.trellis;
    p.lin.svh = (const _Float16*)a.svh;
    p.c[0] = a.c;
    p.M = a.size_m;
    p.K = a.size_k;
    p.N = a.size_n;
    p.out_fp32 = a.out_fp32;
    if (a.out_add && !a.out_fp32) throw std::runtime_error("exl3 gemm: rows are added to an fp32 output only");
    p.out_add = a.out_add;
    p.partials = ws.partials;
    p.counters = ws.counters;
    std::string desc;
    if (plan.ok()) plan.run(p, rotate, a.k_bits, a.codebook, a.stream, desc);
    else dispatch_dense(ws, p, a.k_bits, a.codebook, a.size_m, a.size_k, (a.size_n + 255) / 256, a.stream, desc);
    return d0 + desc + (a.out_fp32 ? " out=f32" : " out=f16");
}

// berth_ops_mgemm with more than 8 rows, or 2..8 where gemm_rows_applies says so: the bundle's linears on the MFMA kernels
// behind one launch that rotates every distinct input (slab s of a_had = Hh(input(s) * suh[s])).
std::string launch_gemm_bundle(const MgemmArgs& m)
{
    if (m.size_k % 128 != 0) throw std::runtime_error("exl3_mgemm: size_k must be a multiple of 128");
    const bool sliced = m.had_src_list != nullptr;
    if (m.host_lists && m.bszm_out > kGemmMaxSlices)
        throw std::runtime_error("exl3_mgemm (host lists): at most " + std::to_string(kGemmMaxSlices) + " slices");
    LaunchScope scope(m.stream);
    Workspace& ws = scope.ws;
    throw_pending_device_fault(ws);
    const int slabs = sliced ? m.num_had_src : m.bszm_out;
    const OperandPlan plan(ws, m.codebook, m.bszm_out, slabs, m.size_m, m.size_k, m.size_n);
    // what the kernel multiplies: the rotated rows, or their copy in operand order
    const size_t slab_stride = plan.ok() ? plan.stride : (size_t)m.size_m * m.size_k;
    const _Float16* const slab0 = (const _Float16*)(plan.ok() ? plan.at : m.a_had);
    GemmRotateParams p{};
    p.fault = ws.fault_dev;
    p.spin_limit = spin_limit();
    p.a_had[0] = slab0;
    p.c[0] = m.c;
    p.M = m.size_m;
    p.K = m.size_k;
    p.N = m.size_n;
    p.out_fp32 = m.c_fp32;
    p.partials = ws.partials;
    p.counters = ws.counters;
    p.num_slices = m.bszm_out;
    p.slab_stride = slab_stride;
    const void* suh_host[kGemmMaxSlices] = {};
    if (m.host_lists) {
        const uint64_t* b = (const uint64_t*)m.b_list;
        const uint64_t* su = (const uint64_t*)m.suh_list;
        const uint64_t* sv = (const uint64_t*)m.svh_list;
        if (slabs > kGemmMaxSlices) throw std::runtime_error("exl3_mgemm (host lists): too many input rotations");
        for (int i = 0; i < slabs; ++i) suh_host[i] = (const void*)su[i];
        for (int i = 0; i < m.bszm_out; ++i) {
            GemmSlice& g = p.slice[i];
            g.trellis = (const uint32_t*)b[i];
            g.svh = (const _Float16*)sv[i];
            if (sliced) {
                const int src = m.had_src_list[i];
                if (src < 0 || src >= m.num_had_src) throw std::runtime_error("exl3_mgemm (host lists): had_src_list entry out of range");
                if (m.size_n_list[i] < 0 || m.size_n_list[i] > m.size_n || m.size_n_list[i] % 128 != 0)
                    throw std::runtime_error("exl3_mgemm (host lists): size_n_list entry must be a multiple of 128 within size_n");
                g.c = (void*)((const uint64_t*)m.c_ptrs)[i];
                g.width = m.size_n_list[i];
                g.n_stride = m.n_stride_list[i];
                g.a_had = slab0 + (size_t)src * slab_stride;
            } else {
                g.c = (char*)m.c + (size_t)i * m.size_m * m.size_n * (m.c_fp32 ? 4 : 2);
                g.width = m.size_n;
                g.n_stride = m.size_n;
                g.a_had = slab0 + (size_t)i * slab_stride;
            }
        }
    } else {
        p.b_list = (const uint64_t*)m.b_list;
        p.svh_list = (const uint64_t*)m.svh_list;
        if (sliced) {
            p.c_ptrs = (const uint64_t*)m.c_ptrs;
            p.size_n_list = m.size_n_list;
            p.n_stride_list = m.n_stride_list;
            p.had_src_list = m.had_src_list;
        }
    }
    RotateArgs rot;
    rot.in = m.a;
    rot.in_stride = (!sliced && m.bszm_in > 1) ? (size_t)m.size_m * m.size_k : 0;
    rot.out = m.a_had;
    rot.out_stride = (size_t)m.size_m * m.size_k;
    rot.suh_list = m.host_lists ? nullptr : m.suh_list;
    rot.suh_host = suh_host;
    rot.slabs = slabs;
    rot.rows = m.size_m;
    rot.cols = m.size_k;
    rot.stream = m.stream;
    if (plan.ok()) {
        rot.operand = plan.at;
        rot.mt = plan.mt();
    }
    const size_t rows_bytes = (size_t)m.size_m * m.size_k * 2, in_bytes = rows_bytes * (rot.in_stride ? slabs : 1);
    const auto output_apart = [&](const void* c, size_t elements) {
        const size_t bytes = elements * (m.c_fp32 ? 4 : 2);
        return apart(m.a, in_bytes, c, bytes) && apart(m.a_had, rows_bytes * slabs, c, bytes);
    };
    bool rotate = plan.rows.ok && plan.rows.rotate && apart(m.a, in_bytes, m.a_had, rows_bytes * slabs);
    // The outputs of slices whose lists are in device memory cannot be looked at here: they may lie over the input or
    // its rotated rows, and a source may have no slice that would leave its slab.  Those keep the two launches.
    if (!sliced) rotate = rotate && output_apart(m.c, (size_t)m.bszm_out * m.size_m * m.size_n);
    else if (m.host_lists) {
        bool used[kGemmMaxSlices] = {};
        for (int i = 0; i < m.bszm_out; ++i) used[m.had_src_list[i]] = true;
        rotate = rotate && std::all_of(used, used + slabs, [](bool u) { return u; });       // every input is some slice's
        for (int i = 0; i < m.bszm_out; ++i)
            rotate = rotate && output_apart(p.slice[i].c, (size_t)(m.size_m - 1) * p.slice[i].n_stride + p.slice[i].width);
    } else {
        rotate = false;
    }
    if (rotate && m.host_lists) {
        bool left[kGemmMaxSlices] = {};
        for (int i = 0; i < m.bszm_out; ++i) {
            const int src = sliced ? m.had_src_list[i] : i;
            GemmRotation& g = p.rotation[i];
            g.suh = (const _Float16*)suh_host[src];
            g.in = (const _Float16*)m.a + (size_t)src * rot.in_stride;
            g.had_out = left[src] ? nullptr : (_Float16*)m.a_had + (size_t)src * rot.out_stride;
            left[src] = true;
        }
    } else if (rotate) {
        p.rot_in = (const _Float16*)m.a;
        p.rot_in_stride = rot.in_stride;
        p.rot_out = (_Float16*)m.a_had;
        p.suh_list = (const uint64_t*)m.suh_list;
    }
    std::string d0 = rotate ? "" : launch_rotate(rot) + " + ";
    const long nblocks = (long)m.bszm_out * ((m.size_n + 255) / 256);
    if (nblocks * ((m.size_m + 31) / 32) > kCounters / 2) throw std::runtime_error("exl3_mgemm: too many output tiles");
    std::string desc;
    if (plan.ok()) plan.run(p, rotate, m.k_bits, m.codebook, m.stream, desc);
    else dispatch_dense(ws, p, m.k_bits, m.codebook, m.size_m, m.size_k, (int)nblocks, m.stream, desc);
    return std::string(sliced ? "sliced x" : "uniform x") + std::to_string(m.bszm_out) + (m.host_lists ? " by value " : " ") + d0 +
           desc + (m.c_fp32 ? " out=f32" : " out=f16");
}

std::string launch_gemm_pair(const PairArgs& a, void* a_had_second, PairNext* next, const Workspace* scratch)
{
    if (a.size_k % 128 != 0) throw std::runtime_error("exl3 linear: size_k must be a multiple of 128");
    std::optional<LaunchScope> scope;
    if (!scratch) scope.emplace(a.stream);
    const Workspace& ws = scratch ? *scratch : scope->ws;
    throw_pending_device_fault(ws);
    const OperandPlan plan(ws, a.codebook, 2, 2, a.size_m, a.size_k, a.size_n, next != nullptr);
    RowsPairParams p{};
    p.fault = ws.fault_dev;
    p.spin_limit = spin_limit();
    p.a_had[0] = (const _Float16*)a.a_had;
    p.c[0] = a.c[0];
    p.M = a.size_m;
    p.K = a.size_k;
    p.N = a.size_n;
    p.out_fp32 = 0;
    p.partials = ws.partials;
    p.counters = ws.counters;
    p.num_slices = 2;
    void* const slabs[2] = {a.a_had, a_had_second};
    for (int i = 0; i < 2; ++i) {
        GemmSlice& g = p.slice[i];
        g.trellis = (const uint32_t*)a.trellis[i];
        g.svh = (const _Float16*)a.svh[i];
        g.c = a.c[i];
        g.width = a.size_n;
        g.n_stride = a.size_n;
        g.a_had = (const _Float16*)slabs[i];
    }
    // What the launch leaves for the next linear: few rows in the launch itself (its partial sums then take twice
    // the room, and the copies of its input in operand order move up), row blocks in the one that finishes their
    // tiles.  The next linear's copy lies behind its partial sums, and behind what of these is still read.
    const OperandPlan after(ws, a.codebook, 1, 1, a.size_m, a.size_n, next ? next->size_n : 128);
    // (Column blocks cut into more than two parts: a pair is handed over by all of them, and the next launch is short.)
    const size_t in_at = plan.rows.operand_at * 2, next_at = std::max(in_at + 2 * plan.stride * 2, after.rows.operand_at);
    const bool pair_rows = next && plan.rows.ok && plan.rows.S <= 2 && !after.block.ok &&
                           next_at + (after.rows.ok ? after.stride * 2 : 0) <= ws.partial_bytes;
    _Float16* const operand = pair_rows ? (_Float16*)((char*)ws.partials + in_at) : plan.at;
    RotateArgs rot;
    rot.in = a.a;
    rot.norm = a.norm;
    rot.suh_host = a.suh;
    rot.out_host = slabs;
    rot.slabs = 2;
    rot.rows = a.size_m;
    rot.cols = a.size_k;
    rot.stream = a.stream;
    if (plan.ok()) {
        rot.operand = operand;
        rot.mt = plan.mt();
        for (int i = 0; i < 2; ++i) p.slice[i].a_had = operand + i * plan.stride;
    }
    std::string d0 = launch_rotate(rot);
    const long nblocks = 2L * ((a.size_n + 255) / 256);
    if (nblocks * ((a.size_m + 31) / 32) > kCounters / 2) throw std::runtime_error("exl3 linear pair: too many output tiles");
    std::string desc;
    const size_t operand_at = std::max(plan.block.operand_at, after.block.operand_at);
    if (pair_rows) {
        p.suh = (const _Float16*)next->suh;
        p.act_had = (_Float16*)next->a_had;
        p.keep_up = next->keep_up;
        if (after.rows.ok) {
            p.operand = (_Float16*)((char*)ws.partials + next_at);
            p.operand_mt = after.mt();
        }
        run_rows(plan.rows, p, false, a.k_bits, a.codebook, a.stream, desc, true);
        next->operand = p.operand;
        next->done = true;
    } else if (next && plan.block.ok && !after.rows.ok && operand_at + after.block.operand_stride * 2 <= ws.partial_bytes) {
        FinishActivation f{(const _Float16*)next->suh, (_Float16*)next->a_had, nullptr, 1};
        if (after.block.ok) {
            f.operand = (_Float16*)((char*)ws.partials + operand_at);
            f.mt = after.mt();
        }
        run_block(plan.block, p, a.k_bits, a.codebook, a.stream, desc, &f);
        next->operand = f.operand;
        next->done = true;
    } else if (plan.ok()) plan.run(p, false, a.k_bits, a.codebook, a.stream, desc);
    else dispatch_dense(ws, p, a.k_bits, a.codebook, a.size_m, a.size_k, (int)nblocks, a.stream, desc);
    return "pair " + d0 + " + " + desc + " out=f16";
}

// Grouped launches of problems of a few rows: room for the column blocks that a workgroup can touch
// when the list is as long as it can get, in as few rounds of one workgroup per compute unit as that
// takes.
struct GroupRowsPlan {
    bool ok = false;
    unsigned grid = 0;
    size_t lds = 0;
};
static GroupRowsPlan plan_group_rows(const Workspace& ws, const GroupedArgs& g)
{
    GroupRowsPlan pl;
    if (g.size_k < 256 || g.small_rows > 16) return pl;
    const unsigned long long TR4 = (unsigned)g.size_k / 64, blocks = (unsigned long long)g.max_problems * g.num_lins * (g.size_n / 128);
    const unsigned long long U = blocks * TR4;
    // (a row's place in a_had is 32 bits there; the list is long enough for all rows)
    if ((unsigned long long)g.max_problems * g.small_rows * g.size_k * 2 >= (1ull << 32)) return pl;
    if (blocks > (unsigned)kCounters / 2 || U * TR4 >= (1ull << 32) || blocks * blocks >= (1ull << 32)) return pl;
    for (unsigned rounds = 1; rounds <= 64; rounds *= 2) {
        const unsigned long long G = (unsigned long long)ws.cu_count * rounds;
        const unsigned long long most = std::max((U + G - 1) / G, 8ull);        // (a short list: 4..7 units each)
        const unsigned long long ncb = (most + TR4 - 2) / TR4 + 1;
        if (ncb > (unsigned)kRowsWaves) continue;
        const size_t lds = rows_group_lds_bytes(g.small_rows, (int)ncb);
        if (lds > 160 * 1024 || G * 2 * g.small_rows * 512 > ws.partial_bytes) continue;
        pl.ok = true;
        pl.grid = (unsigned)G;
        pl.lds = lds;
        return pl;
    }
    return pl;
}

// Workgroups a compute unit up to which the waves of a grouped launch give way (PriorityRamp): one round of four, of gate
// and up together (`pair`) one and a half.  The more bits, the more of the launch waits for the weights instead of for the
// vector pipes, and waves that give way then ask later.  560 random layers of 4..160 tokens at sums of 100 to 2600
// workgroups, the whole layer with and without in turn: gate and up at 2..5 bits 1 to 5 % quicker up to four, 0 to 2 up
// to six, 2 to 5 slower from seven; 6 bits 1 to 3 quicker up to four, then up to 7 slower (112 tokens x 128 experts of
// 3584x1280, 1280 workgroups, 296 -> 308 us; 5 bits as the others, 3INST up to six at 6 and 7 bits too: 1 to 3 quicker); 7 bits 1 to 3
// quicker up to three, then 2 to 5 slower; 8 bits 1 to 3 quicker up to two, 0 to 2 slower up to three, 2 to 6 at four (3INST 1 to 3
// quicker up to three).  Down likewise, with half of each: at 6 bits 1 to 2 % up to four, 7 bits up to 3.9 slower from three, 8 from two.
static int ramp_workgroups(int bits, int codebook, bool pair)
{
    if (codebook == 0) return bits < 8 ? (pair ? 6 : 4) : 3;
    return bits == 8 ? 2 : bits == 7 ? 3 : pair && bits < 6 ? 6 : 4;
}

// grouped: problems of at most 32 rows each (and, in a list of their own, of up to 128); a_had rows are in problem
// order, or found through a_rows
std::string launch_gemm_grouped(const GroupedArgs& g)
{
    constexpr int mb = 1;
    if (g.size_k % 128 != 0 || g.size_n % 128 != 0)
        throw std::runtime_error("moe grouped linear: sizes must be multiples of 128");
    LaunchScope scope(g.stream);
    Workspace& ws = scope.ws;
    throw_pending_device_fault(ws);
    GemmParams p{};
    p.fault = ws.fault_dev;
    p.spin_limit = spin_limit();
    p.a_had[0] = (const _Float16*)g.a_had;
    p.a_had[1] = (const _Float16*)g.a_had2;
    p.a_rows = g.a_rows;
    p.c[0] = g.c0;
    p.c[1] = g.c1;
    p.M = 0;
    p.K = g.size_k;
    p.N = g.size_n;
    p.out_fp32 = g.out_fp32;
    p.experts = (const ExpertLin*)g.experts;
    p.problems = (const GroupProblem*)g.problems;
    p.num_problems = g.num_problems;
    p.lins_per_expert = g.lins_per_expert;
    p.lin_base = g.lin_base;
    p.shared_expert = g.shared ? g.shared_expert : -1;
    if (g.shared) std::memcpy(p.shared, g.shared, sizeof(p.shared));
    p.partials = ws.partials;
    p.counters = ws.counters;
    if (g.small_rows > 0 && g.max_big == 0) {
        const GroupRowsPlan pl = plan_group_rows(ws, g);
        if (pl.ok) {
            const long blocks = (long)g.num_lins * (g.size_n / 128);
            std::string desc;
            p.M = g.small_rows;
            p.cstride = gemm_counter_stride(g.max_problems * blocks);
            p.group_blocks = (int)blocks;
            p.m_rt = magic((unsigned)blocks);
            p.m_tr = magic((unsigned)g.size_k / 64);
            p.m_nb = magic((unsigned)g.size_n / 128);
            p.lds_bytes = (unsigned)pl.lds;
            gemm_bits(p, g.k_bits, g.codebook, -3, g.stream, desc, dim3(pl.grid));
            hip_ok(hipGetLastError(), "exl3_gemm_rows_kernel grouped launch");
            return desc + " grouped";
        }
    }
    if (g.act_had && g.num_lins == 2 && g.max_big == 0 &&
        gemm_split(ws, (long)g.max_problems * (g.size_n / 128), g.size_k / 128, 1) == 1) {
        // whole K in every workgroup: gate, up and the next rotation together
        if (g.max_problems > 65535) throw std::runtime_error("moe grouped linear: too many problems");
        p.act_had = (_Float16*)g.act_had;
        p.group_lins = 1;
        p.ramp_problems = ramp_workgroups(g.k_bits, g.codebook, true) * ws.cu_count / (g.size_n / 128);
        std::string desc;
        gemm_bits(p, g.k_bits, g.codebook, -4, g.stream, desc, group_grid(g.size_n / 128, 1, g.max_problems));
        hip_ok(hipGetLastError(), "exl3_gemm_pair_kernel launch");
        *g.act_done = true;
        return desc + " grouped";
    }
    const int nblocks = (g.size_n + 255) / 256;
    const long tiles = (long)g.max_problems * g.num_lins * nblocks;
    p.cstride = gemm_counter_stride(tiles);
    p.S = gemm_split(ws, tiles, g.size_k / 128, mb);
    if (g.max_problems + g.max_big > 65535) throw std::runtime_error("moe grouped linear: too many problems");
    std::string desc;
    p.group_lins = g.num_lins;
    p.tiles_y = g.max_problems;
    if (g.max_big > 0) {
        // both lists in one launch, whole K per workgroup
        p.big_problems = (const GroupProblem*)g.big_problems;
        p.num_big = g.num_big;
        p.max_big = g.max_big;
        p.S = 1;
        p.places = 2 * ws.cu_count;
        gemm_bits(p, g.k_bits, g.codebook, mb, g.stream, desc,
                  group_grid(nblocks, g.num_lins, g.max_problems + g.max_big + mixed_extra(nblocks * g.num_lins, p.places)));
        hip_ok(hipGetLastError(), "exl3_gemm_mixed_kernel launch");
        return desc + " grouped";
    }
    p.ramp_problems = ramp_workgroups(g.k_bits, g.codebook, false) * ws.cu_count / (nblocks * p.S * g.num_lins);
    gemm_bits(p, g.k_bits, g.codebook, mb, g.stream, desc, group_grid(nblocks * p.S, g.num_lins, g.max_problems));
    hip_ok(hipGetLastError(), "exl3_gemm_kernel grouped launch");
    return desc + " grouped";
}

// ---- plain fp16 GEMM (crates/berth-kernels/csrc/prefill_lin/linear.cu:387-418):
// C[m][ldc] = A[m][k] @ B[k][n], fp32 accumulate.  One wave per 32x32 output
// tile, operands read straight from global memory.
__global__ __launch_bounds__(256) void hgemm_kernel(const _Float16* __restrict__ a,
                                                    const _Float16* __restrict__ b, void* c, int M,
                                                    int K, int N, int ldc, int c_fp32)
{
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int slot = lane & 31, kh = lane >> 5;
    const int m0 = blockIdx.y * 32;
    const int n0 = (blockIdx.x * 4 + wave) * 32;
    if (n0 >= N) return;
    float16_t acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int row = m0 + slot, col = n0 + slot;
    for (int k0 = 0; k0 < K; k0 += 16) {
        half8_t av, bv;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int k = k0 + 8 * kh + i;
            av[i] = (row < M && k < K) ? a[(size_t)row * K + k] : (_Float16)0;
            bv[i] = (col < N && k < K) ? b[(size_t)k * N + col] : (_Float16)0;
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int gm = m0 + 8 * (r >> 2) + 4 * kh + (r & 3);
        if (gm < M && col < N) {
            if (c_fp32) ((float*)c)[(size_t)gm * ldc + col] = acc[r];
            else ((_Float16*)c)[(size_t)gm * ldc + col] = (_Float16)acc[r];
        }
    }
}

std::string launch_hgemm(const void* a, const void* b, void* c, int m, int k, int n, int ldc,
                         int c_fp32, hipStream_t stream)
{
    dim3 grid((n + 127) / 128, (m + 31) / 32);
    hipLaunchKernelGGL(hgemm_kernel, grid, dim3(256), 0, stream, (const _Float16*)a, (const _Float16*)b, c,
                       m, k, n, ldc, c_fp32);
    hip_ok(hipGetLastError(), "hgemm_kernel launch");
    return "hgemm_kernel grid=" + std::to_string(grid.x) + "x" + std::to_string(grid.y) + " block=256" +
           (c_fp32 ? " out=f32" : " out=f16");
}

}  // namespace berth
