// Hadamard rows, SiLU gate.
#include "exl3_decode.cuh"
#include "hadamard.cuh"
#include "launch.h"
#include "rows_operand.cuh"
#include "silu.cuh"

namespace berth {

// crates/berth-kernels/csrc/prefill_lin/reconstruct.cu:31-67: per row and per
// 128 columns, out = Hh(in * scale) (pre) or Hh(in) * scale (post).
template <typename T, bool PRE>
__global__ __launch_bounds__(256) void had_r_128_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                        const _Float16* __restrict__ scale,
                                                        long blocks, int col_blocks)
{
    // sixteen lanes per 128 block, eight consecutive elements per lane (one or two 16-byte
    // accesses): a wave takes four neighbouring blocks at a time and strides over the tensor
    typedef T vec8_t __attribute__((ext_vector_type(8)));
    const int lane = threadIdx.x & 63;
    const int chunk = had_chunk(lane);
    const long waves = (long)gridDim.x * 4;
    const long groups = (blocks + 3) / 4;
    for (long g = (long)blockIdx.x * 4 + (threadIdx.x >> 6); g < groups; g += waves) {
        const long blk = g * 4 + (lane >> 4);
        const bool live = blk < blocks;
        const long b = live ? blk : blocks - 1;             // lanes past the end redo the last block and store nothing
        const int cb = (int)(b % col_blocks);
        const size_t at = (size_t)b * 128 + 8 * chunk;
        const vec8_t x = *(const vec8_t*)(in + at);
        float v[8], sc[8];
        if (scale) {
            const half8_t s8 = *(const half8_t*)(scale + cb * 128 + 8 * chunk);
#pragma unroll
            for (int i = 0; i < 8; ++i) sc[i] = (float)s8[i];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) sc[i] = 1.0f;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = (float)x[i];
            if (PRE) v[i] *= sc[i];
        }
        const float unit = had128_row16(v, lane) * kRsqrt128;
        vec8_t o;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float r = had_scale(v[i], unit);
            if (!PRE) r = rounded(r * sc[i]);
            o[i] = (T)r;
        }
        if (live) *(vec8_t*)(out + at) = o;
    }
}

// The rotated inputs of a launch of the MFMA kernels: Hh(in * suh) per row and 128 columns, for
// one or more slabs (blockIdx.y), whose sign scales come from a device list of pointers or by
// value.  SILU: the input is silu(in) * up with the fp16 steps of silu_mul_kernel, formed here
// instead of in a launch of its own (act_out, when given, still receives it: it may be `up`, whose
// elements a lane has read before it writes them); 6 bytes an element (8 with act_out) against 10
// of the two launches.  `operand`, when given, receives a second copy of the result in the operand
// order of the few-row kernel.
struct RotateTable {
    const _Float16* suh[kBundleMaxSlices];
    _Float16* out[kBundleMaxSlices];        // null: slab s goes to out + s * out_stride
};
struct RotateParams {
    const _Float16* in;
    const _Float16* up;
    _Float16* act_out;
    _Float16* out;
    _Float16* operand;
    const uint64_t* suh_list;
    size_t in_stride, out_stride, operand_stride;
    long blocks;
    int col_blocks, mt;
    RotateTable tab;
};
// values k .. k + 7 of a row of a slab in operand order, row blocks of 16 * mt rows one after the other
__device__ __forceinline__ void store_operand(const RotateParams& p, int slab, int row, int k, half8_t o)
{
    const unsigned block = (unsigned)row / (unsigned)(16 * p.mt);
    *(half8_t*)(p.operand + (size_t)slab * p.operand_stride + block * rows_operand_elements(p.col_blocks * 128, p.mt) +
                rows_operand_offset(row - (int)block * 16 * p.mt, k, p.mt)) = o;
}
template <bool SILU>
__device__ __forceinline__ void rotate_rows(const RotateParams& p)
{
    const int slab = blockIdx.y;
    const _Float16* scale = p.suh_list ? (const _Float16*)p.suh_list[slab] : p.tab.suh[slab];
    const _Float16* in = p.in + (size_t)slab * p.in_stride;
    _Float16* out = (!p.suh_list && p.tab.out[slab]) ? p.tab.out[slab] : p.out + (size_t)slab * p.out_stride;
    const int lane = threadIdx.x & 63;
    const int chunk = had_chunk(lane);
    const long waves = (long)gridDim.x * 4;
    const long groups = (p.blocks + 3) / 4;
    for (long g = (long)blockIdx.x * 4 + (threadIdx.x >> 6); g < groups; g += waves) {
        const long blk = g * 4 + (lane >> 4);
        const bool live = blk < p.blocks;
        const unsigned b = (unsigned)(live ? blk : p.blocks - 1);   // lanes past the end redo the last block and store nothing
        const unsigned row = b / (unsigned)p.col_blocks, cb = b - row * (unsigned)p.col_blocks;
        const size_t at = (size_t)b * 128 + 8 * chunk;
        half8_t x = *(const half8_t*)(in + at);
        const half8_t s8 = *(const half8_t*)(scale + cb * 128 + 8 * chunk);
        if (SILU) {
            const half8_t u = *(const half8_t*)(p.up + at);
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = silu_mul_h(x[i], u[i]);
        }
        float v[8];
        mul_half8(x, s8, v);
        const float unit = had128_row16(v, lane) * kRsqrt128;
        half8_t o;
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = (_Float16)had_scale(v[i], unit);
        if (live) {
            if (SILU && p.act_out) *(half8_t*)(p.act_out + at) = x;
            *(half8_t*)(out + at) = o;
            if (p.operand) store_operand(p, slab, (int)row, (int)cb * 128 + 8 * chunk, o);
        }
    }
}
__global__ __launch_bounds__(256) void had_r_128_slabs_kernel(RotateParams p) { rotate_rows<false>(p); }
__global__ __launch_bounds__(256) void silu_mul_had_r_128_kernel(RotateParams p) { rotate_rows<true>(p); }

// The input of an MLP block's gate and up projections in one pass over the rows: residual add,
// RMS norm (the steps of rms_norm_kernel) and the rotation with each projection's scales.  One
// workgroup per row, eight values a thread and chunk held in registers between the passes, so
// a row is read once and only the residual stream and the rotated rows are written: 20 bytes an
// element against 42 of the four launches (residual add, norm, two rotations).
// With few rows a launch is a chain of waits: row, norm weights and both scales asked for together, and the wave's sum by
// DPP moves, 5 rows of 5120 5.6 -> 5.1 us, 100 rows 7.9 -> 7.4 (traced).
// So with two and four chunks a thread too, for all that these hold 70 and 127 registers (and four of the latter in
// scratch) instead of 46 and 62: 2 / 100 / 600 rows of 9216 8.1 / 10.2 / 21.9 -> 7.3 / 9.6 / 17.7, of 16384 11.2 / 14.5 / 42.6 ->
// 9.2 / 14.0 / 38.9, of 17408 12.4 / 15.8 / 45.5 -> 11.1 / 16.1 / 45.7, of 24576 15.7 / 24.5 / 61.0 -> 13.5 / 21.7 / 58.6, of
// 32768 28.2 / 38.7 / 81.3 -> 22.0 / 27.2 / 76.3 (scales and weight of four chunks behind the sum, no scratch: 25.1 / 33.0 / 76.2).
struct NormParams {
    const float* x;
    const float* res;
    float* res_out;
    const uint16_t* weight;
    int dim, slabs;
    float epsilon, constant_bias, constant_scale;
    int weight_bf16;
};
constexpr int kNormSlabs = 2;           // gate and up
// the sum over a wave by butterflies over lane distances 32 .. 1, the partner's two dwords by DPP moves and the row swaps
// instead of LDS permutes: one row of 2048 / 5120 / 17408 1.91 / 2.18 / 3.48 -> 1.76 / 2.08 / 3.40 us, with the residual 2.10 /
// 2.82 / 5.88 -> 1.90 / 2.64 / 5.73, 48000 fp16 rows of 128 30.0 -> 26.6, 32 of them 2.8 -> 2.6; 1500 rows of 5120 9.1 either way
__device__ __forceinline__ double wave_sum(double v)
{
    auto partner = [](double x, auto move) {
        const uint64_t b = __builtin_bit_cast(uint64_t, x);
        const float lo = move(__builtin_bit_cast(float, (uint32_t)b));
        const float hi = move(__builtin_bit_cast(float, (uint32_t)(b >> 32)));
        return __builtin_bit_cast(double, (uint64_t)__builtin_bit_cast(uint32_t, lo) | ((uint64_t)__builtin_bit_cast(uint32_t, hi) << 32));
    };
    v += partner(v, [](float f) { return lane_xor_swap32(f); });
    v += partner(v, [](float f) { return lane_xor_swap16(f); });
    v += partner(v, [](float f) { return lane_xor_dpp<8>(f); });
    v += partner(v, [](float f) { return lane_xor_dpp<4>(f); });
    v += partner(v, [](float f) { return lane_xor_dpp<2>(f); });
    v += partner(v, [](float f) { return lane_xor_dpp<1>(f); });
    return v;
}
template <int CHUNKS>
__global__ __launch_bounds__(1024) void add_rms_norm_had_r_128_kernel(NormParams n, RotateParams p)
{
    __shared__ double s_part[16];
    const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int mine = (tid & ~15) | had_chunk(lane);        // which eight values of a chunk this thread holds
    const int threads = blockDim.x;
    const size_t base = (size_t)row * n.dim;
    // everything that is read is asked for at once
    float4_t xv[CHUNKS][2], rv[CHUNKS][2];
    half8_t wb[CHUNKS], suh[CHUNKS][kNormSlabs];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int e = 8 * (mine + c * threads), at = e < n.dim ? e : 0;         // (past the end: read and not used)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            xv[c][h] = *(global_ptr<const float4_t>)as_global(n.x + base + at + 4 * h);
            rv[c][h] = *(global_ptr<const float4_t>)as_global(n.res + base + at + 4 * h);
        }
        wb[c] = *(global_ptr<const half8_t>)as_global((const _Float16*)n.weight + at);
#pragma unroll
        for (int s = 0; s < kNormSlabs; ++s)
            suh[c][s] = *(global_ptr<const half8_t>)as_global(p.tab.suh[s < n.slabs ? s : 0] + at);
    }
    float v[CHUNKS][8];
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int e = 8 * (mine + c * threads);
        if (e < n.dim) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4_t sum = {rv[c][h].x + xv[c][h].x, rv[c][h].y + xv[c][h].y, rv[c][h].z + xv[c][h].z, rv[c][h].w + xv[c][h].w};
                *(float4_t*)(n.res_out + base + e + 4 * h) = sum;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v[c][4 * h + j] = sum[j];
                    ss += (double)sum[j] * (double)sum[j];
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[c][j] = 0.0f;
        }
    }
    ss = __shfl(ss, (lane & ~15) | had_chunk(lane), 64);    // summed in the order of the row
    ss = wave_sum(ss);
    if (lane == 0) s_part[tid >> 6] = ss;
    __syncthreads();
    double total = 0.0;
    for (int w = 0; w < (threads >> 6); ++w) total += s_part[w];
    const float rmf = (float)(1.0 / sqrt(total / n.dim + (double)n.epsilon));
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int e = 8 * (mine + c * threads);
        if (e - 8 * had_chunk(lane) >= n.dim) continue;             // the sixteen lanes of a 128 block stay together
        half8_t y;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint16_t bits = __builtin_bit_cast(uint16_t, (_Float16)wb[c][j]);
            const float w = n.weight_bf16 ? __builtin_bit_cast(float, (uint32_t)bits << 16) : (float)(_Float16)wb[c][j];
            float t = v[c][j] * rmf;
            t = t * (w + n.constant_bias);
            t = t * n.constant_scale;
            y[j] = (_Float16)t;
        }
#pragma unroll
        for (int s = 0; s < kNormSlabs; ++s) {
            if (s >= n.slabs) break;
            float r[8];
            mul_half8(y, suh[c][s], r);
            const float unit = had128_row16(r, lane) * kRsqrt128;
            half8_t o;
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = (_Float16)had_scale(r[j], unit);
            _Float16* out = p.tab.out[s] ? p.tab.out[s] : p.out + (size_t)s * p.out_stride;
            *(half8_t*)(out + base + e) = o;
            if (p.operand) store_operand(p, s, row, e, o);
        }
    }
}

static std::string launch_norm_rotate(const RotateArgs& a, const RotateParams& p)
{
    if (a.suh_list || a.slabs > kNormSlabs || a.cols > kNormRotateMaxCols || a.cols % 128)
        throw std::runtime_error("norm + rotation: by-value scales, two slabs and at most " + std::to_string(kNormRotateMaxCols) + " columns");
    const NormInput& in = *a.norm;
    const NormParams n{in.x, in.res, in.res_out, (const uint16_t*)in.weight, a.cols, a.slabs, in.epsilon, in.constant_bias,
                       in.constant_scale, in.weight_bf16};
    const int chunks = (a.cols / 8 + 1023) / 1024;      // 1..4
    const int threads = ((a.cols / 8 + chunks - 1) / chunks + 63) / 64 * 64;
    switch (chunks) {
    case 1: hipLaunchKernelGGL(add_rms_norm_had_r_128_kernel<1>, dim3((unsigned)a.rows), dim3(threads), 0, a.stream, n, p); break;
    case 2: hipLaunchKernelGGL(add_rms_norm_had_r_128_kernel<2>, dim3((unsigned)a.rows), dim3(threads), 0, a.stream, n, p); break;
    default: hipLaunchKernelGGL(add_rms_norm_had_r_128_kernel<4>, dim3((unsigned)a.rows), dim3(threads), 0, a.stream, n, p); break;
    }
    hip_ok(hipGetLastError(), "add + rms_norm + had_r_128 launch");
    return "add_rms_norm_had_r_128_kernel grid=" + std::to_string(a.rows) + " block=" + std::to_string(threads);
}

std::string launch_rotate(const RotateArgs& a)
{
    if (a.slabs < 1 || a.slabs > 65535) throw std::runtime_error("had_r_128 slabs: between 1 and 65535 slabs");
    RotateParams p{};
    p.in = (const _Float16*)a.in;
    p.up = (const _Float16*)a.up;
    p.act_out = (_Float16*)a.act_out;
    p.out = (_Float16*)a.out;
    p.operand = (_Float16*)a.operand;
    p.suh_list = (const uint64_t*)a.suh_list;
    p.in_stride = a.in_stride;
    p.out_stride = a.out_stride;
    p.mt = a.mt;
    p.operand_stride = (size_t)((a.rows + 16 * a.mt - 1) / (16 * a.mt)) * rows_operand_elements(a.cols, a.mt);
    p.col_blocks = a.cols / 128;
    p.blocks = (long)a.rows * p.col_blocks;
    if (p.blocks >= (1L << 31)) throw std::runtime_error("had_r_128 slabs: too many rows");
    if (!a.suh_list) {
        if (a.slabs > kBundleMaxSlices) throw std::runtime_error("had_r_128 slabs: too many slabs for the by-value table");
        for (int i = 0; i < a.slabs; ++i) {
            p.tab.suh[i] = (const _Float16*)a.suh_host[i];
            p.tab.out[i] = a.out_host ? (_Float16*)a.out_host[i] : nullptr;
        }
    }
    if (a.norm) return launch_norm_rotate(a, p);
    const long wgs = (p.blocks + 15) / 16;
    const dim3 grid((unsigned)(wgs < 4096 ? wgs : 4096), (unsigned)a.slabs);
    if (a.up) hipLaunchKernelGGL(silu_mul_had_r_128_kernel, grid, dim3(256), 0, a.stream, p);
    else hipLaunchKernelGGL(had_r_128_slabs_kernel, grid, dim3(256), 0, a.stream, p);
    hip_ok(hipGetLastError(), "had_r_128 slabs launch");
    return std::string(a.up ? "silu_mul_had_r_128_kernel" : "had_r_128_slabs_kernel") + " grid=" + std::to_string(grid.x) +
           "x" + std::to_string(grid.y) + " block=256";
}

std::string launch_had_r_128(const void* in, void* out, const void* scale, int pre_scale,
                             int rows, int cols, int fp32, hipStream_t stream)
{
    const int col_blocks = cols / 128;
    const long blocks = (long)rows * col_blocks;
    const long wgs = (blocks + 15) / 16;                    // four blocks per wave, four waves per workgroup
    const dim3 grid((unsigned)(wgs < 4096 ? wgs : 4096));
    const _Float16* sc = (const _Float16*)scale;
    if (fp32) {
        if (pre_scale) hipLaunchKernelGGL((had_r_128_kernel<float, true>), grid, dim3(256), 0, stream, (const float*)in, (float*)out, sc, blocks, col_blocks);
        else hipLaunchKernelGGL((had_r_128_kernel<float, false>), grid, dim3(256), 0, stream, (const float*)in, (float*)out, sc, blocks, col_blocks);
    } else {
        if (pre_scale) hipLaunchKernelGGL((had_r_128_kernel<_Float16, true>), grid, dim3(256), 0, stream, (const _Float16*)in, (_Float16*)out, sc, blocks, col_blocks);
        else hipLaunchKernelGGL((had_r_128_kernel<_Float16, false>), grid, dim3(256), 0, stream, (const _Float16*)in, (_Float16*)out, sc, blocks, col_blocks);
    }
    hip_ok(hipGetLastError(), "had_r_128 launch");
    return std::string(fp32 ? "had_r_128_kernel<float," : "had_r_128_kernel<half,") + (pre_scale ? "1,0>" : "0,1>") +
           " grid=" + std::to_string(grid.x) + " block=256";
}

// crates/berth-kernels/csrc/ops/act.cu:35-69.  The reference's fixture is
// reproduced bit for bit by half arithmetic with every step rounded to fp16:
// e = exp(-g); s = 1 + e; r = 1 / s; t = g * r; out = t * u.  exp and the
// reciprocal are evaluated in fp32 and rounded once to fp16.
__global__ __launch_bounds__(256) void silu_mul_kernel(const half2_t* __restrict__ gate,
                                                       const half2_t* __restrict__ up,
                                                       half2_t* __restrict__ out, int64_t pairs,
                                                       float act_limit)
{
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pairs) return;
    half2_t g = gate[i], u = up[i], o;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        _Float16 gj = g[j], uj = u[j];
        if (act_limit != 0.0f) {
            float gl = fminf((float)gj, act_limit);
            float ul = fmaxf(fminf((float)uj, act_limit), -act_limit);
            gj = (_Float16)gl;
            uj = (_Float16)ul;
        }
        o[j] = silu_mul_h(gj, uj);
    }
    out[i] = o;
}

std::string launch_silu_mul(const void* gate, const void* up, void* out, int64_t numel,
                            float act_limit, hipStream_t stream)
{
    const int64_t pairs = numel / 2;
    const unsigned blocks = (unsigned)((pairs + 255) / 256);
    hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(256), 0, stream, (const half2_t*)gate,
                       (const half2_t*)up, (half2_t*)out, pairs, act_limit);
    hip_ok(hipGetLastError(), "silu_mul launch");
    return "silu_mul_kernel block=256 grid=" + std::to_string(blocks);
}

// crates/berth-kernels/csrc/ops/add.cu: c = a + b in fp32 (the residual add after the MLP).
__global__ __launch_bounds__(256) void add_f32_kernel(const float* a, const float* b, float* c, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) c[i] = a[i] + b[i];
}

std::string launch_add_f32(const void* a, const void* b, void* c, int n, hipStream_t stream)
{
    const unsigned blocks = (unsigned)((n + 255) / 256);
    hipLaunchKernelGGL(add_f32_kernel, dim3(blocks), dim3(256), 0, stream, (const float*)a, (const float*)b, (float*)c, n);
    hip_ok(hipGetLastError(), "add_f32 launch");
    return "add_f32_kernel block=256 grid=" + std::to_string(blocks);
}

// c[r][j] += bias[j] for a linear that carries a bias (crates/berth-exl3/src/linear.rs:131-133; the
// reference's engine refuses such a linear, crates/berth-engine/src/mlp.rs:67-75).  c is the linear's
// output as written, fp16 or fp32; the sum is formed in fp32 and rounded once to c's type.
template <bool F32>
__global__ __launch_bounds__(256) void add_bias_kernel(void* c, const float* __restrict__ bias, int n, long long total)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const float b = bias[(int)(i % n)];
    if (F32) {
        ((float*)c)[i] += b;
    } else {
        _Float16* h = (_Float16*)c;
        h[i] = (_Float16)((float)h[i] + b);
    }
}

std::string launch_add_bias(void* c, const void* bias, int rows, int n, int c_fp32, hipStream_t stream)
{
    const long long total = (long long)rows * n;
    const unsigned blocks = (unsigned)((total + 255) / 256);
    if (c_fp32)
        hipLaunchKernelGGL(add_bias_kernel<true>, dim3(blocks), dim3(256), 0, stream, c, (const float*)bias, n, total);
    else
        hipLaunchKernelGGL(add_bias_kernel<false>, dim3(blocks), dim3(256), 0, stream, c, (const float*)bias, n, total);
    hip_ok(hipGetLastError(), "add_bias launch");
    return std::string(c_fp32 ? "add_bias_kernel<f32>" : "add_bias_kernel<f16>") + " block=256 grid=" + std::to_string(blocks);
}

// RMS norm of fp32 rows to fp16, optionally with the fused residual
// (crates/berth-kernels/src/ops.rs:398-500, csrc/ops/norm.cu): residual += x in
// place (fp32), then y = fp16((v * rmf) * (w + constant_bias) * constant_scale),
// rmf = fp32(1 / sqrt(mean(v^2) + epsilon)).  The mean is accumulated in double so
// that it does not depend on the order of the reduction.  One workgroup per row.
template <bool RES, bool WBF16>
__global__ __launch_bounds__(256) void rms_norm_kernel(const float* __restrict__ x, const uint16_t* __restrict__ weight,
                                                       _Float16* __restrict__ y, float* residual, int dim,
                                                       float epsilon, float constant_bias, float constant_scale)
{
    __shared__ double s_part[4];
    __shared__ float s_rmf;
    const int row = blockIdx.x, tid = threadIdx.x;
    const float4_t* xr = (const float4_t*)(x + (size_t)row * dim);
    float4_t* rr = RES ? (float4_t*)(residual + (size_t)row * dim) : nullptr;
    double ss = 0.0;
    for (int i = tid; i < dim / 4; i += 256) {
        float4_t v = xr[i];
        if (RES) {
            const float4_t r = rr[i];
            v = float4_t{r.x + v.x, r.y + v.y, r.z + v.z, r.w + v.w};
            rr[i] = v;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) ss += (double)v[j] * (double)v[j];
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_part[tid >> 6] = ss;
    __syncthreads();
    if (tid == 0) {
        const double total = ((s_part[0] + s_part[1]) + s_part[2]) + s_part[3];
        s_rmf = (float)(1.0 / sqrt(total / dim + (double)epsilon));
    }
    __syncthreads();
    const float rmf = s_rmf;
    for (int i = tid; i < dim / 4; i += 256) {
        const float4_t v = RES ? rr[i] : xr[i];     // RES: this thread wrote these four itself
        half4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint16_t wb = weight[4 * i + j];
            const float w = WBF16 ? __builtin_bit_cast(float, (uint32_t)wb << 16)
                                  : (float)__builtin_bit_cast(_Float16, wb);
            float t = v[j] * rmf;
            t = t * (w + constant_bias);
            t = t * constant_scale;
            o[j] = (_Float16)t;
        }
        *(half4_t*)(y + (size_t)row * dim + 4 * i) = o;
    }
}

// The same norm with the row held in registers: eight values a thread and chunk, so that a row is
// read once (RES: read and updated once), the weight is requested along with it and the wait for
// memory is paid once.  Traced: one row of 5120 6.5 -> 4.7 us, 1500 rows 13.6 -> 12.1.
template <int CHUNKS, bool RES, bool WBF16>
__global__ __launch_bounds__(1024) void rms_norm_row_kernel(const float* __restrict__ x, const uint16_t* __restrict__ weight,
                                                            _Float16* __restrict__ y, float* residual, int dim,
                                                            float epsilon, float constant_bias, float constant_scale)
{
    __shared__ double s_part[16];
    const int tid = threadIdx.x, threads = blockDim.x;
    const size_t base = (size_t)blockIdx.x * dim;
    typedef uint16_t u16x8_t __attribute__((ext_vector_type(8)));
    float v[CHUNKS][8];
    u16x8_t wb[CHUNKS];
    double ss = 0.0;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int e = 8 * (tid + c * threads);
        const int at = e < dim ? e : 0;                     // past the end: read and not used
        wb[c] = *(const u16x8_t*)(weight + at);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float4_t t = *(const float4_t*)(x + base + at + 4 * h);
            if (RES) {
                const float4_t r = *(const float4_t*)(residual + base + at + 4 * h);
                t = float4_t{r.x + t.x, r.y + t.y, r.z + t.z, r.w + t.w};
                if (e < dim) *(float4_t*)(residual + base + at + 4 * h) = t;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[c][4 * h + j] = t[j];
                if (e < dim) ss += (double)t[j] * (double)t[j];
            }
        }
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_part[tid >> 6] = ss;
    __syncthreads();
    double total = 0.0;
    for (int w = 0; w < (threads >> 6); ++w) total += s_part[w];
    const float rmf = (float)(1.0 / sqrt(total / dim + (double)epsilon));
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int e = 8 * (tid + c * threads);
        if (e >= dim) break;
        half8_t o;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint16_t b = wb[c][j];
            const float w = WBF16 ? __builtin_bit_cast(float, (uint32_t)b << 16) : (float)__builtin_bit_cast(_Float16, b);
            float t = v[c][j] * rmf;
            t = t * (w + constant_bias);
            t = t * constant_scale;
            o[j] = (_Float16)t;
        }
        *(half8_t*)(y + base + e) = o;
    }
}

template <bool RES, bool WBF16>
static void launch_rms_norm_row(const float* x, const uint16_t* w, _Float16* y, float* r, int rows, int dim, float epsilon,
                                float constant_bias, float constant_scale, hipStream_t stream)
{
    const int chunks = (dim / 8 + 1023) / 1024;             // 1..4
    const dim3 grid((unsigned)rows), block((unsigned)(((dim / 8 + chunks - 1) / chunks + 63) / 64 * 64));
    switch (chunks) {
    case 1: hipLaunchKernelGGL((rms_norm_row_kernel<1, RES, WBF16>), grid, block, 0, stream, x, w, y, r, dim, epsilon, constant_bias, constant_scale); break;
    case 2: hipLaunchKernelGGL((rms_norm_row_kernel<2, RES, WBF16>), grid, block, 0, stream, x, w, y, r, dim, epsilon, constant_bias, constant_scale); break;
    default: hipLaunchKernelGGL((rms_norm_row_kernel<4, RES, WBF16>), grid, block, 0, stream, x, w, y, r, dim, epsilon, constant_bias, constant_scale); break;
    }
}

std::string launch_rms_norm(const void* x, const void* weight, void* y, void* residual, int rows, int dim,
                            float epsilon, float constant_bias, float constant_scale, int weight_bf16,
                            hipStream_t stream)
{
    const dim3 grid((unsigned)rows), block(256);
    const float* xf = (const float*)x;
    const uint16_t* w = (const uint16_t*)weight;
    _Float16* yh = (_Float16*)y;
    float* r = (float*)residual;
    // rows of eight values a thread, sixteen bytes at a time; what does not divide or align takes
    // the four-value kernel
    const bool by_row = dim % 8 == 0 && dim <= 32768 && (((uintptr_t)x | (uintptr_t)weight | (uintptr_t)y | (uintptr_t)residual) & 15) == 0;
    if (by_row) {
        if (residual) {
            if (weight_bf16) launch_rms_norm_row<true, true>(xf, w, yh, r, rows, dim, epsilon, constant_bias, constant_scale, stream);
            else launch_rms_norm_row<true, false>(xf, w, yh, r, rows, dim, epsilon, constant_bias, constant_scale, stream);
        } else {
            if (weight_bf16) launch_rms_norm_row<false, true>(xf, w, yh, r, rows, dim, epsilon, constant_bias, constant_scale, stream);
            else launch_rms_norm_row<false, false>(xf, w, yh, r, rows, dim, epsilon, constant_bias, constant_scale, stream);
        }
    } else if (residual) {
        if (weight_bf16) hipLaunchKernelGGL((rms_norm_kernel<true, true>), grid, block, 0, stream, xf, w, yh, r, dim, epsilon, constant_bias, constant_scale);
        else hipLaunchKernelGGL((rms_norm_kernel<true, false>), grid, block, 0, stream, xf, w, yh, r, dim, epsilon, constant_bias, constant_scale);
    } else {
        if (weight_bf16) hipLaunchKernelGGL((rms_norm_kernel<false, true>), grid, block, 0, stream, xf, w, yh, r, dim, epsilon, constant_bias, constant_scale);
        else hipLaunchKernelGGL((rms_norm_kernel<false, false>), grid, block, 0, stream, xf, w, yh, r, dim, epsilon, constant_bias, constant_scale);
    }
    hip_ok(hipGetLastError(), "rms_norm launch");
    return std::string(by_row ? "rms_norm_row_kernel<" : "rms_norm_kernel<") + (residual ? "2" : "0") + ",float,half," + (weight_bf16 ? "bfloat16" : "half") +
           ",float> grid=" + std::to_string(rows);
}

// RMS norm of fp16 rows to fp16 with a bf16 weight and no residual
// (crates/berth-kernels/src/ops.rs:108-118,600-640, csrc/ops/norm.cu:80-112: the
// normalisation ahead of the MTP input projection).  The fp16 input widens exactly to
// fp32; from there the arithmetic is that of rms_norm_kernel.
__global__ __launch_bounds__(256) void rms_norm_f16_kernel(const _Float16* __restrict__ x, const uint16_t* __restrict__ weight,
                                                           _Float16* __restrict__ y, int dim, float epsilon,
                                                           float constant_bias, float constant_scale)
{
    __shared__ double s_part[4];
    __shared__ float s_rmf;
    const int row = blockIdx.x, tid = threadIdx.x;
    const half4_t* xr = (const half4_t*)(x + (size_t)row * dim);
    double ss = 0.0;
    for (int i = tid; i < dim / 4; i += 256) {
        const half4_t v = xr[i];
#pragma unroll
        for (int j = 0; j < 4; ++j) ss += (double)(float)v[j] * (double)(float)v[j];
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) s_part[tid >> 6] = ss;
    __syncthreads();
    if (tid == 0) {
        const double total = ((s_part[0] + s_part[1]) + s_part[2]) + s_part[3];
        s_rmf = (float)(1.0 / sqrt(total / dim + (double)epsilon));
    }
    __syncthreads();
    const float rmf = s_rmf;
    for (int i = tid; i < dim / 4; i += 256) {
        const half4_t v = xr[i];
        half4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float w = __builtin_bit_cast(float, (uint32_t)weight[4 * i + j] << 16);
            float t = (float)v[j] * rmf;
            t = t * (w + constant_bias);
            t = t * constant_scale;
            o[j] = (_Float16)t;
        }
        *(half4_t*)(y + (size_t)row * dim + 4 * i) = o;
    }
}

std::string launch_rms_norm_f16(const void* x, const void* weight, void* y, int rows, int dim, float epsilon,
                                float constant_bias, float constant_scale, hipStream_t stream)
{
    hipLaunchKernelGGL(rms_norm_f16_kernel, dim3((unsigned)rows), dim3(256), 0, stream, (const _Float16*)x,
                       (const uint16_t*)weight, (_Float16*)y, dim, epsilon, constant_bias, constant_scale);
    hip_ok(hipGetLastError(), "rms_norm_f16 launch");
    return "rms_norm_f16_kernel<0,half,half,bfloat16,half> block=256 grid=" + std::to_string(rows);
}

// Embedding rows (crates/berth-kernels/src/ops.rs:99-127, csrc/ops/embed.cu): out[t] =
// weight[ids[t]], bf16 -> fp32 (an exact widen) or bf16 -> fp16 (the widen, then one
// round-to-nearest-even).  ids are not range-checked, as in the reference.
template <bool F16>
__global__ __launch_bounds__(256) void embed_bf16_kernel(const uint16_t* __restrict__ weight, const int* __restrict__ ids,
                                                         void* __restrict__ out, int hidden)
{
    const int token = blockIdx.x;
    const uint16_t* row = weight + (size_t)ids[token] * hidden;
    for (int i = threadIdx.x; i < hidden; i += 256) {
        const float v = __builtin_bit_cast(float, (uint32_t)row[i] << 16);
        if (F16) ((_Float16*)out)[(size_t)token * hidden + i] = (_Float16)v;
        else ((float*)out)[(size_t)token * hidden + i] = v;
    }
}

std::string launch_embed_tokens(const void* weight, const int* ids, void* out, int hidden, int n, int f16,
                                hipStream_t stream)
{
    if (f16) hipLaunchKernelGGL(embed_bf16_kernel<true>, dim3((unsigned)n), dim3(256), 0, stream, (const uint16_t*)weight, ids, out, hidden);
    else hipLaunchKernelGGL(embed_bf16_kernel<false>, dim3((unsigned)n), dim3(256), 0, stream, (const uint16_t*)weight, ids, out, hidden);
    hip_ok(hipGetLastError(), f16 ? "embed_tokens_f16 launch" : "embed_tokens launch");
    return std::string(f16 ? "embed_bf16_kernel<f16>" : "embed_bf16_kernel<f32>") + " block=256 grid=" + std::to_string(n);
}

// out[row] = embedding[row] followed by hidden[row], fp16 (crates/berth-kernels/src/ops.rs:136-143,
// csrc/ops/copy.cu: the concatenation ahead of the MTP input projection)
__global__ __launch_bounds__(256) void cat_f16_last_kernel(const uint16_t* __restrict__ embedding,
                                                           const uint16_t* __restrict__ hidden,
                                                           uint16_t* __restrict__ out, int width)
{
    const size_t row = blockIdx.x;
    for (int i = threadIdx.x; i < width; i += 256) {
        out[row * 2 * width + i] = embedding[row * width + i];
        out[row * 2 * width + width + i] = hidden[row * width + i];
    }
}

std::string launch_cat_f16_last(const void* embedding, const void* hidden, void* out, int rows, int width,
                                hipStream_t stream)
{
    hipLaunchKernelGGL(cat_f16_last_kernel, dim3((unsigned)rows), dim3(256), 0, stream, (const uint16_t*)embedding,
                       (const uint16_t*)hidden, (uint16_t*)out, width);
    hip_ok(hipGetLastError(), "cat_f16_last launch");
    return "cat_f16_last_kernel block=256 grid=" + std::to_string(rows);
}

// crates/berth-exl3/src/signs.rs:25-46: packed su / sv -> fp16 signs.  Little-endian
// u16 words, bit i of a word is element i of its 16; a set bit is -1.0 (0xBC00),
// a clear bit +1.0 (0x3C00).  One thread per output pair.
__global__ __launch_bounds__(256) void unpack_signs_kernel(const uint16_t* __restrict__ packed,
                                                           uint32_t* __restrict__ out, int64_t pairs)
{
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pairs) return;
    const uint32_t word = packed[i >> 3];
    const uint32_t two = (word >> (2 * (i & 7))) & 3u;
    out[i] = 0x3C003C00u | ((two & 1u) << 15) | ((two & 2u) << 30);
}

std::string launch_unpack_signs(const void* packed, void* out, int64_t words, hipStream_t stream)
{
    const int64_t pairs = words * 8;
    const unsigned blocks = (unsigned)((pairs + 255) / 256);
    hipLaunchKernelGGL(unpack_signs_kernel, dim3(blocks), dim3(256), 0, stream, (const uint16_t*)packed,
                       (uint32_t*)out, pairs);
    hip_ok(hipGetLastError(), "unpack_signs launch");
    return "unpack_signs_kernel block=256 grid=" + std::to_string(blocks);
}

}  // namespace berth
