// producers.hip - the ops that feed an FP8 linear, quantizing their own
// output (gfx950): RMSNorm + activation quantization and SwiGLU +
// activation quantization, for rows of a prefill (or decode) batch.
//
// In the reference every FP8 linear quantizes its bf16 input in a separate
// launch (quantize_act_rows_fp8, src/hephaestus/kernels.mojo:270-287, called
// from linear_fp8 at :449-450) right after the op that produced that input
// (rms_norm, forward.mojo:45-81; silu_mul, kernels.mojo:1243-1278); the
// reference's own notes blame its FP8 GEMM gap on that extra launch and the
// extra pass over the activations. Here the producer writes the E4M3 codes
// and scales itself, bit for bit what heph_rmsnorm (heph_silu_mul) followed
// by heph_fp8_quant_act write, and the linear runs with
// HEPH_FLAG_SKIP_QUANT: one launch and one read of the bf16 activations
// fewer per linear, and the normalized (activated) bf16 row is never
// written.
#include <algorithm>

#include "../../include/hephdecode.h"
#include "heph_kernels.h"

namespace heph {

namespace {

// Longest row the fused ops hold in LDS as bf16 (32 KB).
constexpr int kProdMaxCols = 16384;

__device__ __forceinline__ float f32b(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ float rbf16(float f) { return f32b(f32_to_bf16(f)); }

// Quantizes one row held as bf16 in LDS (yrow, cols elements) into codes
// q[cols] and scales s[cols / group_k], as quant_g128_kernel (group 128:
// 16-lane teams over 8 elements each, amax on bf16 magnitude bits, NaN
// skipped) or quant_row_kernel (group cols) do. Every thread of the
// 256-thread workgroup calls it after the row is in LDS.
__device__ __forceinline__ void quant_row_from_lds(const uint16_t* yrow, int cols, int group_k,
                                                   uint8_t* q, float* s)
{
    const int t = threadIdx.x;
    if (group_k == kChunk) {
        const int G = cols / kChunk, team = t >> 4, j = t & 15;
        for (int g0 = 0; g0 < G; g0 += 16) {
            const int g = g0 + team;
            const bool live = g < G;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (live) v = *reinterpret_cast<const uint4*>(yrow + g * kChunk + j * 8);
            uint32_t mb = absmax_bits8(v);
            for (int o = 1; o < 16; o <<= 1) mb = max(mb, shfl_xor_u(mb, o));
            if (__builtin_amdgcn_ballot_w64(mb > 0x7F80u) != 0) {
                mb = absmax_bits8_skip_nan(v);
                for (int o = 1; o < 16; o <<= 1) mb = max(mb, shfl_xor_u(mb, o));
            }
            float sc, inv;
            group_scale(bf16_bits_f32(mb), sc, inv);
            if (live) {
                *reinterpret_cast<uint2*>(q + g * kChunk + j * 8) = quant8(v, inv);
                if (j == 0) s[g] = sc;
            }
        }
        return;
    }
    __shared__ uint32_t red[4];
    uint32_t m = 0;
    for (int k = t * 8; k < cols; k += 256 * 8)
        m = absmax_bits8_skip_nan(*reinterpret_cast<const uint4*>(yrow + k), m);
    for (int o = 32; o >= 1; o >>= 1) m = max(m, shfl_xor_u(m, o));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = max(max(red[0], red[1]), max(red[2], red[3]));
    float sc, inv;
    group_scale(bf16_bits_f32(m), sc, inv);
    if (t == 0) s[0] = sc;
    for (int k = t * 8; k < cols; k += 256 * 8)
        *reinterpret_cast<uint2*>(q + k) = quant8(*reinterpret_cast<const uint4*>(yrow + k), inv);
}

// One workgroup per row. The norm is heph_rmsnorm's: thread t < 256 sums the
// squares of elements t, t + 256, ... in that order (fma), the 256 sums fold as
// fold256_wave0 does, and y = bf16(gamma * bf16(x * r)). A row of a prefill
// batch is a few KB, so the kernel is a chain of latencies; it is kept to one
// round of 16-byte loads (PPT pieces of 8 elements a thread, the row's and
// gamma's in flight together), one staging of the row in LDS for the sums in
// their order, and two barriers: a thread then normalizes the pieces it still
// holds, and sixteen neighbouring lanes hold a whole 1x128 group, quantized
// where it is. MI355X, graph-replayed, against 2-byte
// loads of elements t, t + 256, .. and a second staging of y for the groups:
// 512 rows of 2560 6.4 -> 4.3 us, 64 of 4096 7.5 -> 3.7, 4096 of 2560 19.7 ->
// 14.5.
template <int PPT>
__global__ __launch_bounds__(1024) void rmsnorm_quant_kernel(uint8_t* q, float* scales,
                                                             const uint16_t* in,
                                                             const uint16_t* gamma, int cols,
                                                             float eps, int group_k)
{
    __shared__ float red[256];
    __shared__ uint32_t redm[16];
    extern __shared__ __attribute__((aligned(16))) uint16_t xrow[];
    const int t = threadIdx.x, nt = blockDim.x, np = cols / 8;
    const uint16_t* x = in + (size_t)blockIdx.x * cols;
    uint4 xv[PPT], gv[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const int p = t + k * nt;
        xv[k] = gv[k] = make_uint4(0, 0, 0, 0);
        if (p < np) {
            xv[k] = ldg16u(x + 8 * p);
            gv[k] = ldg16u(gamma + 8 * p);
        }
    }
#pragma unroll
    for (int k = 0; k < PPT; ++k)
        if (t + k * nt < np) *reinterpret_cast<uint4*>(xrow + 8 * (t + k * nt)) = xv[k];
    __syncthreads();
    float ss = 0.0f;
    if (t < 256) {
#pragma unroll 8
        for (int i = t; i < cols; i += 256) {
            const float v = f32b(xrow[i]);
            ss = __builtin_fmaf(v, v, ss);
        }
    }
    const float r = rms_inv(fold256_every_wave(ss, red), cols, eps);
    uint4 y[PPT];
#pragma unroll
    for (int k = 0; k < PPT; ++k) {
        const uint32_t xd[4] = {xv[k].x, xv[k].y, xv[k].z, xv[k].w};
        const uint32_t gd[4] = {gv[k].x, gv[k].y, gv[k].z, gv[k].w};
        uint32_t yd[4];
#pragma unroll
        for (int d = 0; d < 4; ++d)
            yd[d] = (uint32_t)f32_to_bf16(bf16lo(gd[d]) * rbf16(bf16lo(xd[d]) * r)) |
                    ((uint32_t)f32_to_bf16(bf16hi(gd[d]) * rbf16(bf16hi(xd[d]) * r)) << 16);
        y[k] = make_uint4(yd[0], yd[1], yd[2], yd[3]);
    }
    uint8_t* qr = q + (size_t)blockIdx.x * cols;
    if (group_k == kChunk) {
        // (cols % 128 == 0: a team of 16 lanes is whole or has no piece)
        float* sr = scales + (size_t)blockIdx.x * (cols / kChunk);
#pragma unroll
        for (int k = 0; k < PPT; ++k) {
            const int p = t + k * nt;
            uint32_t mb = absmax_bits8(y[k]);
            if (mb > 0x7F80u) mb = absmax_bits8_skip_nan(y[k]);    // this lane holds a NaN
            mb = lanes_max_u<16>(mb);
            float sc, inv;
            group_scale(bf16_bits_f32(mb), sc, inv);
            if (p < np) {
                *reinterpret_cast<uint2*>(qr + 8 * p) = quant8(y[k], inv);
                if ((p & 15) == 0) sr[p >> 4] = sc;
            }
        }
        return;
    }
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < PPT; ++k) m = absmax_bits8_skip_nan(y[k], m);
    m = lanes_max_u<64>(m);
    if ((t & 63) == 0) redm[t >> 6] = m;
    __syncthreads();
    for (int w = 0; w < nt / 64; ++w) m = max(m, redm[w]);
    float sc, inv;
    group_scale(bf16_bits_f32(m), sc, inv);
    if (t == 0) scales[blockIdx.x] = sc;
#pragma unroll
    for (int k = 0; k < PPT; ++k)
        if (t + k * nt < np) *reinterpret_cast<uint2*>(qr + 8 * (t + k * nt)) = quant8(y[k], inv);
}

// The same for a row or gamma that is not 16-byte aligned: element loads, y
// staged in LDS and quantized from there. It reads the row twice, the second
// time from the cache, and keeps none of it in registers; against a form that
// held 10, 16 or 40 elements a thread (graph-replayed): 4 rows of 2560 5.8 -> 4.8
// us, 4490 of 1024 14.6 -> 11.7, 1608 of 8448 39.7 -> 27.2, 1937 of 12544 63.3 ->
// 60.3.
__global__ __launch_bounds__(256) void rmsnorm_quant_unaligned_kernel(
    uint8_t* q, float* scales, const uint16_t* in, const uint16_t* gamma, int cols, float eps,
    int group_k)
{
    __shared__ float red[256];
    __shared__ float res;
    extern __shared__ __attribute__((aligned(16))) uint16_t yrow[];
    const uint16_t* x = in + (size_t)blockIdx.x * cols;
    const int t = threadIdx.x;
    float ss = 0.0f;
    for (int i = t; i < cols; i += 256) {
        const float v = f32b(x[i]);
        ss = __builtin_fmaf(v, v, ss);
    }
    const float r = rms_inv(fold256_wave0(ss, red, &res), cols, eps);
    for (int i = t; i < cols; i += 256)
        yrow[i] = f32_to_bf16(f32b(gamma[i]) * rbf16(f32b(x[i]) * r));
    __syncthreads();
    quant_row_from_lds(yrow, cols, group_k, q + (size_t)blockIdx.x * cols,
                       scales + (size_t)blockIdx.x * (cols / group_k));
}

__device__ __forceinline__ uint4 swiglu8(const uint4& g, const uint4& u)
{
    const uint32_t gd[4] = {g.x, g.y, g.z, g.w}, ud[4] = {u.x, u.y, u.z, u.w};
    uint32_t r[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
        r[d] = swiglu_bits((uint16_t)gd[d], (uint16_t)ud[d]) |
               (swiglu_bits((uint16_t)(gd[d] >> 16), (uint16_t)(ud[d] >> 16)) << 16);
    return make_uint4(r[0], r[1], r[2], r[3]);
}

// 1x128 groups: one 16-lane team per group of one row, 8 elements a lane,
// the SwiGLU values computed in registers and quantized as
// quant_g128_kernel does. 6 bytes of traffic an element against ~25
// instructions (silu_bf16; ~60 with expf and an IEEE division, which bound the
// kernel): 512 rows of 9728 10.2 -> 7.6 us, 4096 rows 57.3 -> 39.9 (6.0 TB/s).
__global__ __launch_bounds__(256) void silu_mul_quant_g128_kernel(
    uint8_t* __restrict__ q, float* __restrict__ scales, const uint16_t* __restrict__ gate,
    const uint16_t* __restrict__ up, int n, long ld, long n_groups)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long gi = t >> 4;
    const int j = threadIdx.x & 15;
    const bool live = gi < n_groups;
    const int G = n / kChunk;
    const long row = live ? gi / G : 0, g = live ? gi % G : 0;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (live) {
        const size_t off = (size_t)row * ld + (size_t)g * kChunk + j * 8;
        v = swiglu8(ldg16u(gate + off), ldg16u(up + off));
    }
    uint32_t mb = absmax_bits8(v);
    for (int o = 1; o < 16; o <<= 1) mb = max(mb, shfl_xor_u(mb, o));
    if (__builtin_amdgcn_ballot_w64(mb > 0x7F80u) != 0) {
        mb = absmax_bits8_skip_nan(v);
        for (int o = 1; o < 16; o <<= 1) mb = max(mb, shfl_xor_u(mb, o));
    }
    float s, inv;
    group_scale(bf16_bits_f32(mb), s, inv);
    if (live) {
        *reinterpret_cast<uint2*>(q + (size_t)row * n + g * kChunk + j * 8) = quant8(v, inv);
        if (j == 0) scales[row * G + g] = s;
    }
}

// Per-token groups: one workgroup per row, the row's SwiGLU values staged
// in LDS, then quantized as quant_row_kernel does.
__global__ __launch_bounds__(256) void silu_mul_quant_row_kernel(uint8_t* q, float* scales,
                                                                 const uint16_t* gate,
                                                                 const uint16_t* up, int n,
                                                                 long ld)
{
    extern __shared__ __attribute__((aligned(16))) uint16_t yrow[];    // n bf16
    const size_t off = (size_t)blockIdx.x * ld;
    for (int k = threadIdx.x * 8; k < n; k += 256 * 8)
        *reinterpret_cast<uint4*>(yrow + k) = swiglu8(ldg16u(gate + off + k), ldg16u(up + off + k));
    __syncthreads();
    quant_row_from_lds(yrow, n, n, q + (size_t)blockIdx.x * n, scales + blockIdx.x);
}

bool a16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

}  // namespace heph

using namespace heph;

extern "C" {

int heph_rmsnorm_quant_fp8(uint8_t* q, float* scales, const uint16_t* x_bf16,
                           const uint16_t* gamma_bf16, int rows, int cols, float eps, int group_k,
                           void* stream)
{
    if (!q || !scales || !x_bf16 || !gamma_bf16) return HEPH_ERR_NULL;
    if (rows < 1 || cols < kChunk || cols % kChunk) return HEPH_ERR_SHAPE;
    if (group_k != kChunk && group_k != cols) return HEPH_ERR_GROUP;
    if (cols > kProdMaxCols) return HEPH_ERR_UNSUPPORTED;
    if (!a16(q)) return HEPH_ERR_ALIGN;
    if (int st = check_device()) return st;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const size_t lds = (size_t)cols * 2;
    const int np = cols / 8;      // 16-byte pieces; 16384 / 8 = two per thread
    const int nt = std::min(1024, std::max(256, (np + 63) / 64 * 64));
    if (!a16(x_bf16) || !a16(gamma_bf16))
        rmsnorm_quant_unaligned_kernel<<<rows, 256, lds, s>>>(q, scales, x_bf16, gamma_bf16, cols,
                                                              eps, group_k);
    else if (np <= nt)
        rmsnorm_quant_kernel<1><<<rows, nt, lds, s>>>(q, scales, x_bf16, gamma_bf16, cols, eps,
                                                      group_k);
    else
        rmsnorm_quant_kernel<2><<<rows, nt, lds, s>>>(q, scales, x_bf16, gamma_bf16, cols, eps,
                                                      group_k);
    return hipGetLastError() == hipSuccess ? HEPH_OK : HEPH_ERR_LAUNCH;
}

int heph_silu_mul_quant_fp8(uint8_t* q, float* scales, const uint16_t* gate_bf16,
                            const uint16_t* up_bf16, int rows, int n, int ld, int group_k,
                            void* stream)
{
    if (!q || !scales || !gate_bf16 || !up_bf16) return HEPH_ERR_NULL;
    if (rows < 1 || n < kChunk || n % kChunk || ld < n || ld % 8) return HEPH_ERR_SHAPE;
    if (group_k != kChunk && group_k != n) return HEPH_ERR_GROUP;
    if (group_k == n && n > kProdMaxCols) return HEPH_ERR_UNSUPPORTED;
    if (!a16(q) || !a16(gate_bf16) || !a16(up_bf16)) return HEPH_ERR_ALIGN;
    if (int st = check_device()) return st;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (group_k == kChunk) {
        const long n_groups = (long)rows * (n / kChunk);
        const unsigned blocks = (unsigned)((n_groups * 16 + 255) / 256);
        silu_mul_quant_g128_kernel<<<blocks, 256, 0, s>>>(q, scales, gate_bf16, up_bf16, n,
                                                          (long)ld, n_groups);
    } else {
        silu_mul_quant_row_kernel<<<rows, 256, (size_t)n * 2, s>>>(q, scales, gate_bf16, up_bf16,
                                                                    n, (long)ld);
    }
    return hipGetLastError() == hipSuccess ? HEPH_OK : HEPH_ERR_LAUNCH;
}

}  // extern "C"
