// bf16_gemm.hip - unquantized bf16 linear for M > 32.
//
// Replaces the reference's bf16 GEMM for more than one row
// (src/hephaestus/wmma_gfx12.mojo:428-473, wmma_gemm_bf16, reached through
// `linear`, src/hephaestus/kernels.mojo:108-118), e.g. the lm_head over
// every position of a prompt. Rows up to 32 take the weight-streaming
// kernel in bf16_skinny.hip.
//
// The DMA-staged tiles of gemm_big.h and gemm_ring.h in their bf16 form take
// most calls whose operands' byte offsets fit 32 bits: no per-chunk scales,
// so the MFMAs accumulate in place. They are bound by the weight stream (up
// to M of about 100) or by the MFMAs; what costs beside that is rows of the
// last tile past M, a last round of tiles that leaves CUs idle, and the DMA's
// latency at the start of each tile, which the choice of tile trades against
// each other (kBf16Tiles). MI355X, graph-replayed over HBM-streamed weights,
// against the register-staged kernel below: the lm_head (151936 x 2560, f32
// logits) at M = 64 193 -> 178 us, 160 292 -> 188, 257 414 -> 265, 512 570 ->
// 390; 4096 x 6144 x 2560 181 -> 119; M = 45 at 4256 x 1408 21.8 -> 11.0; over
// 51 shapes (M 33 .. 4096) 0.50 to 0.996 of its time, 0.70 in the mean.
//
// The register-staged kernel, for larger operands and where its two tiles on a
// CU beat the ring tiles (bf16_gemm_tile):
//   * 128 x 128 output tile per 256-thread workgroup, 2 x 2 waves of
//     64 x 64, each wave 4 x 4 v_mfma_f32_16x16x32_bf16 per 32-wide K step,
//     two steps per 64-element (128-byte) chunk; the MFMAs accumulate in
//     fp32 across all of K;
//   * the weights are the MFMA's first operand, so lane l's four results
//     are output columns 4*(l >> 4) + i of activation row l & 15: four
//     consecutive outputs per lane, stored together;
//   * chunks are double buffered in LDS with the next chunk's global loads
//     in flight during the MFMAs, one barrier per chunk; LDS rows padded to
//     144 bytes, so the 16 rows of a fragment read fall in distinct banks;
//   * workgroups walk the tiles in groups of 8 tile rows (each weight tile
//     is reused by 8 consecutive workgroups while it is in the L2);
//   * epilogue: the residual (the output buffer's bf16 or f32 values) is
//     added in f32 before the one rounding; rows past M and columns past N
//     are computed on clamped rows and not stored.
#include <algorithm>

#include "gemm_big.h"
#include "gemm_ring.h"

namespace heph {

namespace {
constexpr int kGbM = 128, kGbN = 128;
constexpr int kGbChunk = 64;              // bf16 elements per chunk (128 bytes)
constexpr int kGbLd = 144;                // LDS bytes per row
constexpr int kGbGroup = 8;               // tile rows per group

__device__ __forceinline__ bf16x8 lds_frag(const uint8_t* p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const i32x4*>(p));
}
}  // namespace

__global__ __launch_bounds__(256, 2) void bf16_gemm_kernel(Bf16GemmArgs a)
{
    __shared__ __attribute__((aligned(16))) uint8_t As[2][kGbM * kGbLd];
    __shared__ __attribute__((aligned(16))) uint8_t Bs[2][kGbN * kGbLd];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, slice = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    const int M = a.M, N = a.N, K = a.K, KC = K / kGbChunk;
    const int tiles_m = (M + kGbM - 1) / kGbM, tiles_n = (N + kGbN - 1) / kGbN;
    // grouped order: kGbGroup tile rows sweep each tile column together
    const int bid = blockIdx.x;
    const int width = kGbGroup * tiles_n;
    const int first_m = (bid / width) * kGbGroup;
    const int gsize = min(tiles_m - first_m, kGbGroup);
    const int r = bid % width;
    const int m0 = (first_m + r % gsize) * kGbM, n0 = (r / gsize) * kGbN;

    // global -> LDS staging: 1024 16-byte pieces per operand tile, four per
    // thread; eight consecutive threads cover one 128-byte row chunk. Rows
    // past M (N) are clamped to the last row.
    const int lrow = tid >> 3, lcol = (tid & 7) * 8;    // elements
    const uint16_t* ag[4];
    const uint16_t* bg[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        ag[q] = a.x + (size_t)min(m0 + lrow + 32 * q, M - 1) * K + lcol;
        bg[q] = a.w + (size_t)min(n0 + lrow + 32 * q, N - 1) * K + lcol;
    }
    i32x4 ra[4], rb[4];
    auto gload = [&](int j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            ra[q] = ldg16(ag[q] + (size_t)j * kGbChunk);
            rb[q] = ldg16(bg[q] + (size_t)j * kGbChunk);
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            *reinterpret_cast<i32x4*>(&As[buf][(lrow + 32 * q) * kGbLd + lcol * 2]) = ra[q];
            *reinterpret_cast<i32x4*>(&Bs[buf][(lrow + 32 * q) * kGbLd + lcol * 2]) = rb[q];
        }
    };

    f32x4 acc[4][4];    // [activation row tile][weight column tile]
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0, 0, 0, 0};

    gload(0);
    lstore(0);
    __syncthreads();
    for (int j = 0; j < KC; ++j) {
        const int cur = j & 1;
        if (j + 1 < KC) gload(j + 1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            // lane (r16, slice): elements ks*32 + slice*8 .. +7 of its row
            const int off = ks * 64 + slice * 16;
            bf16x8 xa[4], wb[4];
#pragma unroll
            for (int mi = 0; mi < 4; ++mi)
                xa[mi] = lds_frag(&As[cur][(wm * 64 + mi * 16 + r16) * kGbLd + off]);
#pragma unroll
            for (int ni = 0; ni < 4; ++ni)
                wb[ni] = lds_frag(&Bs[cur][(wn * 64 + ni * 16 + r16) * kGbLd + off]);
#pragma unroll
            for (int mi = 0; mi < 4; ++mi)
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = mfma_bf16(wb[ni], xa[mi], acc[mi][ni]);
        }
        if (j + 1 < KC) lstore(cur ^ 1);
        __syncthreads();
    }

    // lane (r16, slice): row m0 + wm*64 + mi*16 + r16, columns
    // n0 + wn*64 + ni*16 + 4*slice .. +3
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
        const int row = m0 + wm * 64 + mi * 16 + r16;
        if (row >= M) continue;
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
            const int col = n0 + wn * 64 + ni * 16 + 4 * slice;
            if (col >= N) continue;
            f32x4 v = acc[mi][ni];
            const size_t o = (size_t)row * N + col;
            if (a.c_f32) {
                f32x4* c = reinterpret_cast<f32x4*>(static_cast<float*>(a.c) + o);
                if (a.residual) v += *c;
                *c = v;
            } else {
                uint2* c = reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.c) + o);
                if (a.residual) {
                    const uint2 rv = *c;
                    v[0] += bf16lo(rv.x);
                    v[1] += bf16hi(rv.x);
                    v[2] += bf16lo(rv.y);
                    v[3] += bf16hi(rv.y);
                }
                *c = make_uint2((uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16),
                                (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16));
            }
        }
    }
}

namespace {

// Tiles of the DMA-staged kernels and the model that picks one: with n tiles
// on the fullest CU and KC chunks of 64 elements, n g + KC max(c1, n c) + 2 us,
// but at least the weights and the output at 5 TB/s, the rate the tiles reach
// where the stream bounds them. Of two tiles at that bound the one with less
// time of its own is taken among the first three (a call it bounds has few
// rows), else the earlier entry (92 x 119680 x 2304 on 160 x 320 136 us, on the
// register-staged kernel 129; 108 x 127808 x 1408 95.1, on 128 x 256 90.6).
// c1 is a chunk's latency with one workgroup on the CU, c its share of the CU,
// g a tile's prologue and epilogue; fitted to MI355X times at 51 shapes (M 33 ..
// 4096, N 4096 .. 151936, K 1024 .. 2560), over which the choice is on average
// 3 % slower than the fastest tile. (The coefficients are the fit's, not a
// tile's latencies one by one.)
struct Bf16Tile {
    int bm, bn;
    double g, c1, c;
    const char* name;
};
enum { kT160x320, kT160x256, kT128x256, kT256x256, kT288x192, kT128x128, kT64x64, kReg };
constexpr Bf16Tile kBf16Tiles[] = {
    {160, 320, 4.08, 0.109, 1.341, "bf16_gemm_160x320"},
    {160, 256, 3.53, 1.003, 1.159, "bf16_gemm_160x256"},
    {128, 256, 3.46, 0.299, 1.047, "bf16_gemm_128x256"},
    {256, 256, 4.00, 1.005, 1.334, "bf16_gemm_256x256"},
    {288, 192, 4.00, 1.004, 1.156, "bf16_gemm_288x192"},
    {128, 128, 1.92, 0.500, 0.699, "bf16_gemm_128x128"},
    {64, 64, 0.34, 0.410, 0.300, "bf16_gemm_64x64"},
};

}  // namespace

// The 128- to 288-row tiles of gemm_big.h from M = 65 on (up to 64 rows they
// would be at most half full); outputs narrower than 4096 columns, where the
// fit has no shapes, keep the 128 x 128 tile.
// A CU holds two 128 x 128 workgroups of the register-staged kernel, but one
// of the ring's 128 x 128 or two of its 64 x 64. Where the model takes a ring
// tile and there are more than 256 tiles of 128 x 128, the register-staged
// kernel can therefore be the faster one. Its side of the line: short rows
// (K <= 384, where one workgroup's stores hide the other's prologue), and up to
// 64 rows one round that is more than 75 % full, or several more than 65 % full
// against the 128 x 128 tile up to K = 1024. MI355X, register-staged against the
// ring tile: 2528 x 1552 x 128 7.0 and 10.0 us, 65 x 87392 x 256 17.8 and 22.3, 56
// x 59312 x 128 8.8 and 11.9, 62 x 52624 x 2560 62.1 and 67.8, 43 x 96416 x 256
// 17.5 and 20.5. The other side: 157 x 18864 x 256 10.3 and 8.3, one round 67 %
// full 41 x 43808 x 1408 33.8 and 30.4, several 42 x 141632 x 384 33.5 and 30.0 (64
// x 64), 64 x 151936 x 2560 189 and 176. Over 838 drawn shapes (M 33 .. 4096, N 16
// .. 152000, K 128 .. 8192) the choice takes 0.77 of the register-staged kernel's
// time; 19 of them take more than 1.03 (1.12 at worst). (Of 650 shapes drawn
// afterwards two do, 1.05 at worst.)
int bf16_gemm_tile(int M, int N, int K, bool c_f32)
{
    const double floor_us =
        3.0 + (2.0 * N * K + (double)M * N * (c_f32 ? 4 : 2)) / 5.0e6;
    int best = kT128x128;
    double best_t = -1.0, best_own = 0.0;
    for (int i = 0; i <= kT64x64; ++i) {
        const Bf16Tile& t = kBf16Tiles[i];
        if (N < 4096 && i != kT128x128) continue;
        if (M <= 64 && i < kT128x128) continue;
        const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
        const double n = (double)((tiles + kPlanCUs - 1) / kPlanCUs), kc = K / 64;
        const double own = 2.0 + n * t.g + kc * std::max(t.c1, n * t.c);
        const double us = std::max(floor_us, own);
        if (best_t < 0.0 || us < best_t ||
            (us == best_t && i <= kT128x256 && own < best_own)) {
            best_own = own;
            best_t = us;
            best = i;
        }
    }
    const long regs = (long)((M + 127) / 128) * ((N + 127) / 128);
    if (best >= kT128x128 && regs > kPlanCUs) {
        const long slots = 2 * kPlanCUs, rounds = (regs + slots - 1) / slots;
        const bool wide = best == kT128x128;
        const bool few = rounds == 1 ? 4 * regs > 3 * slots
                                     : 20 * regs > 13 * rounds * slots && wide && K <= 1024;
        if (M > 64 ? K <= 384 && (wide || M <= 128) : few)
            return kReg;
    }
    return best;
}

hipError_t launch_bf16_gemm(void* c, bool c_f32, bool residual, const uint16_t* x,
                            const uint16_t* w, int M, int N, int K, hipStream_t stream,
                            const LaunchTiming& t, const char** name)
{
    const bool small_offsets = (long)M * K < (1L << 30) && (long)N * K < (1L << 30);
    const int i = small_offsets ? bf16_gemm_tile(M, N, K, c_f32) : kReg;
    if (i != kReg) {
        Fp8Operands op{};
        op.x = x;
        op.w = reinterpret_cast<const uint8_t*>(w);
        op.c = c;
        op.c_f32 = c_f32;
        op.residual = residual;
        op.M = M;
        op.N = N;
        op.K = K;
        const Bf16Tile& b = kBf16Tiles[i];
        const dim3 grid(((M + b.bm - 1) / b.bm) * ((N + b.bn - 1) / b.bn));
        *name = b.name;
        switch (i) {
        case kT160x320: return launch(fp8_gemm256_kernel<kBigBf16, 160, 320>, grid, dim3(512), 0, stream, t, op);
        case kT160x256: return launch(fp8_gemm256_kernel<kBigBf16, 160, 256>, grid, dim3(512), 0, stream, t, op);
        case kT128x256: return launch(fp8_gemm256_kernel<kBigBf16, 128, 256>, grid, dim3(512), 0, stream, t, op);
        case kT256x256: return launch(fp8_gemm256_kernel<kBigBf16, 256, 256>, grid, dim3(512), 0, stream, t, op);
        case kT288x192: return launch(fp8_gemm256_kernel<kBigBf16, 288, 192>, grid, dim3(512), 0, stream, t, op);
        case kT128x128: return launch(gemm_ring_kernel<kRingBf16, 128, 128, 2, 4>, grid, dim3(256), 0, stream, t, op);
        default: return launch(gemm_ring_kernel<kRingBf16, 64, 64, 2, 4>, grid, dim3(256), 0, stream, t, op);
        }
    }
    const Bf16GemmArgs a{c, x, w, M, N, K, c_f32, residual};
    const long tiles = (long)((M + kGbM - 1) / kGbM) * ((N + kGbN - 1) / kGbN);
    if (tiles > 0x7fffffffL) return hipErrorInvalidValue;
    *name = "bf16_gemm_128x128_reg";
    return launch(bf16_gemm_kernel, dim3((unsigned)tiles), dim3(256), 0, stream, t, a);
}

}  // namespace heph
