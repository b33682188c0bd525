// gemm_ring.h - GEMM tiles for the sizes between batched decode and long
// prefill: a 256-thread workgroup per BM x BN output tile, operands through
// a D-stage LDS ring filled by DMA (included by gemm_ring.hip).
#pragma once

#include <algorithm>

#include "gemm_dma.h"

namespace heph {

namespace {

enum RingType { kRingBlock = 0, kRingChannel = 1, kRingConst = 2, kRingBf16 = 3 };

// s_waitcnt: at most N vector memory instructions and no LDS or scalar one
// left in flight (vmcnt in bits 3:0 and 15:14).
template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
    asm volatile("" ::: "memory");
}

// The wait for a stage with `left` later stages of P instructions in flight.
template <int P, int MAX>
__device__ __forceinline__ void wait_ring(int left)
{
    if constexpr (MAX == 0) {
        wait_vm<0>();
    } else {
        if (left >= MAX) wait_vm<MAX * P>();
        else wait_ring<P, MAX - 1>(left);
    }
}

}  // namespace

template <int SM, int BM, int BN, int WGM, int D>
struct RingTile {
    static constexpr int WGN = 4 / WGM;
    static constexpr int WM = BM / WGM, WN = BN / WGN, MT = WM / 16, NT = WN / 16;
    static constexpr bool SCALES = SM == kRingBlock || SM == kRingChannel;
    static constexpr int SROWS = (BM + 63) / 64;            // waves that hold distinct row scales
    static constexpr int A = BM * 128, B = BN * 128, S = SCALES ? SROWS * 256 : 0;
    static constexpr int STAGE = A + B + S, BYTES = D * STAGE;
    static constexpr int NA = BM / 32, NB = BN / 32;        // 1 KB DMA instructions per wave
    static constexpr int P = NA + NB + (SCALES ? 1 : 0);
    static_assert(BM % (16 * WGM) == 0 && BN % (16 * WGN) == 0 && BM % 32 == 0 && BN % 32 == 0,
                  "whole MFMA blocks per wave, whole DMA instructions per wave");
    static_assert(128 % WN == 0 || SM >= 2, "a wave's columns lie in one weight block");
    static_assert(!SCALES || SROWS <= 4, "a wave moves the scales of 64 rows");
    static_assert(D >= 2 && BYTES <= 160 * 1024, "LDS");
    static constexpr int WGS = BYTES * 2 <= 160 * 1024 ? 2 : 1;    // workgroups per CU
};

template <int SM, int BM, int BN, int WGM, int D>
__global__ __launch_bounds__(256, (RingTile<SM, BM, BN, WGM, D>::WGS)) void gemm_ring_kernel(
    Fp8Operands op)
{
    using T = RingTile<SM, BM, BN, WGM, D>;
    constexpr int MT = T::MT, NT = T::NT;
    __shared__ __attribute__((aligned(16))) uint8_t smem[T::BYTES];    // the only LDS variable

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, slice = lane >> 4;
    const int wm = wave / T::WGN, wn = wave % T::WGN;
    const int M = op.M, N = op.N;
    const uint32_t pitch = SM == kRingBf16 ? 2u * op.K : op.K;          // bytes per row
    const int KC = (int)(pitch >> 7);
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    const int S = op.splits, tiles = tiles_m * tiles_n;
    const int split = blockIdx.x / tiles;
    const int jb = split * KC / S, je = (split + 1) * KC / S;
    int tm, tn;
    tile_of_block(blockIdx.x - split * tiles, tiles_m, tiles_n, &tm, &tn);
    const int m0 = tm * BM, n0 = tn * BN;

    // DMA: wave w moves the 8-row blocks w, w + 4, .. of A and B, one
    // instruction a block; rows past M (N) are clamped, blocks of A wholly
    // past M left out (they feed rows that are never stored).
    const rsrc_t rq = make_rsrc(SM == kRingBf16 ? (const void*)op.x : (const void*)op.q);
    const rsrc_t rw = make_rsrc(op.w), rs = make_rsrc(op.s);
    const int lr = lane >> 3;
    const uint32_t piece = ((lane & 7) ^ lr) * 16;
    uint32_t aoff[T::NA], boff[T::NB];
#pragma unroll
    for (int q = 0; q < T::NA; ++q)
        aoff[q] = (uint32_t)min(m0 + (q * 4 + wave) * 8 + lr, M - 1) * pitch + piece;
#pragma unroll
    for (int q = 0; q < T::NB; ++q)
        boff[q] = (uint32_t)min(n0 + (q * 4 + wave) * 8 + lr, N - 1) * pitch + piece;
    // every wave moves a piece of 64 row scales (the same ones more than
    // once where BM < 256), so that all have P instructions per stage
    const int sp = wave % T::SROWS;
    const uint32_t soff = (uint32_t)min(m0 + sp * 64 + lane, M - 1) * (uint32_t)op.s_ld * 4u;
    const uint32_t s_step = (uint32_t)op.s_step * 4u;
    const bool full = m0 + BM <= M;              // no block of A left out
    const bool live = m0 + wm * T::WM < M;       // this wave has rows to contract
    auto issue = [&](int j, int st) {
        uint8_t* base = smem + st * T::STAGE;
#pragma unroll
        for (int q = 0; q < T::NA; ++q)
            if (full || m0 + (q * 4 + wave) * 8 < M)
                dma16(rq, aoff[q], (uint32_t)j * kChunk, base + (q * 4 + wave) * 1024);
        if constexpr (T::SCALES)
            dma4(rs, soff, (uint32_t)j * s_step, base + T::A + T::B + sp * 256);
#pragma unroll
        for (int q = 0; q < T::NB; ++q)
            dma16(rw, boff[q], (uint32_t)j * kChunk, base + T::A + (q * 4 + wave) * 1024);
    };

    float swc[NT][4];
#pragma unroll
    for (int ni = 0; ni < NT; ++ni)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = min(n0 + wn * T::WN + ni * 16 + slice * 4 + e, N - 1);
            swc[ni][e] = SM == kRingChannel ? op.sw[n] : 0.0f;
        }
    const const_f32_ptr swb =
        (const_f32_ptr)(op.sw + (SM == kRingBlock
                                     ? (size_t)min((n0 + wn * T::WN) >> 7, (N - 1) >> 7) * op.sw_ld
                                     : 0));

    const int sl0 = (slice ^ (r16 & 7)) * 16, sl1 = sl0 ^ 64;
    const int a_row = (wm * T::WM + r16) * kChunk;
    const int b_row = T::A + (wn * T::WN + r16) * kChunk;
    const int s_row = T::A + T::B + (wm * T::WM + r16) * 4;

    f32x4 acc[MT][NT];
#pragma unroll
    for (int mi = 0; mi < MT; ++mi)
#pragma unroll
        for (int ni = 0; ni < NT; ++ni) acc[mi][ni] = f32x4{0, 0, 0, 0};

#pragma unroll
    for (int d = 0; d < D - 1; ++d)
        if (jb + d < je) issue(jb + d, d);
    float sw_cur = SM == kRingBlock ? swb[jb] : 1.0f, sw_nxt = 1.0f;

    int st = 0;
    for (int j = jb; j < je; ++j) {
        // a tile with blocks left out counts the others only (the newest)
        if (full) wait_ring<T::P, D - 2>(je - 1 - j);
        else wait_ring<T::NB + (T::SCALES ? 1 : 0), D - 2>(je - 1 - j);
        stage_barrier();
        const uint8_t* stp = smem + st * T::STAGE;
        auto frag = [&](int off) {
            return join(*reinterpret_cast<const i32x4*>(stp + off + sl0),
                        *reinterpret_cast<const i32x4*>(stp + off + sl1));
        };
        i32x8 b[NT], a[2];
        float sa[2] = {0.0f, 0.0f};
        if (live) {
#pragma unroll
            for (int ni = 0; ni < NT; ++ni) b[ni] = frag(b_row + ni * 16 * kChunk);
            a[0] = frag(a_row);
            if constexpr (T::SCALES) sa[0] = *reinterpret_cast<const float*>(stp + s_row);
        }
        if (j + D - 1 < je) issue(j + D - 1, st == 0 ? D - 1 : st - 1);
        if constexpr (SM == kRingBlock)
            if (j + 1 < je) sw_nxt = swb[j + 1];
        if (live) {
            f32x4 p[2][NT];
            float sc[2] = {0.0f, 0.0f};
            auto rescale = [&](int mi) {
#pragma unroll
                for (int ni = 0; ni < NT; ++ni)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        acc[mi][ni][e] += p[mi & 1][ni][e] *
                                          (SM == kRingBlock ? sc[mi & 1] : sc[mi & 1] * swc[ni][e]);
            };
#pragma unroll
            for (int mi = 0; mi < MT; ++mi) {
                const int cur = mi & 1;
                if (mi + 1 < MT) {
                    a[cur ^ 1] = frag(a_row + (mi + 1) * 16 * kChunk);
                    if constexpr (T::SCALES)
                        sa[cur ^ 1] = *reinterpret_cast<const float*>(stp + s_row + (mi + 1) * 64);
                }
                if constexpr (SM == kRingBf16) {
#pragma unroll
                    for (int ni = 0; ni < NT; ++ni) acc[mi][ni] = mfma_bf16x64(b[ni], a[cur], acc[mi][ni]);
                } else if constexpr (SM == kRingConst) {
#pragma unroll
                    for (int ni = 0; ni < NT; ++ni) acc[mi][ni] = mfma_e4m3(b[ni], a[cur], acc[mi][ni]);
                } else {
                    sc[cur] = sa[cur] * sw_cur;
#pragma unroll
                    for (int ni = 0; ni < NT; ++ni)
                        p[cur][ni] = mfma_e4m3(b[ni], a[cur], f32x4{0, 0, 0, 0});
                    if (mi > 0) rescale(mi - 1);
                }
            }
            if constexpr (T::SCALES) rescale(MT - 1);
        }
        sw_cur = sw_nxt;
        st = st + 1 == D ? 0 : st + 1;
    }

    // lane: row r16 and columns 4 slice .. +3 of each 16x16 block
#pragma unroll
    for (int mi = 0; mi < MT; ++mi) {
        const int row = m0 + wm * T::WM + mi * 16 + r16;
        if (row >= M) continue;
        const float sa = SM == kRingConst ? op.s[row] : 1.0f;
#pragma unroll
        for (int ni = 0; ni < NT; ++ni) {
            const int col = n0 + wn * T::WN + ni * 16 + slice * 4;
            if (col >= N) continue;
            f32x4 v = acc[mi][ni];
            const size_t o = (size_t)row * N + col;
            if (SM != kRingConst && S > 1) {
                *reinterpret_cast<f32x4*>(op.part + (size_t)split * M * N + o) = v;
                continue;
            }
            if constexpr (SM == kRingConst) {
                // the reference's association (wmma_gfx12.mojo:711-712, :848)
                const f32x4 sw = *reinterpret_cast<const f32x4*>(op.sw + col);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = M == 1 ? v[e] * (sa * sw[e]) : (v[e] * sa) * sw[e];
            }
            store4(op, o, v);
        }
    }
}

}  // namespace heph
