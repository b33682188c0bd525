// gemm_ring.h - GEMM tiles for the sizes between batched decode and long
// prefill: a 256-thread workgroup per BM x BN output tile, operands through
// a D-stage LDS ring filled by DMA (included by gemm.hip and bf16_gemm.hip).
//
// At these sizes (M of 33 to a few hundred) the 512-thread tiles of gemm_big.h
// leave most CUs idle, so tiles are small, and a small tile's chunk is short:
// what bounds it is whatever the wave does one after the other. On MI355X a
// 128 x 64 E4M3 chunk costs ~400 cycles of DMA (24 KB into LDS at ~60 B a
// cycle and CU, the L2's rate), 256 of MFMA and ~200 of LDS reads; with the
// chunk's fragments read after its barrier the four waves, in step, paid the
// sum (950 cycles). Hence:
//   * a chunk's fragments are read into registers while the chunk before it is
//     contracted (two sets), and the ring's refill goes out between the row
//     tiles' MFMAs: 456 cycles a chunk;
//   * the steady loop has no branch. The compiler waits for every LDS read in
//     flight (lgkmcnt(0)) at a join of control flow, which serialized the
//     same steps again (tiles inside M, ragged tiles and waves without rows
//     are separate copies of the loop);
//   * no scalar load is in flight beside LDS reads, for the same reason;
//   * the stages are a few more than the DMA's latency needs: two workgroups
//     of 64 KB, or one of up to 150 KB, share a CU.
// M = 333, 4096 x 2560 per-channel: 12.8 -> 9.8 us; M = 48, 2560 x 9728 block
// scales: 18.6 -> 13.9 with its reduction (kernel times, graph-replayed over
// HBM-streamed weights; before: gemm_big.h's 64 x 192 and 64 x 256 x 8 splits).
#pragma once

#include <algorithm>
#include <type_traits>

#include "gemm_dma.h"

namespace heph {

namespace {

// What the tile contracts, as BigType in gemm_big.h.
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
};

template <int SM, int BM, int BN, int WGM, int D>
__global__ __launch_bounds__(256, 2) void gemm_ring_kernel(
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
    // DMA instruction `part` of stage st: A's blocks, the row scales, B's blocks
    auto issue_part = [&](auto fullc, int j, int st, int part) {
        uint8_t* base = smem + st * T::STAGE;
        if (part < T::NA) {
            if (decltype(fullc)::value || m0 + (part * 4 + wave) * 8 < M)
                dma16(rq, aoff[part], (uint32_t)j * kChunk, base + (part * 4 + wave) * 1024);
        } else if (T::SCALES && part == T::NA) {
            dma4(rs, soff, (uint32_t)j * s_step, base + T::A + T::B + sp * 256);
        } else {
            const int q = part - (T::P - T::NB);
            dma16(rw, boff[q], (uint32_t)j * kChunk, base + T::A + (q * 4 + wave) * 1024);
        }
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

    // The fragments of a chunk in registers: read while the MFMAs of the
    // chunk before it run.
    struct Frags {
        i32x8 a[MT], b[NT];
        float sa[MT];
    };
    auto read_a = [&](Frags& f, int st, int mi) {
        const uint8_t* p = smem + st * T::STAGE + a_row + mi * 16 * kChunk;
        f.a[mi] = join(*reinterpret_cast<const i32x4*>(p + sl0),
                       *reinterpret_cast<const i32x4*>(p + sl1));
        if constexpr (T::SCALES)
            f.sa[mi] = *reinterpret_cast<const float*>(smem + st * T::STAGE + s_row + mi * 64);
    };
    auto read_b = [&](Frags& f, int st, int ni) {
        const uint8_t* p = smem + st * T::STAGE + b_row + ni * 16 * kChunk;
        f.b[ni] = join(*reinterpret_cast<const i32x4*>(p + sl0),
                       *reinterpret_cast<const i32x4*>(p + sl1));
    };
    // All of K for one tile. FULL: every row block of A is inside M; else the
    // blocks past it are left out, and a stage's wait counts the others only
    // (the newest). LIVE: this wave has rows to contract. Both are fixed before
    // the loop, whose steady part (the ring not yet draining) then has no
    // branch: across one, the compiler waits for every LDS read in flight.
    auto contract_tile = [&](auto fullc, auto livec) {
        constexpr bool FULL = decltype(fullc)::value, LIVE = decltype(livec)::value;
        constexpr int PW = FULL ? T::P : T::NB + (T::SCALES ? 1 : 0);
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (jb + d < je)
#pragma unroll
                for (int part = 0; part < T::P; ++part) issue_part(fullc, jb + d, d, part);
        float sw_cur = SM == kRingBlock ? swb[jb] : 1.0f;
        Frags f0, f1;
        wait_ring<PW, D - 1>(min(D - 1, je - 1 - jb));
        stage_barrier();
        if constexpr (LIVE) {
#pragma unroll
            for (int ni = 0; ni < NT; ++ni) read_b(f0, 0, ni);
#pragma unroll
            for (int mi = 0; mi < MT; ++mi) read_a(f0, 0, mi);
        }
        // One chunk: wait until the next one is in and every wave has its
        // fragments of this one (the barrier); then, between the row tiles'
        // MFMAs, read the next chunk's fragments and refill this one's stage.
        int st = 0;
        auto step = [&](auto steadyc, Frags& cur, Frags& nxt, int j) {
            constexpr bool STEADY = decltype(steadyc)::value;
            const int sn = st + 1 == D ? 0 : st + 1;
            const bool more = STEADY || j + 1 < je;
            if (more) {
                if constexpr (STEADY) wait_vm<(D - 2) * PW>();
                else wait_ring<PW, D - 2>(je - 2 - j);
                stage_barrier();
            }
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
                if constexpr (LIVE) {
                    if (more) {
#pragma unroll
                        for (int ni = mi * NT / MT; ni < (mi + 1) * NT / MT; ++ni) read_b(nxt, sn, ni);
                        read_a(nxt, sn, mi);
                    }
                    if constexpr (SM == kRingBf16) {
#pragma unroll
                        for (int ni = 0; ni < NT; ++ni)
                            acc[mi][ni] = mfma_bf16x64(cur.b[ni], cur.a[mi], acc[mi][ni]);
                    } else if constexpr (SM == kRingConst) {
#pragma unroll
                        for (int ni = 0; ni < NT; ++ni)
                            acc[mi][ni] = mfma_e4m3(cur.b[ni], cur.a[mi], acc[mi][ni]);
                    } else {
                        sc[mi & 1] = cur.sa[mi] * sw_cur;
#pragma unroll
                        for (int ni = 0; ni < NT; ++ni)
                            p[mi & 1][ni] = mfma_e4m3(cur.b[ni], cur.a[mi], f32x4{0, 0, 0, 0});
                        if (mi > 0) rescale(mi - 1);
                    }
                }
                if constexpr (STEADY) {
#pragma unroll
                    for (int part = mi * T::P / MT; part < (mi + 1) * T::P / MT; ++part)
                        issue_part(fullc, j + D, st, part);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (LIVE && T::SCALES) rescale(MT - 1);
            // after the last LDS read: with a scalar load in flight every wait
            // for LDS would wait for all of it
            if constexpr (SM == kRingBlock)
                if (more) sw_cur = swb[j + 1];
            st = sn;
        };
        int j = jb;
        for (; j + 1 + D < je; j += 2) {
            step(std::true_type{}, f0, f1, j);
            step(std::true_type{}, f1, f0, j + 1);
        }
        for (; j + 1 < je; j += 2) {
            if (j + D < je) step(std::true_type{}, f0, f1, j);
            else step(std::false_type{}, f0, f1, j);
            step(std::false_type{}, f1, f0, j + 1);
        }
        if (j < je) step(std::false_type{}, f0, f1, j);
    };
    if (m0 + BM <= M) contract_tile(std::true_type{}, std::true_type{});
    else if (m0 + wm * T::WM < M) contract_tile(std::false_type{}, std::true_type{});
    else contract_tile(std::false_type{}, std::false_type{});

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
            if (S > 1) {    // the fp32 partial, unscaled for kRingConst
                *reinterpret_cast<f32x4*>(op.part + (size_t)split * M * N + o) = v;
                continue;
            }
            if constexpr (SM == kRingConst) {
                // the reference's association (wmma_gfx12.mojo:711-712, :848)
                const f32x4 sw = ldf4(op.sw + col);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = M == 1 ? v[e] * (sa * sw[e]) : (v[e] * sa) * sw[e];
            }
            store4(op, o, v);
        }
    }
}

}  // namespace heph
