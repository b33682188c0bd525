// gemm_big.h - the large-M GEMM tile, E4M3 and bf16 (included by gemm.hip and
// bf16_gemm.hip).
#pragma once

#include <type_traits>

#include "gemm_dma.h"

namespace heph {

// ---------------------------------------------------------------------------
// Large-M kernel: BMxBN tile per 512-thread workgroup (8 waves of
// (BM/2)x(BN/4), (BM/32)x(BN/64) MFMA 16x16x128 each). The weight fragment is the
// MFMA's first operand, so lane l holds row l&15 of each 16x16 output block
// at columns 4*(l>>4) .. +3: one activation-scale product per row tile and
// chunk, and four consecutive outputs to pack. Operand tiles reach LDS by
// direct DMA (buffer_load_dwordx4 ... lds, 1 KB = 8 rows per instruction,
// no VGPR staging); a 16-byte piece p of row r lands in slot p ^ (r & 7),
// which spreads the fragment reads over the banks. Stages of A BM*128 B,
// B BN*128 B and row scales BM*4 B (two, or three where LDS allows: see
// BigTile); one barrier per 128-wide chunk:
//   wait own DMA of chunk j -> barrier (chunk j visible everywhere, and
//   every wave is done with the stage read in chunk j-1) -> DMA chunk j+1
//   (j+2 with three stages) into that stage -> contract chunk j.
// The chunk loop is unrolled by the stage count so that each stage's LDS
// addresses are fixed registers plus instruction offsets (the B stage of
// the tiles with three B against two A stages is a run-time base), and
// the DMA advances through K
// with a scalar offset only: apart from the rescale (one FMA per
// accumulator and chunk, one multiply per row tile, or per row tile and
// 16-column block where a wave's columns span two weight blocks) the loop holds almost
// no VALU work, because a wave's VALU instructions do not overlap its own
// MFMAs. The block scales come through the scalar cache.
// The compiler does not model the DMA's LDS writes, so the waits are
// explicit s_waitcnt vmcnt(n) plus compiler memory barriers.
// Epilogue, bf16 output: the tile is rounded (v_cvt_pk_bf16_f32), written to
// LDS once as bf16 (8 bytes per lane and block) and stored as coalesced
// 16-byte row pieces. f32 output or a residual: staged in f32, BM/2 rows at
// a time, the residual added before the one rounding.
namespace {

// What the tile contracts: E4M3 with block scales, with per-channel weight
// and per-chunk activation scales, with per-channel / per-token scales
// (nothing varies along K), or unscaled bf16 (a chunk is then 64 elements).
enum BigType { kBigBlock = 0, kBigChannel = 1, kBigConst = 2, kBigBf16 = 3 };

// Tile BM x BN, BM a multiple of 32 up to 288, BN in {192, 256, 320}: the 8
// waves form a 2 x 4 grid of (BM/2) x (BN/4) wave tiles. A smaller tile
// trades MFMA work per chunk for a tile count that fills the CUs (e.g. 256
// tiles of 128 x 320 instead of 160 of 256 x 256 at M = 4096, N = 2560).
template <int BM, int BN, bool SCALES = true>
struct BigTile {
    static_assert(BM % 32 == 0 && BM >= 64 && BM <= 288, "tile height");
    static_assert(BN == 192 || BN == 256 || BN == 320, "tile width");
    // 8 waves in a 2 x 4 grid of WM x WN wave tiles, MT x NT MFMA blocks
    static constexpr int WM = BM / 2, MT = WM / 16, WN = BN / 4, NT = WN / 16;
    // DMA instructions (8 rows each) per wave: NAP of A in as many waves as
    // the tile has rows for (the rescaled types: 32 rows a wave; A spread
    // evenly over all waves ran 1-2 % slower there), NBP of B
    static constexpr int NAP = SCALES ? 4 : (BM / 8 + 7) / 8, NBP = BN / 64;
    // the WN columns of every wave lie in one 128-column weight block
    static constexpr bool ONE_BLOCK = 128 % WN == 0 && BN % WN == 0;
    static constexpr int STAGE_A = BM * kChunk, STAGE_B = BN * kChunk, STAGE_S = SCALES ? BM * 4 : 0;
    static constexpr int STAGE = STAGE_A + STAGE_B + STAGE_S;
    // LDS stages. A short chunk is below the loaded HBM latency, so where
    // LDS allows, the DMA runs two chunks ahead: three whole stages (64 and
    // 128 rows by 256 columns, 64 x 192); else two A/scale stages and three B stages
    // (the weights, streamed from HBM in a real prefill, get the extra
    // chunk: 192 x 256, 256 x 192, 128 x 320); else two (256 x 256).
    static constexpr int kLds = 160 * 1024;
    static constexpr bool FULL3 = 3 * STAGE <= kLds;
    static constexpr bool SPLIT_B = !FULL3 && 2 * (STAGE_A + STAGE_S) + 3 * STAGE_B <= kLds;
    static constexpr int NS = FULL3 ? 3 : 2;                  // A and row-scale stages
    static constexpr int NB = FULL3 || SPLIT_B ? 3 : 2;       // B stages
    static constexpr int BYTES =
        SPLIT_B ? 2 * STAGE_A + 2 * STAGE_S + 3 * STAGE_B : NS * STAGE;
    // Byte offsets of A, B and row-scale stage k.
    static constexpr int a_at(int k) { return SPLIT_B ? k * STAGE_A : k * STAGE; }
    static constexpr int s_at(int k)
    {
        return SPLIT_B ? 2 * STAGE_A + k * STAGE_S : k * STAGE + STAGE_A + STAGE_B;
    }
    static constexpr int b_at(int k)
    {
        return SPLIT_B ? 2 * STAGE_A + 2 * STAGE_S + k * STAGE_B : k * STAGE + STAGE_A;
    }
};

template <int V>
using ic = std::integral_constant<int, V>;

// The chunk-start wait of the large-M kernel: the wave's LDS reads and
// scalar loads done (lgkmcnt(0)) and all its vector memory instructions
// but the newest n (vmcnt(n): with three stages the DMA of the next chunk,
// 3 to 10 instructions of this wave, may stay in flight; any other n waits
// for all).
__device__ __forceinline__ void wait_stage(int n)
{
    switch (n) {
    case 10: __builtin_amdgcn_s_waitcnt(0x007A); break;
    case 9: __builtin_amdgcn_s_waitcnt(0x0079); break;
    case 8: __builtin_amdgcn_s_waitcnt(0x0078); break;
    case 7: __builtin_amdgcn_s_waitcnt(0x0077); break;
    case 6: __builtin_amdgcn_s_waitcnt(0x0076); break;
    case 5: __builtin_amdgcn_s_waitcnt(0x0075); break;
    case 4: __builtin_amdgcn_s_waitcnt(0x0074); break;
    case 3: __builtin_amdgcn_s_waitcnt(0x0073); break;
    default: __builtin_amdgcn_s_waitcnt(0x0070); break;
    }
    asm volatile("" ::: "memory");
}
// Keeps v where the program computes it: the scheduler may not sink the
// rescale FMAs below the next row tile's MFMAs (their partials would then
// all be live at once).
__device__ __forceinline__ void pin(f32x4& v) { asm volatile("" : "+v"(v)); }
}  // namespace

// Epilogue of the large-M kernels: lane l holds C[row r16][cols 4*slice ..
// +3] of each 16x16 block of its (BM/2) x (BN/4) wave tile, already scaled.
// K splits store the fp32 partial tile; bf16 output goes through LDS once
// as bf16 for coalesced 16-byte stores; f32 output or a residual in two
// f32 passes (the residual added before the one rounding); the bf16 contraction
// straight from registers. Every thread of the workgroup calls it; LDS_BYTES of
// smem are free to reuse.
template <int SM, int BM, int BN, int LDS_BYTES>
__device__ __forceinline__ void big_epilogue(const Fp8Operands& op,
                                             f32x4 (&acc)[BM / 32][BN / 64], uint8_t* smem,
                                             int m0, int n0, int split, int S)
{
    constexpr int L_BM = BM, L_WM = BM / 2, L_MT = BM / 32;
    constexpr int L_BN = BN, L_WN = BN / 4, L_NT = BN / 64;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, slice = lane >> 4;
    const int wm = wave >> 2, wn = wave & 3;
    const int M = op.M, N = op.N;
    // Lane l holds C[row r16][cols 4*slice .. +3] of each 16x16 block.
    const int r_lane = wm * L_WM + r16;                  // tile row of (mi = 0)
    const int c_lane = wn * L_WN + slice * 4;            // tile col of (ni = 0)
    if constexpr (SM != kBigConst) {
        if (S > 1) {
            // split over K: the fp32 partial tile goes to the scratch
            // [split][M][N]; splitk_reduce_kernel finishes the output.
            float* pp = op.part + (size_t)split * M * N;
#pragma unroll
            for (int mi = 0; mi < L_MT; ++mi) {
                const int row = m0 + r_lane + mi * 16;
                if (row >= M) continue;
#pragma unroll
                for (int ni = 0; ni < L_NT; ++ni) {
                    const int col = n0 + c_lane + ni * 16;
                    if (col < N) *reinterpret_cast<f32x4*>(pp + (size_t)row * N + col) = acc[mi][ni];
                }
            }
            return;
        }
    }
    if constexpr (SM == kBigBf16) {
        // straight from registers, four consecutive outputs a lane
#pragma unroll
        for (int mi = 0; mi < L_MT; ++mi) {
            const int row = m0 + r_lane + mi * 16;
            if (row >= M) continue;
#pragma unroll
            for (int ni = 0; ni < L_NT; ++ni) {
                const int col = n0 + c_lane + ni * 16;
                if (col < N) store4(op, (size_t)row * N + col, acc[mi][ni]);
            }
        }
        return;
    } else if (!op.residual && !op.c_f32) {
        // bf16 output: the whole tile goes through LDS once as bf16, rows
        // padded by 8 bytes (2 BN + 8: 130 dwords at 256 columns, consecutive
        // rows 2 banks apart), each lane writing 8 bytes per block; then
        // 16-byte coalesced stores.
        constexpr int RB = 2 * L_BN + 8;
        static_assert(L_BM * RB <= LDS_BYTES, "bf16 tile must fit the stage buffers");
        __syncthreads();
#pragma unroll
        for (int mi = 0; mi < L_MT; ++mi) {
            float sa = 1.0f;
            if constexpr (SM == 2) sa = op.s[min(m0 + r_lane + mi * 16, M - 1)];
#pragma unroll
            for (int ni = 0; ni < L_NT; ++ni) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = acc[mi][ni][e];
                    if constexpr (SM == 2)
                    {
                        // reference association: acc*(sa*sw) at M = 1
                        // (wmma_gfx12.mojo:711-712), (acc*sa)*sw otherwise (:848)
                        const float sw = op.sw[min(n0 + c_lane + ni * 16 + e, N - 1)];
                        v[e] = M == 1 ? v[e] * (sa * sw) : (v[e] * sa) * sw;
                    }
                }
                const uint2 pk = make_uint2(pack_bf16_hw(v[0], v[1]), pack_bf16_hw(v[2], v[3]));
                *reinterpret_cast<uint2*>(smem + (r_lane + mi * 16) * RB +
                                          (c_lane + ni * 16) * 2) = pk;
            }
        }
        __syncthreads();
        for (int e = tid; e < L_BM * (L_BN / 8); e += 512) {
            const int r = e / (L_BN / 8);
            const int c8 = (e % (L_BN / 8)) * 8;
            const int grow = m0 + r, gcol = n0 + c8;
            if (grow >= M || gcol >= N) continue;
            *reinterpret_cast<uint4*>(static_cast<uint16_t*>(op.c) + (size_t)grow * N + gcol) =
                *reinterpret_cast<const uint4*>(smem + r * RB + c8 * 2);
        }
        return;
    }
    if constexpr (SM != kBigBf16) {
    // f32 output or residual: two passes of L_WM rows through LDS in f32
    // (the residual is added before the one rounding).
    constexpr int CST = L_BN + 4;
    static_assert(L_WM * CST * 4 <= LDS_BYTES, "epilogue tile must fit the stage buffers");
    float* Cs = reinterpret_cast<float*>(smem);
    float* cw = Cs + r16 * CST + c_lane;
    for (int pass = 0; pass < 2; ++pass) {
        __syncthreads();
        if (wm == pass) {
#pragma unroll
            for (int mi = 0; mi < L_MT; ++mi)
#pragma unroll
                for (int ni = 0; ni < L_NT; ++ni)
                    *reinterpret_cast<f32x4*>(cw + mi * 16 * CST + ni * 16) = acc[mi][ni];
        }
        __syncthreads();
        // L_WM rows x L_BN cols: each thread writes 8 consecutive outputs
        for (int e = tid; e < L_WM * (L_BN / 8); e += 512) {
            const int r = e / (L_BN / 8);
            const int c8 = (e % (L_BN / 8)) * 8;
            const int grow = m0 + pass * L_WM + r;
            const int gcol = n0 + c8;
            if (grow >= M || gcol >= N) continue;
            const f32x4 lo = *reinterpret_cast<const f32x4*>(&Cs[r * CST + c8]);
            const f32x4 hi = *reinterpret_cast<const f32x4*>(&Cs[r * CST + c8 + 4]);
            float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            if constexpr (SM == 2) {
                // reference association: acc*(sa*sw) at M = 1, else (acc*sa)*sw
                const float sa = op.s[grow];
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    v[t] = M == 1 ? v[t] * (sa * op.sw[gcol + t]) : (v[t] * sa) * op.sw[gcol + t];
            }
            const size_t o = (size_t)grow * N + gcol;
            if (op.c_f32) {
                float* c = static_cast<float*>(op.c) + o;
                if (op.residual) {
                    const float4 r0 = *reinterpret_cast<const float4*>(c);
                    const float4 r1 = *reinterpret_cast<const float4*>(c + 4);
                    v[0] += r0.x; v[1] += r0.y; v[2] += r0.z; v[3] += r0.w;
                    v[4] += r1.x; v[5] += r1.y; v[6] += r1.z; v[7] += r1.w;
                }
                *reinterpret_cast<float4*>(c) = make_float4(v[0], v[1], v[2], v[3]);
                *reinterpret_cast<float4*>(c + 4) = make_float4(v[4], v[5], v[6], v[7]);
            } else {
                uint16_t* c = static_cast<uint16_t*>(op.c) + o;
                const uint4 rr = *reinterpret_cast<const uint4*>(c);
                v[0] += bf16lo(rr.x); v[1] += bf16hi(rr.x);
                v[2] += bf16lo(rr.y); v[3] += bf16hi(rr.y);
                v[4] += bf16lo(rr.z); v[5] += bf16hi(rr.z);
                v[6] += bf16lo(rr.w); v[7] += bf16hi(rr.w);
                uint4 out;
                out.x = f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
                out.y = f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
                out.z = f32_to_bf16(v[4]) | ((uint32_t)f32_to_bf16(v[5]) << 16);
                out.w = f32_to_bf16(v[6]) | ((uint32_t)f32_to_bf16(v[7]) << 16);
                *reinterpret_cast<uint4*>(c) = out;
            }
        }
    }
    }
}

template <int SM, int BM, int BN>
__global__ __launch_bounds__(512, 1) void fp8_gemm256_kernel(Fp8Operands op)
{
    using T = BigTile<BM, BN, SM != kBigBf16>;
    constexpr bool RESCALE = SM < kBigConst;    // per-chunk scales
    constexpr int L_BM = BM, L_WM = T::WM, L_MT = T::MT;
    constexpr int L_BN = BN, L_WN = T::WN, L_NT = T::NT, NBP = T::NBP;
    // With three stages, chunk j + 2's DMA goes out in chunk j: a chunk
    // (~0.8 us at 64 rows, ~1.3 us at 192) is below the loaded HBM latency,
    // and weights that are not in the Infinity Cache (each layer of a real
    // prefill) otherwise left every chunk waiting on its DMA (MI355X: M =
    // 512 qkv 16.4 us from the cache, 29.5 us from HBM with two stages).
    constexpr int NS = T::NS, NB = T::NB;
    constexpr bool SPLIT_B = T::SPLIT_B;
    // The kernel's only LDS variable: with a second one the LDS accesses get
    // alias scopes, the compiler then orders every fragment read after all
    // outstanding DMA (vmcnt(0)), and the pipeline serializes (MI355X: +40 %
    // per chunk). Extra LDS state goes into this array.
    __shared__ __attribute__((aligned(16))) uint8_t smem[T::BYTES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, slice = lane >> 4;
    const int wm = wave >> 2, wn = wave & 3;
    const int M = op.M, N = op.N;
    const int K = SM == kBigBf16 ? 2 * op.K : op.K;    // bytes per operand row
    const int KC = K >> 7;
    const int tiles_m = (M + L_BM - 1) / L_BM, tiles_n = (N + L_BN - 1) / L_BN;
    // Split over K: workgroup b takes tile b % tiles and the chunks
    // [split * KC / S, (split + 1) * KC / S) of split b / tiles.
    const int S = op.splits, tiles = tiles_m * tiles_n;
    const int split = blockIdx.x / tiles;
    const int jb = split * KC / S, je = (split + 1) * KC / S;
    int tm, tn;
    tile_of_block(blockIdx.x - split * tiles, tiles_m, tiles_n, &tm, &tn);
    const int m0 = tm * L_BM, n0 = tn * L_BN;

    // DMA sources: wave w moves rows [8 NAP w, 8 NAP (w+1)) of A (one
    // instruction per 8 rows, none past the tile) and rows [8 NBP w, 8 NBP (w+1)) of B (NBP = BN / 64
    // instructions); lane i covers row i >> 3 of a block and global
    // piece (i & 7) ^ (row & 7). Rows past M (N) are clamped to the last
    // row, and loaded: they feed output rows (columns) that are never stored
    // (bf16: nor are the MFMAs of row tiles past M issued). Each lane
    // keeps one 32-bit byte offset per block and operand; chunk j adds the
    // scalar offset 128 * j.
    const rsrc_t rq = make_rsrc(SM == kBigBf16 ? (const void*)op.x : (const void*)op.q);
    const rsrc_t rw = make_rsrc(op.w), rs = make_rsrc(op.s);
    const int lr = lane >> 3;
    const int piece = ((lane & 7) ^ lr) * 16;     // rows 8q + lr share r & 7 = lr
    constexpr int NAP = T::NAP;
    uint32_t aoff[NAP], boff[NBP];
#pragma unroll
    for (int q = 0; q < NAP; ++q)
        aoff[q] = (uint32_t)min(m0 + (wave * NAP + q) * 8 + lr, M - 1) * (uint32_t)K + piece;
#pragma unroll
    for (int q = 0; q < NBP; ++q)
        boff[q] = (uint32_t)min(n0 + wave * 8 * NBP + q * 8 + lr, N - 1) * (uint32_t)K + piece;
    const uint32_t soff = (uint32_t)min(m0 + wave * 64 + lane, M - 1) * (uint32_t)op.s_ld * 4u;
    const uint32_t s_step = (uint32_t)op.s_step * 4u;

    // DMA instruction `part` (0 .. NAP + NBP) of this wave: the first NAP move A
    // rows of chunk ja into A stage abuf, then NBP parts B rows of chunk jw
    // into B stage bbuf and the last the row scales of chunk ja; with
    // separate B stages the row scales come after A's parts and the B rows
    // last, so that the next chunk's wait can leave exactly the NBP B
    // instructions in flight.
    constexpr int kParts = NAP + 1 + NBP;
    constexpr int kFirstB = SPLIT_B ? NAP + 1 : NAP, kScalePart = SPLIT_B ? NAP : NAP + NBP;
    // DMA parts per row tile (MI355X: 2 over the first five of 8 row tiles,
    // 3 over the first three of 6 or 4, fewest cycles per chunk; 5 and 4
    // over the 2 row tiles of BM = 64, so that every part goes out)
    constexpr int kPer = L_MT >= 8 ? 2 : L_MT >= 4 ? 3 : (kParts + L_MT - 1) / L_MT;
    static_assert(kPer * L_MT >= kParts, "every DMA part is issued");
    // A wave's A parts are all inside the tile or all outside it: one test a
    // chunk instead of one a part
    constexpr bool kWholeWaves = L_BM % (8 * NAP) == 0;
    auto issue_part = [&](int ja, int jw, auto abufc, int bbuf, int part) {
        constexpr int abuf = decltype(abufc)::value;
        if (part < NAP) {
            if (kWholeWaves ? wave * NAP * 8 < L_BM : (wave * NAP + part) * 8 < L_BM)
                dma16(rq, aoff[part], (uint32_t)ja * kChunk,
                      smem + T::a_at(abuf) + (wave * NAP + part) * 8 * kChunk);
        } else if (part == kScalePart) {
            if (RESCALE && wave * 64 < L_BM)
                dma4(rs, soff, (uint32_t)ja * s_step, smem + T::s_at(abuf) + wave * 256);
        } else {
            const int q = part - kFirstB;
            dma16(rw, boff[q], (uint32_t)jw * kChunk,
                  smem + T::b_at(bbuf) + (wave * 8 * NBP + q * 8) * kChunk);
        }
    };

    // With the weight fragment as the MFMA's first operand, lane l holds
    // row r16 of each 16x16 block and its columns 4*slice .. 4*slice+3.
    float swc[L_NT][4];
#pragma unroll
    for (int ni = 0; ni < L_NT; ++ni)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = min(n0 + wn * L_WN + ni * 16 + slice * 4 + e, N - 1);
            swc[ni][e] = SM == 1 ? op.sw[n] : 0.0f;
        }
    // A wave whose columns all lie past N still reads a valid scale row
    // (its results are never stored). The rows are uniform per wave: the
    // block scales are scalar loads. Where a wave's columns span two
    // 128-column blocks (WN = 48 or 80), each 16-column block ni has its own.
    constexpr int NSW = T::ONE_BLOCK ? 1 : L_NT;
    const_f32_ptr swb[NSW];
#pragma unroll
    for (int k = 0; k < NSW; ++k)
        swb[k] = (const_f32_ptr)(op.sw + (size_t)min((n0 + wn * L_WN + k * 16) >> 7, (N - 1) >> 7) *
                                             op.sw_ld);

    // Per-lane LDS byte offsets inside a stage: fragment rows of A and B at
    // the two 16-byte slots this lane reads, and the row scale.
    const int sl0 = (slice ^ (r16 & 7)) * 16, sl1 = sl0 ^ 64;
    const int a_row = (wm * L_WM + r16) * kChunk;
    const int b_row = (wn * L_WN + r16) * kChunk;
    const int s_row = (wm * L_WM + r16) * 4;

    const int mt_live = (M - m0 - wm * L_WM + 15) / 16;
    f32x4 acc[L_MT][L_NT];
#pragma unroll
    for (int mi = 0; mi < L_MT; ++mi)
#pragma unroll
        for (int ni = 0; ni < L_NT; ++ni) acc[mi][ni] = f32x4{0, 0, 0, 0};

    float sw_cur[NSW], sw_nxt[NSW];
#pragma unroll
    for (int k = 0; k < NSW; ++k) {
        sw_cur[k] = SM == 0 ? swb[k][jb] : 1.0f;
        sw_nxt[k] = 1.0f;
    }

    // Software pipeline over the row tiles of a wave: the MFMAs of tile mi
    // run while the rescale FMAs of tile mi - 1 execute and the A fragment
    // and row scale of tile mi + 1 are read. The last tile's FMAs are done
    // at the start of the next chunk, so its partials and scale product
    // live across the barrier.
    static_assert(!RESCALE || L_MT % 2 == 0, "rescaled row tiles per wave must be even");
    f32x4 p[2][L_NT];
    float sc[2][NSW] = {};
    auto rescale = [&](int mi, int slot) {
#pragma unroll
        for (int ni = 0; ni < L_NT; ++ni) {
            const float s = sc[slot][NSW == 1 ? 0 : ni];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                acc[mi][ni][e] += p[slot][ni][e] * (SM == 0 ? s : s * swc[ni][e]);
            pin(acc[mi][ni]);
        }
    };

    // DMA instructions a wave issues per chunk (A rows, B rows, row scales).
    const int a_parts = kWholeWaves ? (wave * NAP * 8 < L_BM ? NAP : 0)
                                    : max(0, min(NAP, L_BM / 8 - wave * NAP));
    const int n_parts = a_parts + NBP + (RESCALE && wave * 64 < L_BM ? 1 : 0);

    // One 128-wide chunk j held in A stage buf (a compile-time constant)
    // and B stage bst. The wave's DMA instructions (A rows and scales
    // of chunk j + NS - 1, B rows of chunk j + NB - 1) go out kPer per row
    // tile from the first tile on: issued together right after the barrier,
    // the DMAs of all eight waves stall every wave's instruction issue;
    // spread to the last tile, the late ones are still in flight at the
    // next chunk's wait (MI355X: ~350 of ~3100 cycles a chunk).
    auto chunk = [&](auto bufc, int j, int bst) {
        constexpr int buf = decltype(bufc)::value;
        // with three stages the newest instructions, the next chunk's DMA
        // (n_parts, or its NBP B parts where only B has three stages), may
        // stay in flight; with two, everything lands
        wait_stage(NB == 3 && j + 1 < je ? (SPLIT_B ? NBP : n_parts) : 0);
        stage_barrier();
        const bool more = j + 1 < je;
        const int ja = j + NS - 1, jw = j + NB - 1;
        const int bnext = SPLIT_B ? (bst == 0 ? 2 : bst - 1) : (buf + NB - 1) % NB;
        const uint8_t* sta = smem + T::a_at(buf);
        const uint8_t* sts = smem + T::s_at(buf);
        const uint8_t* stb = smem + T::b_at(bst);
        auto frag = [&](const uint8_t* st, int row_off) {
            return join(*reinterpret_cast<const i32x4*>(st + row_off + sl0),
                        *reinterpret_cast<const i32x4*>(st + row_off + sl1));
        };
        i32x8 b[L_NT];
#pragma unroll
        for (int ni = 0; ni < L_NT; ++ni) b[ni] = frag(stb, b_row + ni * 16 * kChunk);
        float swj[NSW];
#pragma unroll
        for (int k = 0; k < NSW; ++k) swj[k] = sw_cur[k];
        i32x8 a_[2];
        float sa_[2] = {};
        a_[0] = frag(sta, a_row);
        if constexpr (RESCALE) sa_[0] = *reinterpret_cast<const float*>(sts + s_row);
        if constexpr (SM == 0) {
            if (more) {
#pragma unroll
                for (int k = 0; k < NSW; ++k) sw_nxt[k] = swb[k][j + 1];
            }
        }
#pragma unroll
        for (int k = 0; k < NSW; ++k) sw_cur[k] = sw_nxt[k];
#pragma unroll
        for (int mi = 0; mi < L_MT; ++mi) {
            const int cur = mi & 1, prv = cur ^ 1;
            if (mi + 1 < L_MT) {
                a_[prv] = frag(sta, a_row + (mi + 1) * 16 * kChunk);
                if constexpr (RESCALE)
                    sa_[prv] = *reinterpret_cast<const float*>(sts + s_row + (mi + 1) * 64);
            }
            // Waves 4-7 (the second wave of each SIMD) win instruction issue
            // over the first half of the row tiles. Left to the oldest-first
            // arbiter, waves 0-3 finish every chunk ~600 cycles early and the
            // late waves then run alone up to the barrier, with no MFMA of
            // the other wave to hide their VALU work (MI355X: 1.5-3.5 % per
            // shape at M = 4096).
            if (wave >= 4) {
                if (mi == 0) __builtin_amdgcn_s_setprio(1);
                if (mi == L_MT / 2) __builtin_amdgcn_s_setprio(0);
            }
#pragma unroll
            for (int part = 0; part < kParts; ++part) {
                if (part / kPer != mi) continue;
                // the B parts stay behind the A and scale parts in issue
                // order (the next chunk's wait relies on it)
                if (SPLIT_B && part == kFirstB) __builtin_amdgcn_sched_barrier(0);
                if ((part >= kFirstB && part != kScalePart ? jw : ja) < je)
                    issue_part(ja, jw, ic<(buf + NS - 1) % NS>{}, bnext, part);
            }
            if constexpr (SM == kBigBf16) {
                if (mi < mt_live) {    // row tiles past M feed nothing that is stored
#pragma unroll
                    for (int ni = 0; ni < L_NT; ++ni)
                        acc[mi][ni] = mfma_bf16x64(b[ni], a_[cur], acc[mi][ni]);
                }
            } else if constexpr (SM == kBigConst) {
#pragma unroll
                for (int ni = 0; ni < L_NT; ++ni)
                    acc[mi][ni] = mfma_e4m3(b[ni], a_[cur], acc[mi][ni]);
            } else {
#pragma unroll
                for (int k = 0; k < NSW; ++k) sc[cur][k] = sa_[cur] * swj[k];
#pragma unroll
                for (int ni = 0; ni < L_NT; ++ni)
                    p[cur][ni] = mfma_e4m3(b[ni], a_[cur], f32x4{0, 0, 0, 0});
                if (mi > 0) rescale(mi - 1, prv);
                else if (j > jb) rescale(L_MT - 1, prv);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    for (int part = 0; part < kParts; ++part) issue_part(jb, jb, ic<0>{}, 0, part);
    int j = jb;
    if constexpr (SPLIT_B) {
        // chunk jb + 1's B rows, last in issue order
        if (jb + 1 < je) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < NBP; ++q) issue_part(jb, jb + 1, ic<0>{}, 1, kFirstB + q);
        }
    }
    if constexpr (NB == 2) {
        for (; j + 1 < je; j += 2) {
            chunk(ic<0>{}, j, 0);
            chunk(ic<1>{}, j + 1, 1);
        }
        if (j < je) chunk(ic<0>{}, j, 0);
    } else if constexpr (NS == 3) {
        if (jb + 1 < je) {
#pragma unroll
            for (int part = 0; part < kParts; ++part) issue_part(jb + 1, jb + 1, ic<1>{}, 1, part);
        }
        for (; j + 2 < je; j += 3) {
            chunk(ic<0>{}, j, 0);
            chunk(ic<1>{}, j + 1, 1);
            chunk(ic<2>{}, j + 2, 2);
        }
        if (j < je) chunk(ic<0>{}, j, 0);
        if (j + 1 < je) chunk(ic<1>{}, j + 1, 1);
    } else {
        // two A stages, three B stages (the B stage index runs at run time)
        int bst = 0;
        for (; j + 1 < je; j += 2) {
            chunk(ic<0>{}, j, bst);
            bst = bst == 2 ? 0 : bst + 1;
            chunk(ic<1>{}, j + 1, bst);
            bst = bst == 2 ? 0 : bst + 1;
        }
        if (j < je) chunk(ic<0>{}, j, bst);
    }
    if constexpr (RESCALE) rescale(L_MT - 1, (L_MT - 1) & 1);

    big_epilogue<SM, BM, BN, T::BYTES>(op, acc, smem, m0, n0, split, S);
}

}  // namespace heph
