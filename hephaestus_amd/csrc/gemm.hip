// gemm.hip - W8A8 FP8 GEMM for prefill (any M; chosen for M > 32).
//
// Replaces the reference's prefill kernel wmma_gemm_kernel_v3a_fp8
// (src/hephaestus/wmma_gfx12.mojo:756-888: 64x64 tile, BK=16, single LDS
// buffer, two barriers per 16-wide K step, rank-1 scale epilogue). Three
// families, chosen by gemm_plan below: the large DMA-staged tiles of gemm_big.h
// and the ring tiles of gemm_ring.h (33 to 1023 rows) while the operands' byte
// offsets fit 32 bits, and first here the 128x128 kernel for larger operands
// and for K % 128 != 0:
//   * 128x128 output tile per 256-thread workgroup, 2x2 waves of 64x64,
//     each wave 4x4 v_mfma_f32_16x16x128_f8f6f4 per 128-wide K chunk;
//   * K advances one 128-wide chunk per step, which is exactly one
//     activation group and one weight block, so each MFMA result is a
//     chunk partial that is rescaled in registers by sa[m,j] * sw[n/128,j]
//     and accumulated in fp32 (one FMA per accumulator per chunk);
//   * with the reference's granularity (per-channel weight, per-token
//     activation scale) nothing varies along K: the MFMAs accumulate
//     directly and the epilogue applies (acc*sa)*sw as the reference's
//     prefill kernel does (wmma_gfx12.mojo:848; acc*(sa*sw) at M = 1 to
//     match its decode kernel, :711-712);
//   * A/B tiles are double buffered in LDS (one barrier per chunk), with
//     the next chunk's global loads in flight during the MFMAs; LDS rows
//     are padded to 144 bytes to spread the 16-byte fragment reads;
//   * the block -> tile order gives each XCD a contiguous run of tiles in
//     a grouped (8 tile-rows) order, so A and B tiles are reused from that
//     XCD's L2.
#include <algorithm>

#include "gemm_big.h"
#include "gemm_ring.h"

namespace heph {

namespace {
constexpr int BM = 128;
constexpr int BN = 128;
constexpr int LDSTR = kChunk + 16;  // bytes per LDS row

__device__ __forceinline__ i32x4 lds16(const uint8_t* p)
{
    return *reinterpret_cast<const i32x4*>(p);
}

}  // namespace

// SM: 0 = 128x128 weight blocks, 1 = per-channel weights with per-chunk
// activation scales, 2 = per-channel weights and per-token activations.
template <int SM>
__global__ __launch_bounds__(256, 2) void fp8_gemm_kernel(Fp8Operands op)
{
    __shared__ __attribute__((aligned(16))) uint8_t As[2][BM * LDSTR];
    __shared__ __attribute__((aligned(16))) uint8_t Bs[2][BN * LDSTR];
    __shared__ float Ss[2][BM];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, slice = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    // K % 128 != 0 (per-token / per-channel scales only): the last chunk's
    // 16-byte pieces past K are zeros
    const int M = op.M, N = op.N, K = op.K, KC = (K + kChunk - 1) >> 7;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tm, tn;
    tile_of_block(blockIdx.x, tiles_m, tiles_n, &tm, &tn);
    const int m0 = tm * BM, n0 = tn * BN;

    // Global -> LDS staging: 1024 16-byte pieces per operand tile, four per
    // thread; eight consecutive threads cover one 128-byte row.
    const int lrow = tid >> 3, lcol = (tid & 7) * 16;
    const uint8_t* ag[4];
    const uint8_t* bg[4];
    bool aok[4], bok[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = m0 + lrow + 32 * r, n = n0 + lrow + 32 * r;
        aok[r] = m < M;
        bok[r] = n < N;
        ag[r] = op.q + (size_t)(aok[r] ? m : 0) * K + lcol;
        bg[r] = op.w + (size_t)(bok[r] ? n : 0) * K + lcol;
    }
    const bool sok = tid < BM && m0 + tid < M;
    const float* sg = op.s + (size_t)(sok ? m0 + tid : 0) * op.s_ld;

    i32x4 ra[4], rb[4];
    float rs = 0.0f;
    auto gload = [&](int j) {
        const bool kin = j * kChunk + lcol + 16 <= K;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ra[r] = aok[r] && kin ? ldg16(ag[r] + (size_t)j * kChunk) : i32x4{0, 0, 0, 0};
            rb[r] = bok[r] && kin ? ldg16(bg[r] + (size_t)j * kChunk) : i32x4{0, 0, 0, 0};
        }
        rs = sok ? sg[j * op.s_step] : 0.0f;
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            *reinterpret_cast<i32x4*>(&As[buf][(lrow + 32 * r) * LDSTR + lcol]) = ra[r];
            *reinterpret_cast<i32x4*>(&Bs[buf][(lrow + 32 * r) * LDSTR + lcol]) = rb[r];
        }
        if (tid < BM) Ss[buf][tid] = rs;
    };

    float swc[4];
#pragma unroll
    for (int ni = 0; ni < 4; ++ni) {
        const int n = n0 + wn * 64 + ni * 16 + r16;
        swc[ni] = SM == 1 ? op.sw[n < N ? n : 0] : 0.0f;
    }
    const float* swb = op.sw + (size_t)(n0 >> 7) * op.sw_ld;

    f32x4 acc[4][4];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = f32x4{0, 0, 0, 0};

    gload(0);
    lstore(0);
    __syncthreads();

    // The block scale of chunk j + 1 is loaded with chunk j + 1's tiles.
    float sw_cur = SM == 0 ? swb[0] : 1.0f, sw_nxt = 1.0f;
    for (int j = 0; j < KC; ++j) {
        const int cur = j & 1;
        if (j + 1 < KC) {
            gload(j + 1);
            if constexpr (SM == 0) sw_nxt = swb[j + 1];
        }

        i32x8 a[4], b[4];
#pragma unroll
        for (int mi = 0; mi < 4; ++mi) {
            const uint8_t* p = &As[cur][(wm * 64 + mi * 16 + r16) * LDSTR + slice * 16];
            a[mi] = join(lds16(p), lds16(p + 64));
        }
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
            const uint8_t* p = &Bs[cur][(wn * 64 + ni * 16 + r16) * LDSTR + slice * 16];
            b[ni] = join(lds16(p), lds16(p + 64));
        }
        if constexpr (SM == 2) {
#pragma unroll
            for (int mi = 0; mi < 4; ++mi)
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) acc[mi][ni] = mfma_e4m3(a[mi], b[ni], acc[mi][ni]);
        } else {
            const float swj = sw_cur;
            float sc[4][4];
#pragma unroll
            for (int mi = 0; mi < 4; ++mi) {
                const f32x4 s4 =
                    *reinterpret_cast<const f32x4*>(&Ss[cur][wm * 64 + mi * 16 + slice * 4]);
#pragma unroll
                for (int i = 0; i < 4; ++i) sc[mi][i] = s4[i] * swj;
            }
#pragma unroll
            for (int mi = 0; mi < 4; ++mi)
#pragma unroll
                for (int ni = 0; ni < 4; ++ni) {
                    const f32x4 p = mfma_e4m3(a[mi], b[ni], f32x4{0, 0, 0, 0});
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc[mi][ni][i] += p[i] * (SM == 0 ? sc[mi][i] : sc[mi][i] * swc[ni]);
                }
        }

        sw_cur = sw_nxt;
        if (j + 1 < KC) lstore(cur ^ 1);
        __syncthreads();
    }

    // Epilogue: lane holds rows (slice*4 + i) of each 16x16 tile, column r16.
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
        for (int ni = 0; ni < 4; ++ni) {
            const int col = n0 + wn * 64 + ni * 16 + r16;
            if (col >= N) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = m0 + wm * 64 + mi * 16 + slice * 4 + i;
                if (row >= M) continue;
                const size_t o = (size_t)row * N + col;
                float v = acc[mi][ni][i];
                if constexpr (SM == 2) {
                    const float sa = op.s[row], sw = op.sw[col];
                    v = M == 1 ? v * (sa * sw) : (v * sa) * sw;
                }
                if (op.c_f32) {
                    float* c = static_cast<float*>(op.c);
                    c[o] = op.residual ? v + c[o] : v;
                } else {
                    uint16_t* c = static_cast<uint16_t*>(op.c);
                    if (op.residual) v += __uint_as_float((uint32_t)c[o] << 16);
                    c[o] = f32_to_bf16(v);
                }
            }
        }
}

// Sums the K-split partials of a GEMM in split order, applies the scales where
// the partials are unscaled (SCALE: Fp8Operands::scaled_last; (acc*sa)*sw, the
// association of the unsplit tiles), adds the residual and stores bf16 or f32
// (four outputs per thread; N % 16 == 0).
template <bool SCALE>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(Fp8Operands op)
{
    const size_t mn = (size_t)op.M * op.N, n4 = mn / 4;
    const f32x4* part = reinterpret_cast<const f32x4*>(op.part);
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n4;
         i += (size_t)gridDim.x * 256) {
        f32x4 v = part[i];
        for (int s = 1; s < op.splits; ++s) v += part[(size_t)s * n4 + i];
        if constexpr (SCALE) {
            const size_t row = i * 4 / op.N;
            const float sa = op.s[row];
            const f32x4 sw = ldf4(op.sw + (i * 4 - row * op.N));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (v[e] * sa) * sw[e];
        }
        if (op.c_f32) {
            f32x4* c = static_cast<f32x4*>(op.c) + i;
            if (op.residual) v += *c;
            *c = v;
        } else {
            uint2* c = static_cast<uint2*>(op.c) + i;
            if (op.residual) {
                const uint2 r = *c;
                v[0] += bf16lo(r.x);
                v[1] += bf16hi(r.x);
                v[2] += bf16lo(r.y);
                v[3] += bf16hi(r.y);
            }
            *c = make_uint2(pack_bf16_hw(v[0], v[1]), pack_bf16_hw(v[2], v[3]));
        }
    }
}

hipError_t launch_splitk_reduce(const Fp8Operands& op, hipStream_t stream, const LaunchTiming& t)
{
    const size_t n4 = (size_t)op.M * op.N / 4;
    const int blocks = (int)std::min<size_t>((n4 + 255) / 256, 4096);
    if (op.scaled_last())
        return launch(splitk_reduce_kernel<true>, dim3(blocks), dim3(256), 0, stream, t, op);
    return launch(splitk_reduce_kernel<false>, dim3(blocks), dim3(256), 0, stream, t, op);
}

namespace {

template <int BM, int BN>
hipError_t launch_big(const Fp8Operands& op, hipStream_t stream, const LaunchTiming& t)
{
    const int tiles = ((op.M + BM - 1) / BM) * ((op.N + BN - 1) / BN);
    const dim3 grid(tiles * op.splits);
    if (op.splits > 1) {
        // the GEMM carries the start stamp, the reduction the stop stamp
        hipError_t e;
        if (op.w_block)
            e = launch(fp8_gemm256_kernel<0, BM, BN>, grid, dim3(512), 0, stream,
                       LaunchTiming{t.start, nullptr}, op);
        else
            e = launch(fp8_gemm256_kernel<1, BM, BN>, grid, dim3(512), 0, stream,
                       LaunchTiming{t.start, nullptr}, op);
        if (e != hipSuccess) return e;
        return launch_splitk_reduce(op, stream, LaunchTiming{nullptr, t.stop});
    }
    if (op.w_block)
        return launch(fp8_gemm256_kernel<0, BM, BN>, grid, dim3(512), 0, stream, t, op);
    if (op.scaled_last())
        return launch(fp8_gemm256_kernel<2, BM, BN>, grid, dim3(512), 0, stream, t, op);
    return launch(fp8_gemm256_kernel<1, BM, BN>, grid, dim3(512), 0, stream, t, op);
}

template <int SM, int BM, int BN, int D>
hipError_t launch_ring_t(const Fp8Operands& op, hipStream_t stream, const LaunchTiming& t)
{
    const dim3 grid(((op.M + BM - 1) / BM) * ((op.N + BN - 1) / BN) * op.splits);
    if (op.splits == 1)
        return launch(gemm_ring_kernel<SM, BM, BN, 2, D>, grid, dim3(256), 0, stream, t, op);
    hipError_t e = launch(gemm_ring_kernel<SM, BM, BN, 2, D>, grid, dim3(256), 0, stream,
                          LaunchTiming{t.start, nullptr}, op);
    if (e != hipSuccess) return e;
    return launch_splitk_reduce(op, stream, LaunchTiming{nullptr, t.stop});
}

template <int BM, int BN, int D>
hipError_t launch_ring(const Fp8Operands& op, hipStream_t stream, const LaunchTiming& t)
{
    if (op.w_block) return launch_ring_t<kRingBlock, BM, BN, D>(op, stream, t);
    if (op.scaled_last()) return launch_ring_t<kRingConst, BM, BN, D>(op, stream, t);
    return launch_ring_t<kRingChannel, BM, BN, D>(op, stream, t);
}

}  // namespace

// Measured cost per tile (MI355X shader cycles at ~1.9 GHz, random E4M3
// data, weights from HBM): `chunk` per 128-wide chunk and `fixed` per
// workgroup (prologue, epilogue), fitted to the GEMM-only times of the
// config-1 shapes at M = 4096 (o_proj and down: one round of tiles each,
// K = 4096 against 9728); 64 x 256 fitted to M = 512. A bigger tile does
// more MFMA work per chunk, a smaller one fills the CUs in finer steps: at
// M = 4096 the fit ranks the tiles as measured on every config-1 shape
// (qkv 256 x 192 72.6 us against 75.7 at 256 x 256; o_proj 128 x 320 46.5
// against 47.9 at 192 x 256; gate_up 256 x 256 193.0 against 212.2; down
// 128 x 320 100.4 against 104.4), and at M = 512 as well (64 x 192 for qkv,
// 256 tiles, one round: 18.7 against 21.6 us at 64 x 256; 64 x 256 with 3 K
// splits for o_proj; 128 x 320 for gate_up; 128 x 256 with 6 splits for
// down). 64 x 192 is fitted to M = 512 qkv alone.
struct TileCost {
    int bm, bn;
    long chunk, fixed;
};
constexpr TileCost kTileCost[] = {{256, 256, 2535, 16730}, {256, 192, 2569, 11650},
                                  {192, 256, 2440, 12930}, {128, 320, 2327, 13880},
                                  {128, 256, 1734, 9887},  {64, 256, 1550, 7000},
                                  {64, 192, 1300, 6000}};

// Estimated time (us) of the large-M GEMM with tile tc and s K splits:
// rounds of (tile, split) workgroups over the CUs (one 512-thread
// workgroup per CU) times a workgroup's cost (its chunks and the fixed
// part) at ~1.9 GHz; a split adds the reduction: ~8 us of launch and
// per-workgroup set-up, and the partials (M*N*4 bytes a split) read back
// at ~5 TB/s.
static double gemm_estimate(int M, int N, int K, const TileCost& tc, int s, long cus)
{
    const long tiles = (long)((M + tc.bm - 1) / tc.bm) * ((N + tc.bn - 1) / tc.bn);
    const int KC = K / kChunk;
    const long rounds = (tiles * s + cus - 1) / cus;
    double t = (double)rounds * ((double)((KC + s - 1) / s) * tc.chunk + tc.fixed) / 1900.0;
    if (s > 1) t += 8.0 + (double)s * M * N * 4.0 / 5.0e6;
    return t;
}

// The ring tiles (gemm_ring.h) and their cost: with n workgroups on the fullest
// CU, KC chunks each and weights streamed at 5 TB/s at best,
//     max(2 + n g + KC max(c1, n c), 3 + N K / 5e6) us,
// a split's reduction 2.5 us and its partials at 4 TB/s (c1 stands for a chunk's
// latency alone on the CU, c for its share of it: coefficients fitted together to
// 1230 MI355X times at 47 shapes, M 33 .. 1000, N 1024 .. 19456, K 1024 .. 9728,
// 1 .. 8 splits, weights from HBM).
struct RingCost {
    int bm, bn;
    double g, c1, c;
};
constexpr RingCost kRingCost[] = {{64, 64, 1.42, 0.310, 0.274},
                                  {64, 32, 0.65, 0.276, 0.213},
                                  {96, 64, 2.74, 0.242, 0.357},
                                  {64, 128, 3.41, 0.319, 0.424}};

static double ring_estimate(int M, int N, int K, const RingCost& rc, int s)
{
    const long wgs = (long)((M + rc.bm - 1) / rc.bm) * ((N + rc.bn - 1) / rc.bn) * s;
    const double n = (double)((wgs + kPlanCUs - 1) / kPlanCUs);
    const int kc = (K / kChunk + s - 1) / s;
    const double t = std::max(2.0 + n * rc.g + kc * std::max(rc.c1, n * rc.c),
                              3.0 + (double)N * K / 5.0e6);
    return s > 1 ? t + 2.5 + (double)s * M * N * 4.0 / 4.0e6 : t;
}

// Tile and K splits of the large-M GEMM: the pair with the least estimated
// time, splitting into at most 8 splits of at least 4 chunks, and only where
// `scratch` bytes hold the fp32 partials (a ring tile then takes fewer splits,
// a large tile none: a buffer sized for other rows may be any size); ties go
// to the earlier tile of kTileCost, then to fewer splits.
// A forced tile height (gemm_bm) or width (gemm_bn) keeps only the tiles
// that have it. per_token (one activation scale a row, with either weight
// scale): the large tiles do not split.
// From 33 to 511 rows (per-token scales: to 1023, where the alternative is a
// large tile over all of K) a ring tile is taken where its estimate is under
// 0.8 of that, or under 0.7 where the large tile would split a K past 4608. Of
// 1494 drawn calls (M 33 .. 1100, N 16 .. 19456, K 128 .. 16384, every scale
// format, workspaces of several sizes) that a line of 0.8 gave a ring tile, those
// under 0.7 ran at 0.72 of the large tile's time; from 0.7 to 0.8 they ran at
// 0.84 against an unsplit large tile (0.98 at worst), at 1.00 against a split
// one (0.80 to 1.13; 13 of the 14 past 1.015 with K of 4736 and more). Past
// K = 4096 the ring splits first: one workgroup's chain of chunks is then longer
// than a reduction.
GemmPlan gemm_plan(int M, int N, int K, size_t scratch, int forced_bm, int forced_bn,
                   bool per_token)
{
    const auto fits = [&](int s) { return s == 1 || (size_t)s * M * N * 4 <= scratch; };
    // MI355X's 256 CUs, not the visible count: the plan (and the K-split
    // summation order with it) does not change under a CU mask or partition
    const long cus = kPlanCUs;
    const int KC = K / kChunk;
    GemmPlan best{0, 0, 1, false};
    double best_t = -1.0;
    const auto large = [&](int max_splits) {
        best = GemmPlan{0, 0, 1, false};
        best_t = -1.0;
        for (const auto& tc : kTileCost) {
            // 64 x 192 only where its fit holds (M >= 256): below, the K-split
            // plans of the small-M routes stay with the tiles they were measured on
            if (tc.bm == 64 && tc.bn == 192 && M < 256 && forced_bn != 192) continue;
            if (forced_bm >= 64 && tc.bm != forced_bm) continue;
            if (forced_bn && tc.bn != forced_bn) continue;
            for (int s = 1; s <= max_splits; ++s) {
                if (s > 1 && KC / s < 4) break;
                const double t = gemm_estimate(M, N, K, tc, s, cus);
                if (best_t < 0.0 || t < best_t) {
                    best_t = t;
                    best = GemmPlan{tc.bm, tc.bn, s, false};
                }
            }
        }
    };
    large(per_token ? 1 : 8);
    if (!fits(best.splits)) large(1);
    if (best.bm == 0) best = GemmPlan{forced_bm >= 64 ? forced_bm : 256, 256, 1, false};
    if (M <= 32 || M >= (per_token ? 1024 : 512) || forced_bm || forced_bn) return best;
    best_t *= best.splits > 1 && K > 4608 ? 0.7 : 0.8;
    const auto ring = [&](int s0, int s1) {
        for (const auto& rc : kRingCost) {
            for (int s = s0; s <= s1 && fits(s); ++s) {
                if (s > 1 && KC / s < 4) break;
                const double t = ring_estimate(M, N, K, rc, s);
                if (t < best_t) {
                    best_t = t;
                    best = GemmPlan{rc.bm, rc.bn, s, true};
                }
            }
        }
    };
    ring(K > 4096 ? 2 : 1, 8);
    if (!best.ring && best.splits == 1) ring(1, 1);
    return best;
}

bool gemm_splits_ready(const Fp8Operands& op)
{
    return gemm_plan(op.M, op.N, op.K, op.part ? op.part_bytes : 0, op.tune.gemm_bm,
                     op.tune.gemm_bn, op.s_step == 0).splits > 1;
}

size_t gemm_split_bytes(int M, int N, int K)
{
    const int s = gemm_plan(M, N, K, SIZE_MAX).splits;
    return s > 1 ? (size_t)s * M * N * 4 : 0;
}

hipError_t launch_fp8_gemm(const Fp8Operands& op, hipStream_t stream,
                           const LaunchTiming& t, const char** name)
{
    // The DMA-staged tiles for every M (N % 16 == 0 keeps every output group
    // inside the row), splitting K when they leave CUs idle; their 32-bit operand
    // offsets need M*K and N*K below 2^31, else the 128x128 kernel.
    const bool small_offsets = (long)op.M * op.K < (1L << 31) && (long)op.N * op.K < (1L << 31);
    const bool force_128 = op.tune.gemm_bm == 1;
    if (small_offsets && !force_128) {
        Fp8Operands o = op;
        const GemmPlan plan = gemm_plan(o.M, o.N, o.K, o.part ? o.part_bytes : 0, o.tune.gemm_bm,
                                        o.tune.gemm_bn, o.s_step == 0);
        o.splits = plan.splits;
        const bool sk = o.splits > 1;
        if (plan.ring) {
            if (plan.bm == 96) {
                *name = sk ? "fp8_gemm_96x64_splitk" : "fp8_gemm_96x64";
                return launch_ring<96, 64, 6>(o, stream, t);
            }
            if (plan.bn == 64) {
                *name = sk ? "fp8_gemm_64x64_splitk" : "fp8_gemm_64x64";
                return launch_ring<64, 64, 4>(o, stream, t);
            }
            if (plan.bn == 32) {
                *name = sk ? "fp8_gemm_64x32_splitk" : "fp8_gemm_64x32";
                return launch_ring<64, 32, 4>(o, stream, t);
            }
            *name = sk ? "fp8_gemm_64x128_splitk" : "fp8_gemm_64x128";
            return launch_ring<64, 128, 6>(o, stream, t);
        }
        if (plan.bn == 192 && plan.bm == 64) {
            *name = sk ? "fp8_gemm_64x192_splitk" : "fp8_gemm_64x192";
            return launch_big<64, 192>(o, stream, t);
        }
        if (plan.bn == 192) {
            *name = sk ? "fp8_gemm_256x192_splitk" : "fp8_gemm_256x192";
            return launch_big<256, 192>(o, stream, t);
        }
        if (plan.bn == 320) {
            *name = sk ? "fp8_gemm_128x320_splitk" : "fp8_gemm_128x320";
            return launch_big<128, 320>(o, stream, t);
        }
        switch (plan.bm) {
        case 64:
            *name = sk ? "fp8_gemm_64x256_splitk" : "fp8_gemm_64x256";
            return launch_big<64, 256>(o, stream, t);
        case 128:
            *name = sk ? "fp8_gemm_128x256_splitk" : "fp8_gemm_128x256";
            return launch_big<128, 256>(o, stream, t);
        case 192:
            *name = sk ? "fp8_gemm_192x256_splitk" : "fp8_gemm_192x256";
            return launch_big<192, 256>(o, stream, t);
        default:
            *name = sk ? "fp8_gemm_256x256_splitk" : "fp8_gemm_256x256";
            return launch_big<256, 256>(o, stream, t);
        }
    }
    const int tiles = ((op.M + BM - 1) / BM) * ((op.N + BN - 1) / BN);
    *name = "fp8_gemm_128x128";
    if (op.w_block)
        return launch(fp8_gemm_kernel<0>, dim3(tiles), dim3(256), 0, stream, t, op);
    if (op.scaled_last())
        return launch(fp8_gemm_kernel<2>, dim3(tiles), dim3(256), 0, stream, t, op);
    return launch(fp8_gemm_kernel<1>, dim3(tiles), dim3(256), 0, stream, t, op);
}

}  // namespace heph
