// gemm_dma.h - what the DMA-staged GEMM kernels share: the block -> tile
// order, buffer-resource loads straight into LDS, the barrier between
// stages and the bf16 rounding of their epilogues.
#pragma once

#include "heph_kernels.h"

namespace heph {

namespace {

constexpr int GROUP_M = 8;
constexpr int NXCD = 8;

// Block id -> (tile_m, tile_n): contiguous ranges per XCD (blocks are
// handed to the 8 XCDs round robin), then grouped row-major order.
__device__ __forceinline__ void tile_of_block(int bid, int tiles_m, int tiles_n,
                                              int* tm, int* tn)
{
    const int nb = tiles_m * tiles_n;
    const int per = nb / NXCD, rem = nb % NXCD;
    const int x = bid % NXCD, k = bid / NXCD;
    const int lin = x * per + min(x, rem) + k;
    const int width = GROUP_M * tiles_n;
    const int g = lin / width;
    const int first_m = g * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int r = lin % width;
    *tm = first_m + r % gsize;
    *tn = r / gsize;
}

typedef __amdgpu_buffer_rsrc_t rsrc_t;

// Raw buffer resource over [p, p + 2^31): offsets are byte offsets from p.
// Word 3 = 0x00020000 (32-bit data format, as gfx9 raw buffers need).
__device__ __forceinline__ rsrc_t make_rsrc(const void* p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0x7fffffff, 0x00020000);
}
// 16 (4) bytes per lane from base + voff + soff straight into LDS at
// lds + 16 * lane (4 * lane); lds must be uniform.
__device__ __forceinline__ void dma16(rsrc_t r, uint32_t voff, uint32_t soff, void* lds)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16,
                                             voff, soff, 0, 0);
}
__device__ __forceinline__ void dma4(rsrc_t r, uint32_t voff, uint32_t soff, void* lds)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4,
                                             voff, soff, 0, 0);
}

// Workgroup barrier after wait_stage: every wave's DMA into the stage about
// to be read has landed, and its reads of the stage about to be refilled
// are done. No memory fence (the fence of __syncthreads waits for every
// outstanding DMA, the next chunk's included); the clobber keeps the
// compiler from moving LDS accesses across it.
__device__ __forceinline__ void stage_barrier() { asm volatile("s_barrier" ::: "memory"); }

typedef const __attribute__((address_space(4))) float* const_f32_ptr;

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Two floats -> two bf16 (round to nearest even) in one v_cvt_pk_bf16_f32,
// each as f32_to_bf16 rounds it.
__device__ __forceinline__ uint32_t pack_bf16_hw(float a, float b)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t));
}

// Four consecutive outputs v at element o of c: the residual (c's own
// values) added in f32, then one rounding.
__device__ __forceinline__ void store4(const Fp8Operands& op, size_t o, f32x4 v)
{
    if (op.c_f32) {
        f32x4* c = reinterpret_cast<f32x4*>(static_cast<float*>(op.c) + o);
        if (op.residual) v += *c;
        *c = v;
    } else {
        uint2* c = reinterpret_cast<uint2*>(static_cast<uint16_t*>(op.c) + o);
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

}  // namespace

}  // namespace heph
