// Shared device/host definitions for the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/qgemm.h"

namespace qgemm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short us4 __attribute__((ext_vector_type(4)));
// loads and stores of several elements at any address of one: the vector memory path takes any byte address
typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));
typedef float v4f_any __attribute__((ext_vector_type(4), aligned(1)));
typedef int v2i_any __attribute__((ext_vector_type(2), aligned(1)));
typedef unsigned u32_any __attribute__((aligned(1)));
typedef unsigned short u16_any __attribute__((aligned(1)));

// Arithmetic families of the MFMA kernels.
enum Arith : int { AR_I8 = 0, AR_F8 = 1, AR_BF16 = 2, AR_F16 = 3, AR_F8W = 4 };   // F8W: fp8 operands, multiplied as bf16

constexpr int kWave = 64;          // include/gpu_type.h:23 (WAVE_SIZE)
constexpr int kXcds = 8;           // include/gpu_type.h:24 (XCD_SWIZZLE)
constexpr int kScaleBlock = 128;   // hip_mix_gemm_kernel.cpp:46 (SCALE_BLOCK_SIZE)

__host__ __device__ inline int dtype_bytes(int dt) {
    switch (dt) {
        case QGEMM_DT_F32: case QGEMM_DT_I32: return 4;
        case QGEMM_DT_BF16: case QGEMM_DT_F16: return 2;
        case QGEMM_DT_I8: case QGEMM_DT_F8E4M3: return 1;
        default: return 0;
    }
}

// bytes of an element of C (fp32, int32, or one of the 16-bit types)
__device__ inline uint32_t c_elem_bytes(int dt) { return dt == QGEMM_DT_F32 || dt == QGEMM_DT_I32 ? 4 : 2; }

// float -> bf16 bits, round to nearest even with a NaN guard: the intent of
// src/include/fast_quat.h:4-12 (which has no guard).  The compiler lowers the
// cast to v_cvt_pk_bf16_f32 on gfx950.
__device__ inline unsigned short f32_to_bf16_bits(float f) {
    __bf16 h = (__bf16)f;
    return __builtin_bit_cast(unsigned short, h);
}
__device__ inline unsigned short f32_to_f16_bits(float f) {
    _Float16 h = (_Float16)f;
    return __builtin_bit_cast(unsigned short, h);
}
// Four floats -> four bf16 / fp16 values in 8 bytes, element 0 in the low half of component 0.  Two elements per
// v_cvt_pk_*: half the instructions of four scalar conversions, and no packing step afterwards.  (The packing the
// compiler picks for two 16-bit scalars, v_pack_b32_f16, treats its inputs as fp16 numbers and quiets what looks
// like a signalling NaN: a bf16 pattern 0x7c01 .. 0x7dff, a finite value of 2^121 and more, came out with bit 9
// set.  The vector conversions never hold a lone 16-bit value in a register.)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ inline v2i pack4_bf16(float a, float b, float c, float d) {
    return v2i{__builtin_bit_cast(int, __builtin_convertvector(f32x2_t{a, b}, bf16x2_t)),
               __builtin_bit_cast(int, __builtin_convertvector(f32x2_t{c, d}, bf16x2_t))};
}
__device__ inline v2i pack4_f16(float a, float b, float c, float d) {
    return v2i{__builtin_bit_cast(int, __builtin_convertvector(f32x2_t{a, b}, f16x2_t)),
               __builtin_bit_cast(int, __builtin_convertvector(f32x2_t{c, d}, f16x2_t))};
}
// element e (0 .. 3) of such a pack
__device__ inline unsigned short pack4_elem(v2i p, int e) { return (unsigned short)((unsigned)p[e >> 1] >> ((e & 1) * 16)); }

// Four neighbouring elements of a row of C, the first `valid` of them inside it, at any element address
__device__ inline void store_out4(void *C, size_t idx, const float *v, int out_dtype, int valid) {
    if (out_dtype == QGEMM_DT_F32) {
        float *dst = (float *)C + idx;
        if (valid >= 4) *(v4f_any *)dst = v4f{v[0], v[1], v[2], v[3]};
        else
            for (int e = 0; e < 3; ++e)
                if (e < valid) dst[e] = v[e];
        return;
    }
    const v2i h = out_dtype == QGEMM_DT_BF16 ? pack4_bf16(v[0], v[1], v[2], v[3]) : pack4_f16(v[0], v[1], v[2], v[3]);
    unsigned short *dst = (unsigned short *)C + idx;
    if (valid >= 4) *(v2i_any *)dst = h;
    else
        for (int e = 0; e < 3; ++e)
            if (e < valid) dst[e] = pack4_elem(h, e);
}

// W dwords moved down by n bytes (zeros from above); DWORDS: n is a multiple of 4
template <int W, bool DWORDS = false>
__device__ __forceinline__ void move_down(uint32_t *w, uint32_t n) {
    uint32_t v[W + 1];
    const uint32_t q = n >> 2;
#pragma unroll
    for (int i = 0; i <= W; ++i) {
        v[i] = 0;
#pragma unroll
        for (int k = i; k < W; ++k) v[i] = q == (uint32_t)(k - i) ? w[k] : v[i];
    }
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = DWORDS ? v[i] : __builtin_amdgcn_alignbyte(v[i + 1], v[i], n & 3);
}

// four e4m3 values -> four bf16 values (exact; NaNs stay NaNs)
__device__ inline v2i widen_fp8(uint32_t w) {
    return v2i{__builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false)),
               __builtin_bit_cast(int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true))};
}

// A launch whose status is that of the launch itself.  The <<< >>> form passes the sizes through a stack of the runtime and leaves
// the status to hipGetLastError: two calls and 0.1 - 0.3 us of host time more, of 3.3 a product.  A launch that fails leaves nothing in the
// runtime's last error, where the next caller of hipGetLastError, here or in the program, would take it for its own.
template <class... P>
inline hipError_t launch_kernel(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, std::common_type_t<P>... args) {
    void *at[] = {(void *)&args...};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, at, lds, stream);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

// i / d and i % d with inv = inverse_of(d): the estimate is at most one too small.  Four scalar instructions where the values are
// uniform; the compiler's own division by a variable is two dozen, half of them on the vector ALU.
__host__ __device__ inline uint32_t inverse_of(uint32_t d) {
    return d <= 1 ? 0xFFFFFFFFu : (uint32_t)(((uint64_t)1 << 32) / d);
}
__host__ __device__ inline uint32_t div_by_inv(uint32_t i, uint32_t d, uint32_t inv, uint32_t &rem) {
    uint32_t q = (uint32_t)(((uint64_t)i * inv) >> 32);
    rem = i - q * d;
    if (rem >= d) {
        rem -= d;
        ++q;
    }
    return q;
}

// Linear workgroup id -> (tile_m, tile_n).
// Step 1 (XCD remap): the dispatcher deals workgroups to the 8 XCDs round
// robin, so ids {x, x+8, x+16, ..} share an L2.  Renumber so that each XCD
// owns one contiguous range of the raster.
// Step 2 (GROUP_M raster, sm89_gemm_kernel_v3.cu:169-183): walk `group_m`
// tile rows column by column, so that concurrently resident tiles share A
// panels and B panels.  The group-size clamp uses the tile count (the
// reference clamps with M in rows).
// The divisors come with their inverses from the host: every workgroup starts with this map, in front of its first copy.
struct TileMap {
    uint32_t tiles_m, tiles_n, group_m;
    uint32_t inv_group, inv_gm, inv_last;      // of a group's tiles, of group_m, of the rows in the last, shorter group
};
__host__ __device__ inline TileMap make_tile_map(uint32_t tiles_m, uint32_t tiles_n, uint32_t group_m) {
    const uint32_t g = group_m > 1 ? (group_m < tiles_m ? group_m : tiles_m) : 1;
    return TileMap{tiles_m, tiles_n, g, inverse_of(g * tiles_n), inverse_of(g), inverse_of(tiles_m % g)};
}
__host__ __device__ inline void tile_map(uint32_t wg, const TileMap &t, uint32_t &tm, uint32_t &tn) {
    const uint32_t total = t.tiles_m * t.tiles_n;
    uint32_t id = wg;
    if (total >= (uint32_t)kXcds * 2) {
        const uint32_t per = (total + kXcds - 1) / kXcds;           // ids owned by a "tall" XCD
        const uint32_t tall = total % kXcds ? total % kXcds : kXcds;  // XCDs that own `per` ids
        const uint32_t xcd = wg % kXcds, local = wg / kXcds;
        id = xcd < tall ? xcd * per + local : tall * per + (xcd - tall) * (per - 1) + local;
    }
    uint32_t in_group, row;
    const uint32_t start_m = div_by_inv(id, t.group_m * t.tiles_n, t.inv_group, in_group) * t.group_m;
    const uint32_t left = t.tiles_m - start_m;
    tn = div_by_inv(in_group, left < t.group_m ? left : t.group_m, left < t.group_m ? t.inv_last : t.inv_gm, row);
    tm = start_m + row;
}

}  // namespace qgemm
