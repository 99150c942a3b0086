// Kernels around the MFMA GEMM: the transposes, the packing of operands it cannot read as they stand, the
// split-K reduction.
#pragma once
#include "common.h"

namespace qgemm {

// ---------------------------------------------------------------------------
// Transpose of 4-byte elements: out[n*M + m] = in[m*N + n]   (src/transpose/transpose.cu:11-58).
// 64 x 64 element tile through LDS, 256 threads.  The columns of the LDS tile are XOR-swizzled by
// the row, so both the row-wise fill and the column-wise drain touch all banks; no padding column.
// Any M, N.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) transpose_u32_kernel(const uint32_t *__restrict__ in, uint32_t *__restrict__ out, uint32_t M,
                                                            uint32_t N) {
    constexpr int TILE = 64;
    __shared__ uint32_t tile[TILE][TILE];
    const uint32_t m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;   // 64 x 4
    // Every lane loads, those outside from the nearest row and column: behind a branch each of the sixteen loads waited for the
    // one before (us, graph replays: 1120 x 32 5.06 -> 2.51, 2432 x 2368 11.4 -> 8.1).
    const uint32_t from = n0 + tx < N ? n0 + tx : N - 1;
    uint32_t v[TILE / 4];
#pragma unroll
    for (int i = 0; i < TILE / 4; ++i) {
        const uint32_t m = m0 + ty + 4 * i;
        v[i] = in[(size_t)(m < M ? m : M - 1) * N + from];
    }
#pragma unroll
    for (int i = 0; i < TILE / 4; ++i) tile[ty + 4 * i][tx ^ (ty + 4 * i)] = v[i];
    __syncthreads();
    const uint32_t m = m0 + tx;                   // output column
#pragma unroll
    for (int i = 0; i < TILE / 4; ++i) {
        const int r = ty + 4 * i;
        if (n0 + r < N && m < M) out[(size_t)(n0 + r) * M + m] = tile[tx][r ^ tx];
    }
}

// the first `bytes` (below 16) of v at any address, in parts of 8, 4, 2 and 1 bytes
__device__ inline void store_part(void *p, v4i v, uint32_t bytes) {
    char *dst = (char *)p;
    uint32_t e0 = (uint32_t)v[0], e1 = (uint32_t)v[1];
    if (bytes & 8) {
        *(v2i_any *)dst = v2i{v[0], v[1]};
        dst += 8;
        e0 = (uint32_t)v[2];
        e1 = (uint32_t)v[3];
    }
    if (bytes & 4) {
        *(u32_any *)dst = e0;
        dst += 4;
        e0 = e1;
    }
    if (bytes & 2) {
        *(u16_any *)dst = (uint16_t)e0;
        dst += 2;
        e0 >>= 16;
    }
    if (bytes & 1) *(uint8_t *)dst = (uint8_t)e0;
}

// ---------------------------------------------------------------------------
// Byte transpose (the fp8 / int8 operands of the reference layout, packed operands, matrix_transpose).
// 128 x 128 tile, 256 threads.  A thread loads 4 x 4 bytes (four
// rows, one dword each: a wave reads whole 128-byte row pieces), transposes the 4 x 4 block in
// registers with byte permutes, and writes the four resulting dwords (4 consecutive m of one n)
// into the LDS tile [n][m]; the tile leaves as 16-byte pieces of output rows, 128 bytes per row.
// ---------------------------------------------------------------------------
// One 128 x 128 tile of the byte transpose (tile_m, tile_n in tiles).  ALIGNED: M a multiple of 16, N of 4, aligned rows,
// Mout == M.  Otherwise any M, N, ld, pitch and pointers: at a row's end the last whole piece is loaded and moved down, what
// sticks out of the output is stored in parts, and the columns
// M .. Mout - 1 of the output are filled with zeros.
template <bool ALIGNED>
__device__ inline void transpose_bytes_tile(const uint8_t *__restrict__ in, size_t ld, uint8_t *__restrict__ out, size_t pitch,
                                            uint32_t M, uint32_t Mout, uint32_t N, uint32_t tile_m, uint32_t tile_n) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef typename std::conditional<ALIGNED, v4i, v4i_any>::type vec_t;
    typedef typename std::conditional<ALIGNED, uint32_t, u32_any>::type word_t;
    constexpr int T = 128, PITCH = T + 16;        // bytes per LDS row
    __shared__ __attribute__((aligned(16))) uint8_t tile[T * PITCH];
    const uint32_t m0 = tile_m * T, n0 = tile_n * T;
    const int cg = threadIdx.x & 31, rg = threadIdx.x >> 5;      // 32 column groups of 4 bytes x 8 row groups of 16
    const uint32_t n = n0 + cg * 4;
    // Four bytes of one row, zeros outside.  Ragged: every lane with a column and a row loads, from the nearest row and, where its row ends
    // inside the four bytes, from the row's last four, and moves them down (no branch, in which each load would wait for the one before).
    const bool wide = N >= 4, inside = n < N && m0 + rg * 16 < M;
    const uint32_t from = n + 4 <= N ? n : (wide ? N - 4 : 0), down = (n - from) < 4 ? (n - from) * 8 : 32;
    auto load4 = [&](uint32_t m) -> uint32_t {
        const uint8_t *src = in + (size_t)(m < M ? m : M - 1) * ld + from;
        uint32_t w = 0;
        if (wide) {
            w = *(const word_t *)src;
        } else {
            for (uint32_t e = 0; e < N; ++e) w |= (uint32_t)src[e] << (8 * e);
        }
        return m < M && down < 32 ? w >> down : 0;
    };
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
        const uint32_t m = m0 + rg * 16 + ch * 4;
        uint32_t a = 0, b = 0, c = 0, d = 0;
        if constexpr (ALIGNED) {
            if (n < N && m < M) {                 // (M % 4 == 0, the four rows are all inside or all outside)
                const uint8_t *src = in + (size_t)m * ld + n;
                a = *(const word_t *)src;
                b = *(const word_t *)(src + ld);
                c = *(const word_t *)(src + 2 * ld);
                d = *(const word_t *)(src + 3 * ld);
            }
        } else if (inside) {
            a = load4(m);
            b = load4(m + 1);
            c = load4(m + 2);
            d = load4(m + 3);
        }
        // v_perm_b32: selector byte k picks byte k of the result out of {src1 bytes 0-3, src0 bytes 4-7}
        const uint32_t ab_lo = __builtin_amdgcn_perm(b, a, 0x05010400), ab_hi = __builtin_amdgcn_perm(b, a, 0x07030602);
        const uint32_t cd_lo = __builtin_amdgcn_perm(d, c, 0x05010400), cd_hi = __builtin_amdgcn_perm(d, c, 0x07030602);
        const uint32_t o0 = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100), o1 = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302);
        const uint32_t o2 = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100), o3 = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302);
        uint8_t *dst = tile + (cg * 4) * PITCH + rg * 16 + ch * 4;   // [n - n0][m - m0]
        *(uint32_t *)dst = o0;
        *(uint32_t *)(dst + PITCH) = o1;
        *(uint32_t *)(dst + 2 * PITCH) = o2;
        *(uint32_t *)(dst + 3 * PITCH) = o3;
    }
    __syncthreads();
    const int piece = threadIdx.x & 7, row = threadIdx.x >> 3;   // 8 pieces of 16 bytes per output row, 32 rows per pass
#pragma unroll
    for (int ps = 0; ps < 4; ++ps) {
        const int r = row + ps * 32;
        const uint32_t on = n0 + r, om = m0 + piece * 16;
        if (on >= N || om >= Mout) continue;
        const uint8_t *src = tile + r * PITCH + piece * 16;
        uint8_t *dst = out + (size_t)on * pitch + om;
        if (ALIGNED || om + 16 <= Mout) {
            *(vec_t *)dst = *(const v4i *)src;
        } else {
            store_part(dst, *(const v4i *)src, Mout - om);
        }
    }
#endif
}

template <bool ALIGNED>
__global__ void __launch_bounds__(256) transpose_bytes_kernel(const uint8_t *__restrict__ in, uint8_t *__restrict__ out,
                                                              uint32_t M, uint32_t N) {
    transpose_bytes_tile<ALIGNED>(in, N, out, M, M, M, N, blockIdx.y, blockIdx.x);
}

// Two byte transposes in one launch (both operands of the reference fp8 layout: the second launch costs more
// than either transpose takes on mid-size shapes): workgroups 0 .. tiles0-1 take matrix 0, the rest matrix 1.
struct Transpose2Args {
    const uint8_t *in[2];
    uint8_t *out[2];
    uint32_t M[2], N[2], tiles_n[2], tiles0;
};
__global__ void __launch_bounds__(256) transpose_bytes2_kernel(const Transpose2Args a) {
    const uint32_t which = blockIdx.x >= a.tiles0 ? 1u : 0u, t = blockIdx.x - (which ? a.tiles0 : 0u);
    transpose_bytes_tile<true>(a.in[which], a.N[which], a.out[which], a.M[which], a.M[which], a.M[which], a.N[which],
                               t / a.tiles_n[which], t % a.tiles_n[which]);
}

// ---------------------------------------------------------------------------
// 2-byte transpose (matrix_transpose<bf16 / fp16>, src/transpose/transpose.cu:60-74; 16-bit operands
// stored K x N; packed operands).
// No LDS: a lane owns an 8 x 8 block.  It loads eight 16-byte row pieces, interleaves the 16-bit halves
// of vertically adjacent dwords (one v_perm each: 32 per block), and the rest of the transposition is
// which register goes into which output dword.  Lanes 8g..8g+7 hold eight neighbouring column blocks,
// so every load instruction reads 128-byte pieces of 8 rows; lanes g, g+8, .. hold neighbouring row
// blocks, so every store instruction writes 128-byte pieces of 8 output rows.  A wave covers 64 x 64
// elements, a workgroup of four waves 64 rows x 256 columns.
// ---------------------------------------------------------------------------
// ALIGNED: M and N multiples of 8, 16-byte aligned rows, Mout == M.  Otherwise any M, N, ld, pitch and element-aligned
// pointers (1999 x 3001, us: through LDS one element per lane 11.4; so, with a branch around every
// element of a row end 11.3, without 9.7): at a row's end the last whole piece is loaded and moved
// down, what sticks out of the output is stored in parts, the columns M .. Mout - 1 of the output are filled with zeros.
template <bool ALIGNED>
__device__ inline void transpose_u16_tile(const uint16_t *__restrict__ in, size_t ld, uint16_t *__restrict__ out, size_t pitch,
                                          uint32_t M, uint32_t Mout, uint32_t N, uint32_t tile_m, uint32_t tile_n) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef typename std::conditional<ALIGNED, v4i, v4i_any>::type vec_t;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t m = tile_m * 64 + (lane >> 3) * 8;                       // first of this lane's 8 rows
    const uint32_t n = tile_n * 256 + wave * 64 + (lane & 7) * 8;           // first of its 8 columns
    if (m >= Mout || n >= N) return;                                        // (aligned: blocks are wholly in or out)
    const bool cols = ALIGNED || n + 8 <= N, rows = ALIGNED || m + 8 <= Mout;
    v4i row[8];
    if constexpr (ALIGNED) {
        const uint16_t *src = in + (size_t)m * ld + n;
#pragma unroll
        for (int j = 0; j < 8; ++j) row[j] = *(const vec_t *)(src + (size_t)j * ld);
    } else if (N >= 8) {
        // (every lane loads, from the nearest row and, where its row ends inside the piece, the row's last eight elements, which it
        // moves down: no branch, in which each load would wait for the one before.)
        const uint16_t *src = in + (cols ? n : N - 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) row[j] = *(const vec_t *)(src + (size_t)(m + j < M ? m + j : M - 1) * ld);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (__any(!cols)) {
                uint32_t w[4] = {(uint32_t)row[j][0], (uint32_t)row[j][1], (uint32_t)row[j][2], (uint32_t)row[j][3]};
                move_down<4>(w, cols ? 0 : (n + 8 - N) * 2);
                row[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) row[j][k] = m + j < M ? row[j][k] : 0;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 7; ++e)
                if (m + j < M && n + e < N) w[e >> 1] |= (uint32_t)in[(size_t)(m + j) * ld + n + e] << (16 * (e & 1));
            row[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        }
    }
    // pair[i][k] = columns 2k (low perm) and 2k+1 (high perm) of rows 2i, 2i+1
    uint32_t lo[4][4], hi[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t a = (uint32_t)row[2 * i][k], b = (uint32_t)row[2 * i + 1][k];
            lo[i][k] = __builtin_amdgcn_perm(b, a, 0x05040100);     // (a.lo16, b.lo16)
            hi[i][k] = __builtin_amdgcn_perm(b, a, 0x07060302);     // (a.hi16, b.hi16)
        }
    uint16_t *dst = out + (size_t)n * pitch + m;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const v4i v = (k & 1) ? v4i{(int)hi[0][k >> 1], (int)hi[1][k >> 1], (int)hi[2][k >> 1], (int)hi[3][k >> 1]}
                              : v4i{(int)lo[0][k >> 1], (int)lo[1][k >> 1], (int)lo[2][k >> 1], (int)lo[3][k >> 1]};
        if (!cols && n + k >= N) break;
        if (rows) {
            *(vec_t *)(dst + (size_t)k * pitch) = v;
        } else {
            store_part(dst + (size_t)k * pitch, v, (Mout - m) * 2);
        }
    }
#endif
}

template <bool ALIGNED>
__global__ void __launch_bounds__(256) transpose_u16_kernel(const uint16_t *__restrict__ in, uint16_t *__restrict__ out,
                                                            uint32_t M, uint32_t N) {
    transpose_u16_tile<ALIGNED>(in, N, out, M, M, M, N, blockIdx.y, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Operands that the MFMA kernels cannot read as they stand (K bytes not a multiple of 16, rows or pointers that are not
// 16-byte aligned, B stored K x N with such rows): one launch brings one or both of them to rows of `pitch` bytes, K
// contiguous, zeros behind the last element up to the pitch (a multiple of 128), so that the whole of K is whole K steps.
// Bound by memory: every element is read and written once.  Loads are 16 bytes a lane at whatever address the row has
// (the vector memory path takes any byte address).
// ---------------------------------------------------------------------------
struct PackOperand {
    const char *src;
    char *dst;
    uint64_t ld;          // bytes between rows of the source (rows of the operand, or rows of k when k_major)
    uint32_t rows, k;     // of the operand, elements
    uint32_t pitch;       // bytes between rows of dst, a multiple of 128
    uint32_t k_major;     // the source is K x rows
    uint32_t blocks, tiles_k;      // workgroups of this operand; k_major: tiles along k (the slower index is the tile of rows)
    uint32_t inv;                  // inverse_of: k_major: tiles_k, else 16-byte pieces in a row of dst
};
struct PackArgs {
    PackOperand op[2];
};

// rows of the operand as they are: 16 bytes of dst per lane and turn, four turns per workgroup.  Every lane loads: a piece that
// reaches past the end of its row fetches the row's last 16 bytes and moves them down, one behind the end leaves zeros (rows of
// fewer than 16 bytes go element by element).  (Element by element behind branches, each load waited for the one before; with product,
// us: int8 2611 x 2104 x 3960 40.5 -> 36.2, 1531 x 4100 x 3004 36.2 -> 33.8, bf16 3001 x 1000 x 1999 with B stored K x N 34.4 -> 31.1.)
template <int ES>
__device__ inline void pack_rows(const PackOperand &o, uint32_t block) {
    const uint32_t per_row = o.pitch / 16, kbytes = o.k * ES;
    const uint32_t total = o.rows * per_row, first = block * 1024 + threadIdx.x;       // (the host keeps these below 2^32)
    v4i v[4];
    uint32_t at[4];
    const char *row[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t i = first + j * 256, r = div_by_inv(i < total ? i : total - 1, per_row, o.inv, at[j]);
        at[j] *= 16;
        row[j] = o.src + r * o.ld;
    }
    if (kbytes >= 16) {
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = *(const v4i_any *)(row[j] + (at[j] + 16 <= kbytes ? at[j] : kbytes - 16));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (!__any(at[j] + 16 > kbytes)) continue;
            uint32_t w[4] = {(uint32_t)v[j][0], (uint32_t)v[j][1], (uint32_t)v[j][2], (uint32_t)v[j][3]};
            move_down<4>(w, at[j] + 16 <= kbytes ? 0 : (at[j] < kbytes ? at[j] + 16 - kbytes : 16));
            v[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        }
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
            for (int e = 0; e < 16 / ES; ++e)
                if (at[j] + e * ES < kbytes) {
                    const uint32_t x = ES == 2 ? (uint32_t)((const uint16_t *)row[j])[e] : (uint32_t)((const uint8_t *)row[j])[e];
                    w[e * ES / 4] |= x << (8 * (e * ES % 4));
                }
            v[j] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t i = first + j * 256;
        if (i < total) *(v4i *)(o.dst + (size_t)i * 16) = v[j];          // (rows of dst follow each other without a gap)
    }
}

template <int ES>
__global__ void __launch_bounds__(256) pack_kernel(const PackArgs a) {
    const uint32_t which = blockIdx.x >= a.op[0].blocks ? 1u : 0u, block = blockIdx.x - (which ? a.op[0].blocks : 0u);
    const PackOperand &o = a.op[which];
    if (!o.k_major) {
        pack_rows<ES>(o, block);
        return;
    }
    uint32_t tk;
    const uint32_t tr = div_by_inv(block, o.tiles_k, o.inv, tk);
    if constexpr (ES == 2)
        transpose_u16_tile<false>((const uint16_t *)o.src, o.ld / 2, (uint16_t *)o.dst, o.pitch / 2, o.k, o.pitch / 2, o.rows, tk, tr);
    else
        transpose_bytes_tile<false>((const uint8_t *)o.src, o.ld, (uint8_t *)o.dst, o.pitch, o.k, o.pitch, o.rows, tk, tr);
}

// ---------------------------------------------------------------------------
// Split-K second pass: C[m,n] = cast(scale * sum_z part[z][m,n]), z ascending
// (a fixed order, so results do not depend on scheduling; int32 stays exact).
// ---------------------------------------------------------------------------
// Four elements of a row per thread, at any alignment (the last group of a row may be shorter), the loads of up to eight
// planes in flight together, then the sums in the order of the planes.  The launch is bound by latency, not by the
// 5 - 30 MB it reads: one element per thread with a dependent chain of loads took 4.2 us for 160 x 2048 in four planes,
// 11 us for 512 x 4096.
// part: [nsplit][M][N] f32 or i32; inv: inverse_of(groups of four in a row); scaled: the two scales are applied here.
// (Arguments of their own, not a struct: they arrive in scalar registers with the wave, see LaunchHead.)
template <bool IS_I32>
__global__ void __launch_bounds__(256)
splitk_reduce4_kernel(const void *part, void *C, const float *as, const float *bs, uint32_t M, uint32_t N, uint32_t nsplit,
                      uint32_t ldc, uint32_t inv, uint32_t out_dtype, uint32_t scaled) {
    typedef typename std::conditional<IS_I32, v4i, v4f>::type vec_t;
    typedef typename std::conditional<IS_I32, v4i_any, v4f_any>::type vec_any;
    typedef typename std::conditional<IS_I32, int, float>::type elem_t;
    const uint32_t per_row = (N + 3) / 4;
    const size_t plane = (size_t)M * N, total = (size_t)M * per_row, i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const float sa = scaled ? as[0] : 1.0f, sb = scaled ? bs[0] : 1.0f;
    uint32_t m, n;
    if (total >> 32) {
        m = (uint32_t)(i / per_row);
        n = (uint32_t)(i % per_row);
    } else {
        m = div_by_inv((uint32_t)i, per_row, inv, n);
    }
    n *= 4;
    const int valid = N - n < 4 ? (int)(N - n) : 4;
    const size_t idx = (size_t)m * ldc + n;
    const elem_t *src = (const elem_t *)part + (size_t)m * N + n;
    vec_t acc = vec_t{0, 0, 0, 0};
    if (valid == 4) {
        for (uint32_t z0 = 0; z0 < nsplit; z0 += 8) {
            vec_t t[8];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (z0 + j < nsplit) t[j] = __builtin_nontemporal_load((const vec_any *)(src + (size_t)(z0 + j) * plane));
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (z0 + j < nsplit) acc += t[j];
        }
    } else {
        for (uint32_t z = 0; z < nsplit; ++z)
            for (int e = 0; e < 3; ++e)
                if (e < valid) acc[e] += src[z * plane + e];
    }
    if constexpr (IS_I32) {
        if (out_dtype == (uint32_t)QGEMM_DT_I32) {
            int *dst = (int *)C + idx;
            if (valid == 4) *(v4i_any *)dst = acc;
            else
                for (int e = 0; e < valid; ++e) dst[e] = acc[e];
            return;
        }
    }
    const float s = sa * sb;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (float)acc[e] * s;
    store_out4(C, idx, v, (int)out_dtype, valid);
}

}  // namespace qgemm
