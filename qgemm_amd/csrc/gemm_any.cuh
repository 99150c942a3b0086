// The any-shape GEMM: operands at any address, with any distance between rows and any number of elements in them, read where
// they stand.  It asks for no memory but its operands: captured calls and calls on the static scratch, whose kernels may
// overlap with other users of the workspace, run it, as do products too small to be worth packing, fp8 operands (below), and
// whatever exceeds what the other kernels index.  int32 sums for int8, fp32 otherwise; block scales are folded in once per
// 128 elements of K as (P * as) * bs (hip_mix_gemm_kernel.cpp:231-244).
//
// fp8 operands are widened to bf16, which holds every e4m3 number, on their way into LDS: the bf16 matrix instructions add
// in fp32, the fp8 ones keep some 18 bits of the largest product of a step (relative error of a sum over K = 4096 normally
// distributed values: fp32 in sequence 7.1e-8, bf16 instructions 7.5e-8, fp8 ones, of 32 or 128 products, 1.4e-5).
//
// T x T tile, four waves of T/2 x T/2, two LDS buffers of one K step (128 bytes of K as the matrix cores take it).  The
// next step's operands are in flight to registers, 16 bytes a lane at whatever address the row has, while a step is
// computed.  Elements past K are zeroed in registers; rows past M or N repeat the last one and are not stored.
//
// What bounds it: the loads off 16-byte addresses, each of which asks for two cache lines (300 - 650 TFLOP/s; rows packed to
// whole lines reach two to four times that, packing included).  One thread per element, which this replaces / this
// kernel, us: fp8 to fp32 500 x 4608 x 7161 21 495 / 128; graph replays 1 x 1001 x 65 int8 5.5 / 3.9, 16 x 1001 x 33 bf16
// 4.0 / 3.7, 3 x 3 x 3 1.6 / 3.6 (the tail of the only row, byte by byte).
#pragma once
#include "gemm_mfma.cuh"

namespace qgemm {

struct AnyOperand {
    const char *p, *end;      // end: one past the last byte of the last row
    uint64_t ld;              // bytes between rows of the operand or, k_major, between rows of k
    uint32_t rows, k_major;
};
struct AnyArgs {
    AnyOperand a, b;
    void *C;
    const float *as, *bs;
    uint32_t K, tiles_m, tiles_n;
    uint64_t ldc;
    uint32_t as_ms, as_ks, bs_ns, bs_ks;
    int out_dtype, per_matrix_scale;
};

// BYTES bytes at any address, those from `end` on zeros and not read
template <int BYTES, int ES>
__device__ __forceinline__ void load_any(const char *p, const char *end, uint32_t *w) {
    if (p + BYTES <= end) {
        if constexpr (BYTES == 16) {
            const v4i v = *(const v4i_any *)p;
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = (uint32_t)v[i];
        } else if constexpr (BYTES == 8) {
            const v2i v = *(const v2i_any *)p;
            w[0] = (uint32_t)v[0];
            w[1] = (uint32_t)v[1];
        } else {
            w[0] = *(const u32_any *)p;
        }
        return;
    }
    const int left = (int)(end - p);
#pragma unroll
    for (int d = 0; d < BYTES / 4; ++d) {
        uint32_t x = 0;
        if (d * 4 < left) {
            if constexpr (ES == 2) {
                x = *(const uint16_t *)(p + d * 4);
                if (d * 4 + 2 < left) x |= (uint32_t) * (const uint16_t *)(p + d * 4 + 2) << 16;
            } else {
                x = *(const uint8_t *)(p + d * 4);
                if (d * 4 + 1 < left) x |= (uint32_t) * (const uint8_t *)(p + d * 4 + 1) << 8;
                if (d * 4 + 2 < left) x |= (uint32_t) * (const uint8_t *)(p + d * 4 + 2) << 16;
                if (d * 4 + 3 < left) x |= (uint32_t) * (const uint8_t *)(p + d * 4 + 3) << 24;
            }
        }
        w[d] = x;
    }
}

// four e4m3 values -> four bf16 values (exact; NaNs stay NaNs)
__device__ inline v2i widen_fp8(uint32_t w) {
    const f32x2_t lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false), hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
    return v2i{__builtin_bit_cast(int, __builtin_convertvector(lo, bf16x2_t)), __builtin_bit_cast(int, __builtin_convertvector(hi, bf16x2_t))};
}

// One operand of the tile.  LDS: T rows of 128 bytes, chunk c of row r in slot c ^ swz(r): fragment reads (16 rows, one chunk
// each) and the writes of a transposed block (rows 8 apart) both spread over the banks.
// KM: the operand may be K-major (AnyOperand::k_major says so); without, the code that transposes is left out.
template <int IN_DT, int T, bool KM>
struct AnyStage {
    static constexpr int ES = IN_DT == QGEMM_DT_I8 || IN_DT == QGEMM_DT_F8E4M3 ? 1 : 2;
    static constexpr bool WIDEN = IN_DT == QGEMM_DT_F8E4M3;
    static constexpr int KE = IN_DT == QGEMM_DT_I8 ? 128 : 64;                      // elements of K per step
    static constexpr int RB = KE * ES;                                              // ... in bytes of the source
    static constexpr int NR = T * RB / (16 * 256);                                  // 16-byte pieces a thread holds
    // K-major sources: a thread transposes blocks of KL rows of k x LB bytes
    static constexpr int KL = ES == 2 ? 2 : 4, LB = ES == 2 ? 16 : NR * 4, BLOCKS = NR * 16 / (KL * LB), ME = LB / ES;
    static_assert(NR >= 1 && BLOCKS >= 1 && BLOCKS * KL * LB == NR * 16, "");

    uint32_t w[NR * 4];

    __device__ static int slot(int r, int c) { return r * 128 + ((c ^ ((r ^ (r >> 3)) & 7)) << 4); }

    // block j of this thread: its first row of k and of the operand.  A wave takes 8 x 8 blocks, so that it reads 8 pieces in a row.
    __device__ static void block_at(int j, int &k, int &r) {
        constexpr int KQH = KE / KL / 8;
        const int i = threadIdx.x + j * 256, rest = i >> 6;
        k = ((rest % KQH) * 8 + (i & 7)) * KL;
        r = ((rest / KQH) * 8 + ((i >> 3) & 7)) * ME;
    }

    __device__ __forceinline__ void load(const AnyOperand &o, uint32_t row0, uint32_t k0, uint32_t K) {
        if (!KM || !o.k_major) {
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int i = threadIdx.x + j * 256, c = i % (RB / 16);
                const uint32_t r = i / (RB / 16), row = r < o.rows - row0 ? row0 + r : o.rows - 1;
                const int64_t left = (int64_t)(K - k0) * ES - c * 16;                // bytes of the row from here on
                uint32_t *v = w + j * 4;
                if (left > 0) {
                    load_any<16, ES>(o.p + row * o.ld + (uint64_t)k0 * ES + c * 16, o.end, v);
                } else {
                    v[0] = v[1] = v[2] = v[3] = 0;
                }
                if (left < 16) {
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const int n = (int)left - d * 4;
                        if (n < 4) v[d] &= n > 0 ? (1u << (8 * n)) - 1 : 0u;
                    }
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < BLOCKS; ++j) {
                int k, r;
                block_at(j, k, r);
#pragma unroll
                for (int e = 0; e < KL; ++e) {
                    uint32_t *v = w + (j * KL + e) * (LB / 4);
                    if ((uint32_t)r < o.rows - row0 && (uint32_t)(k + e) < K - k0) {
                        load_any<LB, ES>(o.p + (uint64_t)(k0 + k + e) * o.ld + (uint64_t)(row0 + r) * ES, o.end, v);
                    } else {
#pragma unroll
                        for (int d = 0; d < LB / 4; ++d) v[d] = 0;
                    }
                }
            }
        }
    }

    __device__ __forceinline__ void store(const AnyOperand &o, char *lds) const {
        if (!KM || !o.k_major) {
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const int i = threadIdx.x + j * 256, c = i % (RB / 16), r = i / (RB / 16);
                const uint32_t *v = w + j * 4;
                if constexpr (WIDEN) {
                    const v2i a = widen_fp8(v[0]), b = widen_fp8(v[1]), d = widen_fp8(v[2]), e = widen_fp8(v[3]);
                    *(v4i *)(lds + slot(r, 2 * c)) = v4i{a[0], a[1], b[0], b[1]};
                    *(v4i *)(lds + slot(r, 2 * c + 1)) = v4i{d[0], d[1], e[0], e[1]};
                } else {
                    *(v4i *)(lds + slot(r, c)) = v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
                }
            }
        } else {
#pragma unroll
            for (int j = 0; j < BLOCKS; ++j) {
                int k, r;
                block_at(j, k, r);
                const uint32_t *v = w + j * KL * (LB / 4);
                auto put = [&](int m, uint32_t x) { *(uint32_t *)(lds + slot(r + m, k * ES / 16) + k * ES % 16) = x; };
#pragma unroll
                for (int d = 0; d < LB / 4; ++d) {
                    // v_perm_b32: selector byte q picks byte q of the result out of {src1 bytes 0-3, src0 bytes 4-7}
                    if constexpr (ES == 2) {
                        const uint32_t a = v[d], b = v[LB / 4 + d];
                        put(2 * d, __builtin_amdgcn_perm(b, a, 0x05040100));
                        put(2 * d + 1, __builtin_amdgcn_perm(b, a, 0x07060302));
                    } else {
                        const uint32_t a = v[d], b = v[LB / 4 + d], c = v[2 * (LB / 4) + d], e = v[3 * (LB / 4) + d];
                        const uint32_t ab_lo = __builtin_amdgcn_perm(b, a, 0x05010400), ab_hi = __builtin_amdgcn_perm(b, a, 0x07030602);
                        const uint32_t ce_lo = __builtin_amdgcn_perm(e, c, 0x05010400), ce_hi = __builtin_amdgcn_perm(e, c, 0x07030602);
                        const uint32_t x[4] = {__builtin_amdgcn_perm(ce_lo, ab_lo, 0x05040100), __builtin_amdgcn_perm(ce_lo, ab_lo, 0x07060302),
                                               __builtin_amdgcn_perm(ce_hi, ab_hi, 0x05040100), __builtin_amdgcn_perm(ce_hi, ab_hi, 0x07060302)};
#pragma unroll
                        for (int m = 0; m < 4; ++m) {
                            if constexpr (WIDEN) *(v2i *)(lds + slot(r + 4 * d + m, k / 8) + k % 8 * 2) = widen_fp8(x[m]);
                            else put(4 * d + m, x[m]);
                        }
                    }
                }
            }
        }
    }
};

template <int IN_DT, bool BLOCK, int T, bool KM>
__global__ void __launch_bounds__(256, 2) gemm_any_kernel(const AnyArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef AnyStage<IN_DT, T, KM> S;
    constexpr int KE = S::KE, W = T / 2, F = W / 16;                    // wave tile W x W, F x F MFMA tiles
    constexpr bool I8 = IN_DT == QGEMM_DT_I8;
    typedef std::conditional_t<I8, v4i, v4f> part_t;
    typedef std::conditional_t<BLOCK, v4f, part_t> acc_t;
    __shared__ __attribute__((aligned(1024))) char lds[2][2][T * 128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = (wave >> 1) * W, wn = (wave & 1) * W;
    uint32_t tm, tn;
    tile_map(blockIdx.x, p.tiles_m, p.tiles_n, 8, tm, tn);
    const uint32_t row0 = __builtin_amdgcn_readfirstlane(tm) * T, col0 = __builtin_amdgcn_readfirstlane(tn) * T;
    const uint32_t steps = (p.K - 1) / KE + 1;
    auto mma = [](v4i x, v4i y, part_t c) {
        if constexpr (I8) return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, y, c, 0, 0, 0);
        else if constexpr (IN_DT == QGEMM_DT_F16)
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, x), __builtin_bit_cast(v8h, y), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, x), __builtin_bit_cast(v8bf, y), c, 0, 0, 0);
    };
    S sa, sb;
    acc_t acc[F][F];
    part_t part[F][F];
#pragma unroll
    for (int a = 0; a < F; ++a)
#pragma unroll
        for (int b = 0; b < F; ++b) {
            acc[a][b] = acc_t{0, 0, 0, 0};
            part[a][b] = part_t{0, 0, 0, 0};
        }
    sa.load(p.a, row0, 0, p.K);
    sb.load(p.b, col0, 0, p.K);
    sa.store(p.a, lds[0][0]);
    sb.store(p.b, lds[0][1]);
    for (uint32_t s = 0; s < steps; ++s) {
        if (s + 1 < steps) {
            sa.load(p.a, row0, (s + 1) * KE, p.K);
            sb.load(p.b, col0, (s + 1) * KE, p.K);
        }
        __syncthreads();                                                // buffer s & 1 is filled, the other one read
        const char *la = lds[s & 1][0], *lb = lds[s & 1][1];
        float as[F], bs;
        if constexpr (BLOCK) {
            const uint32_t kb = s * KE / kScaleBlock;
            bs = p.bs[(size_t)((col0 + wn) / kScaleBlock) * p.bs_ns + (size_t)kb * p.bs_ks];
#pragma unroll
            for (int a = 0; a < F; ++a) {
                const uint32_t r = wm + a * 16 + (lane & 15), m = r < p.a.rows - row0 ? row0 + r : p.a.rows - 1;
                as[a] = p.as[(size_t)m * p.as_ms + (size_t)kb * p.as_ks];
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            v4i fa[F], fb[F];
#pragma unroll
            for (int i = 0; i < F; ++i) {
                fa[i] = *(const v4i *)(la + S::slot(wm + i * 16 + (lane & 15), h * 4 + (lane >> 4)));
                fb[i] = *(const v4i *)(lb + S::slot(wn + i * 16 + (lane & 15), h * 4 + (lane >> 4)));
            }
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int b = 0; b < F; ++b) {
                    if constexpr (BLOCK) part[a][b] = mma(fb[b], fa[a], part[a][b]);
                    else acc[a][b] = mma(fb[b], fa[a], acc[a][b]);
                }
        }
        if (BLOCK && (I8 || (s & 1) || s + 1 == steps)) {               // 128 elements of K: one step of int8, two of fp8
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int b = 0; b < F; ++b) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[a][b][r] += ((float)part[a][b][r] * as[a]) * bs;
                    part[a][b] = part_t{0, 0, 0, 0};
                }
        }
        if (s + 1 < steps) {
            sa.store(p.a, lds[(s + 1) & 1][0]);
            sb.store(p.b, lds[(s + 1) & 1][1]);
        }
    }
    const float scale = p.per_matrix_scale ? p.as[0] * p.bs[0] : 1.0f;
#pragma unroll
    for (int a = 0; a < F; ++a) {
        const uint32_t m = wm + a * 16 + (lane & 15);
        if (m >= p.a.rows - row0) continue;
#pragma unroll
        for (int b = 0; b < F; ++b) {
            const uint32_t n = wn + b * 16 + (lane >> 4) * 4, left = p.b.rows - col0;
            if (n >= left) continue;
            const size_t idx = ((size_t)row0 + m) * p.ldc + col0 + n;
            const int valid = left - n < 4 ? (int)(left - n) : 4;
            if constexpr (I8 && !BLOCK) {
                if (p.out_dtype == QGEMM_DT_I32) {
                    int *dst = (int *)p.C + idx;
                    if (valid == 4) *(v4i_any *)dst = acc[a][b];
                    else
                        for (int r = 0; r < 3; ++r)
                            if (r < valid) dst[r] = acc[a][b][r];
                    continue;
                }
            }
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (float)acc[a][b][r] * scale;
            store_out4(p.C, idx, v, p.out_dtype, valid);
        }
    }
#endif
}

}  // namespace qgemm
