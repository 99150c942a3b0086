// The any-shape GEMM: operands at any address, with any distance between rows and any number of elements in them, read where
// they stand.  It asks for no memory but its operands: captured calls and calls on the static scratch, whose kernels may
// overlap with other users of the workspace, run it where the MFMA rows do not read their operands as they stand, as do small
// products, and whatever exceeds what the other kernels index.  int32 sums for int8, fp32 otherwise; block scales are folded in once per
// 128 elements of K as (P * as) * bs (hip_mix_gemm_kernel.cpp:231-244), in the form for few rows (gemm_few_kernel, at the end) as
// P * (as * bs), like the kernels for whole rows: two roundings either way.
//
// fp8 operands are widened to bf16, which holds every e4m3 number, on their way into LDS: the bf16 matrix instructions add
// in fp32, the fp8 ones keep some 18 bits of the largest product of a step (relative error of a sum over K = 4096 normally
// distributed values: fp32 in sequence 7.1e-8, bf16 instructions 7.5e-8, fp8 ones, of 32 or 128 products, 1.4e-5).
//
// T x T tile, four waves of T/2 x T/2, two LDS buffers of one K step (128 bytes of K as the matrix cores take it).  The
// operands of the next two steps are in flight to registers, 16 bytes a lane at whatever address the row has, while a step is
// computed.  A piece that would reach past the end of an operand is fetched from the last 16 bytes of it instead and moved
// down in registers, elements past K are zeroed there; rows past M or N repeat the last one and are not stored.
//
// What bounds it: the steps themselves, each with a barrier, fragments out of LDS and MFMAs in turn and two workgroups a CU
// to overlap them, and loads off cache lines that ask for two lines each.  1531 x 4100 x 3004 int8 42 us (900 TFLOP/s),
// 4096 x 4096 x 4001 bf16 191 (700), fp8 4096 x 4608 x 7161 357 (760).  (With a branch around the pieces at the end of an
// operand every load waited for the one before: 94, 473 and 413 us.)  One thread per element took 21 495 us for fp8 to fp32
// 500 x 4608 x 7161, this kernel 102.
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
    uint32_t K;
    TileMap map;
    uint64_t ldc;
    uint32_t as_ms, as_ks, bs_ns, bs_ks;
    int out_dtype, per_matrix_scale;
};

// BYTES (a power of two up to 16) bytes at any address
template <int BYTES>
__device__ __forceinline__ void load_any(const char *p, uint32_t *w) {
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

    // Where piece j of this thread comes from: never past the end of the operand, but moved back from there to the last
    // whole piece of it (`settle` moves the data down again).
    template <int BYTES>
    __device__ static const char *inside(const AnyOperand &o, const char *p) {
        return p + BYTES <= o.end ? p : o.end - BYTES;
    }
    __device__ static const char *row_piece(const AnyOperand &o, uint32_t row0, uint32_t k0, int j) {
        const int i = threadIdx.x + j * 256, c = i % (RB / 16);
        const uint32_t r = i / (RB / 16), row = r < o.rows - row0 ? row0 + r : o.rows - 1;
        return o.p + row * o.ld + (uint64_t)k0 * ES + c * 16;
    }
    __device__ static const char *k_piece(const AnyOperand &o, uint32_t row0, uint32_t k0, int j, int e) {
        int k, r;
        block_at(j, k, r);
        return o.p + ((uint64_t)k0 + k + e) * o.ld + ((uint64_t)row0 + r) * ES;
    }

    // (no branches but uniform ones and nothing that reads what has been loaded: all pieces are in flight together)
    __device__ __forceinline__ void load(const AnyOperand &o, uint32_t row0, uint32_t k0) {
        if (!KM || !o.k_major) {
#pragma unroll
            for (int j = 0; j < NR; ++j) load_any<16>(inside<16>(o, row_piece(o, row0, k0, j)), w + j * 4);
        } else {
#pragma unroll
            for (int j = 0; j < BLOCKS; ++j)
#pragma unroll
                for (int e = 0; e < KL; ++e) load_any<LB>(inside<LB>(o, k_piece(o, row0, k0, j, e)), w + (j * KL + e) * (LB / 4));
        }
    }

    // What a step that reaches past the end of K, or close to the end of the operand, has loaded: pieces moved back are
    // moved down again, elements past K become zeros.
    __device__ __forceinline__ void settle(const AnyOperand &o, uint32_t row0, uint32_t k0, uint32_t K) {
        if (!KM || !o.k_major) {
            if (K - k0 >= (uint32_t)KE) return;
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const char *p = row_piece(o, row0, k0, j);
                uint32_t *v = w + j * 4;
                move_down<4>(v, (uint32_t)(p - inside<16>(o, p)));
                const int left = (int)(K - k0) * ES - (threadIdx.x + j * 256) % (RB / 16) * 16;       // bytes of the row from here on
#pragma unroll
                for (int d = 0; d < 4; ++d) v[d] &= left >= 4 * d + 4 ? ~0u : left > 4 * d ? (1u << (8 * (left - 4 * d))) - 1 : 0u;
            }
        } else {
            if (o.p + ((uint64_t)k0 + KE - 1) * o.ld + ((uint64_t)row0 + T) * ES <= o.end) return;
#pragma unroll
            for (int j = 0; j < BLOCKS; ++j) {
                int k, r;
                block_at(j, k, r);
#pragma unroll
                for (int e = 0; e < KL; ++e) {
                    const char *p = k_piece(o, row0, k0, j, e);
                    uint32_t *v = w + (j * KL + e) * (LB / 4);
                    move_down<LB / 4>(v, (uint32_t)(p - inside<LB>(o, p)));
                    if ((uint32_t)(k + e) >= K - k0) {
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

// How the products of K are added up: in one chain of matrix instructions; in blocks of 128 elements of K from zero, folded into
// fp32 sums with their scales; or a step at a time from zero, added to fp32 sums.  The matrix instructions do not round to
// nearest, so a chain's error grows with its length, where the rows for few rows, which share K among waves, have eight short
// ones.  So 16-bit operands with fp32 output are folded on 64 x 64 tiles, into two sums in turn (relative error, bf16 to fp32,
// eight chains / one chain / one sum / two: 16 x 2048 x 1036 8.4e-8 / 18.4e-8 / 9.1e-8 / 7.8e-8, 64 x 7168 x 2060 10.4e-8 /
// 27.3e-8 / 11.7e-8 / 9.4e-8); on 128 x 128 tiles, where the other kernels have one chain too and more sums do not fit the
// registers, they are not.  A 16-bit output hides the difference.  Blocks of int8 alternate too (512 x 5000 x 3004 to fp32,
// other kernels / one sum / two: 7.5e-8 / 9.4e-8 / 7.4e-8).
enum AnySum : int { ANY_CHAIN = 0, ANY_SCALED = 1, ANY_FOLDED = 2 };

template <int IN_DT, int SUM, int T, bool KM>
__global__ void __launch_bounds__(256, 2) gemm_any_kernel(const AnyArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr bool BLOCK = SUM == ANY_SCALED;
    typedef AnyStage<IN_DT, T, KM> S;
    constexpr int KE = S::KE, W = T / 2, F = W / 16;                    // wave tile W x W, F x F MFMA tiles
    constexpr bool I8 = IN_DT == QGEMM_DT_I8;
    typedef std::conditional_t<I8, v4i, v4f> part_t;
    typedef std::conditional_t<BLOCK, v4f, part_t> acc_t;
    __shared__ __attribute__((aligned(1024))) char lds[2][2][T * 128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = (wave >> 1) * W, wn = (wave & 1) * W;
    uint32_t tm, tn;
    tile_map(blockIdx.x, p.map, tm, tn);
    const uint32_t row0 = tm * T, col0 = tn * T;
    const uint32_t steps = (p.K - 1) / KE + 1;
    auto mma = [](v4i x, v4i y, part_t c) {
        if constexpr (I8) return __builtin_amdgcn_mfma_i32_16x16x64_i8(x, y, c, 0, 0, 0);
        else if constexpr (IN_DT == QGEMM_DT_F16)
            return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, x), __builtin_bit_cast(v8h, y), c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, x), __builtin_bit_cast(v8bf, y), c, 0, 0, 0);
    };
    constexpr int SUMS = SUM == ANY_FOLDED || (BLOCK && I8) ? 2 : 1;    // one of the even and one of the odd steps
    acc_t sums[SUMS][F][F];
    auto &acc = sums[0];
    part_t part[F][F];
#pragma unroll
    for (int i = 0; i < SUMS; ++i)
#pragma unroll
        for (int a = 0; a < F; ++a)
#pragma unroll
            for (int b = 0; b < F; ++b) sums[i][a][b] = acc_t{0, 0, 0, 0};
    struct Stage {
        S a, b;
    } held[2];                                                          // of an even and of an odd step
    auto load = [&](uint32_t s, Stage &r) {
        if (s >= steps) return;
        r.a.load(p.a, row0, s * KE);
        r.b.load(p.b, col0, s * KE);
    };
    auto store = [&](uint32_t s, Stage &r) {
        if (s >= steps) return;
        r.a.settle(p.a, row0, s * KE, p.K);
        r.b.settle(p.b, col0, s * KE, p.K);
        r.a.store(p.a, lds[s & 1][0]);
        r.b.store(p.b, lds[s & 1][1]);
    };
    // step s: `own` brought it and is free, `next` holds step s + 1
    auto turn = [&](uint32_t s, auto odd, Stage &own, Stage &next) {
        load(s + 2, own);
        __syncthreads();                                                // buffer s & 1 is filled, the other one read
        const char *la = lds[odd][0], *lb = lds[odd][1];
        constexpr bool FIRST = I8 || !odd;                              // of a K block: 128 elements are one step of int8, two of fp8
        float f[F];
        if (BLOCK && (I8 || odd || s + 1 == steps)) {
            const uint32_t kb = s * KE / kScaleBlock;
            const float bs = p.bs[(size_t)((col0 + wn) / kScaleBlock) * p.bs_ns + (size_t)kb * p.bs_ks];
#pragma unroll
            for (int a = 0; a < F; ++a) {
                const uint32_t r = wm + a * 16 + (lane & 15), m = r < p.a.rows - row0 ? row0 + r : p.a.rows - 1;
                f[a] = p.as[(size_t)m * p.as_ms + (size_t)kb * p.as_ks] * bs;
            }
        }
        auto frag = [&](const char *l, int r, int h) { return *(const v4i *)(l + S::slot(r + (lane & 15), h * 4 + (lane >> 4))); };
        if constexpr (SUM == ANY_FOLDED) {
            v4i fb[2][F];
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int h = 0; h < 2; ++h) fb[h][i] = frag(lb, wn + i * 16, h);
#pragma unroll
            for (int a = 0; a < F; ++a) {
                const v4i fa0 = frag(la, wm + a * 16, 0), fa1 = frag(la, wm + a * 16, 1);
                part_t q[F];
#pragma unroll
                for (int b = 0; b < F; ++b) q[b] = mma(fb[0][b], fa0, part_t{0, 0, 0, 0});
#pragma unroll
                for (int b = 0; b < F; ++b) q[b] = mma(fb[1][b], fa1, q[b]);
#pragma unroll
                for (int b = 0; b < F; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sums[odd][a][b][r] += q[b][r];
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v4i fa[F], fb[F];
#pragma unroll
                for (int i = 0; i < F; ++i) {
                    fa[i] = frag(la, wm + i * 16, h);
                    fb[i] = frag(lb, wn + i * 16, h);
                }
#pragma unroll
                for (int a = 0; a < F; ++a)
#pragma unroll
                    for (int b = 0; b < F; ++b) {
                        if constexpr (BLOCK) part[a][b] = mma(fb[b], fa[a], FIRST && h == 0 ? part_t{0, 0, 0, 0} : part[a][b]);
                        else acc[a][b] = mma(fb[b], fa[a], acc[a][b]);
                    }
            }
        }
        if (BLOCK && (I8 || odd || s + 1 == steps)) {
#pragma unroll
            for (int a = 0; a < F; ++a)
#pragma unroll
                for (int b = 0; b < F; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sums[SUMS == 2 && odd][a][b][r] += (float)part[a][b][r] * f[a];
        }
        store(s + 1, next);
    };
    load(0, held[0]);
    load(1, held[1]);
    store(0, held[0]);
    for (uint32_t s = 0; s < steps; s += 2) {
        turn(s, std::integral_constant<int, 0>{}, held[0], held[1]);
        if (s + 1 < steps) turn(s + 1, std::integral_constant<int, 1>{}, held[1], held[0]);
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
            for (int r = 0; r < 4; ++r) v[r] = (float)(SUMS == 2 ? acc[a][b][r] + sums[SUMS - 1][a][b][r] : acc[a][b][r]) * scale;
            store_out4(p.C, idx, v, p.out_dtype, valid);
        }
    }
#endif
}

// Few rows: the plan of the skinny-M kernel (gemm_skinny.cuh) on operands at any address.  16 TM rows x 32 columns a workgroup,
// the K steps of 128 bytes dealt to its eight waves in turn, two in flight a wave; nothing is shared until the eight partial sums
// meet in LDS, added in wave order.  The pieces travel through registers, where the last step's are moved and cut (as in
// AnyStage), to the wave's own corner of LDS and from there to the fragments: no barrier in the loop.
// Bound by latency, hence by bytes in flight: 12 KiB a wave and 96 a workgroup, where the kernel above has 16 KiB a workgroup and
// half as many of them.  Up to 16 rows two workgroups share a CU (128 registers a lane; widened blocks of fp8 need more).  us, graph
// replays, kernel above / this: fp8 block scales 16 x 1152 x 4475 39.2 / 9.2, 16 x 7168 x 8001 82.0 / 21.4 (2.7 TB/s), 48 x 4096 x 2001
// 21.6 / 8.6; int8 17 x 1152 x 4475 21.9 / 9.5, bf16 1 x 1176 x 2561 23.8 / 7.1.
template <int ARITH, bool BLOCK, int TM>
__global__ void __launch_bounds__(512, TM == 1 && !(BLOCK && ARITH == AR_F8W) ? 4 : 2) gemm_few_kernel(const AnyArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int TN = 2, NW = 8, PA = 2 * TM, PB = 2 * TN, ES = ARITH == AR_BF16 || ARITH == AR_F16 ? 2 : 1;
    constexpr int AREA = (PA + PB) * 1024;                               // of one step, a wave's own
    static_assert(TM * TN * 1024 <= AREA && NW * AREA <= 65536, "");
    __shared__ __attribute__((aligned(1024))) char lds[NW * AREA];
    typedef typename AccT<ARITH>::type part_t;
    typedef std::conditional_t<BLOCK, v4f, part_t> acc_t;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t row0 = blockIdx.y * (16 * TM), col0 = blockIdx.x * (16 * TN);
    const uint32_t kbytes = p.K * ES, steps = (kbytes + 127) / 128;
    // piece j of a step: rows 8 j .. 8 j + 7, lane l's 16 bytes of row l >> 3 in slot l (rotated by the row: lds_slot)
    const uint32_t chunk = (((lane & 7) - (lane >> 3)) & 7) * 16;
    const char *pa[PA], *pb[PB];
    auto first = [&](const AnyOperand &o, uint32_t r) { return o.p + (r < o.rows ? r : o.rows - 1) * o.ld + chunk; };
#pragma unroll
    for (int j = 0; j < PA; ++j) pa[j] = first(p.a, row0 + 8 * j + (lane >> 3));
#pragma unroll
    for (int j = 0; j < PB; ++j) pb[j] = first(p.b, col0 + 8 * j + (lane >> 3));
    auto inside = [](const AnyOperand &o, const char *q) { return q + 16 <= o.end ? q : o.end - 16; };
    v4i ra[2][PA], rb[2][PB];
    float as[2][TM], bs[2];
    auto load = [&](uint32_t k) {                                        // steps k and k + 8
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const uint32_t kt = k + s * NW;
            if (kt >= steps) return;
#pragma unroll
            for (int j = 0; j < PB; ++j) rb[s][j] = *(const v4i_any *)inside(p.b, pb[j] + (size_t)kt * 128);
#pragma unroll
            for (int j = 0; j < PA; ++j) ra[s][j] = *(const v4i_any *)inside(p.a, pa[j] + (size_t)kt * 128);
            if constexpr (BLOCK) {
#pragma unroll
                for (int a = 0; a < TM; ++a) {
                    const uint32_t m = row0 + a * 16 + (lane & 15);
                    as[s][a] = p.as[(size_t)(m < p.a.rows ? m : p.a.rows - 1) * p.as_ms + (size_t)kt * p.as_ks];
                }
                bs[s] = p.bs[(size_t)(col0 / kScaleBlock) * p.bs_ns + (size_t)kt * p.bs_ks];
            }
        }
    };
    auto settle = [&](const AnyOperand &o, const char *q, uint32_t kt, v4i &r) {
        uint32_t w[4] = {(uint32_t)r[0], (uint32_t)r[1], (uint32_t)r[2], (uint32_t)r[3]};
        q += (size_t)kt * 128;
        move_down<4>(w, (uint32_t)(q - inside(o, q)));
        const int left = (int)(kbytes - kt * 128) - (int)chunk;          // bytes of the row from here on
#pragma unroll
        for (int d = 0; d < 4; ++d) w[d] &= left >= 4 * d + 4 ? ~0u : left > 4 * d ? (1u << (8 * (left - 4 * d))) - 1 : 0u;
        r = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    };
    char *mine = lds + wave * AREA;
    const int off0 = lds_slot(lane & 15, lane >> 4) * 16, off1 = lds_slot(lane & 15, 4 + (lane >> 4)) * 16;
    acc_t acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = acc_t{0, 0, 0, 0};
    v4i fa[TM][2], fb[TN][2];
    float f[TM];
    auto turn = [&](int s, uint32_t kt) {                                // the pieces of step kt to fragments
        if ((kt + 1) * 128 > kbytes) {
#pragma unroll
            for (int j = 0; j < PA; ++j) settle(p.a, pa[j], kt, ra[s][j]);
#pragma unroll
            for (int j = 0; j < PB; ++j) settle(p.b, pb[j], kt, rb[s][j]);
        }
#pragma unroll
        for (int j = 0; j < PA; ++j) *(v4i *)(mine + j * 1024 + lane * 16) = ra[s][j];
#pragma unroll
        for (int j = 0; j < PB; ++j) *(v4i *)(mine + (PA + j) * 1024 + lane * 16) = rb[s][j];
#pragma unroll
        for (int a = 0; a < TM; ++a) {
            fa[a][0] = *(const v4i *)(mine + a * 2048 + off0);
            fa[a][1] = *(const v4i *)(mine + a * 2048 + off1);
            if constexpr (BLOCK) f[a] = as[s][a] * bs[s];
        }
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            fb[b][0] = *(const v4i *)(mine + (TM + b) * 2048 + off0);
            fb[b][1] = *(const v4i *)(mine + (TM + b) * 2048 + off1);
        }
    };
    auto compute = [&]() {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b) {
                if constexpr (BLOCK) {
                    const part_t q = mma128<ARITH>(fb[b][0], fb[b][1], fa[a][0], fa[a][1], part_t{0, 0, 0, 0});
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[a][b][r] += (float)q[r] * f[a];
                } else {
                    acc[a][b] = mma128<ARITH>(fb[b][0], fb[b][1], fa[a][0], fa[a][1], acc[a][b]);
                }
            }
    };
    load(wave);
    const float scale = !BLOCK && p.per_matrix_scale ? p.as[0] * p.bs[0] : 1.0f;
    for (uint32_t k = wave; k < steps; k += 2 * NW) {
        const bool two = k + NW < steps;
        turn(0, k);
        compute();
        if (two) turn(1, k + NW);
        if (k + 2 * NW < steps) load(k + 2 * NW);
        if (two) compute();
    }
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) *(acc_t *)(mine + (a * TN + b) * 1024 + lane * 16) = acc[a][b];
    __syncthreads();
    if (wave >= TM * TN) return;
    acc_t sum = *(const acc_t *)(lds + wave * 1024 + lane * 16);
#pragma unroll
    for (int w = 1; w < NW; ++w) {
        const acc_t o = *(const acc_t *)(lds + w * AREA + wave * 1024 + lane * 16);
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] += o[r];
    }
    const uint32_t m = row0 + wave / TN * 16 + (lane & 15), n = col0 + wave % TN * 16 + (lane >> 4) * 4;
    if (m >= p.a.rows || n >= p.b.rows) return;
    const size_t idx = (size_t)m * p.ldc + n;
    const int valid = p.b.rows - n < 4 ? (int)(p.b.rows - n) : 4;
    if constexpr (ARITH == AR_I8 && !BLOCK) {
        if (p.out_dtype == QGEMM_DT_I32) {
            int *dst = (int *)p.C + idx;
            if (valid == 4) *(v4i_any *)dst = sum;
            else
                for (int r = 0; r < 3; ++r)
                    if (r < valid) dst[r] = sum[r];
            return;
        }
    }
    float v[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = (float)sum[r] * scale;
    store_out4(p.C, idx, v, p.out_dtype, valid);
#endif
}

// One thread per element of C, for fewer than 16 elements of K: an operand may then be shorter than one load of the kernel
// above, and where all of it is small a few loads of single elements are done first (graph replays, this / that, us:
// 3 x 3 x 3 bf16 1.6 / 3.6).  One K block at most, folded as above.
template <int IN_DT, bool BLOCK>
__global__ void __launch_bounds__(256) gemm_short_kernel(const AnyArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    const uint32_t n = (uint32_t)(i % p.b.rows);
    const uint64_t m = i / p.b.rows;
    if (m >= p.a.rows) return;
    auto element = [](const AnyOperand &o, uint64_t row, uint32_t k) {
        constexpr int ES = IN_DT == QGEMM_DT_I8 || IN_DT == QGEMM_DT_F8E4M3 ? 1 : 2;
        const char *q = o.p + (o.k_major ? k * o.ld + row * ES : row * o.ld + (uint64_t)k * ES);
        if constexpr (IN_DT == QGEMM_DT_I8) return (int)*(const int8_t *)q;
        else if constexpr (IN_DT == QGEMM_DT_F8E4M3) return __builtin_amdgcn_cvt_f32_fp8((int)*(const uint8_t *)q, 0);
        else if constexpr (IN_DT == QGEMM_DT_BF16) return __builtin_bit_cast(float, (uint32_t) * (const uint16_t *)q << 16);
        else return (float)*(const _Float16 *)q;
    };
    std::conditional_t<IN_DT == QGEMM_DT_I8, int, float> sum = 0;
    for (uint32_t k = 0; k < p.K; ++k) sum += element(p.a, m, k) * element(p.b, n, k);
    const uint64_t idx = m * p.ldc + n;
    if (IN_DT == QGEMM_DT_I8 && !BLOCK && p.out_dtype == QGEMM_DT_I32) {
        ((int *)p.C)[idx] = (int)sum;
        return;
    }
    float f = p.per_matrix_scale ? p.as[0] * p.bs[0] : 1.0f;
    if (BLOCK) f = p.as[m * p.as_ms] * p.bs[(size_t)(n / kScaleBlock) * p.bs_ns];
    const float v[4] = {(float)sum * f, 0, 0, 0};
    store_out4(p.C, idx, v, p.out_dtype, 1);
#endif
}

}  // namespace qgemm
