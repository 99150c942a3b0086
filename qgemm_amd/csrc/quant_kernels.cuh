// Quantisers: the Q_A / Q_B of C = (A o Q_A) x (B o Q_B) (README.md:1 of the reference, which implements none).
//   per matrix     s = max|x| / 127 (int8) or / 448 (fp8 e4m3);  q = round(x / s), saturated
//   1 x 128 blocks  one scale per row and 128 columns      (the a_scale of hip_mix_gemm_kernel.cpp:149)
//   128 x 128       one scale per 128 x 128 block          (the b_scale of hip_mix_gemm_kernel.cpp:137,164)
// A block (or matrix) of zeros gets s = 1.  x / s is a true division and the rounding is to nearest even,
// so the results are the bits the CPU quantisers give.
//
// What bounds them: memory, once the instructions per element are few.  16-bit input leaves 1.2 ns per element and CU at
// the rate a copy reaches, a dozen vector instructions; element by element, with a test for NaN, infinity and zero and a
// clamp around every quotient, it took 25 and the 1 x 128 quantiser of bf16 ran at 2.9 TB/s.  So:
//   * a lane works on pieces of 16 bytes (8 16-bit or 4 fp32 elements), at any address, a row's end out of its last whole piece;
//   * maxima are integer maxima of the bits without the sign (two at a time for 16-bit input): the order of the numbers,
//     with infinities and NaNs on top, so that one look at a block's maximum tells whether the plain form below will do;
//   * plain form (a finite maximum: no element is NaN or infinite, no quotient exceeds the type's largest value): the
//     quotient of |x| without special cases, the sign moved over afterwards; anything else takes the careful form.
// Before and now, us (to fp8 unless said): 1 x 128 6144 x 7168 bf16 45.7 -> 25.7 (5.1 TB/s, what a copy reaches), 500 x 7200
// 7.3 -> 4.5; 128 x 128 7168 x 6144 fp32 43.4 -> 39.6 (5.6 TB/s); per matrix 1531 x 3004 bf16 to int8 4.9 + 8.5 -> 4.0 + 5.5
// (a trace's times of the two passes; as a graph 11.3 -> 8.5).  A decoder's one row of 2048 1.98 -> 1.85: one trip to memory and back.
#pragma once
#include "common.h"

namespace qgemm {

struct QuantArgs {
    const void *x;        // rows x cols, row stride ld elements
    void *q;              // rows x cols bytes, row stride ldq
    float *scales;        // per matrix: 1 float; blocks: scales[ib*scale_rs + jb*scale_cs]
    uint32_t *partial;    // per matrix: one partial maximum per workgroup of the first pass (bits of |x|; bit 31: NaNs seen)
    uint32_t rows, cols, npartial;
    uint64_t ld, ldq, scale_rs, scale_cs;
    // Work is numbered along rows in units of a piece (per matrix) or of a 1 x 128 block: `per_row` of them in a row,
    // inv = inverse_of(per_row).  blockIdx.y counts slices of rows_per_slice rows, so that a number fits 32 bits.
    uint32_t per_row, inv, rows_per_slice;
    uint32_t share, set, tag, wait; // quant_whole_matrix_kernel: whole pieces of a workgroup; where, under which number and for how long
                                    // (ticks of the 100 MHz clock) maxima meet
};

// What the kernels start with, in front of QuantArgs: arguments of their own arrive in scalar registers with the wave (kernarg
// preloading, see LaunchHead), fields of a struct are a trip to memory in front of the first load.
#define QGEMM_QUANT_HEAD                                                                                                  \
    const void *x, void *q, float *scales, uint64_t ld, uint32_t rows_all, uint32_t cols, uint32_t per_row, uint32_t inv, \
        uint32_t rows_per_slice
#define QGEMM_QUANT_HEAD_OF(a) (a).x, (a).q, (a).scales, (a).ld, (a).rows, (a).cols, (a).per_row, (a).inv, (a).rows_per_slice, a

// ---- 16 bytes of input
template <int IN_DT>
struct Piece {
    static constexpr int ES = IN_DT == QGEMM_DT_F32 ? 4 : 2, VEC = 16 / ES;
    static constexpr int LANES = kScaleBlock / VEC;                  // lanes that cover the 128 columns of a block
    static constexpr uint32_t INF = IN_DT == QGEMM_DT_F32 ? 0x7F800000u : (IN_DT == QGEMM_DT_BF16 ? 0x7F80u : 0x7C00u);

    __device__ static float element(uint32_t bits) {
        if constexpr (IN_DT == QGEMM_DT_F32) return __builtin_bit_cast(float, bits);
        else if constexpr (IN_DT == QGEMM_DT_BF16) return __builtin_bit_cast(float, bits << 16);
        else return (float)__builtin_bit_cast(_Float16, (unsigned short)bits);
    }
    // Elements idx .. idx + VEC - 1 of a row that has `valid` of them left.  Where the row ends inside the piece load_whole fetches
    // the last whole piece of the row instead, and `settle` moves its end down and leaves zeros behind it: nothing waits and
    // nothing branches between the loads of a lane.  (Element by element behind a branch each, every load waited for the one
    // before: 128 x 128 blocks of 500 x 7195 bf16 11.3 us, 7.0 so, 1 x 128 5.3 and 4.7, per matrix 9.9 and 8.3.)  Rows of fewer than VEC elements: load_elements.
    __device__ static v4i load_whole(const void *base, size_t idx, uint32_t valid) {
        return *(const v4i_any *)((const char *)base + idx * ES - (valid ? missing(valid) * ES : 0));
    }
    __device__ static v4i load_elements(const void *base, size_t idx, uint32_t valid) {          // (valid: 1 or more)
        const char *p = (const char *)base + idx * ES;
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll 1
        for (uint32_t e = valid; e-- > 0;) {
#pragma unroll
            for (int i = 3; i > 0; --i) w[i] = ES == 4 ? w[i - 1] : (w[i] << 16 | w[i - 1] >> 16);
            if constexpr (ES == 4) w[0] = ((const uint32_t *)p)[e];
            else w[0] = w[0] << 16 | ((const uint16_t *)p)[e];
        }
        return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
    // RAGGED: the row may end inside a piece
    template <bool RAGGED>
    __device__ static v4i load(const void *base, size_t idx, uint32_t valid, bool wide) {
        if constexpr (!RAGGED) return *(const v4i_any *)((const char *)base + idx * ES);
        else return wide ? load_whole(base, idx, valid) : load_elements(base, idx, valid);
    }
    // element e + 1 to where element e is
    __device__ static void next_element(v4i &r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t up = i < 3 ? (uint32_t)r[i < 3 ? i + 1 : 3] : 0u, at = (uint32_t)r[i];
            r[i] = (int)(ES == 4 ? up : (at >> 16 | up << 16));
        }
    }
    __device__ static uint32_t missing(uint32_t valid) { return valid < (uint32_t)VEC ? VEC - valid : 0; }
    __device__ static void settle(v4i &r, uint32_t valid) {
        if (!__any(valid != 0 && valid < (uint32_t)VEC)) return;
        uint32_t w[4] = {(uint32_t)r[0], (uint32_t)r[1], (uint32_t)r[2], (uint32_t)r[3]};
        move_down<4, ES == 4>(w, valid ? missing(valid) * ES : 0);
        r = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
    __device__ static uint32_t bits(v4i r, int e) {
        if constexpr (ES == 4) return (uint32_t)r[e];
        else return ((uint32_t)r[e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
    }
    // bits of the largest |x| of the piece, NaNs above everything
    __device__ static uint32_t max_bits(v4i r) {
        if constexpr (ES == 4) {
            const uint32_t k = 0x7FFFFFFFu, a = r[0] & k, b = r[1] & k, c = r[2] & k, d = r[3] & k;
            const uint32_t m = a > b ? a : b, n = c > d ? c : d;
            return m > n ? m : n;
        } else {
            typedef unsigned short us2 __attribute__((ext_vector_type(2)));
            auto h = [&](int i) { return __builtin_bit_cast(us2, (uint32_t)r[i] & 0x7FFF7FFFu); };
            const us2 m = __builtin_elementwise_max(__builtin_elementwise_max(h(0), h(1)), __builtin_elementwise_max(h(2), h(3)));
            const uint32_t u = __builtin_bit_cast(uint32_t, m), hi = u >> 16, lo = u & 0xFFFFu;
            return hi > lo ? hi : lo;
        }
    }
    // acc = the larger |x| of acc and r, element by element; max_bits(acc) is the maximum in the end
    __device__ static void fold_max(v4i &acc, v4i r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (ES == 4) {
                const uint32_t b = (uint32_t)r[i] & 0x7FFFFFFFu;
                acc[i] = (int)(b > (uint32_t)acc[i] ? b : (uint32_t)acc[i]);
            } else {
                typedef unsigned short us2 __attribute__((ext_vector_type(2)));
                const uint32_t old = (uint32_t)acc[i], bits = (uint32_t)r[i] & 0x7FFF7FFFu;
                acc[i] = __builtin_bit_cast(int, __builtin_elementwise_max(__builtin_bit_cast(us2, old), __builtin_bit_cast(us2, bits)));
            }
        }
    }
    // max_bits over the elements that are numbers
    __device__ static uint32_t max_bits_of_numbers(v4i r) {
        // (rolled, an element a turn out of the low bits: unrolled and hoisted out of its rare branch it took up to 235 registers of
        // the kernels that hold several pieces, and with them the waves that keep memory busy: 128 x 128 blocks of 6144 x 7168
        // fp16 95.7 us, 27.8 with this and the loads of quant_square_block_kernel)
        uint32_t m = 0;
#pragma unroll 1
        for (int e = 0; e < VEC; ++e) {
            const uint32_t b = (uint32_t)r[0] & (ES == 4 ? 0x7FFFFFFFu : 0x7FFFu);
            if (b <= INF && b > m) m = b;
            next_element(r);
        }
        return m;
    }
};

// e4m3 (OCP): saturate to +-448, then round to nearest even; NaN -> 0x7F with the sign kept.
__device__ inline uint32_t f32_to_fp8_careful(float a) {
    if (a != a) return 0x7Fu | ((__builtin_bit_cast(uint32_t, a) >> 24) & 0x80u);
    const float c = __builtin_fminf(__builtin_fmaxf(a, -448.0f), 448.0f);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, c, 0, false) & 0xFFu;
}

__device__ inline uint32_t f32_to_i8_careful(float v) {
    float r = __builtin_rintf(v);                 // ties to even
    r = r > 127.0f ? 127.0f : r;
    r = r < -127.0f ? -127.0f : r;
    return (uint32_t)(int)r & 0xFFu;              // NaN: the comparisons are false, the cast gives 0
}

// x / s for many x and one s (a scale: positive).  The compiler expands every fp32 division into a
// reciprocal, two refinements of it and three of the quotient, all on values scaled by v_div_scale so that nothing
// leaves the normal range.  With s between 2^-60 and 2^60 and |x| at most a few hundred s (the quantisers divide by
// max|x| / 448 or / 127) that scaling is the identity unless the quotient is below 2^-100, which every output type
// here turns into a zero of the quotient's sign whatever its low bits: so the reciprocal is refined once per scale
// and the quotient steps are the same fused multiply-adds on the same values: the same bits as x / s, about half
// the instructions per element.  (A zero comes out as +0: the callers carry the sign.)
struct Divisor {
    float s, r;
    bool plain;           // the quotients may take the short way: s in range and every x finite
};
__device__ inline Divisor make_divisor(float s, bool finite) {
    Divisor d;
    d.s = s;
    d.plain = finite && s >= 0x1p-60f && s <= 0x1p60f;
    const float r0 = __builtin_amdgcn_rcpf(s);
    d.r = __builtin_fmaf(__builtin_fmaf(-s, r0, 1.0f), r0, r0);
    return d;
}
__device__ inline float div_plain(float x, const Divisor &d) {
    float q = x * d.r;
    q = __builtin_fmaf(__builtin_fmaf(-d.s, q, x), d.r, q);
    return __builtin_fmaf(__builtin_fmaf(-d.s, q, x), d.r, q);
}

// the VEC quantised bytes of a piece, element 0 in the low byte of component 0
template <int IN_DT, int OUT_DT>
__device__ inline v2i quant_piece(v4i r, const Divisor &dv) {
    typedef Piece<IN_DT> P;
    uint32_t w[2] = {0, 0};
    asm volatile("" : "+v"(r));             // (a piece at a time: nothing of the next pieces' conversions moves in front of this one)
    if (dv.plain) {
#pragma unroll
        for (int h = 0; h < P::VEC / 4; ++h) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = P::element(P::bits(r, 4 * h + e));
            if constexpr (OUT_DT == QGEMM_DT_F8E4M3) {
                // |x| / s is at most 448 and half an ulp: it rounds to at most 448
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float q = div_plain(__builtin_fabsf(v[e]), dv);
                    v[e] = P::ES == 4 ? __builtin_copysignf(q, v[e]) : q;
                }
                uint32_t p = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
                p = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], (int)p, true);
                if constexpr (P::ES == 2)        // the four sign bits at once, out of the high bytes of the elements
                    p |= __builtin_amdgcn_perm((uint32_t)r[2 * h + 1], (uint32_t)r[2 * h], 0x07050301) & 0x80808080u;
                w[h] = p;
            } else {
                // adding 1.5 * 2^23 rounds to the nearest integer, ties to even, and leaves it in the low byte; |x| / s is
                // at most 127 and half an ulp
                uint32_t b[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) b[e] = __builtin_bit_cast(uint32_t, div_plain(v[e], dv) + 12582912.0f);
                const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0C0C0400), hi = __builtin_amdgcn_perm(b[3], b[2], 0x0C0C0400);
                w[h] = lo | (hi << 16);
            }
        }
    } else {
        // (an element a turn out of the low bits)
#pragma unroll 1
        for (int e = 0; e < P::VEC; ++e) {
            const float v = P::element(P::ES == 4 ? (uint32_t)r[0] : (uint32_t)r[0] & 0xFFFFu) / dv.s;
            const uint32_t q = OUT_DT == QGEMM_DT_F8E4M3 ? f32_to_fp8_careful(v) : f32_to_i8_careful(v);
            if constexpr (P::ES == 4) {
                w[0] = w[0] >> 8 | q << 24;
            } else {
                w[0] = w[0] >> 8 | w[1] << 24;
                w[1] = w[1] >> 8 | q << 24;
            }
            P::next_element(r);
        }
    }
    return v2i{(int)w[0], (int)w[1]};
}

template <int IN_DT>
__device__ inline void store_piece(void *q, size_t idx, v2i w, uint32_t valid) {
    uint8_t *p = (uint8_t *)q + idx;
    if (valid >= (uint32_t)Piece<IN_DT>::VEC) {
        if constexpr (Piece<IN_DT>::VEC == 8) *(v2i_any *)p = w;
        else *(u32_any *)p = (uint32_t)w[0];
        return;
    }
    uint32_t b = (uint32_t)w[0];                                  // the parts of 4, 2 and 1 bytes that the row still has
    if (valid & 4) {
        *(u32_any *)p = b;
        p += 4;
        b = (uint32_t)w[1];
    }
    if (valid & 2) {
        *(u16_any *)p = (uint16_t)b;
        p += 2;
        b >>= 16;
    }
    if (valid & 1) *p = (uint8_t)b;
}

// maximum over groups of 16, 32 or 64 neighbouring lanes, in every lane, on the vector ALU alone: lane exchanges inside a
// row of 16 ride on the max instruction (DPP), rows are exchanged with lane swaps.  (Every __shfl_xor is a trip through
// the LDS crossbar with its address arithmetic.)
template <int LANES>
__device__ inline uint32_t lanes_max(uint32_t m) {
    auto with = [&](uint32_t o) { m = o > m ? o : m; };
    auto dpp = [&](auto ctrl) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, decltype(ctrl)::value, 0xF, 0xF, true); };
    with(dpp(std::integral_constant<int, 0xB1>{}));      // quad_perm [1,0,3,2]: lane ^ 1
    with(dpp(std::integral_constant<int, 0x4E>{}));      // quad_perm [2,3,0,1]: lane ^ 2
    with(dpp(std::integral_constant<int, 0x141>{}));     // row_half_mirror: lane -> 7 - lane within 8
    with(dpp(std::integral_constant<int, 0x140>{}));     // row_mirror: lane -> 15 - lane within 16
    if constexpr (LANES >= 32) {
        const auto sw = __builtin_amdgcn_permlane16_swap(m, m, false, false);      // (R0 R0 R2 R2), (R1 R1 R3 R3)
        const uint32_t a = sw[0], b = sw[1];
        m = a > b ? a : b;
    }
    if constexpr (LANES == 64) {
        const auto sw = __builtin_amdgcn_permlane32_swap(m, m, false, false);
        const uint32_t a = sw[0], b = sw[1];
        m = a > b ? a : b;
    }
    return m;
}

template <int OUT_DT>
__device__ inline float scale_of(float amax) {
    return amax > 0.0f ? amax / (OUT_DT == QGEMM_DT_F8E4M3 ? 448.0f : 127.0f) : 1.0f;
}

constexpr uint32_t kQuantNan = 0x80000000u;
constexpr int kQuantTurn = 4;                    // pieces a lane has in flight (per-matrix passes)

// ---- per matrix.  The host hands over a matrix without gaps as a single row (QuantArgs::per_row pieces), which saves the
// divisions and all row ends but one.  RAGGED: rows may end inside a piece; where they do not, nothing has to be settled, and a single
// row's maximum is that of its whole pieces and of its last one (start to now, us, graph replays: 500 x 7200 bf16 with gaps 7.6 -> 6.8,
// 1435 x 3368 fp32 with gaps 11.7 -> 10.5, 64 x 2048 6.1 -> 4.9, 41 x 1001 5.1 -> 4.8).
// Where piece i of `total` lies, loads and stores of it
template <int IN_DT, bool ONE_ROW, bool RAGGED>
struct MatrixPieces {
    typedef Piece<IN_DT> P;
    struct Place {
        uint32_t r, c, valid;        // row, element of it, elements that the row has from there on (0: past the last piece)
    };
    const QuantArgs &p;
    uint32_t row0, total;
    bool wide;
    __device__ MatrixPieces(const QuantArgs &a, uint32_t slice) : p(a) {
        row0 = slice * a.rows_per_slice;
        total = (a.rows - row0 < a.rows_per_slice ? a.rows - row0 : a.rows_per_slice) * a.per_row;
        wide = !RAGGED || a.cols >= (uint32_t)P::VEC;
    }
    // the whole pieces of a single row that ends inside one
    __device__ explicit MatrixPieces(const MatrixPieces<IN_DT, ONE_ROW, true> &o) : p(o.p), row0(0), total(o.total - 1), wide(true) {}
    __device__ Place place(uint32_t i) const {
        const bool in = i < total;
        Place o;
        o.r = 0;
        o.c = in ? i : 0;
        if constexpr (!ONE_ROW) o.r = row0 + div_by_inv(o.c, p.per_row, p.inv, o.c);
        o.c *= P::VEC;
        o.valid = in ? p.cols - o.c : 0;
        return o;
    }
    // as they come from memory, requested together; `settle` leaves zeros past the end  (WIDE: known to be `wide`)
    template <int N, bool WIDE = false>
    __device__ void request(v4i (&v)[N], const Place (&at)[N]) const {
        auto idx = [&](int j) { return ONE_ROW ? (size_t)at[j].c : at[j].r * p.ld + at[j].c; };
        if (WIDE || wide) {
#pragma unroll
            for (int j = 0; j < N; ++j) v[j] = P::template load<RAGGED>(p.x, idx(j), at[j].valid, true);
        } else {
#pragma unroll
            for (int j = 0; j < N; ++j) v[j] = at[j].valid ? P::load_elements(p.x, idx(j), at[j].valid) : v4i{0, 0, 0, 0};
        }
    }
    template <int N, bool WIDE = false>
    __device__ void settle(v4i (&v)[N], const Place (&at)[N]) const {
        if (!WIDE && !wide) return;
#pragma unroll
        for (int j = 0; j < N; ++j)
            if (!at[j].valid) v[j] = v4i{0, 0, 0, 0};
        if constexpr (RAGGED) {
#pragma unroll
            for (int j = 0; j < N; ++j) P::settle(v[j], at[j].valid);
        }
    }
    // both, for N pieces, `stride` apart
    template <int N>
    __device__ void load(v4i (&v)[N], Place (&at)[N], uint32_t first, uint32_t stride) const {
#pragma unroll
        for (int j = 0; j < N; ++j) at[j] = place(first + j * stride);
        if (wide) {
            request<N, true>(v, at);
            settle<N, true>(v, at);
        } else {
            request<N>(v, at);
        }
    }
    __device__ void store(const Place &at, v2i w) const {
        if (at.valid) store_piece<IN_DT>(p.q, at.r * p.ldq + at.c, w, RAGGED ? at.valid : P::VEC);
    }
    // bits of the largest |x| that is a number, bit 31 set where there is something else, of N pieces, `stride` apart, from
    // `first` on, N from first + `turn` on, ...; a single row's last piece, if it is cut short, where `last` says so
    template <int N>
    __device__ uint32_t maximum(uint32_t first, uint32_t stride, uint32_t turn, bool last) const {
        if constexpr (ONE_ROW && RAGGED) {
            v4i end[1] = {v4i{0, 0, 0, 0}};
            const Place at[1] = {place(total - 1)};
            if (last) request<1>(end, at);
            const uint32_t m = MatrixPieces<IN_DT, true, false>(*this).template maximum<N>(first, stride, turn, false);
            if (last) settle<1>(end, at);
            uint32_t b = P::max_bits(end[0]);
            if (b > P::INF) b = P::max_bits_of_numbers(end[0]) | kQuantNan;
            const uint32_t v = m & ~kQuantNan, w = b & ~kQuantNan;
            return (v > w ? v : w) | ((m | b) & kQuantNan);
        }
        v4i acc = v4i{0, 0, 0, 0}, v[N];
        Place at[N];
        for (uint32_t i = first; i < total; i += turn) {
            load<N>(v, at, i, stride);
#pragma unroll
            for (int j = 0; j < N; ++j) P::fold_max(acc, v[j]);
        }
        uint32_t m = P::max_bits(acc);
        if (m <= P::INF) return m;
        m = 0;
        for (uint32_t i = first; i < total; i += turn)
            for (int j = 0; j < N; ++j) {
                v4i one[1];
                Place there[1];
                load<1>(one, there, i + j * stride, 0);
                const uint32_t b = P::max_bits_of_numbers(one[0]);
                m = b > m ? b : m;
            }
        return m | kQuantNan;
    }
};
// the same over the workgroup's waves; bit 31 as above
template <int WAVES>
__device__ inline uint32_t workgroup_maximum(uint32_t m) {
    __shared__ uint32_t red[WAVES];
    m = lanes_max<64>(m & ~kQuantNan) | (__any((m & kQuantNan) != 0) ? kQuantNan : 0u);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = red[threadIdx.x % WAVES];                                   // (the 16 lanes of a row hold all of them)
    return lanes_max<16>(m & ~kQuantNan) | (__any((m & kQuantNan) != 0) ? kQuantNan : 0u);
}
template <int IN_DT, int OUT_DT>
__device__ inline Divisor matrix_divisor(uint32_t m) {
    const uint32_t b = m & ~kQuantNan;
    return make_divisor(scale_of<OUT_DT>(Piece<IN_DT>::element(b)), m < Piece<IN_DT>::INF);
}

// Small: one launch, no workspace.  Every workgroup takes the maximum of the whole matrix, then quantises its own 1024 pieces.
// A workgroup reads some 100 GB/s, so this ends where the exchange of quant_whole_matrix_kernel, which a call has to look for a capture for (0.25 us
// of host time, and calls of this size are bound by that), is ahead of it by as much: bf16, us a call among others / on the GPU alone, this: 48 x 2048
// (192 KiB) 5.0 / 7.2, exchange 5.1 / 6.5; 128 x 2048 (512 KiB) 7.1 / 9.4 and 6.7 / 7.2.  With gaps between the rows and a division for every piece it
// ends where two passes are ahead (kQuantSmallRowsBytes; graph replays, us, this / two passes: 64 x 512 (64 KiB) 4.3 / 4.8, 64 x 1024 4.4 / 5.2,
// 40 x 2176 (170 KiB) 7.6 / 5.2), but for a stream that is being captured, which has no more workspace than is there.
constexpr uint64_t kQuantSmallBytes = 256 << 10, kQuantSmallRowsBytes = 128 << 10;
template <int IN_DT, int OUT_DT, bool ONE_ROW, bool RAGGED>
__global__ void __launch_bounds__(1024) quant_small_matrix_kernel(const QuantArgs p) {
    const MatrixPieces<IN_DT, ONE_ROW, RAGGED> x(p, 0);
    const uint32_t mine = blockIdx.x * 1024 + threadIdx.x;
    v4i own[1];
    typename MatrixPieces<IN_DT, ONE_ROW, RAGGED>::Place at[1] = {x.place(mine)};
    x.template request<1>(own, at);                  // (settled behind the maximum: here it would wait for the piece in front of all others)
    const Divisor dv = matrix_divisor<IN_DT, OUT_DT>(workgroup_maximum<16>(x.template maximum<8>(threadIdx.x, 1024, 8 * 1024, threadIdx.x == 0)));
    x.template settle<1>(own, at);
    if (mine == 0) p.scales[0] = dv.s;
    x.store(at[0], quant_piece<IN_DT, OUT_DT>(own[0], dv));
}

// One launch for a matrix without gaps that the chip can hold: every lane keeps its pieces in registers, the workgroups exchange their
// maxima through memory and each quantises what it holds.  The matrix is read once and a launch saved, for an exchange of some 2 us.
// Eager calls one after another, bf16 to int8, us, two passes / so: 50 x 5296 7.9 / 5.3, 378 x 4632 9.2 / 6.6, 1531 x 3004 7.7 / 7.1, 1000 x
// 7168 8.6 / 7.9, 4096 x 4096 14.1 / 12.9; fp32 50 x 5296 7.9 / 5.1, 500 x 4096 7.4 / 6.1, 2048 x 4096 11.0 / 9.9.  Bound by the exchange up to
// some 10 MiB, by memory above.
// A workgroup writes its maximum and the launch's number as one 64-bit word, with the device's scope, and reads everybody's words
// until they carry that number: nothing has to be reset, ordered or fenced (a fence of that scope writes back the L2: 27 us), and a
// word is either this launch's or it is not.  The two streams that launch it at a time (may_exchange_maxima) have half of the sets each, which
// their launches take in turn; should another stream take a place over before the last one's launches are done, should workgroups not all
// find room beside another program's kernels, the wait ends after QuantArgs::wait and the workgroup takes the
// maximum of the whole matrix itself: slow, and the same result.  A replayed graph would bring the same number again: captured calls take the two passes below.
constexpr int kQuantSets = 64, kQuantGroups = 256, kQuantMostPieces = 8;
static __device__ uint64_t quant_words[kQuantSets][kQuantGroups];
// maximum of all workgroups' m (as workgroup_maximum gives it), false where some of them did not come in time
__device__ inline bool launch_maximum(uint32_t &m, uint32_t set, uint32_t tag, uint32_t wait) {
    uint64_t *const words = quant_words[set];
    const uint32_t t = threadIdx.x;
    if (t == 0) __hip_atomic_store(words + blockIdx.x, (uint64_t)tag << 32 | m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    uint64_t w = 0;
    bool late = false;
    if (t < gridDim.x) {
        const uint64_t start = __builtin_amdgcn_s_memrealtime();
        while (w = __hip_atomic_load(words + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), (uint32_t)(w >> 32) != tag) {
            late = __builtin_amdgcn_s_memrealtime() - start > wait;
            if (late) break;
        }
    } else if (blockIdx.x == 0 && t < (uint32_t)kQuantGroups) {          // (numbers come round: no old word stays for longer than a place's sets)
        __hip_atomic_store(words + t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    late = __syncthreads_or(late);
    m = workgroup_maximum<16>((uint32_t)w);
    return !late;
}
template <int IN_DT, int OUT_DT, int N>
__global__ void __launch_bounds__(1024, 8) quant_whole_matrix_kernel(const QuantArgs p) {
    typedef Piece<IN_DT> P;
    const MatrixPieces<IN_DT, true, true> x(p, 0);
    const uint32_t whole = p.cols / P::VEC, first = blockIdx.x * p.share;
    const uint32_t mine = first < whole ? (whole - first < p.share ? whole - first : p.share) : 0;
    // (lanes past the workgroup's share are out of the buffer's range and get zeros: no branch between the loads)
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>((const char *)p.x + (size_t)first * 16), 0, mine * 16, 0x00020000);
    v4i v[N];
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, threadIdx.x * 16, j * 1024 * 16, 0));
    // the last piece of a matrix that ends inside one is one lane's
    const bool last = whole < x.total && blockIdx.x == 0 && threadIdx.x == 0;
    v4i end[1] = {v4i{0, 0, 0, 0}};
    const typename MatrixPieces<IN_DT, true, true>::Place at[1] = {x.place(x.total - 1)};
    if (last) x.template request<1>(end, at);
    v4i acc = v4i{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < N; ++j) P::fold_max(acc, v[j]);
    if (last) {
        x.template settle<1>(end, at);
        P::fold_max(acc, end[0]);
    }
    uint32_t m = P::max_bits(acc);
    if (m > P::INF) {
        m = P::max_bits_of_numbers(end[0]);
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const uint32_t b = P::max_bits_of_numbers(v[j]);
            m = b > m ? b : m;
        }
        m |= kQuantNan;
    }
    m = workgroup_maximum<16>(m);
    if (!launch_maximum(m, p.set, p.tag, p.wait)) {
        __syncthreads();
        m = workgroup_maximum<16>(x.template maximum<1>(threadIdx.x, 1024, 1024, threadIdx.x == 0));
    }
    const Divisor dv = matrix_divisor<IN_DT, OUT_DT>(m);
    if (blockIdx.x == 0 && threadIdx.x == 0) p.scales[0] = dv.s;
#pragma unroll
    for (int j = 0; j < N; ++j)
        if (j * 1024 + threadIdx.x < mine)
            store_piece<IN_DT>(p.q, (size_t)(first + j * 1024 + threadIdx.x) * P::VEC, quant_piece<IN_DT, OUT_DT>(v[j], dv), P::VEC);
    if (last) x.store(at[0], quant_piece<IN_DT, OUT_DT>(end[0], dv));
}

// pass 1: one partial maximum per workgroup
template <int IN_DT, bool ONE_ROW, bool RAGGED>
__global__ void __launch_bounds__(256) quant_amax_kernel(const QuantArgs p) {
    const MatrixPieces<IN_DT, ONE_ROW, RAGGED> x(p, blockIdx.y);
    const uint32_t m = workgroup_maximum<4>(x.template maximum<kQuantTurn>(blockIdx.x * 256 * kQuantTurn + threadIdx.x, 256, gridDim.x * 256 * kQuantTurn,
                                                                                 blockIdx.x == 0 && threadIdx.x == 0));
    if (threadIdx.x == 0) p.partial[blockIdx.y * gridDim.x + blockIdx.x] = m;
}

// pass 2: every workgroup reduces the partial maxima again (a few KB, L2 resident), then
// quantises its share; workgroup 0 writes the scale
template <int IN_DT, int OUT_DT, bool ONE_ROW, bool RAGGED>
__global__ void __launch_bounds__(256) quant_matrix_kernel(const QuantArgs p) {
    const MatrixPieces<IN_DT, ONE_ROW, RAGGED> x(p, blockIdx.y);
    uint32_t m = 0, nan = 0;
    for (uint32_t i = threadIdx.x; i < p.npartial; i += 256) {
        const uint32_t b = p.partial[i];
        nan |= b & kQuantNan;
        m = (b & ~kQuantNan) > m ? (b & ~kQuantNan) : m;
    }
    const Divisor dv = matrix_divisor<IN_DT, OUT_DT>(workgroup_maximum<4>(m | nan));
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) p.scales[0] = dv.s;
    auto quantise = [&](const auto &pieces) {
        for (uint32_t first = blockIdx.x * 256 * kQuantTurn; first < pieces.total; first += gridDim.x * 256 * kQuantTurn) {
            v4i v[kQuantTurn];
            typename std::decay_t<decltype(pieces)>::Place at[kQuantTurn];
            pieces.template load<kQuantTurn>(v, at, first + threadIdx.x, 256);
#pragma unroll
            for (int j = 0; j < kQuantTurn; ++j) pieces.store(at[j], quant_piece<IN_DT, OUT_DT>(v[j], dv));
        }
    };
    if constexpr (ONE_ROW && RAGGED) {               // as in `maximum`
        const bool last = blockIdx.x == 0 && threadIdx.x == 0;
        v4i end[1];
        const typename MatrixPieces<IN_DT, ONE_ROW, RAGGED>::Place at[1] = {x.place(x.total - 1)};
        if (last) x.template request<1>(end, at);
        quantise(MatrixPieces<IN_DT, true, false>(x));
        if (!last) return;
        x.template settle<1>(end, at);
        x.store(at[0], quant_piece<IN_DT, OUT_DT>(end[0], dv));
    } else {
        quantise(x);
    }
}

// scale and divisor of a block whose maximum is in every lane that works on it; `numbers`: the maximum without its NaNs
template <int IN_DT, int OUT_DT, class F>
__device__ inline Divisor block_divisor(uint32_t m, F numbers) {
    const bool finite = m < Piece<IN_DT>::INF;
    if (m > Piece<IN_DT>::INF) m = numbers();
    return make_divisor(scale_of<OUT_DT>(Piece<IN_DT>::element(m)), finite);
}

// ---- 1 x 128 blocks: Piece::LANES lanes (16 or 32) per block, one piece a lane.  What keeps memory busy is waves: with four
// pieces in flight per lane and a quarter of the waves, as it was from 65536 blocks on, 1500 x 7168 bf16 took 10.9 us and takes
// 7.8, 6144 x 7168 29.5 and 25.7 (5.1 TB/s, what a copy reaches).
template <int IN_DT, int OUT_DT, bool RAGGED>
__device__ __forceinline__ void quant_row_block(QGEMM_QUANT_HEAD, const QuantArgs &p) {
    typedef Piece<IN_DT> P;
    const uint32_t row0 = blockIdx.y * rows_per_slice;
    const uint32_t rows = rows_all - row0 < rows_per_slice ? rows_all - row0 : rows_per_slice, total = rows * per_row;
    const uint32_t lane = threadIdx.x % P::LANES, i = blockIdx.x * (256 / P::LANES) + threadIdx.x / P::LANES;
    uint32_t jb;
    const uint32_t r = row0 + div_by_inv(i, per_row, inv, jb), c = jb * kScaleBlock + lane * P::VEC;
    const uint32_t valid = (i < total && c < cols) ? cols - c : 0;
    v4i v = v4i{0, 0, 0, 0};
    const bool wide = cols >= (uint32_t)P::VEC;
    if (valid) v = P::template load<RAGGED>(x, (size_t)r * ld + c, valid, wide);
    uint64_t ldq = p.ldq, scale_rs = p.scale_rs, scale_cs = p.scale_cs;
    asm volatile("" : "+s"(ldq), "+s"(scale_rs), "+s"(scale_cs));          // (fetched here, while the load flies, not where they are used)
    if (RAGGED && wide) P::settle(v, valid);
    const uint32_t m = lanes_max<P::LANES>(P::max_bits(v));
    const Divisor dv = block_divisor<IN_DT, OUT_DT>(m, [&] { return lanes_max<P::LANES>(P::max_bits_of_numbers(v)); });
    if (i >= total) return;                                                // (whole groups of lanes leave together)
    if (lane == 0) scales[(size_t)r * scale_rs + (size_t)jb * scale_cs] = dv.s;
    if (valid) store_piece<IN_DT>(q, (size_t)r * ldq + c, quant_piece<IN_DT, OUT_DT>(v, dv), valid);
}
// The arguments of a launch with preloaded ones cost it 0.07 us, which more than a few hundred workgroups gain back (256 x 7168
// 3.69 -> 3.52 us, 500 x 7200 4.81 -> 4.51; 128 x 4096 2.90 against 2.96): kQuantManyGroups.
constexpr uint32_t kQuantManyGroups = 640;
template <int IN_DT, int OUT_DT, bool RAGGED>
__global__ void __launch_bounds__(256) quant_row_block_kernel(QGEMM_QUANT_HEAD, const QuantArgs p) {
    quant_row_block<IN_DT, OUT_DT, RAGGED>(x, q, scales, ld, rows_all, cols, per_row, inv, rows_per_slice, p);
}
template <int IN_DT, int OUT_DT, bool RAGGED>
__global__ void __launch_bounds__(256) quant_few_blocks_kernel(const QuantArgs p) {
    quant_row_block<IN_DT, OUT_DT, RAGGED>(QGEMM_QUANT_HEAD_OF(p));
}

// ---- 128 x 128 blocks: one workgroup per block, which it holds in registers
template <int IN_DT, int OUT_DT, bool RAGGED, int BLOCK_ROWS>
__device__ __forceinline__ void quant_square_block(QGEMM_QUANT_HEAD, const QuantArgs &p) {
    typedef Piece<IN_DT> P;
    constexpr int ROWS = 256 / P::LANES, TURNS = BLOCK_ROWS / ROWS;
    __shared__ uint32_t red[4];
    const uint32_t nbc = (cols + 127) / 128;
    const uint32_t ib = blockIdx.x / nbc, jb = blockIdx.x % nbc;
    const uint32_t c = jb * 128 + (threadIdx.x % P::LANES) * P::VEC;
    const uint32_t r0 = ib * 128 + threadIdx.x / P::LANES;               // rows r0, r0 + ROWS, ...
    const uint32_t valid = c < cols ? cols - c : 0;
    auto workgroup_max = [&](uint32_t m) {
        m = lanes_max<64>(m);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
        __syncthreads();
        const uint32_t a = red[0] > red[1] ? red[0] : red[1], b = red[2] > red[3] ? red[2] : red[3];
        return a > b ? a : b;
    };
    v4i v[TURNS];
    if (!RAGGED || cols >= (uint32_t)P::VEC) {
        // (every lane loads, those outside from the nearest row or the start of a row: with a branch around each load the compiler
        // copied the array at each of them, up to 235 registers, and the waves that keep memory busy were gone: 6144 x 7168 fp16 95.7 us, 27.8 so)
        const uint32_t from = valid ? c : 0;
#pragma unroll
        for (int i = 0; i < TURNS; ++i) {
            const uint32_t r = r0 + i * ROWS;
            v[i] = P::template load<RAGGED>(x, (size_t)(r < rows_all ? r : rows_all - 1) * ld + from, valid, true);
        }
#pragma unroll
        for (int i = 0; i < TURNS; ++i) {
            const bool in = r0 + i * ROWS < rows_all && valid;
            if (RAGGED && jb + 1 == nbc) P::settle(v[i], in ? valid : 0);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[i][k] = in ? v[i][k] : 0;
        }
    } else {
#pragma unroll
        for (int i = 0; i < TURNS; ++i) {
            const uint32_t r = r0 + i * ROWS;
            v[i] = r < rows_all && valid ? P::load_elements(x, (size_t)r * ld + c, valid) : v4i{0, 0, 0, 0};
        }
    }
    uint64_t ldq = p.ldq, scale_rs = p.scale_rs, scale_cs = p.scale_cs;
    asm volatile("" : "+s"(ldq), "+s"(scale_rs), "+s"(scale_cs));
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < TURNS; ++i) {
        const uint32_t b = P::max_bits(v[i]);
        m = b > m ? b : m;
    }
    m = workgroup_max(m);
    const Divisor dv = block_divisor<IN_DT, OUT_DT>(m, [&] {
        uint32_t n = 0;
        for (int i = 0; i < TURNS; ++i) {
            const uint32_t b = P::max_bits_of_numbers(v[i]);
            n = b > n ? b : n;
        }
        __syncthreads();                                                 // (m is the same in every lane of the workgroup)
        return workgroup_max(n);
    });
    if (threadIdx.x == 0) scales[(size_t)ib * scale_rs + (size_t)jb * scale_cs] = dv.s;
#pragma unroll
    for (int i = 0; i < TURNS; ++i) {
        const uint32_t r = r0 + i * ROWS;
        if (r < rows_all && valid) store_piece<IN_DT>(q, (size_t)r * ldq + c, quant_piece<IN_DT, OUT_DT>(v[i], dv), valid);
    }
}

template <int IN_DT, int OUT_DT, bool RAGGED>
__global__ void __launch_bounds__(256) quant_square_block_kernel(QGEMM_QUANT_HEAD, const QuantArgs p) {
    quant_square_block<IN_DT, OUT_DT, RAGGED, 128>(x, q, scales, ld, rows_all, cols, per_row, inv, rows_per_slice, p);
}
// Up to kQuantFewRows rows: without the rows that are not there, which every lane fetched and quantised as well, and without preloaded
// arguments, which a launch of a few workgroups does not gain back.  us, graph replays, 128 rows a block / so: fp32 1 x 967 3.41 / 2.42,
// 8 x 1025 3.44 / 2.46; bf16 16 x 1985 3.37 / 2.58, 2 x 128 at odd addresses 2.80 / 2.16, 12 x 7168 2.66 / 2.48.
constexpr uint32_t kQuantFewRows = 32;
template <int IN_DT, int OUT_DT, bool RAGGED>
__global__ void __launch_bounds__(256) quant_low_block_kernel(const QuantArgs p) {
    quant_square_block<IN_DT, OUT_DT, RAGGED, kQuantFewRows>(QGEMM_QUANT_HEAD_OF(p));
}

}  // namespace qgemm
