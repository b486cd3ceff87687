// One step of 64 keys for one wave of the 16-bit matrix-core kernels with position tables (head_dim 64, MFMA 16x16x32).
//
// The wave owns 16 QG consecutive query rows.  Scores are kept transposed, S^T[key][query]: a lane has one query (n = lane & 15)
// of each of the QG groups and the keys 4 g + t (g = lane >> 4) of each of the four groups of 16, so that the streaming
// softmax reduces inside the lane and over the four lane rows, and the probabilities are the B operand of O^T += V^T.P^T
// as they stand.
//
// The position terms are functions of r = i - j and have to be skewed into (i, j).  They never leave the registers:
//   * both are computed for six (QG = 1: five) tiles of 16 relative positions.  The product
//     P'[key][r] = K_key . Q_r[delta(r)] has its lanes along r; for a fixed key the scores of 16 consecutive queries are 16
//     consecutive r, i.e. two neighbouring tiles, cut at a lane that depends on the key, and turned by as many lanes.  The key of an
//     accumulator is 4 g + t: one select between the two tiles under a mask that depends on t, one rotation of the lane rows by t and
//     two more by 4 and 8 under row masks (row g turns by 4 g) bring it to the lanes of its queries.
//   * C'[query][r] = Q_query . K_r[delta(r)], its columns in the opposite order, turns into C[query][key], lanes along the keys, in the
//     same way; the product that adds it to S^T transposes it.
//   * a dword holds two values (16 bits, as the model rounds these terms) that turn alike: p2c of two key groups, c2p of two query groups
//     (one query group: of two key groups).  p2c is where the score products start from; c2p is added to them by products with an identity (exact: one addend each).
// Against a scratch in LDS (results stored, read back element by element or through a ring, as in attn_mfma.hip) this costs three
// vector instructions per dword and a product, and saves the stores, the reads, their waits and the barriers between the waves that
// compute positions and those that compute scores: here every wave does the same, with one barrier a step for the keys.
//
// A near step is bound by its SIMD: about 430 vector instructions and 80 matrix ones of a wave of 32 rows.  Measured there: a matrix
// instruction of this shape takes 16.5 clk; conversions, selects, lane moves and shifts 4.3; exponentials 8.5; additions, products and
// masks 4.3 too, but those of the two waves at the same time.  Vector instructions beside a stream of matrix instructions go at half their
// rate, so the two together take about the sum of their times.
//
// Such a product multiplies every element of a row with a zero but one, so an infinity or a NaN among the c2p terms spoils its
// neighbours' scores.  The maximum of a row tells: if a score is not a number, the step's scores are computed again, the finite terms
// and indicators of the others apart (CAREFUL).
//
// The bits of a row are those of the kernels of 32 x 32 tiles (attn_mfma.hip, attn_short.hip), which take other launches: the same
// roundings, every product over the same elements in the same order, sums of probabilities in the same order, a step of the same 64 keys.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "tdb_internal.h"

namespace tdb_step {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

constexpr int BN = 64;                  // keys per step
constexpr int ROW = 128;                // bytes of a row of 64 values: LDS rows are not padded, their 16-byte chunks are permuted

template <int DT>
struct Elem;
template <>
struct Elem<TDB_BF16> {
    using T = __bf16;
    using X2 = bf16x2;
    using X8 = bf16x8;
    static __device__ __forceinline__ f32x4 mfma(X8 a, X8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
    static constexpr uint32_t ONE = 0x3f80, EXPONENT = 0x7f80, MANTISSA = 0x7f, DOUBLE = 0x80;
    static __device__ __forceinline__ float low(uint32_t x) { return __builtin_bit_cast(float, x << 16); }
    static __device__ __forceinline__ float high(uint32_t x) { return __builtin_bit_cast(float, x & 0xffff0000u); }
};
template <>
struct Elem<TDB_F16> {
    using T = _Float16;
    using X2 = f16x2;
    using X8 = f16x8;
    static __device__ __forceinline__ f32x4 mfma(X8 a, X8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
    static constexpr uint32_t ONE = 0x3c00, EXPONENT = 0x7c00, MANTISSA = 0x3ff, DOUBLE = 0x400;
    static __device__ __forceinline__ float low(uint32_t x) { return float(__builtin_bit_cast(X2, x)[0]); }
    static __device__ __forceinline__ float high(uint32_t x) { return float(__builtin_bit_cast(X2, x)[1]); }
};

template <typename E>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typename E::X2 v = {(typename E::T)lo, (typename E::T)hi};
    return __builtin_bit_cast(uint32_t, v);
}
// The same, opaque to the optimiser: it would turn a select between two packed pairs into two selects and a pack for each use.
template <typename E>
__device__ __forceinline__ uint32_t packed2(float lo, float hi) {
    uint32_t x = pack2<E>(lo, hi);
    asm("" : "+v"(x));
    return x;
}

// Where 16-byte chunk `chunk` of row `row` lies.  Operand rows (keys, table rows): 16 rows at the same chunk are on distinct banks.
// Values: the transposing read takes 4 rows x 32 bytes per 16 lanes, 8 such rows are on distinct banks.
__device__ __forceinline__ uint32_t operand_at(uint32_t row, uint32_t chunk) { return row * ROW + ((chunk * 16) ^ ((row * 8) & 0x70)); }
__device__ __forceinline__ uint32_t value_at(uint32_t row, uint32_t chunk) { return row * ROW + ((chunk * 16) ^ ((row * 16) & 0x60)); }

// (By value: the cast of a vector's element would take the vector's first.)
__device__ __forceinline__ uint32_t bits(float x) { return __builtin_bit_cast(uint32_t, x); }
// (By value: `c ? x : y` of two array elements would select an address.)
__device__ __forceinline__ uint32_t either(bool c, uint32_t x, uint32_t y) { return c ? x : y; }

// Word t: `on` where bit t of the lane's masks says so, else `before`; then lane row g turned right by 4 g + first + t lanes.
// (All four words side by side: a DPP move may not follow the instruction that made its source.)
template <int FIRST>
__device__ __forceinline__ u32x4 turned(const bool (&in)[5], const uint32_t (&on)[4], const uint32_t (&before)[4]) {
    u32x4 x;
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = either(in[FIRST + t], on[t], before[t]);
    if constexpr (FIRST == 1) x[0] = __builtin_amdgcn_mov_dpp(x[0], 0x121, 0xf, 0xf, true);     // row_ror:1
    x[1] = __builtin_amdgcn_mov_dpp(x[1], 0x121 + FIRST, 0xf, 0xf, true);
    x[2] = __builtin_amdgcn_mov_dpp(x[2], 0x122 + FIRST, 0xf, 0xf, true);
    x[3] = __builtin_amdgcn_mov_dpp(x[3], 0x123 + FIRST, 0xf, 0xf, true);
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = __builtin_amdgcn_update_dpp(x[t], x[t], 0x124, 0xa, 0xf, false);     // rows 1 and 3
#pragma unroll
    for (int t = 0; t < 4; ++t) x[t] = __builtin_amdgcn_update_dpp(x[t], x[t], 0x128, 0xc, 0xf, false);     // rows 2 and 3
    return x;
}

// Maxima: NaN if one of the values is, or (NUMBERS) of the others.
template <bool NUMBERS>
__device__ __forceinline__ float largest(float a, float b, float c) {
    if constexpr (NUMBERS) return fmaxf(fmaxf(a, b), c);
    else return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
// The largest of a value over the four lane rows, and the sum.
template <bool NUMBERS>
__device__ __forceinline__ float rows_max(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const float a = __builtin_bit_cast(float, uint32_t(r[0])), b = __builtin_bit_cast(float, uint32_t(r[1]));
    const uint32_t w = __builtin_bit_cast(uint32_t, largest<NUMBERS>(a, b, b));
    const auto s = __builtin_amdgcn_permlane32_swap(w, w, false, false);
    const float c = __builtin_bit_cast(float, uint32_t(s[0])), d = __builtin_bit_cast(float, uint32_t(s[1]));
    return largest<NUMBERS>(c, d, d);
}
template <int N>
using Int = std::integral_constant<int, N>;
// What stands between two of these is scheduled by itself: `products` matrix instructions, each followed by `each` vector ones.
template <int products, int each>
__device__ __forceinline__ void stage_end() {
    if constexpr (products > 0) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, each, 0);
        stage_end<products - 1, each>();
    } else {
        __builtin_amdgcn_sched_barrier(0);
    }
}
// This lane row's value and that of the row two on; of the neighbouring rows.
__device__ __forceinline__ float halves_sum(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __builtin_bit_cast(float, uint32_t(r[0])) + __builtin_bit_cast(float, uint32_t(r[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return __builtin_bit_cast(float, uint32_t(r[0])) + __builtin_bit_cast(float, uint32_t(r[1]));
}

// EXACT: steps whose relative positions all have one table row keep their position terms in 32 bits.
template <bool C2P, bool P2C, int DT, int QG, bool EXACT>
struct Wave {
    using E = Elem<DT>;
    using X8 = typename E::X8;
    static constexpr int NT = QG + 4;       // position tiles of a step: tile i holds r = q0 - k0 + 16 (i - 4) + n
    static constexpr int UQ = 16 * QG;      // query rows
    static constexpr bool POS = C2P || P2C;

    int n, g;                               // lane & 15, lane >> 4
    uint32_t kr_base;                       // LDS offset of the K_r rows (the Q_r rows lie at rows_base)
    uint32_t k_lane, v_lane;                // this lane's place in a block of keys / values
    bool in[5];                             // n + 4 g + t < 16
    u32x4 one;                              // identity, first half: value 2 t of lane (n, g) is 1 where n = 4 g + t
    X8 q[QG][2];                            // query n, columns 32 h + 8 g .. + 7: A operand (c2p) and B operand (scores)
    f32x4 o[4][QG];                         // O^T: d = 16 dt + 4 g + t of query n
    float m[QG], l[QG];
    uint32_t a[NT];                         // LDS offsets of row r of each tile (chunk g) among the Q_r rows
    // c2p of the highest tile of each query group, which is the lowest of the step before: packed (QG = 2) or as it is (QG = 1)
    u32x4 carry;
    bool carried;
    uint32_t far_row;                       // EXACT: the row whose c2p values are in `carry` instead

    __device__ __forceinline__ void init(int lane, uint32_t kr_base_) {
        n = lane & 15, g = lane >> 4;
        kr_base = kr_base_;
        k_lane = operand_at(n, g);
        v_lane = value_at(4 * g + (n >> 2), 0) + 8 * (n & 3);
#pragma unroll
        for (int t = 0; t < 5; ++t) in[t] = n + 4 * g + t < 16;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint32_t x = n == 4 * g + t ? E::ONE : 0;
            asm volatile("" : "+v"(x));     // (or each product would build its operand anew)
            one[t] = x;
        }
    }
    __device__ __forceinline__ void open() {
        carried = false, far_row = ~0u;
#pragma unroll
        for (int x = 0; x < QG; ++x) {
            m[x] = -INFINITY, l[x] = 0.f;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) o[dt][x] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    // LDS offset of table row `delta`, chunk g
    __device__ __forceinline__ uint32_t row_at(int delta) const { return (uint32_t(delta) << 7) ^ ((uint32_t(delta) << 3) & 0x70) ^ (uint32_t(g) << 4); }
    // (The kernels that use this have dynamic LDS only: it starts at 0.  Through the array's address the compiler adds that 0 to each offset.)
    static __device__ __forceinline__ X8 frag(uint32_t at) { return *(const __attribute__((address_space(3))) X8*)at; }
    __device__ __forceinline__ X8 identity(int half) const {
        return __builtin_bit_cast(X8, half ? u32x4{one[0] << 16, one[1] << 16, one[2] << 16, one[3] << 16} : one);
    }
    static __device__ __forceinline__ f32x4 dot(const X8 (&x)[2], const X8 (&y)[2], f32x4 c) { return E::mfma(x[1], y[1], E::mfma(x[0], y[0], c)); }

    // Non-finite values of a dword: taken out of it, and as indicators 1 (NaN), 2 (+infinity), 4 (-infinity).
    static __device__ __forceinline__ uint32_t take_out(uint32_t& x) {
        uint32_t out = 0;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const uint32_t v = (x >> (16 * half)) & 0xffff;
            if ((v & E::EXPONENT) == E::EXPONENT) {
                out |= (E::ONE + E::DOUBLE * ((v & E::MANTISSA) ? 0 : (v >> 15) ? 2 : 1)) << (16 * half);
                x &= half ? 0x0000ffffu : 0xffff0000u;
            }
        }
        return out;
    }

    // K_r rows of a tile, columns mirrored (at: this lane's offset among the Q_r rows)
    __device__ __forceinline__ void mirrored(X8 (&r)[2], uint32_t at) const {
        const uint32_t m = uint32_t(__builtin_amdgcn_mov_dpp(at, 0x140 /* row_mirror */, 0xf, 0xf, true)) + kr_base;
        r[0] = frag(m), r[1] = frag(m ^ 64);
    }
    static __device__ __forceinline__ void plain(X8 (&r)[2], uint32_t at) { r[0] = frag(at), r[1] = frag(at ^ 64); }

    __device__ __forceinline__ void keys(X8 (&kf)[4][2], uint32_t k_at) const {
#pragma unroll
        for (int kg = 0; kg < 4; ++kg)
#pragma unroll
            for (int h = 0; h < 2; ++h) kf[kg][h] = frag(k_at + 16 * ROW * kg + (k_lane ^ (64 * h)));
    }

    // Scores of a step whose relative positions meet several table rows.  In stages: the products of one beside the vector
    // instructions that the results of the one before need.
    //   p2c  p[kg][y]: tile QG - 1 - kg - y; query group x takes y = QG - 1 - x, from lane 4 g + t on, and y + 1.  Turned in 32 bits, as
    //        the accumulators that the score products start from.
    //   c2p  c[x][y]: tile x - y, columns mirrored; key group kg takes y = kg + 1, from lane 4 g + t + 1 on, and y = kg.  y = 0 has been
    //        the y = 4 of the step before.
    template <bool CAREFUL>
    __device__ __forceinline__ void scores(f32x4 (&s)[4][QG], uint32_t k_at) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        // (Opaque the second time: what was read the first time shall not stay in registers for it.)
        uint32_t rows[NT];
#pragma unroll
        for (int i = 0; i < NT; ++i) {
            rows[i] = a[i];
            if constexpr (CAREFUL) asm volatile("" : "+v"(rows[i]));
        }
        if constexpr (CAREFUL) asm volatile("" : "+s"(k_at));
        X8 kf[4][2], kr[NT][2], qr[NT][2];
        f32x4 c[QG][5], p[4][QG + 1];
        u32x4 cw[2 * QG];                 // QG = 2: word kg holds both query groups; QG = 1: word kg / 2 two key groups
        auto c_product = [&](auto ii) {
            constexpr int i = decltype(ii)::value;
#pragma unroll
            for (int x = 0; x < QG; ++x) {
                const int y = x + 4 - i;
                if (y >= (CAREFUL ? 0 : 1) && y <= 4) c[x][y] = dot(q[x], kr[i], zero);
            }
        };
        auto p_products = [&](auto cc) {
            constexpr int first = decltype(cc)::value;
            if constexpr (P2C) {
#pragma unroll
                for (int i = QG + 3 - first; i >= 2 - first; --i)
#pragma unroll
                    for (int kg = first; kg < first + 2; ++kg) {
                        const int y = QG + 3 - kg - i;
                        if (y >= 0 && y <= QG) p[kg][y] = dot(kf[kg], qr[i], zero);
                    }
            }
        };
        auto p_turn = [&](auto cc) {
            constexpr int first = decltype(cc)::value;
            if constexpr (P2C) {
                // A word has two key groups, so that a tile is packed once for both query groups that take it (of one key group and two
                // query groups it was 32 conversions a step for 24: 1.0 to 1.6 %).  To add the words by products with an identity instead
                // of unpacking them saves 32 instructions for 8 products and is not faster: of either there is as much to do.
                uint32_t w[QG + 1][4];
#pragma unroll
                for (int y = 0; y <= QG; ++y)
#pragma unroll
                    for (int t = 0; t < 4; ++t) w[y][t] = packed2<E>(p[first][y][t], p[first + 1][y][t]);
#pragma unroll
                for (int x = 0; x < QG; ++x) {
                    const u32x4 to = turned<0>(in, w[QG - 1 - x], w[QG - x]);
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        s[first][x][t] = E::low(to[t]);
                        s[first + 1][x][t] = E::high(to[t]);
                    }
                }
            }
        };
        auto c_turn = [&]() {
            if constexpr (C2P && QG == 2) {
                uint32_t w[5][4];
#pragma unroll
                for (int y = 0; y <= 4; ++y)
#pragma unroll
                    for (int t = 0; t < 4; ++t) w[y][t] = y == 0 && !CAREFUL ? carry[t] : packed2<E>(c[0][y][t], c[1][y][t]);
                if constexpr (!CAREFUL) carry = u32x4{w[4][0], w[4][1], w[4][2], w[4][3]};
#pragma unroll
                for (int kg = 0; kg < 4; ++kg) cw[kg] = turned<1>(in, w[kg + 1], w[kg]);
            } else if constexpr (C2P) {
                if constexpr (!CAREFUL) {
                    c[0][0] = __builtin_bit_cast(f32x4, carry);
                    carry = __builtin_bit_cast(u32x4, c[0][4]);
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    uint32_t on[4], before[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        on[t] = packed2<E>(c[0][2 * k + 1][t], c[0][2 * k + 2][t]);
                        before[t] = packed2<E>(c[0][2 * k][t], c[0][2 * k + 1][t]);
                    }
                    cw[k] = turned<1>(in, on, before);
                }
            }
        };
        if constexpr (C2P && !CAREFUL) {
            if (!carried) {                 // the first step of a unit, or behind a far one
                f32x4 top[QG];
#pragma unroll
                for (int x = 0; x < QG; ++x) {
                    X8 r[2];
                    mirrored(r, rows[4 + x]);
                    top[x] = dot(q[x], r, zero);
                }
#pragma unroll
                for (int t = 0; t < 4; ++t) carry[t] = QG == 2 ? packed2<E>(top[0][t], top[QG - 1][t]) : bits(top[0][t]);
            }
            carried = true;
        }
        if constexpr (C2P) {
#pragma unroll
            for (int i = CAREFUL ? NT - 1 : QG + 2; i >= 0; --i) mirrored(kr[i], rows[i]);
        }
        keys(kf, k_at);
        if constexpr (P2C) {
#pragma unroll
            for (int i = NT - 1; i >= 0; --i) plain(qr[i], rows[i]);
        }
        if constexpr (C2P) {
            if constexpr (CAREFUL) c_product(Int<NT - 1>{});
            if constexpr (QG == 2) c_product(Int<4>{});
            c_product(Int<3>{});
            c_product(Int<2>{});
            c_product(Int<1>{});
            c_product(Int<0>{});
        }
        __builtin_amdgcn_sched_barrier(0);
        p_products(Int<0>{});
        c_turn();
        stage_end<CAREFUL || !C2P || !P2C ? 0 : 4 * (QG + 1), 6>();
        p_products(Int<2>{});
        p_turn(Int<0>{});
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!P2C) {
#pragma unroll
            for (int kg = 0; kg < 4; ++kg)
#pragma unroll
                for (int x = 0; x < QG; ++x) s[kg][x] = zero;
        }
#pragma unroll
        for (int kg = 0; kg < 2; ++kg)
#pragma unroll
            for (int x = 0; x < QG; ++x) s[kg][x] = dot(kf[kg], q[x], s[kg][x]);
        p_turn(Int<2>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kg = 2; kg < 4; ++kg)
#pragma unroll
            for (int x = 0; x < QG; ++x) s[kg][x] = dot(kf[kg], q[x], s[kg][x]);
        if constexpr (C2P) {
#pragma unroll
            for (int k = 0; k < 2 * QG; ++k) {
                u32x4 odd;
                if constexpr (CAREFUL) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        uint32_t v = cw[k][t];
                        odd[t] = take_out(v);
                        cw[k][t] = v;
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int kg = QG == 2 ? k : 2 * k + h, x = QG == 2 ? h : 0;
                    s[kg][x] = E::mfma(__builtin_bit_cast(X8, cw[k]), identity(h), s[kg][x]);
                    if constexpr (CAREFUL) {
                        const f32x4 bad = E::mfma(__builtin_bit_cast(X8, odd), identity(h), zero);
#pragma unroll
                        for (int t = 0; t < 4; ++t) {
                            const float b = bad[t];
                            s[kg][x][t] += b == 1.f ? NAN : b == 2.f ? INFINITY : b == 4.f ? -INFINITY : 0.f;
                        }
                    }
                }
            }
        }
    }

    // Scores of a step all of whose relative positions have one table row (at LDS offset `row`, chunk 0): a c2p value per query and a
    // p2c value per key.  EXACT: both stay in 32 bits, c2p is returned in `add` and kept for the next step of this row; otherwise the bits
    // are those of scores().
    __device__ __forceinline__ void far_scores(f32x4 (&s)[4][QG], float (&add)[QG], uint32_t k_at, uint32_t row) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        X8 kf[4][2];
        keys(kf, k_at);
        const uint32_t at = row ^ (g << 4);
        X8 r[2];
        f32x4 p[4];
#pragma unroll
        for (int kg = 0; kg < 4; ++kg) p[kg] = zero;
        if constexpr (P2C) {
            plain(r, at);
#pragma unroll
            for (int kg = 0; kg < 4; ++kg) p[kg] = dot(kf[kg], r, zero);
            if constexpr (!EXACT) {
#pragma unroll
                for (int kg = 0; kg < 4; ++kg) {
                    const uint32_t w0 = pack2<E>(p[kg][0], p[kg][1]), w1 = pack2<E>(p[kg][2], p[kg][3]);
                    p[kg] = f32x4{E::low(w0), E::high(w0), E::low(w1), E::high(w1)};
                }
            }
        }
#pragma unroll
        for (int kg = 0; kg < 4; ++kg)
#pragma unroll
            for (int x = 0; x < QG; ++x) s[kg][x] = dot(kf[kg], q[x], p[kg]);
        if constexpr (C2P) {
            if constexpr (EXACT) {
                if (row != far_row) {
                    plain(r, at + kr_base);
#pragma unroll
                    for (int x = 0; x < QG; ++x) {
                        const f32x4 c = tdb_settled(dot(r, q[x], zero));
                        carry[x] = bits(c[0]);
                    }
                    far_row = row;
                }
#pragma unroll
                for (int x = 0; x < QG; ++x) {
                    const uint32_t kept = carry[x];     // (the cast of the element itself is that of element 0)
                    add[x] = __builtin_bit_cast(float, kept);
                }
            } else {
                plain(r, at + kr_base);
                f32x4 c[QG];
                u32x4 w;
#pragma unroll
                for (int x = 0; x < QG; ++x) c[x] = dot(q[x], r, zero);
#pragma unroll
                for (int t = 0; t < 4; ++t) w[t] = pack2<E>(c[0][t], c[QG - 1][t]);
#pragma unroll
                for (int kg = 0; kg < 4; ++kg)
#pragma unroll
                    for (int x = 0; x < QG; ++x) s[kg][x] = E::mfma(__builtin_bit_cast(X8, w), identity(x), s[kg][x]);
            }
        }
    }

    // Keys from `left` on do not exist.
    __device__ __forceinline__ void mask(f32x4 (&s)[4][QG], int left) const {
        const int lim = left - 4 * g;
#pragma unroll
        for (int kg = 0; kg < 4; ++kg)
#pragma unroll
            for (int x = 0; x < QG; ++x)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (16 * kg + t >= lim) s[kg][x][t] = -INFINITY;
    }
    template <bool NUMBERS>
    __device__ __forceinline__ float maximum(const f32x4 (&s)[4][QG], int x) const {
        float part[4];
#pragma unroll
        for (int kg = 0; kg < 4; ++kg) part[kg] = largest<NUMBERS>(s[kg][x][0], s[kg][x][1], s[kg][x][2]);
#pragma unroll
        for (int kg = 0; kg < 4; kg += 2) part[kg] = largest<NUMBERS>(largest<NUMBERS>(part[kg], s[kg][x][3], s[kg + 1][x][3]), part[kg + 1], part[kg + 1]);
        return rows_max<NUMBERS>(largest<NUMBERS>(part[0], part[2], part[2]));
    }
    // Probabilities under the running maxima, and this lane's sums of them.
    __device__ __forceinline__ void probabilities(const f32x4 (&s)[4][QG], const float (&add)[QG], float c_exp, X8 (&pb)[QG][2], float (&sum)[QG]) const {
#pragma unroll
        for (int x = 0; x < QG; ++x) {
            const float mc = (m[x] - add[x]) * c_exp;
            float total[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f32x4& v = s[2 * c + (e >> 1)][x];
                    const float p0 = __builtin_amdgcn_exp2f(fmaf(v[2 * (e & 1)], c_exp, -mc)), p1 = __builtin_amdgcn_exp2f(fmaf(v[2 * (e & 1) + 1], c_exp, -mc));
                    total[c] = e ? total[c] + (p0 + p1) : p0 + p1;
                    w[e] = pack2<E>(p0, p1);
                }
                pb[x][c] = __builtin_bit_cast(X8, u32x4{w[0], w[1], w[2], w[3]});
            }
            sum[x] = total[0] + total[1];
        }
    }

    // One step: keys at LDS offset k_at, values at v_at, `left` keys from its first one to the end of the sequence.  far: all its relative
    // positions have the table row at LDS offset `row`.
    __device__ __forceinline__ void step(uint32_t k_at, uint32_t v_at, int left, float c_exp, bool first, bool far, uint32_t row) {
        f32x4 s[4][QG];
        float add[QG], sum[QG];
        X8 pb[QG][2];
#pragma unroll
        for (int x = 0; x < QG; ++x) add[x] = 0.f;
        // A wave in its scores, whose matrix instructions feed one another, goes before the other wave of its SIMD in its softmax (the
        // other way about 64 x 512 keys take 5 % more).
        __builtin_amdgcn_s_setprio(1);
        if (far) {
            far_scores(s, add, k_at, row);
            carried = false;
        } else {
            far_row = ~0u;
            scores<false>(s, k_at);
        }
        if (left < BN) mask(s, left);
        __builtin_amdgcn_s_setprio(0);
        // V^T through the transposing read: the lane provides the address of four columns of one key.
        s16x8 vf[2][4];
        uint32_t v_from[4];
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            v_from[dt] = v_at + (v_lane ^ (32 * dt));
            asm("" : "+v"(v_from[dt]));     // (or every read has an addition of its own, instead of an offset)
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                const uint32_t at = v_from[dt] + 32 * ROW * c;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)at);
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(at + 16 * ROW));
                vf[c][dt] = s16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
        // The running maximum of a row is only raised (and its accumulators rescaled) when the row exceeds it by more than 2^8; until
        // then the probabilities may be as large as 256, which the element types and the sums carry as exactly.  Rows decide
        // separately: a row's result does not depend on its neighbours.  The maximum itself is looked for only where some lane's sum says
        // that a probability may be larger, or is not a number.
        bool look = first;
        if (!first) {
            probabilities(s, add, c_exp, pb, sum);
            bool over = false;
#pragma unroll
            for (int x = 0; x < QG; ++x) over = over || !(sum[x] <= 255.f);
            look = __builtin_amdgcn_ballot_w64(over) != 0;
        }
        if (look) {
            float mx[QG];
#pragma unroll
            for (int x = 0; x < QG; ++x) mx[x] = maximum<!C2P>(s, x);
            if constexpr (C2P) {
                bool nan = false;
#pragma unroll
                for (int x = 0; x < QG; ++x) nan = nan || mx[x] != mx[x];
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(nan) != 0, 0)) {
                    if (!far || !EXACT) {
                        scores<true>(s, k_at);
                        if (left < BN) mask(s, left);
                    }
#pragma unroll
                    for (int x = 0; x < QG; ++x) mx[x] = maximum<true>(s, x);
                }
            }
#pragma unroll
            for (int x = 0; x < QG; ++x) {
                const float m_new = fmaxf(m[x], mx[x] + add[x]);
                const bool up = (m_new - m[x]) * c_exp > 8.f;
                const float alpha = up ? __builtin_amdgcn_exp2f((m[x] - m_new) * c_exp) : 1.f;
                l[x] *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) o[dt][x] *= alpha;
                m[x] = up ? m_new : m[x];
            }
            probabilities(s, add, c_exp, pb, sum);
        }
#pragma unroll
        for (int x = 0; x < QG; ++x) {
            l[x] += halves_sum(sum[x]);     // (a lane of the kernels of 32 x 32 tiles has these keys)
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) o[dt][x] = E::mfma(__builtin_bit_cast(X8, vf[c][dt]), pb[x][c], o[dt][x]);
        }
    }

    // Normalised output rows in 16-byte stores: one swap between neighbouring lane rows gives each lane eight consecutive d.
    // Row x 16 + n of the unit is written if it is under `rows`, as zeros from `live` on.
    __device__ __forceinline__ void store(char* out, uint32_t stride, int rows, int live) const {
#pragma unroll
        for (int x = 0; x < QG; ++x) {
            const float inv = 1.f / rows_sum(l[x]);
            const int row = 16 * x + n;
            char* const at = out + uint32_t(row) * stride + 32 * (g & 1) + 16 * (g >> 1);
#pragma unroll
            for (int d2 = 0; d2 < 2; ++d2) {
                u32x2 r[2];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const f32x4 v = o[2 * d2 + k][x] * inv;
                    r[k] = row < live ? u32x2{pack2<E>(v[0], v[1]), pack2<E>(v[2], v[3])} : u32x2{0, 0};
                }
                const auto y = __builtin_amdgcn_permlane16_swap(r[0][0], r[1][0], false, false);
                const auto z = __builtin_amdgcn_permlane16_swap(r[0][1], r[1][1], false, false);
                if (row < rows) *reinterpret_cast<u32x4*>(at + 64 * d2) = u32x4{y[0], z[0], y[1], z[1]};
            }
        }
    }
};

}  // namespace tdb_step
