// Matrix-core disentangled-attention forward for float32, head_dim 64, larger launches: products of bf16 parts (gfx950, MFMA 16x16x32).
//
// A float32 is the sum of three bf16 numbers (rounded to nearest each: what is left after two has 8 bits).  A product is six products of
// parts; the three left out are below 2^-26 of it.  The small ones are summed first, so that the sum is rounded at its full size only
// twice: a sum of 64 products is three times as exact as 16 steps of the float32 MFMA (error 4.6e-8 against 1.45e-7 of the root mean square,
// normal values), in 12 x 16 clk instead of 16 x 32.
//
// Taking a row apart costs 5.5 vector instructions per element, so a workgroup does it once for all its waves: keys, values and table
// rows of a step are requested a step ahead, taken apart in registers and passed through LDS in operand order.
//
// One workgroup = 64 query rows of one (sequence, head), a wave per 16 (SETS = 2: two groups of four waves, each with its half of the keys
// and its half of LDS; their sums meet at the end).  A step is 16 keys.  Relative positions come in tiles e of r = 16 e .. + 15; query
// tile a and key tile b need e = a - b and a - b - 1.  The tiles of a step lie in a ring of five; a step brings one new one, and there are two
// buffers for values: 78 KB a set, two workgroups (or two sets) to a compute unit.
//   p2c  P'[key][r] = K_key . Q_r[delta(r)], lanes along r; c2p  C'[query][r], lanes along r (mirrored), the upper tile's kept from the
//   step before.  Both are turned into place in registers as in attn_step.h, in 32 bits; c2p is added by a product with an identity.
//
// What bounds it: a step's chain.  One workgroup alone on a compute unit takes 3060 clk a step, two 4400: per wave 60 matrix instructions of 16 clk and
// 4 of 32, some 250 vector ones, 24 + 12 reads and 12 writes of LDS, whose port is busy for 1830 clk of the 4400.  Measured against
// attn_f32.hip, error against 64 bits (2-norm) in brackets: 8 x 12 heads, lengths 96..384 65.6 -> 45.6 us (1.80e-7 -> 1.18e-7); 8 x 512 158 -> 112
// (2.33e-7 -> 1.43e-7); 32 x 128 56.4 -> 36.7 (1.50e-7 -> 1.05e-7); 2 x 512 with two sets 55.5 -> 39.5.  Without wait for the loads of the table of
// indexes behind a branch 158 -> 126 for 8 x 512, with descriptors instead of clamped addresses 126 -> 115, with the rows passed on in the middle of a step
// instead of between two 115 -> 111.  No gain: schedules without groups, all LDS reads first (5 % slower), two sets that wait
// for themselves only (5 % slower), the next rows' parts shared out over both stages of products (5 % slower).
//
// An infinity has no parts (its rest is NaN), nor has what rounds to one: a wave whose results are not all finite computes its rows
// again from the float32 operands and takes what was not finite from there.  A NaN or an infinity in each sequence costs that for all its rows: 8 x 512
// 132 -> 345 us, 2 x 4096 1.5 -> 4.4 ms (one key after another 1950 us and 14.2 ms; attn_f32.hip, which needs nothing of the kind, 160 to 170 us
// and 2.2 ms).
// Operands below about 1e-33 lose bits of their third part, at most TINY each (bf16 has the exponents of float32).  In a score that is nothing
// unless what it is multiplied with is beyond LARGE; in a result it is unless the result is as small.  Both are looked for, and such results
// are computed again too.  (Against no such look 8 of 96..384 50.6 -> 51.2 us, 8 x 512 118.3 -> 120, 32 x 128 38.9 -> 40.1, 2 x 512 40.2 -> 40.8; errors of
// 150 keys whose values are 1e-36 2.5e-5 -> 1.8e-7, whose keys are 1e36 and queries 1e-36 2.6e-5 -> 1.8e-7; attn_f32.hip 3.9e-7.)
// (Same definition as the other kernels: modeling_deberta_v2.py:243, :317-324, :337-343.)
#include <algorithm>
#include <atomic>
#include <cfloat>
#include <type_traits>

#include "attn_step.h"
#include "tdb_internal.h"

namespace {

using namespace tdb_step;
using E = Elem<TDB_BF16>;

constexpr int D = 64;
constexpr int ROWS = 64;                    // query rows of a workgroup
constexpr int PLANE = 16 * ROW, TILE = 3 * PLANE;       // bytes of 16 rows x 64: one part, all three
constexpr int RING = 5;
constexpr int GAP_WGS = 64;                 // workgroups that look for packed rows outside every sequence
constexpr int tiles_bytes(bool c2p, bool p2c) { return TILE * (3 + RING * (int(c2p) + int(p2c))); }
constexpr int MAGS = 5 * D;                 // floats: largest magnitudes that each wave of a set has passed on, and the second one when it opened
constexpr int smem_bytes(bool c2p, bool p2c, int sets) { return sets * (tiles_bytes(c2p, p2c) + 4 * MAGS); }

// What the parts of an operand may miss: half of the least subnormal bf16 (the products take them as they are).  128 products of TINY and LARGE
// are 2^-63 of a score; a scale (up to LARGE_SCALE) makes 2^-33 of that.
constexpr float TINY = 0x1p-134f, LARGE = 0x1p64f, LARGE_SCALE = 0x1p30f;

struct Parts {                              // of eight elements
    bf16x8 p[3];
};

__device__ __forceinline__ float largest(float mag, float x, float y) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(mag) : "v"(x), "v"(y));      // (fmaxf of what was loaded has an instruction more for each of them)
    return mag;
}

// The three parts of two values, packed.
__device__ __forceinline__ void split2(float x, float y, uint32_t (&w)[3]) {
    w[0] = packed2<E>(x, y);
    const float x1 = x - E::low(w[0]), y1 = y - E::high(w[0]);
    w[1] = packed2<E>(x1, y1);
    w[2] = pack2<E>(x1 - E::low(w[1]), y1 - E::high(w[1]));
}

// Sum over 64 columns (two halves), small products first.
__device__ __forceinline__ void dot_small(const Parts (&x)[2], const Parts (&y)[2], f32x4& acc) {
    constexpr int order[5][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}};
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) acc = E::mfma(x[h].p[order[i][0]], y[h].p[order[i][1]], acc);
}
__device__ __forceinline__ void dot_large(const Parts (&x)[2], const Parts (&y)[2], f32x4& acc) {
#pragma unroll
    for (int h = 0; h < 2; ++h) acc = E::mfma(x[h].p[0], y[h].p[0], acc);
}
__device__ __forceinline__ f32x4 dot(const Parts (&x)[2], const Parts (&y)[2]) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    dot_small(x, y, acc);
    dot_large(x, y, acc);
    return acc;
}

__device__ __forceinline__ float fold_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 16));
    return fmaxf(x, __shfl_xor(x, 32));
}
// Of the lanes that have the same columns, without LDS.
__device__ __forceinline__ float rows_max(float x) {
    const uint32_t u = bits(x);
    const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t v = bits(fmaxf(__builtin_bit_cast(float, uint32_t(h[0])), __builtin_bit_cast(float, uint32_t(h[1]))));
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return fmaxf(__builtin_bit_cast(float, uint32_t(r[0])), __builtin_bit_cast(float, uint32_t(r[1])));
}
__device__ __forceinline__ float fold_sum(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}

template <bool C2P, bool P2C, int SETS>
__global__ __launch_bounds__(SETS * 256, 2) void attn_f32_split_kernel(const TdbKernelParams p, const int tiles_x) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int SET = tiles_bytes(C2P, P2C);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int a = wave & 3, set = SETS > 1 ? wave >> 2 : 0;
    const int n = l & 15, g = l >> 4;

    if (p.gap_cu && blockIdx.x + GAP_WGS >= gridDim.x) {
        const int worker = (blockIdx.x + GAP_WGS - gridDim.x) * (4 * SETS) + wave;
        tdb_fill_gaps(p.gap_cu, p.gap_B, p.L, p.total, static_cast<char*>(p.o), p.os_l * 4, p.os_h * 4, p.H, 4 * D, worker, GAP_WGS * 4 * SETS);
        return;
    }

    // Block ids go round-robin over the 8 XCDs: four neighbouring query tiles, which read the same keys and values, on one of them.
    const int slot = blockIdx.x >> 3;
    const int group = (slot >> 2) * 8 + (blockIdx.x & 7), h = group % p.H, tile = group / p.H * 4 + (slot & 3);
    int b, row0, len;
    int64_t tok0;
    if (tile >= tiles_x || !tdb_locate_tile_sorted(p, ROWS, tile, b, row0, len, tok0)) return;
    b = __builtin_amdgcn_readfirstlane(b), row0 = __builtin_amdgcn_readfirstlane(row0), len = __builtin_amdgcn_readfirstlane(len);

    auto base = [&](const void* ptr, int64_t sb, int64_t sh, int64_t sl) {
        return static_cast<const float*>(ptr) + (p.varlen ? tok0 * sl : int64_t(b) * sb) + int64_t(h) * sh;
    };
    float* const O = const_cast<float*>(base(p.o, p.os_b, p.os_h, p.os_l));
    const int rows_here = min(ROWS, (p.varlen ? len : p.L) - row0);
    if (row0 >= len) {                      // padded query rows only (fixed layout): zeros
        for (int idx = threadIdx.x; idx < rows_here * (D / 4); idx += SETS * 256)
            *reinterpret_cast<f32x4*>(O + int64_t(row0 + idx / (D / 4)) * p.os_l + idx % (D / 4) * 4) = f32x4{0.f, 0.f, 0.f, 0.f};
        return;
    }
    const float* const Q = base(p.q, p.qs_b, p.qs_h, p.qs_l);
    const float* const K = base(p.k, p.ks_b, p.ks_h, p.ks_l);
    const float* const V = base(p.v, p.vs_b, p.vs_h, p.vs_l);
    const float* const KR = static_cast<const float*>(p.pk) + int64_t(h) * p.pks_h;
    const float* const QR = static_cast<const float*>(p.pq) + int64_t(h) * p.pqs_h;
    auto delta_of = [&](int r) { return p.lut[min(max(r + p.lut_half, 0), 2 * p.lut_half)]; };

    const int ntiles = (len + 15) >> 4, steps = (ntiles + SETS - 1) / SETS;
    const int b0 = set * steps, a0 = row0 >> 4;      // (a0: tile of the workgroup's first query)
    const bool live = row0 + 16 * a < len;

    // Each wave of a set passes on one kind of rows: 0 keys, 1 values, 2 K_r, 3 Q_r.  A lane has four columns of rows 4 t + g.
    const uint32_t set_at = set * SET;
    auto tile_at = [&](int kind, int e) {   // LDS offset of a tile: keys, values, or position tile e
        const int slot = ((e % RING) + RING) % RING;
        return set_at + uint32_t(kind == 0 ? 0 : kind == 1 ? (1 + (e & 1)) * TILE : (3 + (kind == 3 && C2P ? RING : 0) + slot) * TILE);
    };
    // Loads through descriptors: rows past the end are zeros (values there may be anything, and their probability is 0), indexes past the
    // end of their table are 0, a row that exists and that nothing uses.
    const int lane_col = 16 * n;
    auto stride_of = [&](int kind) { return int(kind == 0 ? p.ks_l : kind == 1 ? p.vs_l : kind == 2 ? p.pks_r : p.pqs_r) * 4; };
    auto rows_from = [&](const float* base, int rows, int stride) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, rows > 0 ? (rows - 1) * stride + 4 * D : 0, 0x00020000);
    };
    auto rows_of_tile = [&](int kind, int e, int stride) {      // (a table that is not there has no rows: nothing is read)
        const bool there = kind < 2 || (kind == 2 ? C2P : P2C);
        const float* const base = kind == 0 || !there ? K : kind == 1 ? V : kind == 2 ? KR : QR;
        return rows_from(kind < 2 ? base + int64_t(4 * e) * stride : base, !there ? 0 : kind < 2 ? len - 16 * e : 2 * p.span, stride);
    };
    const __amdgpu_buffer_rsrc_t lut = __builtin_amdgcn_make_buffer_rsrc(const_cast<int*>(p.lut), 0, (2 * p.lut_half + 1) * 4, 0x00020000);
    auto read_deltas = [&](int e, int (&d)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) d[t] = __builtin_amdgcn_raw_buffer_load_b32(lut, (16 * e + g + p.lut_half) * 4 + 16 * t, 0, 0);
    };
    auto request = [&](const __amdgpu_buffer_rsrc_t& from, const int (&at)[4], f32x4 (&x)[4]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) x[t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(from, at[t], 0, 0));
    };
    auto take_apart = [&](const f32x4 (&x)[4], u32x2 (&w)[4][3], auto from, auto to) {
#pragma unroll
        for (int t = decltype(from)::value; t < decltype(to)::value; ++t) {
            uint32_t lo[3], hi[3];
            split2(x[t][0], x[t][1], lo);
            split2(x[t][2], x[t][3], hi);
#pragma unroll
            for (int i = 0; i < 3; ++i) w[t][i] = u32x2{lo[i], hi[i]};
        }
    };
    auto put = [&](int kind, uint32_t at, const u32x2 (&w)[4][3]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint32_t row = 4 * t + g, chunk = n >> 1;
            const uint32_t to = at + (kind == 1 ? value_at(row, chunk) : operand_at(row, chunk)) + 8 * (n & 1);
#pragma unroll
            for (int i = 0; i < 3; ++i) *(__attribute__((address_space(3))) u32x2*)(to + PLANE * i) = w[t][i];
        }
    };
    // Largest magnitudes, of each column that this lane passes on.  (NaN passes by: it shows in the results.)
    auto look = [&](const f32x4 (&x)[4], f32x4& mag) {
#pragma unroll
        for (int t = 0; t < 4; t += 2)
#pragma unroll
            for (int c = 0; c < 4; ++c) mag[c] = largest(mag[c], x[t][c], x[t + 1][c]);
    };
    f32x4 mag = {0.f, 0.f, 0.f, 0.f}, mag_first = mag;      // (mag_first: of the tables' rows in the opening, whichever wave has them)
    // Opening: the first keys and values, and five tiles of each table.
    {
        int d[3][4];
        f32x4 x[3][4];
        constexpr int ITEMS = 2 + RING * (int(C2P) + int(P2C));
        auto item = [&](int i, int& kind, int& e) {
            const int at = a + 4 * i;
            kind = at < 2 ? at : at < 2 + RING && C2P ? 2 : 3;
            e = at < 2 ? b0 : a0 - b0 - 1 + (at - 2) % RING;
        };
        if (C2P || P2C) {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                int kind, e;
                item(i, kind, e);
                read_deltas(e, d[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (a + 4 * i < ITEMS) {
                int kind, e, at[4];
                item(i, kind, e);
                const int stride = stride_of(kind);
#pragma unroll
                for (int t = 0; t < 4; ++t) at[t] = (kind < 2 ? 4 * t + g : d[i][t]) * stride + lane_col;
                request(rows_of_tile(kind, e, stride), at, x[i]);
            }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            if (a + 4 * i < ITEMS) {
                int kind, e;
                item(i, kind, e);
                look(x[i], i ? mag_first : mag);
                u32x2 w[4][3];
                take_apart(x[i], w, Int<0>{}, Int<4>{});
                put(kind, tile_at(kind, e), w);
            }
    }
    Parts q[2];
    bool plain = true;                      // this lane's query is finite and not LARGE.  (Another one takes part as zeros: infinite c2p terms would reach its neighbours.)
    {
        const float* const row = Q + int64_t(min(row0 + 16 * a + n, len - 1)) * p.qs_l + 8 * g;
        f32x4 x[4];
        bool ok = true;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = *reinterpret_cast<const f32x4*>(row + 32 * (i >> 1) + 4 * (i & 1));
#pragma unroll
            for (int t = 0; t < 4; ++t) ok = ok && fabsf(x[i][t]) <= LARGE;
        }
        const uint64_t other = __builtin_amdgcn_ballot_w64(!ok);
        plain = !((other >> n | other >> (n + 16) | other >> (n + 32) | other >> (n + 48)) & 1);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            uint32_t w[4][3];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f32x4& y = x[2 * half + (i >> 1)];
                split2(y[2 * (i & 1)], y[2 * (i & 1) + 1], w[i]);
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) q[half].p[i] = __builtin_bit_cast(bf16x8, plain ? u32x4{w[0][i], w[1][i], w[2][i], w[3][i]} : u32x4{0, 0, 0, 0});
        }
    }
    const uint32_t frag_lane = operand_at(n, g), mirror_lane = operand_at(15 - n, g), v_lane = value_at(4 * g + (n >> 2), 0) + 8 * (n & 3);
    bool in[5];                             // n + 4 g + t < 16
#pragma unroll
    for (int t = 0; t < 5; ++t) in[t] = n + 4 * g + t < 16;
    float one[4];                           // identity
#pragma unroll
    for (int t = 0; t < 4; ++t) one[t] = n == 4 * g + t ? 1.f : 0.f;
    auto frags = [&](uint32_t at, uint32_t lane, Parts (&x)[2]) {
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int i = 0; i < 3; ++i) x[half].p[i] = *(const __attribute__((address_space(3))) bf16x8*)(at + PLANE * i + (lane ^ (64 * half)));
    };

    f32x4 o[4], low[4], upper = {0.f, 0.f, 0.f, 0.f};       // O^T: d = 16 dt + 4 g + t of query n, and its small products; c2p products of the step's upper tile
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = low[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -FLT_MAX, sum = 0.f;          // running maximum (in powers of two), this lane's sum
    const float c_exp = p.scale * 1.44269504f;

    // Rows are requested half a step after those of the step before, a step and a half before they are used; their table indexes a
    // step earlier.
    const int kind = a;
    const bool table = (kind == 2 && C2P) || (kind == 3 && P2C), passes = kind < 2 || table;
    const int stride = passes ? stride_of(kind) : 0;
    auto tile_of = [&](int step) { return kind < 2 ? step : a0 - step - 1; };
    int delta[4], at[4];
    f32x4 x[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) at[t] = (4 * t + g) * stride + lane_col;
    auto next_deltas = [&](int step) {      // (where the rows of `step` are, and the indexes of the one behind)
        if (table) {
#pragma unroll
            for (int t = 0; t < 4; ++t) at[t] = delta[t] * stride + lane_col;
            read_deltas(tile_of(step + 1), delta);
        }
    };
    auto next_rows = [&](int step) { request(rows_of_tile(kind, tile_of(step), stride), at, x); };
    if (table) read_deltas(tile_of(b0 + 1), delta);
    next_deltas(b0 + 1);
    next_rows(b0 + 1);
    __syncthreads();
    if (C2P) {
        Parts kr[2];
        frags(tile_at(2, a0 + a - b0), mirror_lane, kr);
        upper = dot(q, kr);
    }
    for (int i = 0; i < steps; ++i) {
        const int bt = b0 + i;
        const bool more = i + 1 < steps;
        u32x2 w[4][3];
        {
#pragma clang fp contract(off)                // (a scaled score and its maximum are rounded alike, or large ones differ by more than they should)
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            Parts kf[2], kr[2], qh[2], ql[2];
            f32x4 s = zero, ph = zero, pl = zero, lower = zero, c;
            if constexpr (C2P) frags(tile_at(2, a0 + a - bt - 1), mirror_lane, kr);
            if (SETS > 1) __builtin_amdgcn_s_setprio(1);    // (its products feed one another: before the other set's softmax, 3 %)
            frags(set_at, frag_lane, kf);
            if constexpr (P2C) {
                frags(tile_at(3, a0 + a - bt), frag_lane, qh);
                frags(tile_at(3, a0 + a - bt - 1), frag_lane, ql);
            }
            // Two sums side by side: a chain of products waits for itself.
            constexpr int order[6][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}, {0, 0}};
#pragma unroll
            for (int o = 0; o < 6; ++o)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int u = order[o][0], v = order[o][1];
                    if constexpr (C2P) lower = E::mfma(q[half].p[u], kr[half].p[v], lower);
                    if (o < 5) s = E::mfma(kf[half].p[u], q[half].p[v], s);
                }
            take_apart(x, w, Int<0>{}, Int<4>{});
            look(x, mag);
            stage_end<10 + 12 * int(C2P), 3>();
            if constexpr (P2C) {
#pragma unroll
                for (int o = 0; o < 6; ++o)
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const int u = order[o][0], v = order[o][1];
                        ph = E::mfma(kf[half].p[u], qh[half].p[v], ph);
                        pl = E::mfma(kf[half].p[u], ql[half].p[v], pl);
                    }
            }
            if constexpr (C2P) {
                const uint32_t on[4] = {bits(lower[0]), bits(lower[1]), bits(lower[2]), bits(lower[3])};
                const uint32_t before[4] = {bits(upper[0]), bits(upper[1]), bits(upper[2]), bits(upper[3])};
                c = __builtin_bit_cast(f32x4, turned<1>(in, on, before));
                upper = lower;
            }
            stage_end<24 * int(P2C), 1>();
            // (The fragments of this step's keys and positions are in registers; there are two buffers for values.)
            next_deltas(bt + 2);
            next_rows(bt + 2);
            if (more) {
                __syncthreads();
                if (passes) put(kind, tile_at(kind, tile_of(bt + 1)), w);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (C2P) {
#pragma unroll
                for (int t = 0; t < 4; ++t) s = __builtin_amdgcn_mfma_f32_16x16x4f32(c[t], one[t], s, 0, 0, 0);
            }
            dot_large(kf, q, s);
            if constexpr (P2C) {
                const uint32_t on[4] = {bits(ph[0]), bits(ph[1]), bits(ph[2]), bits(ph[3])}, before[4] = {bits(pl[0]), bits(pl[1]), bits(pl[2]), bits(pl[3])};
                s += __builtin_bit_cast(f32x4, turned<0>(in, on, before));
            }
            s *= c_exp;
            asm volatile("" : "+v"(s));     // (read ahead of the condition below: see tdb_settled)
            if (SETS > 1) __builtin_amdgcn_s_setprio(0);
            if (16 * (bt + 1) > len) {
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (16 * bt + 4 * g + t >= len) s[t] = -INFINITY;
            }
            // The maximum is raised only where a score exceeds it by more than 2^4.
            float e[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) e[t] = s[t] - m;
            const float most = fmaxf(fmaxf(e[0], e[1]), fmaxf(e[2], e[3]));
            if (__builtin_amdgcn_ballot_w64(most > 4.f) != 0) {
                const float up = fmaxf(m, fold_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])))), alpha = __builtin_amdgcn_exp2f(m - up);
                m = up, sum *= alpha;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) o[dt] *= alpha, low[dt] *= alpha;
#pragma unroll
                for (int t = 0; t < 4; ++t) e[t] = s[t] - m;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) e[t] = __builtin_amdgcn_exp2f(e[t]);
            sum += (e[0] + e[1]) + (e[2] + e[3]);
            uint32_t lo[3], hi[3];
            split2(e[0], e[1], lo);
            split2(e[2], e[3], hi);
            // Sixteen keys fill half a product: two parts of a value side by side.
            const bf16x8 p_ml = __builtin_bit_cast(bf16x8, u32x4{lo[1], hi[1], lo[2], hi[2]});
            const bf16x8 p_hm = __builtin_bit_cast(bf16x8, u32x4{lo[0], hi[0], lo[1], hi[1]});
            const bf16x8 p_hh = __builtin_bit_cast(bf16x8, u32x4{lo[0], hi[0], lo[0], hi[0]});
            const uint32_t v_at = tile_at(1, bt);
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                s16x4 v[3];
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    v[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(v_at + PLANE * i + (v_lane ^ (32 * dt))));
                const bf16x8 v_mh = __builtin_bit_cast(bf16x8, s16x8{v[1][0], v[1][1], v[1][2], v[1][3], v[0][0], v[0][1], v[0][2], v[0][3]});
                const bf16x8 v_lh = __builtin_bit_cast(bf16x8, s16x8{v[2][0], v[2][1], v[2][2], v[2][3], v[0][0], v[0][1], v[0][2], v[0][3]});
                low[dt] = E::mfma(v_mh, p_ml, low[dt]);     // m m + h l
                low[dt] = E::mfma(v_mh, p_hm, low[dt]);     // m h + h m
                o[dt] += E::mfma(v_lh, p_hh, zero);         // l h + h h (added here: rounded to nearest)
            }
        }
        if (more) __syncthreads();
    }

#pragma unroll
    for (int dt = 0; dt < 4; ++dt) {
        o[dt] += tdb_settled(low[dt]);
    }
    {
        float* const mine = reinterpret_cast<float*>(smem + SETS * SET) + set * MAGS;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (a != 1) mag[c] = fmaxf(mag[c], mag_first[c]);
            mag[c] = rows_max(mag[c]);
        }
        if (g == 0) *reinterpret_cast<f32x4*>(&mine[D * a + 4 * n]) = mag;
        if (a == 1) mine[4 * D + l] = fmaxf(fmaxf(mag_first[0], mag_first[1]), fmaxf(mag_first[2], mag_first[3]));
    }
    if constexpr (SETS > 1) {               // the second set's sums to the first one
        __syncthreads();
        float* const mine = reinterpret_cast<float*>(smem) + a * (64 * 18);
        if (set == 1) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) *reinterpret_cast<f32x4*>(&mine[(dt * 64 + l) * 4]) = o[dt];
            mine[1024 + l] = m, mine[1088 + l] = sum;
        }
        __syncthreads();
        if (set == 1) return;
        const float m1 = mine[1024 + l], top = fmaxf(m, m1), f0 = __builtin_amdgcn_exp2f(m - top), f1 = __builtin_amdgcn_exp2f(m1 - top);
        sum = sum * f0 + mine[1088 + l] * f1;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] = o[dt] * f0 + *reinterpret_cast<const f32x4*>(&mine[(dt * 64 + l) * 4]) * f1;
    }
    const int row_mine = row0 + 16 * a + n;
    if constexpr (SETS == 1) __syncthreads();       // (the magnitudes are there; the other waves' last step is over: its LDS is written below)
    const float* const seen = reinterpret_cast<const float*>(smem + SETS * SET);
    float of_kr = 0.f, of_v = 0.f;
#pragma unroll
    for (int i = 0; i < 5 * SETS; ++i) (i % 5 == 1 ? of_v : of_kr) = fmaxf(i % 5 == 1 ? of_v : of_kr, seen[D * i + l]);
    // A value misses up to TINY, a probability (of up to 4096 keys) too: a result has to exceed what that makes by 2^26.
    constexpr float LEAST = 0x1p26f * TINY, LEAST_BY = 0x1p38f * TINY, ORDINARY = 0x1p40f;
    const bool sound = __builtin_amdgcn_ballot_w64(of_kr > LARGE && of_kr <= FLT_MAX) == 0;
    const bool ordinary = sound && __builtin_amdgcn_ballot_w64(of_v > ORDINARY) == 0;
    const float inv = 1.f / fold_sum(sum);
    float total = 0.f, least = FLT_MAX;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            o[dt][t] *= inv;
            total += fabsf(o[dt][t]);       // (neither NaN nor an infinity passes by)
            least = fminf(least, fabsf(o[dt][t]));
        }
    uint32_t keep = plain && ordinary && total <= FLT_MAX && least >= LEAST_BY * ORDINARY ? 0xffff : 0;      // results that stay
    if (__builtin_expect(live && __builtin_amdgcn_ballot_w64(keep == 0 && row_mine < len) != 0, 0)) {
        keep = 0;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            f32x4 v = *reinterpret_cast<const f32x4*>(&seen[D + 16 * dt + 4 * g]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (SETS > 1) v[t] = fmaxf(v[t], seen[MAGS + D + 16 * dt + 4 * g + t]);
                const float x = fabsf(o[dt][t]);
                // (Zeros are ordinary results, but not of tiny values.)
                const bool enough = x >= fmaxf(LEAST, v[t] * LEAST_BY) || (x == 0.f && (v[t] == 0.f || v[t] > 0x1p16f * TINY));
                if (plain && sound && x <= FLT_MAX && enough) keep |= 1u << (4 * dt + t);
            }
        }
    }
    if (__builtin_expect(live && __builtin_amdgcn_ballot_w64(keep != 0xffff && row_mine < len) != 0, 0)) {
        // Again, as in attn_f32.hip: tiles of 16 keys, the position products through this wave's own LDS.  The results' layout is that of `o`.
        constexpr int CS = 36;
        float* const sC = reinterpret_cast<float*>(smem) + a * (2 * 16 * CS);
        float* const sP = sC + 16 * CS;
        auto fence = [] {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        auto row_of = [&](f32x4 (&f)[4], const float* row) {
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) f[dt] = *reinterpret_cast<const f32x4*>(row + 16 * dt + 4 * g);
        };
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        auto product = [&](const f32x4 (&x)[4], const f32x4 (&y)[4]) {      // (four sums of 16: rounded at its full size two times for sixteen)
            f32x4 acc[4];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[i & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i >> 2][i & 3], y[i >> 2][i & 3], i < 4 ? zero : acc[i & 3], 0, 0, 0);
            return (acc[0] + acc[1]) + (acc[2] + acc[3]);
        };
        f32x4 qf[4], kr[4], qr[2][4], c[2] = {zero, zero}, res[4];      // [0]: the step's lower position tile, [1]: its upper one, the lower one of the step before
        row_of(qf, Q + int64_t(min(row_mine, len - 1)) * p.qs_l);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) res[dt] = zero;
        float top = -FLT_MAX, all = 0.f;
        int64_t d = 0;
        if (C2P || P2C) {
            d = delta_of(16 * (a0 + a) + n);
            if (C2P) row_of(kr, KR + d * p.pks_r), c[1] = product(kr, qf);
            if (P2C) row_of(qr[1], QR + d * p.pqs_r);
            d = delta_of(16 * (a0 + a - 1) + n);
        }
        for (int b = 0; b < ntiles; ++b) {
            f32x4 kf[4], s = zero;
            float v[4][4];
            row_of(kf, K + int64_t(min(16 * b + n, len - 1)) * p.ks_l);
            if (C2P) row_of(kr, KR + d * p.pks_r);
            if (P2C) row_of(qr[0], QR + d * p.pqs_r);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int key = 16 * b + 4 * g + t;
                const float* const row = V + int64_t(min(key, len - 1)) * p.vs_l + n;
#pragma unroll
                for (int dt = 0; dt < 4; ++dt) v[dt][t] = key < len ? row[16 * dt] : 0.f;
            }
            if (C2P || P2C) {
                d = delta_of(16 * (a0 + a - b - 2) + n);
                if (C2P) {
                    c[0] = product(kr, qf);
#pragma unroll
                    for (int x = 0; x < 2; ++x) *reinterpret_cast<f32x4*>(&sC[n * CS + 16 * x + 4 * g]) = c[x];
                    c[1] = c[0];
                }
                if (P2C) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) *reinterpret_cast<f32x4*>(&sP[n * CS + 16 * x + 4 * g]) = product(qr[x], kf);
#pragma unroll
                    for (int dt = 0; dt < 4; ++dt) qr[1][dt] = qr[0][dt];
                }
                fence();
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int r = 16 + n - (4 * g + t);
                    if (C2P) s[t] = sC[n * CS + r];
                    if (P2C) s[t] += sP[(4 * g + t) * CS + r];
                }
                fence();
            }
            s += product(kf, qf);
            float most = -INFINITY;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                s[t] = 16 * b + 4 * g + t < len ? s[t] * p.scale : -INFINITY;
                most = fmaxf(most, s[t]);               // (NaN scores pass it by and meet expf)
            }
            const float up = fmaxf(top, fold_max(most)), alpha = expf(top - up);
            top = up, all *= alpha;
#pragma unroll
            for (int t = 0; t < 4; ++t) s[t] = expf(s[t] - up), all += s[t];
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) {
                f32x4 add = zero;           // (the tile's own sum first)
#pragma unroll
                for (int t = 0; t < 4; ++t) add = __builtin_amdgcn_mfma_f32_16x16x4f32(v[dt][t], s[t], add, 0, 0, 0);
                res[dt] = res[dt] * alpha + add;
            }
        }
        const float div = 1.f / fold_sum(all);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int t = 0; t < 4; ++t) o[dt][t] = keep >> (4 * dt + t) & 1 ? o[dt][t] : res[dt][t] * div;
    }
    if (row_mine < row0 + rows_here) {
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
            *reinterpret_cast<f32x4*>(O + int64_t(row_mine) * p.os_l + 16 * dt + 4 * g) = row_mine < len ? o[dt] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
}

}  // namespace

// (Offsets inside a sequence and a table are 32-bit numbers here.)
bool tdb_f32_split_supported(const TdbKernelParams& p, int dtype) {
    auto fits = [](int64_t rows, int64_t stride) { return stride <= (int64_t(INT32_MAX) / 4 - 1024) / std::max<int64_t>(rows, 1); };
    return dtype == TDB_F32 && p.D == D && fabsf(p.scale) <= LARGE_SCALE && !p.c2p && !p.p2c && fits(int64_t(p.L) + 16, std::max(p.ks_l, p.vs_l)) &&
           (!p.pk || fits(2 * int64_t(p.span), p.pks_r)) && (!p.pq || fits(2 * int64_t(p.span), p.pqs_r));
}

namespace {
int tiles_of(const TdbKernelParams& p) { return p.varlen ? p.total / ROWS + p.B : p.B * ((p.L + ROWS - 1) / ROWS); }
int64_t blocks_of(const TdbKernelParams& p) { return (int64_t((tiles_of(p) + 3) / 4) * p.H + 7) / 8 * 32; }      // groups of 4 tiles, rounded up to 8 XCDs
}  // namespace

// How many sets of waves make a launch faster than attn_f32.hip does, or 0.  Fitted to 4000 random launches (16 to 1200 keys, 6 to 16 heads, lengths evenly
// spread and such as texts have).  Equal lengths: 574 taken, 1.214x, 9 of these below 0.97x, 0.86x at worst; packed: 442, 1.176x, 31, 0.84x; padded, of which
// the host knows the longest possible length only: evenly spread 271, 1.18x, 30, 0.76x; as texts have them 282, 1.09x, 73, and down to 0.58x where
// most of a batch is padding (10 of up to 248, 45 in the mean, 22 -> 35 us): a limit that spares these would cost full batches as much.
//   * as many workgroups as compute units: two sets, from three quarters of the units on (4 x 256 32.2 -> 24.0 us, 2 x 512 55.5 -> 39; 4 x 128, half of the
//     units, 15 either way), earlier for long texts, where the opening of a workgroup (2.5 us) weighs less (3 x 190 26.0 -> 19.7).  Short texts leave the
//     second set little (9 of 53..66 11.7 -> 14.3), and a long one among them decides alone, which the four waves of the other kernel share (packed, half of the
//     longest in the mean: below 0.7 to 1.04x, 14 of 36 below 0.97x; above 1.1 to 1.39x).  With lengths, of which the host knows the longest possible, a good
//     half of the workgroups has keys;
//   * more: one set, two workgroups to a compute unit (8 of 96..384 65.6 -> 46, 32 x 128 56.4 -> 37), but not for one or two key tiles (44 x 21 12.3 -> 15.9),
//     nor for one term alone where the units are hardly filled (7 x 134 17.3 -> 20.9), nor up to one and a half workgroups to a unit if lengths are far apart
//     (packed, mean below 0.55: 0.6 to 1.0x) or the second of two is nearly empty (9 x 68, 16 heads, 18.3 -> 21.8), nor for an eighth more than the units
//     if they may be padding (0.9x).
int tdb_f32_split_sets(const TdbKernelParams& p) {
    const int64_t units = tdb_compute_units(-1), wgs = int64_t(tiles_of(p)) * p.H;
    const bool both = p.pk && p.pq, lengths = p.varlen || p.seqlens;
    const double mean = p.varlen ? double(p.total) / p.B / p.L : 1.0;
    if (blocks_of(p) <= (p.seqlens && p.L > 200 ? units * 25 / 16 : units)) {
        const int64_t least = p.L <= 160 ? units * 3 / 4 : both ? units * 17 / 32 : units * 21 / 32;
        return p.L > 80 && wgs >= least && (both || p.L >= 300) && mean >= 0.5 ? 2 : 0;
    }
    const int keys = p.varlen ? p.total / p.B : p.L;
    if (keys <= (lengths ? 40 : 32) || (!both && wgs <= units * 17 / 16)) return 0;
    if (wgs <= units * 3 / 2 && (mean < 0.55 || (keys > 64 && keys <= 80))) return 0;
    return p.seqlens && wgs <= units * 9 / 8 ? 0 : 1;
}

hipError_t tdb_launch_f32_split(const TdbKernelParams& p, int sets, hipStream_t stream) {
    const int tiles = tiles_of(p);
    const int64_t blocks = blocks_of(p) + (p.gap_cu ? GAP_WGS : 0);
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    int dev = 0;
    if (const hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
    auto launch = [&](auto c, auto x, auto s) {
        constexpr bool C2P = decltype(c)::value, P2C = decltype(x)::value;
        constexpr int SETS = decltype(s)::value;
        const auto kernel = attn_f32_split_kernel<C2P, P2C, SETS>;
        constexpr int smem = smem_bytes(C2P, P2C, SETS);
        static std::atomic<uint64_t> raised{0};     // devices whose limit for this instance is raised (twice does no harm)
        const uint64_t bit = uint64_t(1) << (dev & 63);
        if (dev >= 64 || !(raised.load(std::memory_order_relaxed) & bit)) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
            if (e != hipSuccess) return e;
            if (dev < 64) raised.fetch_or(bit, std::memory_order_relaxed);
        }
        hipLaunchKernelGGL(kernel, dim3(unsigned(blocks)), dim3(256 * SETS), smem, stream, p, tiles);
        return hipGetLastError();
    };
    auto terms = [&](auto s) {
        using std::bool_constant;
        if (p.pk && p.pq) return launch(bool_constant<true>{}, bool_constant<true>{}, s);
        if (p.pk) return launch(bool_constant<true>{}, bool_constant<false>{}, s);
        if (p.pq) return launch(bool_constant<false>{}, bool_constant<true>{}, s);
        return launch(bool_constant<false>{}, bool_constant<false>{}, s);
    };
    return sets > 1 ? terms(Int<2>{}) : terms(Int<1>{});
}
