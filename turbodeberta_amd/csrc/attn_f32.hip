// Matrix-core disentangled-attention forward for float32, head_dim 64 (gfx950, wave64, MFMA 16x16x4 f32).
//
// float32 is the type checkpoints load in.  Products and sums are float32 FMAs, on the matrix cores (152 TFLOP/s measured for a large
// product; the packed vector forms that would reach that rate are not used here).  Larger launches with tables are attn_f32_split.hip's: here
// a wave reads its own operands, and taking them apart for bf16 products would cost it what those products save.
//
// What bounds it: the matrix pipe.  A 16 x 16 x 64 tile product takes 16 MFMAs = 512 clk, sixteen times a bf16 one, so
// everything else is chosen to be simple rather than cheap: operands go straight from global memory to registers (a
// fragment is four 16-byte loads whose lanes cover 64 contiguous bytes of 16 rows), the two position terms are shifted
// through a wave's own LDS scratch with plain 4-byte reads, and no wave waits for another until the end.
//
// Measured (vector-ALU kernel before): 1 x 20 x 12 heads 24 -> 5.6 us; 2 x 128 84 -> 9.1 (bound by its chain of loads and products, with
// three waves to a compute unit).  What launches above its present ones took here, before they went to attn_f32_split.hip: 8 x 12 heads, lengths
// 96..384, 66 us; 8 x 512 full 157 us = 83 TFLOP/s without credit for the half-used outer tiles, 103 with (matrix pipe busy 65 % of the time; what
// is left is the start and end of a workgroup, a tenth, and L2 latency that two waves per SIMD do not quite cover).
//
// One workgroup = QT*16 query rows of one (sequence, head); its four waves share out the KEYS (blocks of two
// 16-key tiles, in turn) and merge their partial softmax sums through LDS at the end.  Splitting the keys rather than the
// queries gives a 2 x 128 x 12 head call 768 waves of work instead of 96.  QT = 2 spends 1.25x the products the
// formulation cannot do without (a 16-wide position tile serves 16 + 16 query-key diagonals, and the outer ones of a
// block are only half used), QT = 1 1.375x but twice the workgroups: see tdb_launch_f32 for the rule.
//
// Relative positions come in 16-wide tiles as well: tile e covers r = 16e .. 16e+15, and the (query tile a, key tile b)
// pair needs r = 16(a-b)-15 .. 16(a-b)+15, i.e. tiles a-b-1 and a-b.  A block of QT query tiles and KT key tiles needs
// QT+KT position tiles; each of their table rows K_r[delta(r)], Q_r[delta(r)] is loaded once per block and contracted
// with the query tiles (c2p) and the key tiles (p2c) that reach it.
//   c2p  C'^T[r, i] = K_r[delta(r)].Q_i   lane = query, registers = 4 positions -> scratch C[query][r]
//   p2c  P'^T[r, j] = Q_r[delta(r)].K_j   lane = key,   registers = 4 positions -> scratch P[key][r]
// The score tile S^T[j, i] (lane = query, registers = 4 keys) then starts from C[i][i-j] + P[j][i-j].
// With strips the two starting values are read from the caller's arrays instead.
// (Same definition as the other kernels: modeling_deberta_v2.py:243, :317-324, :337-343.)
#include <cfloat>
#include <type_traits>

#include "tdb_internal.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int WAVES = 4;
constexpr int D = 64;
constexpr int GAP_WGS = 64;                 // workgroups that look for packed rows outside every sequence
constexpr int pos_stride(int n) { return 16 * (n + 1) + 4; }     // floats of a scratch row: n + 1 position tiles
constexpr int scratch_floats(int qt, int kt) { return qt * 16 * pos_stride(kt) + kt * 16 * pos_stride(qt); }      // per wave
// the merge needs QT * 1024 floats of partial sums per wave, and 2 * QT * 16 of maxima and denominators
constexpr int wave_floats(int qt, int kt) { return scratch_floats(qt, kt) > qt * (1024 + 32) ? scratch_floats(qt, kt) : qt * (1024 + 32); }

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Lanes of one wave exchange data through LDS: DS instructions of a wave execute in order, so only the compiler has to
// be kept from moving accesses across.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Value of the three lanes that share (l & 15), folded: lanes l ^ 16 and l ^ 32.
__device__ __forceinline__ float fold_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 16));
    return fmaxf(x, __shfl_xor(x, 32));
}
// exp(x) for x <= 0 to about one unit in the last place: the hardware's base-2 exponential of the rounded x log2(e),
// corrected to first order by what the rounding (and log2(e)'s own) left out.  A third of the instructions of expf, whose
// range handling the softmax does not need; arguments below -1e4 (masked keys, the first block's old maximum) give 0, NaN
// gives NaN (fmaxf would make a 0 of it, and of a key that is none a finite answer).
__device__ __forceinline__ float exp_neg(float x) {
    x = __builtin_elementwise_maximum(x, -1e4f);
    const float h = x * 1.44269502f;                                              // float(log2 e)
    const float e = fmaf(x, 1.92596303e-8f, fmaf(x, 1.44269502f, -h));            // + the rest of log2 e
    const float y = __builtin_amdgcn_exp2f(h);
    return fmaf(y, e * 0.693147182f, y);
}
__device__ __forceinline__ float fold_sum(float x) {
    x += __shfl_xor(x, 16);
    return x + __shfl_xor(x, 32);
}

// Fragment of 16 rows x 64: lane (row = l & 15, g = l >> 4) holds columns 16t + 4g .. +3, t = 0..3.  Both operands of a
// product use this order, so MFMA (t, e) contracts columns {16t + 4g + e}: any order of the sum is a valid one.
__device__ __forceinline__ void load_frag(f32x4 (&f)[4], const float* row, int g) {
#pragma unroll
    for (int t = 0; t < 4; ++t) f[t] = *reinterpret_cast<const f32x4*>(row + 16 * t + 4 * g);
}

// KT: key tiles of 16 per block.
template <int QT, int KT, bool STRIP, bool C2P, bool P2C>
__global__ __launch_bounds__(WAVES * 64, STRIP || QT > 1 ? 2 : 3) void attn_f32_kernel(const TdbKernelParams p, const int tiles_x) {
    extern __shared__ __attribute__((aligned(16))) float smem_f[];
    constexpr int CST = pos_stride(KT), PST = pos_stride(QT), WAVE = wave_floats(QT, KT);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int c = l & 15, g = l >> 4;       // column (or row) of a tile, group of four rows
    float* const sC = smem_f + wave * WAVE;
    float* const sP = sC + QT * 16 * CST;

    if (p.gap_cu && blockIdx.x + GAP_WGS >= gridDim.x) {
        const int worker = (blockIdx.x + GAP_WGS - gridDim.x) * WAVES + wave;
        tdb_fill_gaps(p.gap_cu, p.gap_B, p.L, p.total, static_cast<char*>(p.o), p.os_l * 4, p.os_h * 4, p.H, 4 * D, worker, GAP_WGS * WAVES);
        return;
    }

    // Block ids go round-robin over the 8 XCDs: four neighbouring query tiles, which read the same keys and values,
    // are kept on one of them.  The heads of a tile group follow each other (and not the tile groups of a head), so
    // that every XCD gets its share of every sequence, however their lengths differ.
    const int slot = blockIdx.x >> 3;
    const int group = (slot >> 2) * 8 + (blockIdx.x & 7), h = group % p.H, tile = group / p.H * 4 + (slot & 3);
    int b, row0, len;
    int64_t tok0;
    if (tile >= tiles_x || !tdb_locate_tile_sorted(p, QT * 16, tile, b, row0, len, tok0)) return;
    b = __builtin_amdgcn_readfirstlane(b), row0 = __builtin_amdgcn_readfirstlane(row0), len = __builtin_amdgcn_readfirstlane(len);

    auto base = [&](const void* ptr, int64_t sb, int64_t sh, int64_t sl) {
        return static_cast<const float*>(ptr) + (p.varlen ? tok0 * sl : int64_t(b) * sb) + int64_t(h) * sh;
    };
    float* const O = const_cast<float*>(base(p.o, p.os_b, p.os_h, p.os_l));
    const int rows_here = min(QT * 16, (p.varlen ? len : p.L) - row0);
    if (row0 >= len) {                      // padded query rows only (fixed layout): zeros
        for (int idx = threadIdx.x; idx < rows_here * (D / 4); idx += WAVES * 64)
            *reinterpret_cast<f32x4*>(O + int64_t(row0 + idx / (D / 4)) * p.os_l + idx % (D / 4) * 4) = f32x4{0.f, 0.f, 0.f, 0.f};
        return;
    }
    const float* const Q = base(p.q, p.qs_b, p.qs_h, p.qs_l);
    const float* const K = base(p.k, p.ks_b, p.ks_h, p.ks_l);
    const float* const V = base(p.v, p.vs_b, p.vs_h, p.vs_l);
    const float* const C = STRIP ? base(p.c2p, p.c2s_b, p.c2s_h, p.c2s_l) : static_cast<const float*>(p.pk) + int64_t(h) * p.pks_h;
    const float* const P = STRIP ? base(p.p2c, p.p2s_b, p.p2s_h, p.p2s_l) : static_cast<const float*>(p.pq) + int64_t(h) * p.pqs_h;
    const int lut_max = 2 * p.lut_half;
    auto delta_of = [&](int r) { return p.lut[min(max(r + p.lut_half, 0), lut_max)]; };

    // This wave's key tiles: blocks of KT, dealt to the waves in turn (the position rows of neighbouring blocks overlap
    // by half, and waves that work on neighbours at the same time find them in L1); of the last, incomplete round single tiles, if it has
    // no more than one for each wave.  (Pairs there gave 12 tiles to the waves as 4, 4, 2, 2 instead of 3 each.)
    const int ntiles = (len + 15) >> 4, rest = ntiles % (WAVES * KT), behind = ntiles - rest, in_rest = rest > WAVES ? KT * wave : wave;
    const bool pair_in_rest = rest > WAVES && in_rest + 1 < rest;
    const int pairs = KT > 1 ? ntiles / (WAVES * KT) + (pair_in_rest ? 1 : 0) : 0;      // then a single tile, if it exists (KT = 1: one after the other)
    const int single = KT > 1 ? (!pair_in_rest && in_rest < rest ? behind + in_rest : ntiles) : wave;
    const int first = pairs > 0 ? KT * wave : single;

    // Table rows of position tile x of the block that starts at key tile bt: r = row0 - 16 bt + 16 (x - KT) + c.
    int dl[QT + KT];
    auto read_deltas = [&](int bt) {
#pragma unroll
        for (int x = 0; x < QT + KT; ++x) dl[x] = delta_of(row0 - 16 * bt + 16 * (x - KT) + c);
    };
    if (!STRIP && (C2P || P2C) && first < ntiles) read_deltas(first);

    f32x4 qf[QT][4];
#pragma unroll
    for (int a = 0; a < QT; ++a) load_frag(qf[a], Q + int64_t(min(row0 + 16 * a + c, len - 1)) * p.qs_l, g);

    f32x4 oacc[QT][4];                      // [query tile][u]: row m of tile u is d = 4m + u
    float m_run[QT], l_run[QT];             // l_run: this lane's keys only
#pragma unroll
    for (int a = 0; a < QT; ++a) {
        m_run[a] = -FLT_MAX, l_run[a] = 0.f;        // finite: a block whose scores are all -inf leaves no NaN behind
#pragma unroll
        for (int u = 0; u < 4; ++u) oacc[a][u] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // Operands are requested one use ahead: a fragment of position rows while the one before it is contracted, the
    // values under the score products, the next block's keys and first position rows under the softmax.
    f32x4 kf[KT][4], pf[2][4];              // keys; position rows of this phase and the next
    auto load_keys = [&](int bt, bool pair) {
#pragma unroll
        for (int bi = 0; bi < KT; ++bi)
            if (bi == 0 || pair) load_frag(kf[bi], K + int64_t(min(16 * (bt + bi) + c, len - 1)) * p.ks_l, g);
    };
    // phases of a block: position tile x = ph / TERMS, one term after the other (c2p first)
    constexpr int TERMS = int(C2P) + int(P2C), PHASES = STRIP ? 0 : TERMS * (QT + KT);
    auto load_pos = [&](int ph, int slot) {
        const int x = ph / (TERMS > 0 ? TERMS : 1);
        if (C2P && (!P2C || ph % 2 == 0)) load_frag(pf[slot], C + int64_t(dl[x]) * p.pks_r, g);
        else load_frag(pf[slot], P + int64_t(dl[x]) * p.pqs_r, g);
    };
    // Nothing moves across: left alone, the scheduler sinks every load to just before its use (one exposed L2 round
    // trip per 16 bytes: 190 us instead of 138 at batch 8 x 512).
    auto issued = [] { __builtin_amdgcn_sched_barrier(0); };
    // Keys and first position rows of a block (one of a single tile has no use for the lowest position tile).
    auto load_first = [&](int bt, bool pair) {
        load_keys(bt, pair);
        if (!PHASES) return;
        if (KT > 1 && pair) load_pos(0, 0);
        else load_pos(TERMS * (KT - 1), 0);
    };
    if (first < ntiles) load_first(first, pairs > 0);
    auto block = [&](int bt, int after, bool after_pair, auto pair_tag) {    // after: the block that this wave has next
        constexpr bool PAIR = decltype(pair_tag)::value;
        constexpr int TILES = PAIR ? KT : 1, LOWEST = KT - TILES;
        int c_ = c, g_ = g;                 // (opaque for the last tile: address terms that both blocks share would not leave the registers)
        if (!PAIR) asm volatile("" : "+v"(c_), "+v"(g_));
        const int c = c_, g = g_;
        f32x4 s[QT][TILES];
#pragma unroll
        for (int a = 0; a < QT; ++a)
#pragma unroll
            for (int bi = 0; bi < TILES; ++bi) s[a][bi] = f32x4{0.f, 0.f, 0.f, 0.f};

        if (STRIP) {
#pragma unroll
            for (int a = 0; a < QT; ++a)
#pragma unroll
                for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int i = min(row0 + 16 * a + c, len - 1), j = min(16 * (bt + bi) + 4 * g + t, len - 1);
                        const int d = delta_of(i - j);
                        if (C2P) s[a][bi][t] += C[int64_t(i) * p.c2s_l + d];
                        if (P2C) s[a][bi][t] += P[int64_t(j) * p.p2s_l + d];
                    }
        } else if (C2P || P2C) {
            // c2p: query tile a reaches position tiles a .. a+KT; p2c: key tile bi reaches KT-1-bi .. QT+KT-1-bi.
            // (A product with a single tile is summed in two halves: a dependent MFMA waits longer than the pipe is busy.)
#pragma unroll
            for (int ph = LOWEST * TERMS; ph < PHASES; ++ph) {
                const int x = ph / TERMS;
                const int slot = (ph - LOWEST * TERMS) & 1;
                if (ph + 1 < PHASES) load_pos(ph + 1, slot ^ 1);
                issued();
                const f32x4(&f)[4] = pf[slot];
                if (C2P && (!P2C || ph % 2 == 0)) {
                    constexpr int HALVES = QT * TILES == 1 ? 2 : 1;
                    f32x4 acc[QT][HALVES];
#pragma unroll
                    for (int a = 0; a < QT; ++a)
#pragma unroll
                        for (int n = 0; n < HALVES; ++n) acc[a][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int te = 0; te < 16; ++te)
#pragma unroll
                        for (int a = 0; a < QT; ++a)
                            if (x >= a + LOWEST && x <= a + KT) acc[a][te % HALVES] = mfma(f[te >> 2][te & 3], qf[a][te >> 2][te & 3], acc[a][te % HALVES]);
#pragma unroll
                    for (int a = 0; a < QT; ++a)
                        if (x >= a + LOWEST && x <= a + KT)
                            *reinterpret_cast<f32x4*>(&sC[(16 * a + c) * CST + 16 * (x - a) + 4 * g]) = HALVES > 1 ? acc[a][0] + acc[a][HALVES - 1] : acc[a][0];
                } else {
                    constexpr int HALVES = TILES == 1 ? 2 : 1;
                    f32x4 acc[TILES][HALVES];
#pragma unroll
                    for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
                        for (int n = 0; n < HALVES; ++n) acc[bi][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int te = 0; te < 16; ++te)
#pragma unroll
                        for (int bi = 0; bi < TILES; ++bi)
                            if (x >= KT - 1 - bi && x <= QT + KT - 1 - bi) acc[bi][te % HALVES] = mfma(f[te >> 2][te & 3], kf[bi][te >> 2][te & 3], acc[bi][te % HALVES]);
#pragma unroll
                    for (int bi = 0; bi < TILES; ++bi)
                        if (x >= KT - 1 - bi && x <= QT + KT - 1 - bi)
                            *reinterpret_cast<f32x4*>(&sP[(16 * bi + c) * PST + 16 * (x + bi - (KT - 1)) + 4 * g]) = HALVES > 1 ? acc[bi][0] + acc[bi][HALVES - 1] : acc[bi][0];
                }
            }
            if (after < ntiles) read_deltas(after);
            wave_fence();
            // query 16a + c, key 16bi + jl: position i - j sits at 16 (KT - bi) + c - jl of C's row and at 16 (a + 1) + c - jl of P's
#pragma unroll
            for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int jl = 4 * g + t;
#pragma unroll
                    for (int a = 0; a < QT; ++a) {
                        float x = 0.f;
                        if (C2P) x = sC[(16 * a + c) * CST + 16 * (KT - bi) + c - jl];
                        if (P2C) x += sP[(16 * bi + jl) * PST + 16 * (a + 1) + c - jl];
                        s[a][bi][t] = x;
                    }
                }
            wave_fence();
        }
        f32x4 vf[TILES][4];                 // V[key 4g + t][4c .. 4c+3]
#pragma unroll
        for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
            for (int t = 0; t < 4; ++t) vf[bi][t] = *reinterpret_cast<const f32x4*>(V + int64_t(min(16 * (bt + bi) + 4 * g + t, len - 1)) * p.vs_l + 4 * c);
        issued();
        auto score = [&](int bi) {
            constexpr int HALVES = QT * TILES == 1 ? 2 : 1;
            f32x4 rest = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int te = 0; te < 16; ++te)
#pragma unroll
                for (int a = 0; a < QT; ++a) {
                    f32x4& sum = te % HALVES ? rest : s[a][bi];
                    sum = mfma(kf[bi][te >> 2][te & 3], qf[a][te >> 2][te & 3], sum);
                }
            if (HALVES > 1) s[0][0] += rest;
            if (STRIP) asm volatile("" : "+v"(s[0][bi]));      // (added up ahead of the conditions below: see tdb_settled)
        };
        score(0);
        if (TILES > 1) score(TILES - 1);
        if (after < ntiles) load_first(after, after_pair);
        issued();
        // Values past the end are zeros, not the last row again: that may be infinite, and its probability there is 0.
        if (16 * (bt + TILES) > len) {
#pragma unroll
            for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    if (16 * (bt + bi) + 4 * g + t >= len) vf[bi][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        // streaming softmax: this lane has keys 16 bi + 4g + t of query c
#pragma unroll
        for (int a = 0; a < QT; ++a) {
            float mx = -INFINITY;
#pragma unroll
            for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const bool in = 16 * (bt + bi) + 4 * g + t < len;
                    s[a][bi][t] = in ? s[a][bi][t] * p.scale : -INFINITY;
                    mx = fmaxf(mx, s[a][bi][t]);        // (NaN scores pass it by and meet exp_neg)
                }
            const float mn = fmaxf(m_run[a], fold_max(mx));
            const float alpha = exp_neg(m_run[a] - mn);            // (0 on the first block)
            float sum = 0.f;
#pragma unroll
            for (int bi = 0; bi < TILES; ++bi)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    s[a][bi][t] = exp_neg(s[a][bi][t] - mn);
                    sum += s[a][bi][t];
                }
            l_run[a] = l_run[a] * alpha + sum;
            m_run[a] = mn;
#pragma unroll
            for (int u = 0; u < 4; ++u) oacc[a][u] *= alpha;
        }
        // O^T[d, q] += V^T P^T: MFMA t contracts keys 4g + t, whose probabilities the lane already holds
        auto pv = [&](int bi) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int a = 0; a < QT; ++a)
#pragma unroll
                    for (int u = 0; u < 4; ++u) oacc[a][u] = mfma(vf[bi][t][u], s[a][bi][t], oacc[a][u]);
        };
        pv(0);
        if (TILES > 1) pv(TILES - 1);
    };
    if constexpr (KT > 1) {
        for (int i = 0; i < pairs; ++i) {
            const bool more = i + 1 < pairs;
            block(KT * (WAVES * i + wave), more ? KT * (WAVES * (i + 1) + wave) : single, more, std::true_type{});
        }
        if (single < ntiles) block(single, ntiles, false, std::false_type{});
    } else {
        for (int bt = single; bt < ntiles; bt += WAVES) block(bt, bt + WAVES, false, std::true_type{});
    }

    // Merge of the four waves: partial sums [QT][4][64 lanes] x 16 B, then maxima and denominators of the queries.
    float* const mine = smem_f + wave * WAVE;
    wave_fence();                           // (the scratch above is this wave's own)
#pragma unroll
    for (int a = 0; a < QT; ++a) {
#pragma unroll
        for (int t = 0; t < 4; ++t)         // lane (c, g): d = 16g + 4t + u of query c
            *reinterpret_cast<f32x4*>(&mine[((a * 4 + t) * 64 + l) * 4]) = f32x4{oacc[a][0][t], oacc[a][1][t], oacc[a][2][t], oacc[a][3][t]};
        const float l_all = fold_sum(l_run[a]);
        if (g == 0) {
            mine[QT * 1024 + a * 32 + c] = m_run[a];
            mine[QT * 1024 + a * 32 + 16 + c] = l_all;
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < QT; ++a) {
        float f[WAVES], m = -FLT_MAX, den = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) m = fmaxf(m, smem_f[w * WAVE + QT * 1024 + a * 32 + c]);
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            f[w] = exp_neg(smem_f[w * WAVE + QT * 1024 + a * 32 + c] - m);      // (0 for a wave without keys)
            den += f[w] * smem_f[w * WAVE + QT * 1024 + a * 32 + 16 + c];
        }
        const int row = row0 + 16 * a + c;
        const float inv = row < len ? 1.f / den : 0.f;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += *reinterpret_cast<const f32x4*>(&smem_f[w * WAVE + ((a * 4 + wave) * 64 + l) * 4]) * f[w];
        if (row >= len) sum = f32x4{0.f, 0.f, 0.f, 0.f};
        if (row < row0 + rows_here) *reinterpret_cast<f32x4*>(O + int64_t(row) * p.os_l + 16 * g + 4 * wave) = sum * inv;
    }
}

}  // namespace

bool tdb_f32_supported(const TdbKernelParams& p, int dtype) {
    return dtype == TDB_F32 && p.D == D && !((p.c2p || p.p2c) && (p.pk || p.pq));
}

hipError_t tdb_launch_f32(const TdbKernelParams& p, hipStream_t stream) {
    auto tiles_of = [&](int rows) { return p.varlen ? p.total / rows + p.B : p.B * ((p.L + rows - 1) / rows); };
    // 32 query rows per workgroup need a tenth fewer products than 16 and half the operand traffic (8 x 512: 160 us against
    // 200), as long as there are enough workgroups to give every CU its two (2 x 512, 384 of them: 56 us either way).
    const bool wide = int64_t(tiles_of(32)) * p.H >= 512;
    const bool strip = p.c2p || p.p2c;
    const int tiles = tiles_of(wide ? 32 : 16);
    const int64_t blocks = (int64_t((tiles + 3) / 4) * p.H + 7) / 8 * 32 + (p.gap_cu ? GAP_WGS : 0);      // groups of 4 tiles, rounded up to 8 XCDs
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    // Up to 64 tokens a wave has a single key tile: blocks of two would spend a third of their loads and products on a
    // second one that is not there (1 x 64 8.2 -> 6.8 us).  With five tiles, two waves of which would have a pair, single ones pay in large
    // launches (32 x 80 40.8 -> 39.9, 24 of 40..80 29.4 -> 23.8) and not in small ones (2 x 80 7.9 against 8.8).
    const bool single = p.L <= 16 * WAVES || (wide && p.L <= 16 * (WAVES + 1));
    const dim3 grid{unsigned(blocks)}, block(WAVES * 64);
    const size_t smem = sizeof(float) * WAVES * wave_floats(wide ? 2 : 1, single ? 1 : 2);
    const bool c2p = strip ? p.c2p != nullptr : p.pk != nullptr, p2c = strip ? p.p2c != nullptr : p.pq != nullptr;
    auto launch = [&](auto qt, auto kt, auto s, auto c, auto x) {
        hipLaunchKernelGGL((attn_f32_kernel<decltype(qt)::value, decltype(kt)::value, decltype(s)::value, decltype(c)::value, decltype(x)::value>), grid, block, smem, stream, p, tiles);
    };
    using std::bool_constant;
    auto terms = [&](auto qt, auto kt) {
        if (strip && c2p && p2c) launch(qt, kt, bool_constant<true>{}, bool_constant<true>{}, bool_constant<true>{});
        else if (strip && c2p) launch(qt, kt, bool_constant<true>{}, bool_constant<true>{}, bool_constant<false>{});
        else if (strip) launch(qt, kt, bool_constant<true>{}, bool_constant<false>{}, bool_constant<true>{});
        else if (c2p && p2c) launch(qt, kt, bool_constant<false>{}, bool_constant<true>{}, bool_constant<true>{});
        else if (c2p) launch(qt, kt, bool_constant<false>{}, bool_constant<true>{}, bool_constant<false>{});
        else if (p2c) launch(qt, kt, bool_constant<false>{}, bool_constant<false>{}, bool_constant<true>{});
        else launch(qt, kt, bool_constant<false>{}, bool_constant<false>{}, bool_constant<false>{});
    };
    constexpr std::integral_constant<int, 1> one;
    constexpr std::integral_constant<int, 2> two;
    if (wide) single ? terms(two, one) : terms(two, two);
    else single ? terms(one, one) : terms(one, two);
    return hipGetLastError();
}
