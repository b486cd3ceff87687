// Matrix-core disentangled-attention forward for SHORT sequences in bf16 / fp16, head_dim 64 (gfx950, MFMA 32x32x16).
//
// The persistent kernel (attn_mfma.hip) works in tiles of 128 query rows with eight waves in lock step, two barriers per
// 64 keys.  A sequence of 50 tokens fills less than half of such a tile, and a tile costs five steps to open and close
// for the one it runs: 300 sequences of 4 to 96 tokens x 12 heads took 118 us where their bytes take 19.
// Here a WAVE owns 32 query rows of one (sequence, head) and nothing else in the workgroup waits for it:
//   * a workgroup belongs to one head and keeps that head's table rows K_r[delta(r)], Q_r[delta(r)] for EVERY relative
//     position the launch can meet (2 * 32 T of them, T = ceil(max length / 32) <= 5) in LDS, loaded once;
//   * its waves take (sequence, query tile) units from a counter in LDS -- units differ in cost --, all tiles of a
//     sequence going to one workgroup, so that its keys and values come from HBM once;
//   * keys, position products and values pass through one scratch area of the wave, one after the other.
// Measured, persistent kernel before (12 heads, bf16): 1 x 29 8.1 -> 4.5 us, 1 x 128 9.8 -> 9.3, 32 x 64 12.7 -> 7.0,
// 128 x 96 42 -> 28, 128 x 128 43 -> 37; packed 64 of 4..32 tokens 21 -> 9, 64 of 32..128 28.6 -> 21.9, 300 of 4..96
// 120 -> 34.7.  What bounds it now: a small call, the instructions and memory
// round trips in front of its one step; a large one, LDS instructions (some 700 clk per CU and wave step) under two waves
// per SIMD.  160 tokens are the limit because the tables of 320 relative positions and seven waves' scratch fill the LDS; many_tiles
// below says from where they pay.
// The arithmetic is the persistent kernel's, operation for operation (64 keys per softmax step; MFMA chains over the same
// columns in the same order; position products rounded to the element type, p2c as the initial accumulator, c2p added
// after the score products): a sequence gives the same bits in whichever launch it travels.
//
// Position terms: 32-wide tiles of relative positions.  A step of 32 queries x 64 keys meets three of them, tile y =
// r - (row0 - k0 - 64 + 32 y) in 0..31; key tile jt (32 keys) needs y = 1 - jt and 2 - jt.
//   c2p  C'^T[r, i] = K_r'[r].Q_i, lane = query -> scratch C[query][r], 8-byte stores; element (i, j) is C[i][i - j]
//   p2c  P'^T[r, j] = Q_r'[r].K_j, lane = key   -> scratch P[key][r];                  element (i, j) is P[j][i - j]
// The shifts read dwords and pick the halves with a byte permute whose selector depends on the lane's parity.
//
// STRIP: the caller has the position terms as strips (c2p[i][delta], p2c[j][delta]).  The persistent kernel's position waves
// move them in tiles of 128; here the wave gathers the 2 x 32 x 64 elements of its step itself, into registers, a step or unit
// ahead -- four waves a workgroup for their sake.  Measured (12 heads, bf16), persistent kernel before: 1 x 16 10.4 -> 4.8 us,
// 30 x 64 12.3 -> 6.7, 8 x 100 10.5 -> 9.3, 32 x 96 18.4 -> 15.4, 32 x 128 18.8 -> 18.3.  Bound: the 64 gathers of a step.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "tdb_internal.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

#define TDB_LDS(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr int D = 64;
constexpr int UQ = TDB_SHORT_TILE;      // query rows of a unit
constexpr int BN = 64;                  // keys per step
constexpr int MAX_T = 5;                // query tiles of the longest sequence
constexpr int MAX_WAVES = 8;            // two per SIMD
constexpr int STRIP_WAVES = 4;          // of the strip instances, which hold the gathered elements of a step in registers
constexpr int RS = 72;                  // LDS row stride of 16-bit rows of 64 (144 B: conflict-free 16-byte reads)
constexpr int CS = 100;                 // row stride of C[32 queries][96 positions]: 8-byte stores of 16 lanes on distinct banks
constexpr int PS = 68;                  // row stride of P[64 keys][64 positions]
constexpr int SCRATCH = BN * RS * 2;    // bytes per wave: keys, C, P, values in turn
static_assert(UQ * CS * 2 <= SCRATCH && BN * PS * 2 <= SCRATCH, "C and P fit the wave's scratch");

template <int DT>
struct Elem;
template <>
struct Elem<TDB_BF16> {
    using T = __bf16;
    using X2 = bf16x2;
    using X8 = bf16x8;
    static __device__ __forceinline__ f32x16 mfma(X8 a, X8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
    // one half of a dword as fp32: selectors for the lower and the upper
    static constexpr uint32_t LOW = 0x01000c0cu, HIGH = 0x03020c0cu, ONE = 0x3f80;
    static __device__ __forceinline__ float pick(uint32_t pair, uint32_t sel) { return __builtin_bit_cast(float, __builtin_amdgcn_perm(pair, pair, sel)); }
};
template <>
struct Elem<TDB_F16> {
    using T = _Float16;
    using X2 = f16x2;
    using X8 = f16x8;
    static __device__ __forceinline__ f32x16 mfma(X8 a, X8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
    static constexpr uint32_t LOW = 0x0c0c0100u, HIGH = 0x0c0c0302u, ONE = 0x3c00;
    static __device__ __forceinline__ float pick(uint32_t pair, uint32_t sel) {
        return (float)__builtin_bit_cast(X2, __builtin_amdgcn_perm(pair, pair, sel))[0];
    }
};

template <typename E>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typename E::X2 v = {(typename E::T)lo, (typename E::T)hi};
    return __builtin_bit_cast(uint32_t, v);
}

// Lanes of one wave exchange data through LDS: its DS instructions execute in order, so only the compiler has to be kept
// from moving accesses across.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_sched_barrier(0);
}

// What this lane and lane ^ 32 hold, in an order that depends on the half.
__device__ __forceinline__ void both_halves(float x, float& a, float& b) {
    const uint32_t u = __builtin_bit_cast(uint32_t, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    a = __builtin_bit_cast(float, uint32_t(r[0]));
    b = __builtin_bit_cast(float, uint32_t(r[1]));
}

// What the kernel needs, in three cache lines: byte strides (32 bits), the head dimension of the grid, and the scheme of
// the lengths as a template parameter.  A short call is bound by the number of instructions on the way to its first
// loads -- a single wave per SIMD issues one in 4 to 8 clk -- and 64-bit strides, divisions and branches on the layout had
// made that a thousand of them (2 of the 5 us that 29 tokens took on the GPU).
struct ShortArgs {
    const char *q, *k, *v;
    char* o;
    const char *pk, *pq;
    const int32_t *lut, *bounds;            // bounds: lengths or cu_seqlens
    uint32_t qb, qh, ql, kb, kh, kl, vb, vh, vl, ob, oh, ol;      // batch (packed: token), head, row
    uint32_t pkh, pkr, pqh, pqr;            // tables: head, row; strips: head, row of pk / pq ...
    uint32_t pkb, pqb;                      // ... and batch (packed: token)
    int32_t span;
    int32_t B, L, total, lut_half;
    float c_exp;                            // scale * log2(e): softmax in base 2
    int32_t T, tshift;                      // units of a sequence: tiles 0 .. T-1 of 2^tshift numbers
    int32_t waves;                          // per workgroup
    int32_t single;                         // every unit has a wave of its own
    int32_t gaps;                           // packed: zeros for the rows outside every sequence
};
enum { FIXED = 0, LENGTHS = 1, PACKED = 2 };

template <bool C2P, bool P2C, int DT, int MODE, bool STRIP>
__global__ __launch_bounds__((STRIP ? STRIP_WAVES : MAX_WAVES) * 64) void attn_short_kernel(const ShortArgs p) {
#pragma clang fp contract(off)              // (a product and a sum are fused here and there where the persistent kernel's are)
    using E = Elem<DT>;
    using X8 = typename E::X8;
    asm volatile("" ::"s"(p.q), "s"(p.qb), "s"(p.B));       // (all three lines in one round trip)
    extern __shared__ __attribute__((aligned(16))) char smem_s[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int h = blockIdx.x, wg = blockIdx.y, per_head = gridDim.y;
    const int rows = 2 * UQ * p.T;          // relative positions -32T .. 32T - 1
    // LDS: counter, tables (strips: their columns, for positions from 64 before the first), the waves' scratch
    int* const counter = reinterpret_cast<int*>(smem_s);
    uint16_t* const sKr = reinterpret_cast<uint16_t*>(smem_s + 16);
    uint16_t* const sQr = sKr + (C2P ? rows * RS : 0);
    int* const sD = reinterpret_cast<int*>(smem_s + 16);
    uint16_t* const scratch = (STRIP ? sKr + 2 * (BN + rows) : sQr + (P2C ? rows * RS : 0)) + wave * (SCRATCH / 2);

    if (!p.single) {
        if (tid == 0) *counter = p.waves;           // (the waves' first units are their own numbers)
        __syncthreads();
    }
    const char *const qh = p.q + uint64_t(h) * p.qh, *const kh = p.k + uint64_t(h) * p.kh, *const vh = p.v + uint64_t(h) * p.vh;
    char* const oh = p.o + uint64_t(h) * p.oh;

    // Units: tile t0 of sequence wg + n per_head has number (n << tshift) + t0.  Numbers without live query rows are passed
    // over; tiles that hold padded rows only get their zeros on the way.
    struct Unit {
        int seq, row0, len;                 // seq < 0: none
        uint32_t at;                        // what the batch strides are multiplied with
    };
    auto take = [&](int number) {
        while (true) {
            Unit u;
            u.seq = wg + (number >> p.tshift) * per_head;
            u.row0 = UQ * (number & ((1 << p.tshift) - 1));
            u.len = p.L;
            u.at = u.seq;
            if (u.seq >= p.B || number < 0) {
                u.seq = -1;
                return u;
            }
            if (MODE == PACKED) {
                const int lo = __builtin_amdgcn_readfirstlane(p.bounds[u.seq]), hi = __builtin_amdgcn_readfirstlane(p.bounds[u.seq + 1]);
                u.len = lo < 0 || hi < lo || hi > p.total ? 0 : min(hi - lo, p.L);      // malformed entry: no rows
                u.at = lo;
            } else if (MODE == LENGTHS) {
                u.len = min(max(__builtin_amdgcn_readfirstlane(p.bounds[u.seq]), 0), p.L);
            }
            if (u.row0 < u.len) return u;
            if (MODE == LENGTHS) {
                char* const Oz = oh + uint64_t(u.at) * p.ob + uint32_t(u.row0) * p.ol;
                for (int idx = l; idx < min(UQ, p.L - u.row0) * (D / 8); idx += 64)
                    *reinterpret_cast<u32x4*>(Oz + (idx >> 3) * p.ol + (idx & 7) * 16) = u32x4{0, 0, 0, 0};
            }
            number = -1;                    // (nothing else for this wave)
            if (!p.single) {
                if (l == 0) number = atomicAdd(counter, 1);
                number = __builtin_amdgcn_readfirstlane(number);
            }
        }
    };

    // Buffer loads: the buffer starts at the block's first row and ends with the last row of the sequence, so rows past
    // the end read as zeros and the per-lane offsets are the same for every block.
    auto rows_from = [&](const Unit& u, const char* src, uint32_t stride, int r0) {
        const int left = u.len - r0;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(src + uint32_t(r0) * stride), 0, left > 0 ? (left - 1) * stride + 2 * D : 0, 0x00020000);
    };
    X8 qf[4];                               // B operand: lane = query il, columns 16 c + 8 hh .. +7
    u32x4 kr[8], vr[8];                     // rows 8 n + (l >> 3) of a step, chunk l & 7; the upper four only where it has them
    auto load_q = [&](const Unit& u) {
        const auto rsrc = rows_from(u, qh + uint64_t(u.at) * p.qb, p.ql, u.row0);
        const uint32_t off = (l & 31) * p.ql + 16 * (l >> 5);
#pragma unroll
        for (int c = 0; c < 4; ++c) qf[c] = __builtin_bit_cast(X8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 32 * c, 0, 0));
    };
    auto load_block = [&](const Unit& u, u32x4 (&dst)[8], const char* src, uint32_t stride, int k0) {
        const auto rsrc = rows_from(u, src, stride, k0);
        const uint32_t off = (l >> 3) * stride + (l & 7) * 16;
#pragma unroll
        for (int n = 0; n < 4; ++n) dst[n] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 8 * n * stride, 0, 0);
        if (u.len > k0 + 32) {
#pragma unroll
            for (int n = 4; n < 8; ++n) dst[n] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off + 8 * n * stride, 0, 0);
        }
    };
    auto load_k = [&](const Unit& u, int k0) { load_block(u, kr, kh + uint64_t(u.at) * p.kb, p.kl, k0); };
    auto load_v = [&](const Unit& u, int k0) { load_block(u, vr, vh + uint64_t(u.at) * p.vb, p.vl, k0); };
    auto store_block = [&](const u32x4 (&src)[8], bool two) {
        uint16_t* const at = scratch + (l >> 3) * RS + (l & 7) * 8;
#pragma unroll
        for (int n = 0; n < 4; ++n) *reinterpret_cast<u32x4*>(at + 8 * n * RS) = src[n];
        if (two) {
#pragma unroll
            for (int n = 4; n < 8; ++n) *reinterpret_cast<u32x4*>(at + 8 * n * RS) = src[n];
        }
    };

    // Strips: the elements that a step needs, as 16-bit loads.  c2p: lane = key, query row0 + t; a load reads neighbouring
    // columns of one row, and the scratch turns them.  p2c: lane = query, the keys that the lane's accumulator has; a load reads
    // neighbouring columns of two rows.  Rows past the sequence read as zeros.
    uint16_t cv[STRIP && C2P ? UQ : 1], pv[STRIP && P2C ? 2 : 1][16];
    auto gather = [&](const Unit& u, int k0) {
        const bool two = u.len > k0 + 32;
        const int first = u.row0 - k0 + UQ * p.T + BN;      // sD index of row0 - k0
        if (STRIP && P2C) {
            const char* const base = p.pq + uint64_t(h) * p.pqh + uint64_t(u.at) * p.pqb;
            const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, (u.len - 1) * p.pqr + 4 * p.span, 0x00020000);
            const int* const d = sD + first + (l & 31) - 4 * (l >> 5) - 63;
            const uint32_t row = 4 * (l >> 5) * p.pqr;
#pragma unroll
            for (int jt = 0; jt < 2; ++jt)
                if (jt == 0 || two) {
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int key = 32 * jt + 8 * (e >> 2) + (e & 3);
                        pv[jt][e] = uint16_t(__builtin_amdgcn_raw_buffer_load_b16(rsrc, row + (k0 + key) * p.pqr + d[63 - key], 0, 0));
                    }
                }
        }
        if (STRIP && C2P) {
            const char* const base = p.pk + uint64_t(h) * p.pkh + uint64_t(u.at) * p.pkb;
            const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, (u.len - 1) * p.pkr + 4 * p.span, 0x00020000);
            const int* const d = sD + first - l;
#pragma unroll
            for (int t = 0; t < UQ; ++t) cv[t] = uint16_t(__builtin_amdgcn_raw_buffer_load_b16(rsrc, (u.row0 + t) * p.pkr + d[t], 0, 0));
        }
    };

    // Table rows: every delta value first, then the first unit's rows, then every table row (thread: chunk tid & 7 of rows
    // (tid >> 3) + n 8 p.waves; up to four query tiles the launcher brings enough waves for four passes).  No branches around the loads, or each
    // would wait for the last; what lies past the delta table reads as row 0.
    constexpr int N = !STRIP && (C2P || P2C) ? 4 : 0;
    const int per_pass = 8 * p.waves;
    int d[4];
    auto read_deltas = [&](int first) {
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(p.lut), 0, (2 * p.lut_half + 1) * 4, 0x00020000);
        const int off = (first + (tid >> 3) - UQ * p.T + p.lut_half) * 4;
#pragma unroll
        for (int n = 0; n < N; ++n) d[n] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off + n * per_pass * 4, 0, 0);
    };
    read_deltas(0);
    if (STRIP) {
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(p.lut), 0, (2 * p.lut_half + 1) * 4, 0x00020000);
        for (int i = tid; i < BN + rows; i += 64 * p.waves)
            sD[i] = 2 * __builtin_amdgcn_raw_buffer_load_b32(rsrc, (i - BN - UQ * p.T + p.lut_half) * 4, 0, 0);
    }
    Unit cur = take(wave);
    if (cur.seq >= 0) {
        load_k(cur, 0);
        load_q(cur);
        load_v(cur, 0);
    }
    __builtin_amdgcn_sched_barrier(0);      // (left alone, the scheduler sinks every load to its use)
    if (N) {
        const uint32_t ch = (tid & 7) * 16;
        const char *const pk = p.pk + uint64_t(h) * p.pkh, *const pq = p.pq + uint64_t(h) * p.pqh;
        for (int first = 0;;) {
            u32x4 wk[4], wq[4];
#pragma unroll
            for (int n = 0; n < N; ++n) {
                if (C2P) wk[n] = *reinterpret_cast<const u32x4*>(pk + (uint32_t(d[n]) * p.pkr + ch));
                if (P2C) wq[n] = *reinterpret_cast<const u32x4*>(pq + (uint32_t(d[n]) * p.pqr + ch));
            }
            __builtin_amdgcn_sched_barrier(0);
            const int row = first + (tid >> 3), el = row * RS + (tid & 7) * 8;
#pragma unroll
            for (int n = 0; n < N; ++n)
                if (row + n * per_pass < rows) {
                    if (C2P) *reinterpret_cast<u32x4*>(sKr + el + n * per_pass * RS) = wk[n];
                    if (P2C) *reinterpret_cast<u32x4*>(sQr + el + n * per_pass * RS) = wq[n];
                }
            first += 4 * per_pass;
            if (first >= rows) break;       // (five query tiles take a second turn)
            read_deltas(first);
        }
        __syncthreads();
    }
    if (STRIP) {
        __syncthreads();
        if (cur.seq >= 0) gather(cur, 0);
    }

    if (MODE == PACKED && p.gaps && wave == p.waves - 1)
        tdb_fill_gaps(p.bounds, p.B, p.L, p.total, p.o, p.ol, p.oh, gridDim.x, 2 * D, wg * gridDim.x + h, gridDim.x * per_head);

    const float c_exp = p.c_exp;
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    while (cur.seq >= 0) {
        const int len = cur.len, row0 = cur.row0;
        Unit nxt;
        nxt.seq = -1, nxt.row0 = nxt.len = 0, nxt.at = 0;
        if (!p.single) {
            int number = 0;
            if (l == 0) number = atomicAdd(counter, 1);
            nxt = take(__builtin_amdgcn_readfirstlane(number));
        }
        f32x16 oacc[2] = {zero16, zero16};  // lane = query; register 4a + t of tile dt: d = 32 dt + 8 a + 4 hh + t
        float m_run = -INFINITY, l_run = 0.f;

        // One step; TWO: it has keys beyond its first 32.
        auto step = [&](int k0, auto two_tag) {
            constexpr bool TWO = decltype(two_tag)::value;
            constexpr int JT = TWO ? 2 : 1;
            // (The lane's coordinates, opaque to the optimiser: address terms are redone in each step instead of living in
            // registers across it.)
            int il = l & 31, hh = l >> 5;
            asm volatile("" : "+v"(il), "+v"(hh));
            store_block(kr, TWO);
            wave_fence();
            X8 kf[2][4];                    // lane = key il: A operand of the scores, B operand of p2c
#pragma unroll
            for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                for (int c = 0; c < 4; ++c) kf[jt][c] = *reinterpret_cast<const X8*>(scratch + (32 * jt + il) * RS + 16 * c + 8 * hh);
            wave_fence();
            // Fragments of table tiles are read well before their products, and two products run side by side: one after the
            // other, each waits for its reads and for its own last result (32 x 128 14.1 -> 13.4 us with the early keys below).
            const int prow = row0 - k0 - 64 + UQ * p.T;      // LDS row of the first position of tile 0
            auto read_rows = [&](X8 (&f)[4], const uint16_t* table, int first_row) {
                const char* const at = reinterpret_cast<const char*>(table + first_row * RS) + __umul24(il, 2 * RS) + 16 * hh;
#pragma unroll
                for (int c = 0; c < 4; ++c) f[c] = *reinterpret_cast<const X8*>(at + 32 * c);
            };
            auto two_products = [&](f32x16 (&acc)[2], const X8 (&f0)[4], const X8 (&f1)[4], const X8 (&b)[4]) {
                acc[0] = E::mfma(f0[0], b[0], zero16);
                acc[1] = E::mfma(f1[0], b[0], zero16);
#pragma unroll
                for (int c = 1; c < 4; ++c) {
                    acc[0] = E::mfma(f0[c], b[c], acc[0]);
                    acc[1] = E::mfma(f1[c], b[c], acc[1]);
                }
            };
            auto put = [&](uint16_t* at, const f32x16& acc) {
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    *reinterpret_cast<u32x2*>(at + 8 * a) = u32x2{pack2<E>(acc[4 * a], acc[4 * a + 1]), pack2<E>(acc[4 * a + 2], acc[4 * a + 3])};
            };
            f32x16 s[2] = {zero16, zero16};
            if (STRIP && P2C) {
#pragma unroll
                for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) s[jt][e] = E::pick(pv[jt][e], E::LOW);
            }
            X8 cf[2][4];                    // of tiles 0, 1 (TWO) or 1, 2
            auto read_c = [&]() {
                if (!STRIP && C2P) {
#pragma unroll
                    for (int y = 0; y < 2; ++y) read_rows(cf[y], sKr, prow + 32 * (y + (TWO ? 0 : 1)));
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if (!P2C) read_c();
            if (!STRIP && P2C) {
                X8 pf[2][4];
                auto read_p = [&](int jt) {
#pragma unroll
                    for (int z = 0; z < 2; ++z) read_rows(pf[z], sQr, prow + 32 * (z + 1 - jt));
                    __builtin_amdgcn_sched_barrier(0);
                };
                read_p(0);
#pragma unroll
                for (int jt = 0; jt < JT; ++jt) {
                    f32x16 acc[2];
                    two_products(acc, pf[0], pf[1], kf[jt]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (jt + 1 < JT) read_p(jt + 1);
#pragma unroll
                    for (int z = 0; z < 2; ++z) put(scratch + (32 * jt + il) * PS + 32 * z + 4 * hh, acc[z]);
                }
                wave_fence();
                asm volatile("" : "+v"(il), "+v"(hh));
                read_c();
                // key jl = 32 jt + jr sits at jl (PS - 1) + 32 jt + il + 32: the word of its dword alternates with the key
                const uint32_t even = (il & 1) ? E::HIGH : E::LOW, odd = (il & 1) ? E::LOW : E::HIGH;
                const auto* at_even = TDB_LDS(const uint32_t, scratch) + ((il + 32) >> 1) + 2 * hh * (PS - 1);
                const auto* at_odd = TDB_LDS(const uint32_t, scratch) + ((il + 32 + PS - 1) >> 1) + 2 * hh * (PS - 1);
#pragma unroll
                for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int jc = 32 * jt + 8 * (e >> 2) + (e & 3);
                        const uint32_t d = (jc & 1) ? at_odd[(jc - 1) / 2 * (PS - 1) + 16 * jt] : at_even[jc / 2 * (PS - 1) + 16 * jt];
                        s[jt][e] = E::pick(d, (jc & 1) ? odd : even);
                    }
                wave_fence();
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int jt = 0; jt < JT; ++jt) s[jt] = E::mfma(kf[jt][c], qf[c], s[jt]);
            // (the keys of the next step or unit: their registers are free, and they are needed first)
            if (k0 + 32 * JT < len) load_k(cur, k0 + BN);
            else if (nxt.seq >= 0) load_k(nxt, 0);
            if (C2P) {                      // (after the score products, which read no scratch)
                asm volatile("" : "+v"(il), "+v"(hh));
                uint32_t w[JT][8];
                if (STRIP) {
#pragma unroll
                    for (int t = 0; t < UQ; ++t) scratch[t * PS + l] = cv[t];
                    wave_fence();
#pragma unroll
                    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                        for (int a = 0; a < 4; ++a) {
                            const u32x2 x = *reinterpret_cast<const u32x2*>(scratch + il * PS + 32 * jt + 8 * a + 4 * hh);
                            w[jt][2 * a] = x[0], w[jt][2 * a + 1] = x[1];
                        }
                } else {
                f32x16 acc[2];
                two_products(acc, cf[0], cf[1], qf);
                if (TWO) read_rows(cf[0], sKr, prow + 64);
                __builtin_amdgcn_sched_barrier(0);
                uint16_t* const at_c = scratch + il * CS + 4 * hh + (TWO ? 0 : 32);
                put(at_c, acc[0]);
                if (TWO) {
                    acc[0] = E::mfma(cf[0][0], qf[0], zero16);
#pragma unroll
                    for (int c = 1; c < 4; ++c) acc[0] = E::mfma(cf[0][c], qf[c], acc[0]);
                }
                put(at_c + 32, acc[1]);
                if (TWO) put(at_c + 64, acc[0]);
                wave_fence();
                // Keys 8a + 4hh + t of tile jt: positions x0 + 3 - t, x0 = 61 + il - 32 jt - 8 a - 4 hh, in three dwords.  They
                // are added by an MFMA against an identity whose columns stand in the order the lane has the keys in:
                // two byte permutes per group of four and no unpacking.
                const uint32_t swap = (il & 1) ? 0x01000302u : 0x03020504u;       // (x0 is even where il is odd)
                const auto* at = TDB_LDS(const uint32_t, scratch) + il * (CS / 2) + ((61 + il) >> 1) - 2 * hh;
#pragma unroll
                for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                    for (int a = 0; a < 4; ++a) {
                        const uint32_t d0 = at[-16 * jt - 4 * a], d1 = at[-16 * jt - 4 * a + 1], d2 = at[-16 * jt - 4 * a + 2];
                        w[jt][2 * a] = __builtin_amdgcn_perm(d2, d1, swap);
                        w[jt][2 * a + 1] = __builtin_amdgcn_perm(d1, d0, swap);
                    }
                }
#pragma unroll
                for (int c2 = 0; c2 < 2; ++c2) {
                    // row il: key 16 c2 + 8 (e >> 2) + 4 hh + (e & 3)
                    const int at_one = il - 16 * c2 - 4 * hh;
                    u32x4 bits;
#pragma unroll
                    for (int w4 = 0; w4 < 4; ++w4) {
                        const uint32_t n = uint32_t(at_one - 8 * (w4 >> 1) - 2 * (w4 & 1));
                        bits[w4] = n < 2 ? E::ONE << (16 * n) : 0;
                    }
                    const X8 one = __builtin_bit_cast(X8, bits);
#pragma unroll
                    for (int jt = 0; jt < JT; ++jt)
                        s[jt] = E::mfma(one, __builtin_bit_cast(X8, u32x4{w[jt][4 * c2], w[jt][4 * c2 + 1], w[jt][4 * c2 + 2], w[jt][4 * c2 + 3]}), s[jt]);
                }
                wave_fence();
            }
            asm volatile("" : "+v"(il), "+v"(hh));
            store_block(vr, TWO);
            // the rows after these: of the next step, or of the next unit (the last reader of the queries was c2p)
            if (k0 + 32 * JT < len) {
                load_v(cur, k0 + BN);
            } else if (nxt.seq >= 0) {
                load_q(nxt);
                load_v(nxt, 0);
            }
            if (STRIP) {
                if (k0 + 32 * JT < len) gather(cur, k0 + BN);
                else if (nxt.seq >= 0) gather(nxt, 0);
            }
            wave_fence();
            X8 vf[2][2][2];                 // V^T through the transposing read: [key tile][16 keys][dim tile]
            {
                const int g = l >> 4, ll = l & 15;
                const uint16_t* vbase = scratch + ((ll >> 2) + 4 * (g >> 1)) * RS + 16 * (g & 1) + 4 * (ll & 3);
#pragma unroll
                for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                    for (int c = 0; c < 2; ++c)
#pragma unroll
                        for (int dt = 0; dt < 2; ++dt) {
                            const uint16_t* src = vbase + (32 * jt + 8 * c) * RS + 32 * dt;
                            const s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(TDB_LDS(s16x4, src));
                            const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(TDB_LDS(s16x4, src + 16 * RS));
                            const s16x8 both = {lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                            vf[jt][c][dt] = __builtin_bit_cast(X8, both);
                        }
            }
            if (k0 + 32 * JT > len) {
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (k0 + 32 * (JT - 1) + 8 * (e >> 2) + 4 * hh + (e & 3) >= len) s[JT - 1][e] = -INFINITY;
            }
            float mx = s[0][0];
#pragma unroll
            for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[jt][e]);
            float m_a, m_b;
            both_halves(mx, m_a, m_b);
            const float m_new = fmaxf(m_run, fmaxf(m_a, m_b));       // finite: the step's first key exists
            if (k0 == 0) {
                m_run = m_new;              // (the accumulators are still zero)
            } else if ((m_new - m_run) * c_exp > 8.f) {
                const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c_exp);
                l_run *= alpha;
#pragma unroll
                for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                    for (int e = 0; e < 16; ++e) oacc[dt][e] *= alpha;
                m_run = m_new;
            }
            const float mc = m_run * c_exp;
            float psum[2];                  // (sums and value products in the order of the kernel with resident tables)
#pragma unroll
            for (int jt = 0; jt < JT; ++jt)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    uint32_t pw[4];
                    float part = 0.f;
#pragma unroll
                    for (int h2 = 0; h2 < 4; ++h2) {
                        const int e = 4 * c + 8 * (h2 >> 1) + 2 * (h2 & 1);
                        const float p0 = __builtin_amdgcn_exp2f(fmaf(s[jt][e], c_exp, -mc));
                        const float p1 = __builtin_amdgcn_exp2f(fmaf(s[jt][e + 1], c_exp, -mc));
                        part += p0 + p1;
                        pw[h2] = pack2<E>(p0, p1);
                    }
                    psum[c] = jt == 0 ? part : psum[c] + part;
                    const X8 pb = __builtin_bit_cast(X8, u32x4{pw[0], pw[1], pw[2], pw[3]});
#pragma unroll
                    for (int dt = 0; dt < 2; ++dt) oacc[dt] = E::mfma(vf[jt][c][dt], pb, oacc[dt]);
                }
            l_run += psum[0] + psum[1];
            wave_fence();                   // the next step's keys reuse the scratch
        };
        int k0 = 0;
        for (; k0 + 32 < len; k0 += BN) step(k0, std::true_type{});
        if (k0 < len) step(k0, std::false_type{});

        // Rows go out in 16-byte stores: one swap between the lane halves gives each lane eight consecutive d.
        float l_a, l_b;
        both_halves(l_run, l_a, l_b);
        const float inv = 1.f / (l_a + l_b);
        const int qi = l & 31, rows_here = min(UQ, (MODE == LENGTHS ? p.L : len) - row0);
        if (qi < rows_here) {
            const bool live = row0 + qi < len;              // (padded rows of a fixed layout: zeros)
            char* const at = oh + uint64_t(cur.at) * p.ob + uint32_t(row0 + qi) * p.ol + 16 * (l >> 5);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int a2 = 0; a2 < 2; ++a2) {
                    u32x2 r[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const int a = 2 * a2 + t;
                        r[t] = u32x2{0, 0};
                        if (live) r[t] = u32x2{pack2<E>(oacc[dt][4 * a] * inv, oacc[dt][4 * a + 1] * inv), pack2<E>(oacc[dt][4 * a + 2] * inv, oacc[dt][4 * a + 3] * inv)};
                    }
                    const auto x = __builtin_amdgcn_permlane32_swap(r[0][0], r[1][0], false, false);
                    const auto y = __builtin_amdgcn_permlane32_swap(r[0][1], r[1][1], false, false);
                    *reinterpret_cast<u32x4*>(at + 64 * dt + 32 * a2) = u32x4{x[0], y[0], x[1], y[1]};
                }
        }
        cur = nxt;
    }
}

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
bool g_attr_set[kMaxDevices][48] = {{false}};

template <int DT, int MODE, bool STRIP>
const void* kernel_of(bool c2p, bool p2c) {
    return c2p ? (p2c ? reinterpret_cast<const void*>(&attn_short_kernel<true, true, DT, MODE, STRIP>) : reinterpret_cast<const void*>(&attn_short_kernel<true, false, DT, MODE, STRIP>))
               : (p2c ? reinterpret_cast<const void*>(&attn_short_kernel<false, true, DT, MODE, STRIP>) : reinterpret_cast<const void*>(&attn_short_kernel<false, false, DT, MODE, false>));
}
template <int DT, bool STRIP>
const void* kernel_of(bool c2p, bool p2c, int mode) {
    return mode == FIXED ? kernel_of<DT, FIXED, STRIP>(c2p, p2c) : mode == LENGTHS ? kernel_of<DT, LENGTHS, STRIP>(c2p, p2c) : kernel_of<DT, PACKED, STRIP>(c2p, p2c);
}

}  // namespace

// Above 128 tokens the persistent kernel has two tiles of 128 rows per sequence, each two key steps dearer than its three; one
// round of tiles over the CUs is still quicker than three steps of a wave here (8 x 160: 11.5 against 13.7 us), two are not
// (11 x 160 18.1 against 13.8, packed 150 of 10..160, three launches there, 73.9 against 43.9).  Where the lengths differ a tile
// is half as many steps and the line lies higher (packed 32 of 30..140: 17 either way).  Strips stay there (4 x 140 12.6 against
// 18.2: their gathers are shared out over four waves).
static bool many_tiles(const TdbKernelParams& p) {
    if (p.c2p || p.p2c) return false;
    const int64_t BH = int64_t(p.B) * p.H, cus = tdb_compute_units(-1);
    if (p.varlen ? 10 * int64_t(p.total) > 9 * int64_t(p.B) * p.L : !p.seqlens) return 2 * BH > cus;
    return (p.varlen ? int64_t(p.H) * (p.total / 128) + BH / 2 : BH * 3 / 2) > cus * 7 / 4;
}

bool tdb_short_supported(const TdbKernelParams& p, int dtype) {
    if ((dtype != TDB_BF16 && dtype != TDB_F16) || p.D != D || p.L > UQ * MAX_T || ((p.pk || p.pq) && (p.c2p || p.p2c))) return false;
    if (p.L > 128 && !many_tiles(p)) return false;
    // byte strides in 32 bits, byte offsets inside a sequence and inside a head's table in 31
    const int64_t lim = int64_t(1) << 31, outer[] = {p.qs_b, p.qs_h, p.ks_b, p.ks_h, p.vs_b, p.vs_h, p.os_b, p.os_h, p.pks_h, p.pqs_h, p.c2s_b, p.c2s_h, p.p2s_b, p.p2s_h};
    for (int64_t s : outer)
        if (s >= lim) return false;
    for (int64_t s : {p.qs_l, p.ks_l, p.vs_l, p.os_l, p.c2s_l, p.p2s_l})
        if (s * 2 * (UQ * MAX_T) >= lim) return false;
    return int64_t(2) * p.span * p.pks_r * 2 < lim && int64_t(2) * p.span * p.pqs_r * 2 < lim && 2 * int64_t(p.lut_half) + 1 < lim / 4;
}

hipError_t tdb_launch_short(const TdbKernelParams& p, int dtype, hipStream_t stream) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    const bool strip = p.c2p || p.p2c, c2p = p.pk || p.c2p, p2c = p.pq || p.p2c;
    const int mode = p.varlen ? PACKED : p.seqlens ? LENGTHS : FIXED;
    ShortArgs a;
    a.q = static_cast<const char*>(p.q), a.k = static_cast<const char*>(p.k), a.v = static_cast<const char*>(p.v), a.o = static_cast<char*>(p.o);
    a.pk = static_cast<const char*>(strip ? p.c2p : p.pk), a.pq = static_cast<const char*>(strip ? p.p2c : p.pq);
    a.lut = p.lut, a.bounds = p.varlen ? p.cu_seqlens : p.seqlens;
    auto bytes = [](int64_t s) { return uint32_t(2 * s); };
    a.qb = bytes(p.varlen ? p.qs_l : p.qs_b), a.qh = bytes(p.qs_h), a.ql = bytes(p.qs_l);
    a.kb = bytes(p.varlen ? p.ks_l : p.ks_b), a.kh = bytes(p.ks_h), a.kl = bytes(p.ks_l);
    a.vb = bytes(p.varlen ? p.vs_l : p.vs_b), a.vh = bytes(p.vs_h), a.vl = bytes(p.vs_l);
    a.ob = bytes(p.varlen ? p.os_l : p.os_b), a.oh = bytes(p.os_h), a.ol = bytes(p.os_l);
    a.pkh = bytes(strip ? p.c2s_h : p.pks_h), a.pkr = bytes(strip ? p.c2s_l : p.pks_r);
    a.pqh = bytes(strip ? p.p2s_h : p.pqs_h), a.pqr = bytes(strip ? p.p2s_l : p.pqs_r);
    a.pkb = bytes(p.varlen ? p.c2s_l : p.c2s_b), a.pqb = bytes(p.varlen ? p.p2s_l : p.p2s_b), a.span = p.span;
    a.B = p.B, a.L = p.L, a.total = p.total, a.lut_half = p.lut_half;
    a.c_exp = p.scale * 1.4426950408889634f;
    a.T = (p.L + UQ - 1) / UQ;
    a.tshift = a.T > 4 ? 3 : a.T > 2 ? 2 : a.T - 1;
    const void* fn = dtype == TDB_F16 ? (strip ? kernel_of<TDB_F16, true>(c2p, p2c, mode) : kernel_of<TDB_F16, false>(c2p, p2c, mode))
                                      : (strip ? kernel_of<TDB_BF16, true>(c2p, p2c, mode) : kernel_of<TDB_BF16, false>(c2p, p2c, mode));
    const int cus = tdb_compute_units(dev);
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        bool& set = g_attr_set[dev][(strip ? 24 : 0) + mode * 8 + (dtype == TDB_F16 ? 4 : 0) + (c2p ? 2 : 0) + (p2c ? 1 : 0)];
        if (!set) {
            e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return e;
            set = true;
        }
    }
    // One workgroup per CU, shared out over the heads; no more waves than there are units, but enough to load the tables in
    // four passes.  (T = 4: 8 waves and the tables fill 147 KB of LDS.)
    const int per_head = std::min(p.B, std::max(1, cus / p.H));
    const int units = (p.B + per_head - 1) / per_head << a.tshift;
    const int waves = std::min(strip ? STRIP_WAVES : a.T > 4 ? MAX_WAVES - 1 : MAX_WAVES, std::max(std::max(4, 2 * a.T), units));
    a.gaps = p.gap_cu != nullptr;
    a.waves = waves, a.single = units <= waves;
    const size_t smem = 16 + (strip ? (BN + 2 * UQ * a.T) * sizeof(int) : (int(c2p) + int(p2c)) * size_t(2 * UQ * a.T * RS * 2)) + size_t(waves) * SCRATCH;
    void* args[] = {&a};
    return hipLaunchKernel(fn, dim3(unsigned(p.H), unsigned(per_head)), dim3(waves * 64), args, smem, stream);
}
