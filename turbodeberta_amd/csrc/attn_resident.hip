// Matrix-core disentangled-attention forward for bf16 and fp16, head_dim 64, position terms as per-head tables of up to 512 rows (gfx950).
//
// A workgroup keeps the K_r and Q_r rows of its head in LDS (128 KiB without padding, 16-byte chunks swizzled) and lets keys and values
// pass through the other 32 KiB: fetched two steps of 64 keys ahead into registers, staged one step ahead, one barrier a step.  Eight
// waves take 16 or 32 consecutive query rows each and do all that a step has (attn_step.h).  160 KiB are all there is, so one workgroup
// a compute unit, and tiles are dealt so that it mostly keeps its head: the tables are read once for many tiles.
//
// Microseconds at 12 heads, both terms, bf16, against the persistent kernel of attn_mfma.hip, whose waves compute windows of positions
// for each other through LDS: 64 x 512 keys 187 -> 166, 32 x 1024 315 -> 264, 8 x 4096 977 -> 700; c2p alone 64 x 512 131 -> 117, p2c
// alone 138 -> 120, neither 104 -> 77.  1 x 512 18.2 -> 16, 1 x 180 11.8 -> 10.
#include <algorithm>
#include <mutex>
#include <numeric>

#include "attn_step.h"
#include "tdb_internal.h"

namespace {

using namespace tdb_step;

constexpr int WAVES = 8, HALF = WAVES / 2, NTHREADS = 64 * WAVES;
constexpr int BLOCK = BN * ROW;             // bytes of the keys or values of a step
constexpr int MAX_ROWS = 512;               // table rows that fit the LDS beside two steps of keys and values

struct ResidentArgs {
    const char *q, *k, *v;
    char* o;
    const char *pk, *pq;
    const int32_t *lut, *bounds, *gap_cu;   // bounds: lengths or cu_seqlens
    uint64_t qb, kb, vb, ob;                // byte strides: batch (packed: token) ...
    uint32_t qh, ql, kh, kl, vh, vl, oh, ol;    // ... head, row
    uint32_t pkh, pkr, pqh, pqr;
    int32_t mode, gap_B;
    int32_t B, H, L, total, lut_half, rows; // rows: of a table
    float c_exp;
    int32_t per_group, heads;               // workgroups and heads of a group that deals its tiles among itself
};
enum { FIXED = 0, LENGTHS = 1, PACKED = 2 };

// Time of a step of a tile: of up to WAVES units (every SIMD has two waves) and of up to HALF, by query groups per unit.  (3.1 and 2.1 us
// of the whole chip at 32 rows a unit, 2.0 and 1.35 at 16.)
template <int QG>
struct StepCost {
    static constexpr int whole = QG == 2 ? 9 : 6, half = QG == 2 ? 6 : 4;
};

__device__ __forceinline__ int scan(int v) {        // sums over the lanes up to this one
    v += __builtin_amdgcn_update_dpp(0, v, 0x111 /* row_shr:1 */, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142 /* row_bcast:15 */, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143 /* row_bcast:31 */, 0xc, 0xf, false);
    return v;
}
// Tiles of the sequences up to this lane's, over all heads of a group: those of more than HALF units, and the ends of up to HALF.
struct Upto {
    int whole, half;
};
template <int QG>
__device__ __forceinline__ Upto tiles_upto(int n, int heads) {
    const int units = (n + 16 * QG - 1) / (16 * QG), end = units % WAVES;
    return {scan((units / WAVES + (end > HALF ? 1 : 0)) * heads), scan((end > 0 && end <= HALF ? 1 : 0) * heads)};
}
// One workgroup's tiles.  s_at, s_n, s_upto: of the sequence of this lane, in order of decreasing length: what the batch strides are
// multiplied with, its length, its tiles.
template <bool C2P, bool P2C, int DT, int QG, bool EQUAL, bool LONG>
__device__ __forceinline__ void run(const ResidentArgs& p, const int s_at, const int s_n, const Upto s_upto) {
#pragma clang fp contract(off)
    using W = Wave<C2P, P2C, DT, QG, LONG>;
    using X8 = typename W::X8;
    constexpr int UQ = W::UQ, NT = W::NT;
    constexpr bool POS = W::POS;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t table = uint32_t(p.rows) * ROW;
    const uint32_t kr_base = P2C ? table : 0, kv_base = (int(C2P) + int(P2C)) * table;

    // ---- tiles: up to eight units of UQ query rows of one (sequence, head), a wave each --------------------------------------
    // Lane i of every wave works out the i-th tile of the workgroup (of the 64 that start at `listed`); a tile is then a few
    // readlanes away, and its divisions are done once and for all lanes together.
    const int per_xcd = gridDim.x >> 3, number = int(blockIdx.x & 7) * per_xcd + int(blockIdx.x >> 3);      // neighbours share an XCD
    const int group = number / p.per_group, mine = number - group * p.per_group;
    // Sequences of different lengths: how many of them end at or before tile k of their kind.
    const int wholes = EQUAL ? 0 : __builtin_amdgcn_readlane(s_upto.whole, 63), all = EQUAL ? 0 : wholes + __builtin_amdgcn_readlane(s_upto.half, 63);
    auto before = [&](int k) {
        const bool whole = k < wholes;
        const int among = whole ? k : k - wholes;
        int from = 0;
#pragma unroll
        for (int step = 32; step > 0; step >>= 1) {         // (reads of other lanes, by all lanes)
            const int a = __builtin_amdgcn_ds_bpermute((from + step - 1) * 4, s_upto.whole), b = __builtin_amdgcn_ds_bpermute((from + step - 1) * 4, s_upto.half);
            if ((whole ? a : b) <= among) from += step;
        }
        return from;
    };
    // The last, incomplete round: whole tiles go by halves if there are workgroups for that, also only the longest of them where the next
    // is clearly shorter, and the costliest to the least loaded workgroup.  Without: 7 packed texts of 1100 89 -> 103 us, 32 padded ones
    // of 64 to 512 53.7 -> 57.  What workgroups have is reckoned after one or two rounds, and after up to five where lengths of more than
    // 512 are far apart and less than seven eighths of a round are left (900 launches of 8 to 24 heads: 1.025x there, 0.96 to 1.17x; with more
    // left a quarter of them are slower).  It takes a microsecond or two, too much for texts up to 320 and elsewhere (39 texts of 384 to 512
    // 2 % slower), and a lane per workgroup.  Otherwise the order stays, and whoever had the cheaper tile of the round before gets the
    // costlier one.
    const int full = all - all % p.per_group, rounds = full / p.per_group, rest = all - full;
    const int longest = EQUAL ? 0 : __builtin_amdgcn_readlane(s_n, 0), shortest = EQUAL ? 0 : __builtin_amdgcn_readlane(s_n, p.B - 1);
    const bool far_apart = longest > 8 * BN && 2 * shortest < longest && 8 * rest < 7 * p.per_group;
    const bool reckon = longest > 5 * BN && rest > 0 && p.per_group <= 64 && rounds > 0 && rounds <= (far_apart ? 5 : 2);
    int halved = EQUAL ? 0 : max(wholes - full, 0);
    if (rest + halved > p.per_group) {
        halved = p.per_group - rest;
        if (reckon) {
            const int n = __builtin_amdgcn_ds_bpermute(before(full + (lane ? halved : 0)) * 4, s_n);
            if (10 * __builtin_amdgcn_readlane(n, 1) > 9 * __builtin_amdgcn_readlane(n, 0)) halved = 0;
        } else if (rounds > 0) halved = 0;
    }
    auto last_tile = [&](int i) { return full + (i < 2 * halved ? i >> 1 : i - halved); };
    auto cost = [&](int n, bool half) { return ((n + BN - 1) / BN + 1) * (half ? StepCost<QG>::half : StepCost<QG>::whole); };
    int last = (rounds & 1) ? p.per_group - 1 - mine : mine;
    if (reckon) {
        int load = lane < p.per_group ? 0 : 1 << 30;
        for (int j = 0; j < rounds; ++j) {
            const int k = j * p.per_group + ((j & 1) ? p.per_group - 1 - lane : lane), n = __builtin_amdgcn_ds_bpermute(before(k) * 4, s_n);
            if (lane < p.per_group) load += cost(n, k >= wholes);
        }
        const int own = __builtin_amdgcn_readlane(load, mine);
        last = __builtin_popcountll(__builtin_amdgcn_ballot_w64(load < own || (load == own && lane < mine)));
        if (halved > 0) {                   // (without halves the order of the costs is that of the tiles, or nearly)
            const int k = last_tile(lane), n = __builtin_amdgcn_ds_bpermute(before(k) * 4, s_n);
            const int key = k < all ? cost(n, lane < 2 * halved || k >= wholes) * 64 + 63 - lane : -1;
            int rank = k < all ? 0 : 64;
#pragma unroll
            for (int i = 0; i < 64; ++i) rank += __builtin_amdgcn_readlane(key, i) > key ? 1 : 0;
            const uint64_t it = __builtin_amdgcn_ballot_w64(rank == last);
            last = it ? __builtin_ctzll(it) : p.per_group;
        }
    }
    int t_head, t_at, t_len, t_first, t_units, listed = 0;          // t_len = 0: no tile
    auto list_tiles = [&]() {
        const int j = listed + lane;
        int head, units_from, units_to;
        if (EQUAL) {
            // Each workgroup takes an equal run of half tiles, most of it in one head, and makes tiles of two of them where both are in
            // one sequence; or one whole tile, where these are no more than the workgroups.
            const int per_head = (p.L + UQ * HALF - 1) / (UQ * HALF), pairs = (per_head + 1) >> 1;
            const int64_t seqs = int64_t(p.heads) * p.B, all = seqs * per_head;
            int begin = int(all * mine / p.per_group), end = int(all * (mine + 1) / p.per_group);
            if (all > p.per_group && seqs * pairs <= p.per_group) {
                begin = mine / pairs * per_head + 2 * (mine % pairs);
                end = mine < int(seqs) * pairs ? min(begin + 2, (mine / pairs + 1) * per_head) : begin;
            }
            const int next = (begin / per_head + 1) * per_head, pairs0 = (min(next, end) - begin + 1) >> 1;     // of the sequence that the run starts in
            const int more = max(j - pairs0, 0) / pairs;
            const int k = j < pairs0 ? begin + 2 * j : next + more * per_head + 2 * (j - pairs0 - more * pairs);
            const int seq = k / per_head;
            head = seq / p.B;
            t_at = seq - head * p.B;
            t_len = k < end ? p.L : 0;
            units_from = HALF * (k - seq * per_head);
            units_to = units_from + HALF * min(2, end - k);
        } else {
            // Whole tiles by decreasing length of their sequence, then the ends by decreasing length, dealt back and forth: whoever got
            // the costlier tile of one round gets the cheaper one of the next.
            const bool half = j == rounds && last < 2 * halved;
            const int k = j < rounds ? j * p.per_group + ((j & 1) ? p.per_group - 1 - mine : mine) : j == rounds ? last_tile(last) : all;
            const bool whole = k < wholes;
            const int among = whole ? k : k - wholes, from = before(k);
            const int n = __builtin_amdgcn_ds_bpermute(from * 4, s_n), upto = __builtin_amdgcn_ds_bpermute(from * 4, s_upto.whole),
                      upto_half = __builtin_amdgcn_ds_bpermute(from * 4, s_upto.half);
            t_at = __builtin_amdgcn_ds_bpermute(from * 4, s_at);
            t_len = k < all ? n : 0;
            const int units = (n + UQ - 1) / UQ, end = units % WAVES, per_head = units / WAVES + (end > HALF ? 1 : 0);
            if (whole) {
                const int within = among - (upto - per_head * p.heads);
                head = within / max(per_head, 1);
                units_from = WAVES * (within - head * per_head);
            } else {
                head = among - (upto_half - p.heads);
                units_from = units - end;
            }
            units_to = units_from + WAVES;
            if (half) {
                if (last & 1) units_from += HALF;
                else units_to -= HALF;
            }
        }
        t_head = group * p.heads + head;
        t_first = units_from;
        t_units = min(units_to, (t_len + UQ - 1) / UQ) - units_from;
    };
    list_tiles();

    // ---- keys and values: two steps ahead in registers, one step ahead in LDS -----------------------------------------------
    const int srow = tid >> 3, sch = tid & 7;
    const uint32_t k_off = uint32_t(srow) * p.kl + 16 * sch, v_off = uint32_t(srow) * p.vl + 16 * sch;
    const uint32_t k_to = operand_at(srow, sch), v_to = value_at(srow, sch);
    u32x4 pre_k = {0, 0, 0, 0}, pre_v = {0, 0, 0, 0};
    auto rows_from = [&](const char* base, uint32_t stride, int left) {     // rows past the end read as zeros
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, left > 0 ? (left - 1) * stride + ROW : 0, 0x00020000);
    };
    // what is fetched next: keys from k_from and values from v_from on, of which left_from remain in the sequence; tile fj follows
    const char *k_from = nullptr, *v_from = nullptr;
    int left_from = 0, fj = 0;
    auto fetch = [&]() {
        if (left_from <= 0) {
            const int i = fj - listed;      // (two steps ahead: at most three tiles)
            left_from = __builtin_amdgcn_readlane(t_len, i);
            if (left_from <= 0) return;
            ++fj;
            const uint32_t head = __builtin_amdgcn_readlane(t_head, i);
            const int64_t at = __builtin_amdgcn_readlane(t_at, i);
            k_from = p.k + at * p.kb + uint64_t(head) * p.kh;
            v_from = p.v + at * p.vb + uint64_t(head) * p.vh;
        }
        pre_k = __builtin_amdgcn_raw_buffer_load_b128(rows_from(k_from, p.kl, left_from), k_off, 0, 0);
        pre_v = __builtin_amdgcn_raw_buffer_load_b128(rows_from(v_from, p.vl, left_from), v_off, 0, 0);
        k_from += uint64_t(BN) * p.kl, v_from += uint64_t(BN) * p.vl, left_from -= BN;
    };
    auto stage = [&](int buf) {
        char* const at = smem + kv_base + buf * 2 * BLOCK;
        *reinterpret_cast<u32x4*>(at + k_to) = pre_k;
        *reinterpret_cast<u32x4*>(at + BLOCK + v_to) = pre_v;
    };

    if (p.gap_cu && wave == WAVES - 1)
        tdb_fill_gaps(p.gap_cu, p.gap_B, p.L, p.total, p.o, p.ol, p.oh, p.H, ROW, blockIdx.x, gridDim.x);
    if (!EQUAL && p.mode == LENGTHS) {
        // rows behind the last unit of each sequence
        for (int i = blockIdx.x; i < p.B * p.H; i += gridDim.x) {
            const int b = i / p.H, n = min(max(__builtin_amdgcn_readfirstlane(p.bounds[b]), 0), p.L), r0 = (n + UQ - 1) / UQ * UQ;
            char* const zeros = p.o + uint64_t(b) * p.ob + uint64_t(i - b * p.H) * p.oh + uint64_t(r0) * p.ol;
            for (int idx = tid; idx < (p.L - r0) * (ROW / 16); idx += NTHREADS)
                *reinterpret_cast<u32x4*>(zeros + uint64_t(idx >> 3) * p.ol + 16 * (idx & 7)) = u32x4{0, 0, 0, 0};
        }
    }
    if (__builtin_amdgcn_readlane(t_len, 0) <= 0) return;
    fetch();

    const auto lut = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t*>(p.lut), 0, POS ? (2 * p.lut_half + 1) * 4 : 0, 0x00020000);
    // (Relative positions that no pair of the launch has may lie outside the table: they read as row 0.)
    auto delta = [&](int r) { return __builtin_amdgcn_raw_buffer_load_b32(lut, (r + p.lut_half) * 4, 0, 0); };
    // A step is far if its relative positions have one table row (delta is monotone: the two ends decide), in long sequences those of the
    // whole block of 128 rows, as in the persistent kernel: its far steps keep the position terms in 32 bits.
    auto ends_of = [&](int q0, int k0) {
        const int from = LONG ? q0 & -128 : q0, to = LONG ? from + 127 : from + UQ - 1;
        return delta(min(max((lane & 1 ? to : from - (BN - 1)) - k0, -p.lut_half), p.lut_half));
    };
    auto load_tables = [&](int head) {
        const int hi = p.rows - 1;
        const auto kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.pk + uint64_t(head) * p.pkh), 0, C2P ? hi * p.pkr + ROW : 0, 0x00020000);
        const auto qr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.pq + uint64_t(head) * p.pqh), 0, P2C ? hi * p.pqr + ROW : 0, 0x00020000);
        for (int r0 = 0; r0 <= hi; r0 += 4 * 64) {
            u32x4 x[4], y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t row = r0 + 64 * i + srow;
                if (C2P) x[i] = __builtin_amdgcn_raw_buffer_load_b128(kr, row * p.pkr + 16 * sch, 0, 0);
                if (P2C) y[i] = __builtin_amdgcn_raw_buffer_load_b128(qr, row * p.pqr + 16 * sch, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int row = r0 + 64 * i + srow;
                if (row <= hi) {
                    if (C2P) *reinterpret_cast<u32x4*>(smem + kr_base + operand_at(row, sch)) = x[i];
                    if (P2C) *reinterpret_cast<u32x4*>(smem + operand_at(row, sch)) = y[i];
                }
            }
        }
    };

    W w;
    w.init(lane, kr_base);
    int buf = 0, tables = -1;               // whose tables are in LDS
    for (int j = 0;; ++j) {
        if (j - listed >= 32) {
            listed = j;
            list_tiles();
        }
        const int len = __builtin_amdgcn_readlane(t_len, j - listed);
        if (len <= 0) break;
        const int head = __builtin_amdgcn_readlane(t_head, j - listed);
        const int q0 = UQ * (__builtin_amdgcn_readlane(t_first, j - listed) + wave);
        const int units = __builtin_amdgcn_readlane(t_units, j - listed);      // wave < units: this wave has one
        int ends = 0, ends_next = 0;        // even lanes: table row at the lower end of the step's window, odd lanes: at the upper end
        if (wave < units) {
            w.open();
            if (POS) ends = ends_of(q0, 0);
            if (POS && LONG) ends_next = ends_of(q0, BN);
            const char* const qt = p.q + int64_t(__builtin_amdgcn_readlane(t_at, j - listed)) * p.qb + uint64_t(head) * p.qh + uint64_t(q0) * p.ql;
            const auto rsrc = rows_from(qt, p.ql, len - q0);
#pragma unroll
            for (int x = 0; x < QG; ++x)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    w.q[x][h] = __builtin_bit_cast(X8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (16 * x + w.n) * p.ql + 64 * h + 16 * w.g, 0, 0));
            if (POS) {
#pragma unroll
                for (int i = 0; i < NT; ++i) w.a[i] = w.row_at(delta(q0 + 16 * (i - 4) + w.n));
            }
        }
        if (POS && head != tables) {
            if (tables >= 0) __syncthreads();       // everybody is done with them
            load_tables(head);
            __syncthreads();
            tables = head;
        }
        if (j == 0) {
            stage(0);
            fetch();
        }
        // Where L allows runs of far steps (LONG), a step knows two ahead whether there is one table row, so that far steps need neither the
        // rows of the tiles of the next (all of them are read anew before a near one) nor their addresses: with the c2p values kept from one
        // far step to the next 195 -> 163 vector instructions and 44 -> 40 products a step:
        // 4 x 4096 keys (12 heads) 390 -> 355 us, 2 x 8192 711 -> 621, 8 x 1536 177 -> 173.  The loads for the next steps stand behind those of
        // keys and values (before them each step waited for what it had just asked for: 370).  Scores of a step beside the softmax of the one
        // before in one wave (448, registers spilled) or half a step between the two waves of a SIMD, by barriers (374): slower.
        int low = __builtin_amdgcn_readlane(ends, 0), high = __builtin_amdgcn_readlane(ends, 1);
        int low_next = __builtin_amdgcn_readlane(ends_next, 0), high_next = __builtin_amdgcn_readlane(ends_next, 1);
        for (int k0 = 0; k0 < len; k0 += BN) {
            __syncthreads();                // step k0 is in LDS, and nobody reads the other buffer any more
            stage(buf ^ 1);
            fetch();
            if (wave < units) {
                const uint32_t at = kv_base + buf * 2 * BLOCK;
                int raw[NT];                // the position rows of the next step, whose lowest four tiles are new
                if (POS && (!LONG || low_next != high_next)) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) raw[i] = delta(q0 - k0 - BN + 16 * (i - 4) + w.n);
                    if (LONG && low == high) {
#pragma unroll
                        for (int i = 4; i < NT; ++i) raw[i] = delta(q0 - k0 - BN + 16 * (i - 4) + w.n);
                    }
                }
                if (POS) ends = ends_of(q0, k0 + (LONG ? 2 : 1) * BN);
                w.step(at, at + BLOCK, len - k0, p.c_exp, k0 == 0, POS && low == high, (uint32_t(low) << 7) ^ ((uint32_t(low) << 3) & 0x70));
                if (POS && (!LONG || low_next != high_next)) {
#pragma unroll
                    for (int i = 0; i < QG; ++i) w.a[4 + i] = w.a[i];
                    if (LONG && low == high) {
#pragma unroll
                        for (int i = 4; i < NT; ++i) w.a[i] = w.row_at(raw[i]);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) w.a[i] = w.row_at(raw[i]);
                }
                if (LONG) low = low_next, high = high_next;
                (LONG ? low_next : low) = __builtin_amdgcn_readlane(ends, 0);
                (LONG ? high_next : high) = __builtin_amdgcn_readlane(ends, 1);
            }
            buf ^= 1;
        }
        if (wave < units) {
            char* const ot = p.o + int64_t(__builtin_amdgcn_readlane(t_at, j - listed)) * p.ob + uint64_t(head) * p.oh + uint64_t(q0) * p.ol;
            w.store(ot, p.ol, (p.mode == PACKED ? len : p.L) - q0, len - q0);
        }
    }
}

// Units of 16 QG query rows; sequences that are all equal, or up to 64 of different lengths, which the device alone may know.
template <bool C2P, bool P2C, int DT, int QG, bool EQUAL, bool LONG>
__global__ __launch_bounds__(NTHREADS) void attn_resident_kernel(const ResidentArgs p) {
    if constexpr (EQUAL) {
        run<C2P, P2C, DT, QG, true, LONG>(p, 0, 0, Upto{0, 0});
        return;
    }
    const int lane = threadIdx.x & 63;
    int n = 0, at = lane;
    if (lane < p.B) {
        if (p.mode == LENGTHS) {
            n = min(max(p.bounds[lane], 0), p.L);
        } else {
            at = p.bounds[lane];
            const int hi = p.bounds[lane + 1];
            n = at < 0 || hi < at || hi > p.total ? 0 : min(hi - at, p.L);          // malformed entry: no tiles
        }
    }
    const int key = n * 64 + 63 - lane;
    int rank = lane < p.B ? 0 : lane;
    for (int b = 0; b < p.B; ++b) {
        const int other = __builtin_amdgcn_readlane(key, b);
        if (lane < p.B) rank += other > key ? 1 : 0;
    }
    at = __builtin_amdgcn_ds_permute(rank * 4, at);
    n = __builtin_amdgcn_ds_permute(rank * 4, n);
    run<C2P, P2C, DT, QG, false, LONG>(p, at, n, tiles_upto<QG>(n, p.heads));
}

// What equal sequences cost: see how run() deals them.
template <int QG>
int64_t equal_cost(int64_t seqs, int L, int per_group) {
    const int64_t per_head = (L + 16 * QG * HALF - 1) / (16 * QG * HALF), all = seqs * per_head, each = (all + per_group - 1) / per_group;
    constexpr int whole = StepCost<QG>::whole, half = StepCost<QG>::half;
    if (all <= per_group) return half;
    if (seqs * ((per_head + 1) / 2) <= per_group) return whole;
    const bool split = each % 2 == 0 && (per_head % 2 || all % (2 * per_group));        // the run of some workgroup begins and ends with half a tile
    return each / 2 * whole + each % 2 * half + (split ? 2 * half - whole : 0);
}

// Workgroups, in groups that each take some of the heads.
struct Grid {
    int wgs, per_group, heads;
};
Grid grid_of(int device, int H, int limit) {
    int wgs = std::max(tdb_compute_units(device), 8) / 8 * 8;
    if (limit > 0 && limit < wgs) wgs = limit;
    const int groups = std::gcd(wgs, H);
    return {wgs, wgs / groups, H / groups};
}

constexpr int MAX_SEQS = 64;                // of different lengths in a launch: one per lane
int sequences_of(const TdbKernelParams& p) {
    const int parts = p.varlen || p.seqlens ? (p.B + MAX_SEQS - 1) / MAX_SEQS : 1;
    return (p.B + parts - 1) / parts;
}
// Sequences of different lengths: rounds of tiles of 128 rows of a launch, as far as the host can tell (p: the whole batch).
double ragged_rounds(const TdbKernelParams& p, const Grid& g) {
    return (p.varlen ? p.total / 128.0 / p.B + 0.5 : double((p.L + 127) / 128)) * sequences_of(p) * g.heads / g.per_group;
}
// Whether a unit has 32 rows, which read keys and values once where units of 16 read them twice but fill a round or two better.  In packed
// batches the mean length tells how the sequences end: short ones far below the longest leave units of 32 rows mostly idle (44 of 10 to 233
// tokens, 83 in the mean: 30.1 -> 24.4 us with 16), long ones of similar lengths end in few half tiles (2 of 1835 and 3059 with 8 heads:
// 105 -> 78 with 32).  With a mask the host knows the longest possible length only.
bool wide_units(const TdbKernelParams& p, const Grid& g) {
    if (!p.varlen && !p.seqlens) {
        const int64_t seqs = int64_t(g.heads) * p.B;
        return equal_cost<2>(seqs, p.L, g.per_group) <= equal_cost<1>(seqs, p.L, g.per_group);
    }
    double from = 1.25;
    if (p.varlen) {
        const double mean = double(p.total) / p.B / p.L;
        if (p.L <= 4 * BN) from = mean < 0.5 ? 3.2 : mean < 0.65 ? 1.8 : 1.25;
        else if (p.L >= TDB_FAR_MIN_LEN && mean > 0.65) from = 1.1;
    }
    return ragged_rounds(p, g) > from;
}

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
bool g_attr_set[kMaxDevices][64] = {{false}};

template <bool C2P, bool P2C, int DT, int QG, bool LONG>
const void* kernel_of(bool equal) {
    return equal ? reinterpret_cast<const void*>(&attn_resident_kernel<C2P, P2C, DT, QG, true, LONG>)
                 : reinterpret_cast<const void*>(&attn_resident_kernel<C2P, P2C, DT, QG, false, LONG>);
}
template <bool C2P, bool P2C, int DT>
const void* kernel_of(bool wide, bool equal, bool far) {
    if constexpr (C2P || P2C)
        if (far) return wide ? kernel_of<C2P, P2C, DT, 2, true>(equal) : kernel_of<C2P, P2C, DT, 1, true>(equal);
    return wide ? kernel_of<C2P, P2C, DT, 2, false>(equal) : kernel_of<C2P, P2C, DT, 1, false>(equal);
}
template <int DT>
const void* kernel_of(bool c2p, bool p2c, bool wide, bool equal, bool far) {
    return c2p ? (p2c ? kernel_of<true, true, DT>(wide, equal, far) : kernel_of<true, false, DT>(wide, equal, far))
               : (p2c ? kernel_of<false, true, DT>(wide, equal, far) : kernel_of<false, false, DT>(wide, equal, far));
}

}  // namespace

bool tdb_resident_supported(const TdbKernelParams& p, int dtype) {
    if ((dtype != TDB_BF16 && dtype != TDB_F16) || p.D != 64 || p.c2p || p.p2c) return false;
    if ((p.pk || p.pq) && 2 * int64_t(p.span) > MAX_ROWS) return false;
    // byte offsets inside a sequence and inside a head's table in 31 bits, head strides in 32
    const int64_t lim = int64_t(1) << 31;
    for (int64_t s : {p.qs_l, p.ks_l, p.vs_l, p.os_l})
        if (s * 2 * (int64_t(p.L) + 64) >= lim) return false;
    for (int64_t s : {p.qs_h, p.ks_h, p.vs_h, p.os_h, p.pks_h, p.pqs_h})
        if (s >= lim) return false;
    return (p.pks_r + p.pqs_r) * 2 * (MAX_ROWS + 256) < lim && int64_t(p.B) * p.H * (p.L / 64 + 1) < lim;
}

bool tdb_resident_wide(const TdbKernelParams& p) { return wide_units(p, grid_of(-1, p.H, 0)); }

// The persistent kernel (attn_mfma.hip) has tiles of 128 rows only and loads no whole tables: it is ahead where those tiles nearly fill
// one round of workgroups, and where few rounds leave many workgroups with less than the longest share.  Measured against that kernel as it
// was when it took every launch, over 5000 random ones of 161 to 4096 keys (6 to 24 heads; both terms, one or none; equal lengths, evenly
// spread ones and such as texts have): 1.09x by this rule, 1.115x if the fastest of the two kernels and both heights of units were known.
// Equal lengths 0.978x at worst; packed 2.5 % of the launches below 0.97x, 0.73x at worst (one of 3619 among 4 texts, 6 heads: 82 -> 113 us);
// padded, of which the host knows the longest possible length only, 2 % if lengths are evenly spread and 9 % if most are far below it, 0.73x
// (18 of up to 974, 359 in the mean, 8 heads: 37.5 -> 51).  No limit in L and rounds tells these from padded batches of nearly full texts, which
// would lose as much (1250 launches: limits of 3400 to 5000, 16-row units up to 2 to 4 rounds, the other kernel below 2.2 to 3.5 of them).
// From TDB_FAR_MIN_LEN on the far steps here take less time than there, and limits of their own hold, from random launches of up to
// 3.6 rounds: equal lengths all but one round of whole tiles (0.97x; two of them at 12 to 2: 1.05x); packed ones all but nearly a round, and
// what the limits at the end leave to the other kernel of lengths far apart (of 3000, evenly spread and such as texts have, 404 change, by 1.11x; 23 of these are
// below 0.97x, 0.845x at worst: 5 of 559 to 1700, 6 heads, 54 -> 64 us.  All of more than 1.3 rounds: 0.72x where the mean is below half of the
// longest, one of 2322 among 11, 370 in the mean, 52 -> 69); padded ones all but 1.2 to 1.75 rounds (of 3000 503 change, by 1.06x; 30 of these below
// 0.97x, 0.895x at worst; in between 1.05x, but 12 % below 0.97x).
bool tdb_resident_pays(const TdbKernelParams& p) {
    if (!p.pk && !p.pq) return true;        // (no tables to load: 1.21x over 708 such launches, 1.12x before this line)
    const Grid g = grid_of(-1, p.H, 0);
    const int64_t B = sequences_of(p), seqs = g.heads * B;
    const bool far = p.L >= TDB_FAR_MIN_LEN;
    if (!p.varlen && !p.seqlens) {          // (5.2, 5.8: a step of the persistent kernel's tile in units of StepCost)
        const int64_t rounds = (seqs * ((p.L + 127) / 128) + g.per_group - 1) / g.per_group;
        return std::min(equal_cost<1>(seqs, p.L, g.per_group), equal_cost<2>(seqs, p.L, g.per_group)) * 10 <= (far ? 58 : 52) * rounds;
    }
    const double rounds = ragged_rounds(p, g), mean = p.varlen ? double(p.total) / p.B / p.L : 1.0;
    if (far) {
        if (!p.varlen) return rounds <= 1.2 || rounds >= 1.75 || rounds * p.L >= 3400;
        if (rounds <= (mean > 0.9 ? 0.6 : 0.8)) return true;
        if (rounds <= 1.0) return false;
        if (mean > 0.65 || (mean >= 0.5 && rounds > 1.3)) return true;
    } else {
        if (p.L <= 4 * BN || rounds <= (p.L <= 900 ? 0.6 : 0.45)) return true;
        // Workgroups that keep one head load its tables once: launches of 257 to 1535 keys below the limits of the next line.  Packed, from a third of
        // the longest in the mean on, 785 of 3000 change, by 1.077x (below 2.25 rounds 0.98x); 24 of these are below 0.97x, 0.926x at worst (shorter
        // ones 0.78 to 1.02x: 53 of up to 1092, 120 in the mean, 51 -> 61 us).  Padded 1.085x if lengths are evenly spread, 0.95x at worst (3 to
        // 3.5 rounds 1.02x, and a quarter of them slower); such as texts have 1.02x, but 0.72x where most of a batch is padding (14 of up to 605, 145 in the
        // mean, 27 -> 37 us), which the host does not know.  With three heads 1.02x and 1.035x, but up to an eighth of them slower.
        if (g.heads == 1 && (p.varlen ? rounds >= 2.25 && mean >= 0.35 : rounds >= 3.5)) return true;
    }
    // (Of few rounds of very different lengths the longest alone decide: 2 of 650 and 2600 0.82x.  With a mask the lengths are only bounded.)
    return rounds * p.L >= (rounds >= (p.varlen ? 1.4 : 1.75) ? 3000 : 3400);
}

// All sequences of one length, or up to MAX_SEQS of different ones.
static hipError_t launch_part(const TdbKernelParams& p, bool wide, const Grid& g, int dev, int dtype, hipStream_t stream) {
    ResidentArgs a;
    a.q = static_cast<const char*>(p.q), a.k = static_cast<const char*>(p.k), a.v = static_cast<const char*>(p.v), a.o = static_cast<char*>(p.o);
    a.pk = static_cast<const char*>(p.pk), a.pq = static_cast<const char*>(p.pq);
    a.lut = p.lut, a.gap_cu = p.gap_cu, a.gap_B = p.gap_B;
    a.mode = p.varlen ? PACKED : p.seqlens ? LENGTHS : FIXED;
    a.bounds = p.varlen ? p.cu_seqlens : p.seqlens;
    auto bytes = [](int64_t s) { return uint32_t(2 * s); };
    a.qb = 2 * uint64_t(p.varlen ? p.qs_l : p.qs_b), a.qh = bytes(p.qs_h), a.ql = bytes(p.qs_l);
    a.kb = 2 * uint64_t(p.varlen ? p.ks_l : p.ks_b), a.kh = bytes(p.ks_h), a.kl = bytes(p.ks_l);
    a.vb = 2 * uint64_t(p.varlen ? p.vs_l : p.vs_b), a.vh = bytes(p.vs_h), a.vl = bytes(p.vs_l);
    a.ob = 2 * uint64_t(p.varlen ? p.os_l : p.os_b), a.oh = bytes(p.os_h), a.ol = bytes(p.os_l);
    a.pkh = bytes(p.pks_h), a.pkr = bytes(p.pks_r), a.pqh = bytes(p.pqs_h), a.pqr = bytes(p.pqs_r);
    a.B = p.B, a.H = p.H, a.L = p.L, a.total = p.total, a.lut_half = p.lut_half;
    const bool c2p = p.pk != nullptr, p2c = p.pq != nullptr;
    a.rows = c2p || p2c ? 2 * p.span : 0;
    a.c_exp = p.scale * 1.4426950408889634f;
    a.per_group = g.per_group, a.heads = g.heads;
    const bool equal = a.mode == FIXED, far = p.L >= TDB_FAR_MIN_LEN;
    const void* fn = dtype == TDB_F16 ? kernel_of<TDB_F16>(c2p, p2c, wide, equal, far) : kernel_of<TDB_BF16>(c2p, p2c, wide, equal, far);
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        bool& set = g_attr_set[dev][(far ? 32 : 0) + (wide ? 16 : 0) + (equal ? 8 : 0) + (dtype == TDB_F16 ? 4 : 0) + (c2p ? 2 : 0) + (p2c ? 1 : 0)];
        if (!set) {
            const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return e;
            set = true;
        }
    }
    const size_t lds = (int(c2p) + int(p2c)) * size_t(a.rows) * ROW + 4 * BLOCK;
    void* args[] = {&a};
    return hipLaunchKernel(fn, dim3(unsigned(g.wgs)), dim3(NTHREADS), args, lds, stream);
}

hipError_t tdb_launch_resident(const TdbKernelParams& whole, int dtype, hipStream_t stream) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    const Grid g = grid_of(dev, whole.H, tdb_mfma_workgroup_limit());
    const bool wide = wide_units(whole, g);
    const int per = sequences_of(whole);
    if (per == whole.B) return launch_part(whole, wide, g, dev, dtype, stream);
    for (int first = 0; first < whole.B; first += per) {        // in even parts
        TdbKernelParams part = whole;
        if (first > 0) part.gap_cu = nullptr;
        part.B = std::min(per, whole.B - first);
        if (whole.varlen) {
            part.cu_seqlens = whole.cu_seqlens + first;
        } else {
            auto at = [first](const void* base, int64_t stride_b) { return static_cast<const uint16_t*>(base) + first * stride_b; };
            part.seqlens = whole.seqlens + first;
            part.q = at(whole.q, whole.qs_b);
            part.k = at(whole.k, whole.ks_b);
            part.v = at(whole.v, whole.vs_b);
            part.o = const_cast<uint16_t*>(at(whole.o, whole.os_b));
        }
        e = launch_part(part, wide, g, dev, dtype, stream);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
