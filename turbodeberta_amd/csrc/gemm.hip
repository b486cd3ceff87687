// Dense products of an encoder layer, 16-bit in and out, float32 sums: y[M, N] = x[M, K] w[N, K]^T + bias, GELU on request.
//
// Bound: matrix cores where there are rows enough (the power limit leaves about 1.3 PFLOP/s), latency below some 2000 rows.
// The library's products take 9.5 us for 600 x 3072 x 768, its GELU another pass over the output, and its large ones leave
// the last round of tiles mostly empty.  Here:
//   * a workgroup computes one BM x BN tile, 64 columns of the contraction at a time.  Stages go from global memory straight
//     into LDS (16 bytes per lane, no registers in between) two or three steps ahead; fragments of the next 16 columns are
//     read, and loads issued, between the products of these, in the 32 clk that each keeps the matrix pipe busy; the barrier
//     of a step lies before its last products, whose operands are in registers by then.  One tile of 256 x 256 alone on a CU
//     steps at 89 % of the matrix pipe's rate, 128 x 256 at 85 %; with the loads in one burst behind the barrier: 65 %.
//   * the tile comes from a small cost model, the contraction is split where the output has too few tiles; the reader of the
//     output (residual + LayerNorm) adds up the parts.
//   * bias and GELU are applied to the float32 sums; results leave through LDS in whole rows.
//   * with more large tiles than compute units, a workgroup takes one after another, and the first stages of the next are on their
//     way while the last products of this one are made: a tile of 12 to 16 steps otherwise spends a third of its time on its start
//     and end (8190 x 3072 x 1024, weights in HBM, 53.1 -> 47.4 us; 8190 x 2304 x 768 39.3 -> 33.1; 8190 x 3072 x 768 with GELU 53.7 -> 49.5).
// A layer's four products and GELU (768 wide, library against these): 128 rows 39 / 23 us, 512 47 / 31, 1024 54 / 40, 4352
// 109 / 88, 8192 169 / 147; 1024 wide, 5000 rows 174 / 153.
#include <atomic>
#include <type_traits>

#include "tdb_encoder.h"
#include "tdb_internal.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <int DT>
struct Elem;
template <>
struct Elem<TDB_BF16> {
    using T = __bf16;
    using X8 = bf16x8;
    static __device__ __forceinline__ f32x16 mfma(X8 a, X8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Elem<TDB_F16> {
    using T = _Float16;
    using X8 = f16x8;
    static __device__ __forceinline__ f32x16 mfma(X8 a, X8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};

struct GemmArgs {
    const void *x, *w, *bias;
    void* y;
    int M, N, K, splits;
};

constexpr int BK = 64;                      // 128 bytes of a row: whole cache lines

// 64 lanes x 16 bytes from base + off (per lane) to 1 KB of LDS at `lds` (nothing else in this file uses m0)
__device__ __forceinline__ void load_lds(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
// one dword per lane, for its cache line's sake
__device__ __forceinline__ void touch_lds(uint32_t lds, const void* base, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LOOP: as many workgroups as compute units, each takes tile after tile.
template <int DT, int BM, int BN, int WM, int WN, int NS, bool GELU, bool PART, bool LOOP>
__global__ __launch_bounds__(WM* WN * 64, 2) void gemm_kernel(GemmArgs p) {
    using E = Elem<DT>;
    using T = typename E::T;
    using X8 = typename E::X8;
    typedef __attribute__((ext_vector_type(4))) T T4;
    constexpr int WAVES = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr int JX = BM / 8 / WAVES, JW = BN / 8 / WAVES;              // 1 KB loads of a wave per stage
    constexpr int STAGE = (BM + BN) * BK * 2;
    // The weights come from HBM (those of a whole model are more than the caches hold), and the two or three stages ahead are
    // less than its latency: with larger tiles every workgroup first asks for its share of all of them, a load per cache line.
    constexpr bool TOUCH = BM * BN > 64 * 64;
    static_assert(JX * 8 * WAVES == BM && JW * 8 * WAVES == BN, "");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int wm = wave / WN, wn = wave % WN;

    // tile: blocks of one XCD (ids equal mod 8) take neighbouring ones, eight rows of tiles at a time
    const int mt = (p.M + BM - 1) / BM, nt = (p.N + BN - 1) / BN, tiles = mt * nt;
    int m0, n0, split = 0;
    auto locate = [&](int b) {
        const int all = tiles * (PART ? p.splits : 1), q = all >> 3, r = all & 7, xcd = b & 7;
        b = xcd * q + min(xcd, r) + (b >> 3);
        if (PART) {
            split = b / tiles;
            b -= split * tiles;
        }
        const int group = b / (8 * nt), in = b - group * 8 * nt, rows = min(8, mt - 8 * group);
        const int n = in / rows;
        m0 = (group * 8 + in - n * rows) * BM;
        n0 = n * BN;
    };
    int number = blockIdx.x;
    locate(number);
    const int steps_all = p.K / BK;
    const int k0 = PART ? steps_all * split / p.splits : 0, k1 = PART ? steps_all * (split + 1) / p.splits : steps_all, steps = k1 - k0;

    // A row is 8 chunks of 16 bytes; chunk c of row r lies at c ^ (r / 2 % 8): fragment reads (16 rows, one chunk) are free of
    // bank conflicts, and a load still covers whole rows.
    uint32_t xo[JX], wo[JW];
    auto rows_of = [&](int m, int n) {      // where the loads of the tile at row m and column n start
#pragma unroll
        for (int j = 0; j < JX; ++j) {
            const int row = (wave * JX + j) * 8 + (l >> 3);
            xo[j] = uint32_t(min(m + row, p.M - 1)) * uint32_t(p.K * 2) + (((l & 7) ^ ((row >> 1) & 7)) << 4);
        }
#pragma unroll
        for (int j = 0; j < JW; ++j) {
            const int row = (wave * JW + j) * 8 + (l >> 3);
            wo[j] = uint32_t(min(n + row, p.N - 1)) * uint32_t(p.K * 2) + (((l & 7) ^ ((row >> 1) & 7)) << 4);
        }
    };
    rows_of(m0, n0);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)smem)));
    constexpr int L = JX + JW;
    auto load = [&](int step, int stage, int lo, int hi) {              // loads lo .. hi - 1 of the L of a stage
        const char* const xb = static_cast<const char*>(p.x) + int64_t(k0 + step) * (BK * 2);
        const char* const wb = static_cast<const char*>(p.w) + int64_t(k0 + step) * (BK * 2);
        const uint32_t at = lds0 + stage * STAGE + wave * (JX * 1024), bt = lds0 + stage * STAGE + BM * 128 + wave * (JW * 1024);
#pragma unroll
        for (int j = 0; j < L; ++j)
            if (j >= lo && j < hi) {
                if (j < JX) load_lds(at + j * 1024, xb, xo[j < JX ? j : 0]);
                else load_lds(bt + (j - JX) * 1024, wb, wo[j < JX ? 0 : j - JX]);
            }
    };
    f32x16 acc[TM][TN];
    auto clear = [&]() {
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
    };
    clear();
    const int h = l >> 5;
    int frag[4];                            // chunk 2 kk + h of row l % 32
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) frag[kk] = (l & 31) * 128 + (((2 * kk + h) ^ ((l >> 1) & 7)) << 4);

    // The loads of stage s + NS are issued in parts: 0 behind the last products of step s, the others behind those of step s + 1
    // (with two stages, where they have to be back at its end, in its first quarter).
    constexpr int PARTS = NS == 2 ? 2 : 4;
    auto from = [](int part) { return part >= PARTS ? L : L * part / PARTS; };
#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
        if (s < steps) load(s, s, 0, L);
    if (TOUCH) {
        const uint32_t lines = uint32_t(p.N) * uint32_t(steps_all), threads = gridDim.x * (WAVES * 64);
        for (uint32_t i = blockIdx.x * (WAVES * 64) + threadIdx.x; i < lines; i += threads) {
            const uint32_t k = i / uint32_t(p.N), n = i - k * uint32_t(p.N);
            touch_lds(lds0 + NS * STAGE, p.w, n * uint32_t(p.K * 2) + k * (BK * 2));
        }
    }
    if (NS - 1 < steps) load(NS - 1, NS - 1, 0, from(1));
    X8 a[2][TN], b[2][TM];
    auto read = [&](int stage, int kk, int set, int op) {               // fragment `op` of TN + TM
        if (op < TN) a[set][op] = *reinterpret_cast<const X8*>(smem + stage * STAGE + BM * 128 + wn * (TN * 32 * 128) + frag[kk] + op * 4096);
        else b[set][op - TN] = *reinterpret_cast<const X8*>(smem + stage * STAGE + wm * (TM * 32 * 128) + frag[kk] + (op - TN) * 4096);
    };
    // Products of fragment set kk % 2; between them the reads of the next set and a part of the loads: the matrix pipe is busy
    // for 32 clk per product, an instruction in its shadow costs nothing.
    auto multiply = [&](int kk, auto READ, int rstage, auto LOAD, int lstep, int lstage, int part) {
        constexpr int OPS = TM * TN, R = TM + TN;
        const int lo = from(part), n = from(part + 1) - lo;
#pragma unroll
        for (int op = 0; op < OPS; ++op) {
            acc[op / TN][op % TN] = E::mfma(a[kk & 1][op % TN], b[kk & 1][op / TN], acc[op / TN][op % TN]);
            __builtin_amdgcn_sched_barrier(0);
            if (decltype(READ)::value) {
#pragma unroll
                for (int r = R * op / OPS; r < R * (op + 1) / OPS; ++r) read(rstage, (kk + 1) & 3, (kk + 1) & 1, r);
            }
            if (decltype(LOAD)::value) load(lstep, lstage, lo + n * op / OPS, lo + n * (op + 1) / OPS);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    constexpr std::true_type yes;
    constexpr std::false_type no;
    if (steps >= NS) wait_loads<(NS - 2) * L + L / PARTS>();
    else wait_loads<0>();
    barrier();
#pragma unroll
    for (int r = 0; r < TM + TN; ++r) read(0, 0, 0, r);
    int stage = 0, before = NS - 1;         // of this step, of the one before it
    auto step = [&](int s, auto REST, auto NEXT, auto MORE) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 3; ++kk) multiply(kk, yes, stage, REST, s + NS - 1, before, kk + 1);
        // The next stage has landed (at most the NS - 2 after it are under way) and everybody has read this one.
        if (decltype(MORE)::value) {
            if (decltype(REST)::value) wait_loads<(NS - 2) * L>();
            else wait_loads<0>();
            barrier();
        }
        before = stage;
        stage = stage == NS - 1 ? 0 : stage + 1;
        multiply(3, MORE, stage, NEXT, s + NS, before, 0);
    };
    // The finished tile, by way of the weights' part of stage `at` that this wave itself loads: rows of COLS columns, their 16-byte chunks
    // exchanged by the row's middle bits and, in the upper half of the rows, the chunks' halves too, so that writes of 8 bytes to 32 rows
    // meet every bank once.  (Everybody has read that stage.)
    auto finish = [&](int m, int n0, int at) {
        T4 bias[TN][4];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                bias[j][g] = *reinterpret_cast<const T4*>(static_cast<const T*>(p.bias) + min(n0 + (wn * TN + j) * 32 + 8 * g + 4 * h, p.N - 4));
        constexpr int COLS = TN * 32, LANES = COLS / 8, LOW = LANES == 8 ? 1 : 2;       // lanes per row of the way out
        static_assert(32 * COLS * 2 <= JW * 1024 && (LANES == 8 || LANES == 4), "");
        char* const mine = smem + at * STAGE + BM * 128 + wave * (JW * 1024);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    T4 out;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        float v = acc[i][j][4 * g + e] + float(bias[j][g][e]);
                        if (GELU) v = tdb_gelu(v);
                        out[e] = T(v);
                    }
                    *reinterpret_cast<T4*>(mine + (l & 31) * (COLS * 2) + (((j * 4 + g) ^ (l >> LOW & (LANES - 1))) << 4) + 8 * (h ^ (l >> 4 & 1))) = out;
                }
#pragma unroll
            for (int r = 0; r < 32 * LANES / 64; ++r) {
                const int row = r * (64 / LANES) + l / LANES, c = l % LANES;
                uint4 v = *reinterpret_cast<const uint4*>(mine + row * (COLS * 2) + ((c ^ (row >> LOW & (LANES - 1))) << 4));
                if (row & 16) v = uint4{v.z, v.w, v.x, v.y};
                const int to = m + (wm * TM + i) * 32 + row, n = n0 + wn * COLS + c * 8;
                if (to < p.M && n < p.N) *reinterpret_cast<uint4*>(static_cast<T*>(p.y) + int64_t(to) * p.N + n) = v;
            }
        }
    };

    int s = 0;
    if constexpr (LOOP) {
        // The stages of the next tile follow those of this one as if they were its next steps; only the last part of the way, behind the last
        // products, waits for the tile to leave through its stage.  (steps > NS)
        while (number + int(gridDim.x) < tiles) {
            const int m = m0, n = n0;
            for (s = 0; s < steps - NS; ++s) step(s, yes, yes, yes);
            number += gridDim.x;
            locate(number);
            step(s++, yes, no, yes);        // its last loads
            rows_of(m0, n0);
            load(0, before, 0, from(1));
            for (; s < steps - 1; ++s) step(s - steps, yes, yes, yes);
            step(s - steps, yes, no, yes);
            finish(m, n, before);
            load(NS - 1, before, 0, from(1));
            clear();
        }
    }
    for (s = 0; s < steps - NS; ++s) step(s, yes, yes, yes);
    if (s == steps - NS && s < steps - 1) step(s++, yes, no, yes);
    for (; s < steps - 1; ++s) step(s, no, no, yes);
    step(s, no, no, no);

    // Lane l holds, of token row l % 32 of its tile, columns 8 g + 4 h .. +3.
    if (PART) {
        float* const y = static_cast<float*>(p.y) + int64_t(split) * p.M * p.N;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = m0 + (wm * TM + i) * 32 + (l & 31);
            if (row < p.M)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int col = n0 + (wn * TN + j) * 32 + 8 * g + 4 * h;
                        f32x4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                        if (col < p.N) *reinterpret_cast<f32x4*>(y + int64_t(row) * p.N + col) = v;
                    }
        }
        return;
    }
    barrier();
    finish(m0, n0, before);
}

// What a launch of each tile takes, in us:
//   base + fill round + n (steps step + [GELU] gelu)
// with n = the most tiles that a CU gets, fill = tiles per CU, steps = K / 64.  Fitted to measurements of N and K from 768 to
// 4096 and 80 to 8192 rows, weights in HBM; the tile of least cost is on average within 0.5 % of the best one there.
struct Cost {
    int bm, bn;
    float base, round, step, gelu;
};
// (192 x 128 is for outputs that give the other large tiles a nearly empty last round.  Of 144 products of 1200 to 9000 rows, 512 to 1536 wide,
// 43 take it, 1.093x as fast as what they took before: 1900 x 2304 x 768 11.7 -> 10.3 us, 5800 x 768 x 3072 32.4 -> 29.6, 4100 x 1024 x 1024
// 13.6 -> 12.2, 7500 x 2304 x 768 40.4 -> 29.8.  3700 x 3072 x 768 with GELU 28.3 -> 29.8 and 2600 x 1024 x 4096 28.1 -> 29.1 are the two
// below 0.97x; the other 101 products 1.016x.)
constexpr Cost COST[] = {{32, 64, 2.96f, 0.62f, 0.148f, 0.07f},  {64, 64, 2.86f, 0.76f, 0.205f, 0.f},   {128, 64, 3.22f, 1.37f, 0.29f, 0.11f},
                         {128, 128, 2.59f, 4.38f, 0.402f, 0.93f}, {128, 256, 2.67f, 7.89f, 0.601f, 2.59f}, {256, 256, 3.55f, 3.7f, 1.195f, 11.09f},
                         {192, 128, 3.3f, 6.f, 0.47f, 1.9f}};
// 128 x 256 and 192 x 128 where workgroups take one tile after another.
constexpr Cost LOOP_COST[] = {{128, 256, 3.5f, 3.9f, 0.65f, 3.6f}, {192, 128, 2.35f, 5.f, 0.45f, 2.2f}};
constexpr int TILES = 7;
constexpr int SPLITS[] = {1, 2, 3, 4, 6, 8};

float cost(int tile, int splits, int M, int N, int K, bool gelu, int cus) {
    const int64_t blocks = int64_t((M + COST[tile].bm - 1) / COST[tile].bm) * ((N + COST[tile].bn - 1) / COST[tile].bn) * splits;
    const Cost& c = (tile == 4 || tile == 6) && splits == 1 && blocks > cus ? LOOP_COST[tile / 6] : COST[tile];
    const float steps = float(K / BK) / float(splits), n = float((blocks + cus - 1) / cus), fill = float(blocks) / float(cus);
    // Partial sums are written, and read by the kernel after this one, at some 5 bytes per ns.
    const float parts = splits > 1 ? float(splits * 8 - 4) * float(M) * float(N) / 5e6f : 0.f;
    return c.base + fill * c.round + n * (steps * c.step + (gelu ? c.gelu : 0.f)) + parts;
}

struct Choice {
    int tile, splits;
};
Choice choose(int M, int N, int K, bool gelu, int splits) {             // splits 0: any
    Choice best{1, 1};
    float least = 1e30f;
    const int cus = tdb_compute_units(-1);
    for (int t = 0; t < TILES; ++t)
        for (int s : SPLITS) {
            if (splits ? s != splits : s > 1 && s > K / BK / 2) continue;
            if (const float c = cost(t, s, M, N, K, gelu, cus); c < least) least = c, best = {t, s};
        }
    return best;
}

bool takes(int M, int N, int K, int dtype) {
    return (dtype == TDB_BF16 || dtype == TDB_F16) && M >= 1 && N >= 8 && N % 8 == 0 && K >= BK && K % BK == 0 && int64_t(M) * K <= 1 << 30 && int64_t(N) * K <= 1 << 30;
}

template <int DT, int BM, int BN, int WM, int WN, int NS>
int launch(const GemmArgs& a, bool gelu, hipStream_t s) {
    constexpr int smem = NS * (BM + BN) * BK * 2 + 256;
    const int blocks = (a.M + BM - 1) / BM * ((a.N + BN - 1) / BN) * a.splits, cus = tdb_compute_units(-1) & -8;
    auto go = [&](auto kernel, std::atomic<uint64_t>& raised, int grid) {
        int dev = 0;
        if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return int(e);
        if (!(raised.load(std::memory_order_acquire) >> dev & 1)) {     // (twice does no harm)
            if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, smem); e != hipSuccess) return int(e);
            raised.fetch_or(uint64_t(1) << dev, std::memory_order_release);
        }
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(WM * WN * 64), smem, s, a);
        return int(hipGetLastError());
    };
    static std::atomic<uint64_t> raised[5];
    if (a.splits > 1) return go(gemm_kernel<DT, BM, BN, WM, WN, NS, false, true, false>, raised[0], blocks);
    if constexpr (BM * BN >= 192 * 128)
        if (blocks > cus && cus >= 8 && a.K / BK > NS)
            return gelu ? go(gemm_kernel<DT, BM, BN, WM, WN, NS, true, false, true>, raised[3], cus) : go(gemm_kernel<DT, BM, BN, WM, WN, NS, false, false, true>, raised[4], cus);
    if (gelu) return go(gemm_kernel<DT, BM, BN, WM, WN, NS, true, false, false>, raised[1], blocks);
    return go(gemm_kernel<DT, BM, BN, WM, WN, NS, false, false, false>, raised[2], blocks);
}

template <int DT>
int launch_tile(int tile, const GemmArgs& a, bool gelu, hipStream_t s) {
    switch (tile) {
        case 0: return launch<DT, 32, 64, 1, 2, 6>(a, gelu, s);
        case 1: return launch<DT, 64, 64, 2, 2, 4>(a, gelu, s);
        case 2: return launch<DT, 128, 64, 2, 2, 3>(a, gelu, s);
        case 3: return launch<DT, 128, 128, 2, 4, 4>(a, gelu, s);
        case 4: return launch<DT, 128, 256, 2, 4, 3>(a, gelu, s);
        case 5: return launch<DT, 256, 256, 2, 4, 2>(a, gelu, s);
        default: return launch<DT, 192, 128, 2, 4, 3>(a, gelu, s);
    }
}

}  // namespace

extern "C" {

int tdb_enc_gemm_splits(int M, int N, int K, int dtype) { return takes(M, N, K, dtype) ? choose(M, N, K, false, 0).splits : 0; }

int tdb_enc_gemm(const void* x, const void* w, const void* bias, int flags, int splits, int M, int N, int K, int dtype, void* y, void* stream) {
    if (!takes(M, N, K, dtype) || splits < 1 || splits > K / BK || (splits > 1 && flags & TDB_ENC_GELU)) return int(hipErrorInvalidValue);
    const bool gelu = flags & TDB_ENC_GELU;
    const int forced = flags >> TDB_ENC_TILE_SHIFT;
    if (forced > TILES) return int(hipErrorInvalidValue);
    const int tile = forced > 0 ? forced - 1 : choose(M, N, K, gelu, splits).tile;
    const GemmArgs a{x, w, bias, y, M, N, K, splits};
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dtype == TDB_BF16 ? launch_tile<TDB_BF16>(tile, a, gelu, s) : launch_tile<TDB_F16>(tile, a, gelu, s);
}

}  // extern "C"
