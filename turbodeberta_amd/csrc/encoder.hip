// The kernels around attention in an encoder layer: embeddings, residual + LayerNorm, products with few rows, mask scan,
// unpacking.  Products with more rows are in gemm.hip; what is here is bound by memory traffic or by latency:
//   * residual + LayerNorm in one pass, a wave per row with the row in registers: three arrays of traffic instead of five.
//   * products with at most 64 rows (a single text): the library takes 8-10 us for 48 x 768 x 768 where the weights are
//     read in well under one.  Here a workgroup takes 16 output columns and its waves share out the contraction, so that all
//     of the weight matrix is requested at once; sums of the waves meet in LDS.  Where the output has too few columns to
//     fill the chip (hidden-sized ones), the contraction is split over workgroups as well, and the residual + LayerNorm
//     that follows adds the parts up in a fixed order.
#include <algorithm>
#include <type_traits>

#include "tdb_encoder.h"
#include "tdb_internal.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

template <int DT>
struct Elem;
template <>
struct Elem<TDB_BF16> {
    using T = __bf16;
    using X8 = bf16x8;
    static __device__ __forceinline__ f32x4 mfma(X8 a, X8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <>
struct Elem<TDB_F16> {
    using T = _Float16;
    using X8 = f16x8;
    static __device__ __forceinline__ f32x4 mfma(X8 a, X8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <>
struct Elem<TDB_F32> {
    using T = float;
};

constexpr int MAX_SPLITS = 8;

// eight consecutive elements as float32, and back
template <int DT>
__device__ __forceinline__ void load8(const void* p, int64_t at, float (&v)[8]) {
    using T = typename Elem<DT>::T;
    typedef __attribute__((ext_vector_type(8))) T T8;
    const T8 x = *reinterpret_cast<const T8*>(static_cast<const T*>(p) + at);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = float(x[i]);
}
template <int DT>
__device__ __forceinline__ void store8(void* p, int64_t at, const float (&v)[8]) {
    using T = typename Elem<DT>::T;
    typedef __attribute__((ext_vector_type(8))) T T8;
    T8 x;
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = T(v[i]);
    *reinterpret_cast<T8*>(static_cast<T*>(p) + at) = x;
}

// Rows of activations, in element offsets of chunk `chunk` (eight columns) of row t.  mt = 0: row after row.  mt > 0, used
// between the kernels of a short call: in the order in which the products load them -- 32 columns x 16 rows after another,
// mt of them per 32 columns --, so that a load instruction covers 1 KB in one piece.  (In row order its 64 lanes touch 16 rows,
// consecutive lanes different ones, and it occupies the CU's load path for 54 clk instead of 16: 48 x 3072 x 768 6.1 us.)
__device__ __forceinline__ int64_t row_at(int t, int chunk, int hidden, int mt) {
    return mt == 0 ? int64_t(t) * hidden + chunk * 8 : int64_t((((chunk >> 2) * mt + (t >> 4)) * 64 + (chunk & 3) * 16 + (t & 15)) * 8);
}

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    return x;
}

// LayerNorm of a row held by a wave: lane l has the chunks of eight l, l + 64, ...; chunks past the row hold zeros.
// (The caller loads the scale and shift with the row: behind the sums they would be another round trip.)
template <int DT, int CH>
__device__ __forceinline__ void load_affine(float (&w)[CH][8], float (&b)[CH][8], int chunks, const void* gamma, const void* beta) {
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const int el = min(l + 64 * c, chunks - 1) * 8;
        load8<DT>(gamma, el, w[c]);
        load8<DT>(beta, el, b[c]);
    }
}
template <int DT, int CH>
__device__ __forceinline__ void norm_row(float (&v)[CH][8], const float (&w)[CH][8], const float (&b)[CH][8], int chunks, int hidden, float eps,
                                         void* out, int t, int mt) {
    const int l = threadIdx.x & 63;
    float sum = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += v[c][i];
    const float mean = wave_sum(sum) / float(hidden);
    float sq = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c)
        if (l + 64 * c < chunks) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float d = v[c][i] - mean;
                sq += d * d;
            }
        }
    const float rstd = rsqrtf(wave_sum(sq) / float(hidden) + eps);
#pragma unroll
    for (int c = 0; c < CH; ++c)
        if (l + 64 * c < chunks) {
            float y[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) y[i] = (v[c][i] - mean) * rstd * w[c][i] + b[c][i];
            store8<DT>(out, row_at(t, l + 64 * c, hidden, mt), y);
        }
}

// Row t, columns 4 c4 .. + 3 of rows in float32 (see norm_gemm_kernel), in the order in which the products load them: 1 KB in one piece for a load instruction.
__device__ __forceinline__ int64_t x_at(int t, int c4, int mt) { return int64_t((((c4 >> 3) * mt + (t >> 4)) * 2 + (c4 & 1)) * 64 + ((c4 >> 1) & 3) * 16 + (t & 15)) * 4; }

// ROWS: the row before its LayerNorm (`out`, `stats`) for the products that normalise what they load.
template <int DT, int CH, bool ROWS>
__global__ __launch_bounds__(256) void embed_kernel(const void* ids, int ids64, const void* table, int64_t vocab, const void* gamma,
                                                    const void* beta, float eps, const int32_t* cu, int B, int L, int T, int hidden,
                                                    int mt, void* out, float2* stats) {
    const int t = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63, chunks = hidden / 8;
    if (t >= T) return;
    int64_t at = t;
    if (cu) {                               // packed token t: the sequence b with cu[b] <= t < cu[b+1]
        int lo = 0, hi = B;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (cu[mid] <= t) lo = mid;
            else hi = mid;
        }
        at = min(max(int64_t(lo) * L + (t - cu[lo]), int64_t(0)), int64_t(B) * L - 1);     // (a caller's boundaries may not fit)
    }
    const int64_t id = ids64 ? static_cast<const int64_t*>(ids)[at] : static_cast<const int32_t*>(ids)[at];
    const bool ok = id >= 0 && id < vocab;
    float v[CH][8], w[CH][8], b[CH][8];
    if constexpr (!ROWS) load_affine<DT, CH>(w, b, chunks, gamma, beta);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[c][i] = 0.f;
        if (l + 64 * c < chunks) {
            if (ok) load8<DT>(table, id * hidden + (l + 64 * c) * 8, v[c]);
            else v[c][0] = __builtin_nanf("");          // an id outside the table: the row says so
        }
    }
    if constexpr (ROWS) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            float sum = 0.f, dev = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) sum += v[c][i];
            const float mid = (sum + __shfl_xor(sum, 1)) * (1.f / 16.f);
#pragma unroll
            for (int i = 0; i < 8; ++i) dev += (v[c][i] - mid) * (v[c][i] - mid);
            dev += __shfl_xor(dev, 1);
            const int chunk = l + 64 * c;
            if (chunk < chunks) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + x_at(t, 2 * chunk + h, mt)) = f32x4{v[c][4 * h], v[c][4 * h + 1], v[c][4 * h + 2], v[c][4 * h + 3]};
                if (!(l & 1)) stats[(chunk >> 1) * 16 * mt + t] = float2{mid, dev};
            }
        }
    } else {
        norm_row<DT, CH>(v, w, b, chunks, hidden, eps, out, t, mt);
    }
}

template <int DT, int CH, int PARTS>      // PARTS: 0, or the most partial sums
__global__ __launch_bounds__(256) void add_norm_kernel(const void* x, int splits, const void* bias, const void* residual, const void* gamma,
                                                       const void* beta, float eps, int T, int hidden, int mt_in, int mt_out, void* out) {
    const int t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6), l = threadIdx.x & 63, chunks = hidden / 8;
    if (t >= T) return;
    const int64_t at = int64_t(t) * hidden;
    float v[CH][8], w[CH][8], b[CH][8];
    load_affine<DT, CH>(w, b, chunks, gamma, beta);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[c][i] = 0.f;
        const int el = (l + 64 * c) * 8;
        if (l + 64 * c < chunks) {
            float r[8];
            load8<DT>(residual, row_at(t, l + 64 * c, hidden, mt_in), r);
            if constexpr (PARTS > 0) {
                float y[PARTS][8], add[8];             // all requested before the first is added; past the last: it again
#pragma unroll
                for (int s = 0; s < PARTS; ++s) load8<TDB_F32>(x, int64_t(min(s, splits - 1)) * T * hidden + at + el, y[s]);
                load8<DT>(bias, el, add);
#pragma unroll
                for (int s = 0; s < PARTS; ++s)
                    if (s < splits) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) v[c][i] += y[s][i];
                    }
#pragma unroll
                for (int i = 0; i < 8; ++i) v[c][i] += add[i];
            } else {
                load8<DT>(x, at + el, v[c]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) v[c][i] += r[i];
        }
    }
    norm_row<DT, CH>(v, w, b, chunks, hidden, eps, out, t, mt_out);
}

// Fragments of 16 rows x 32 columns whose rows lie apart (weights): a load in operand order, consecutive lanes in different rows, occupies the
// CU's load path for 54 clk; here four lanes share a row (16 clk), and the wave's own LDS brings the chunks to their lanes.  (Replayed as a graph, operand order ->
// this: 12 layers of 768, 48 rows 357 -> 351 us, 24 of 1024 862 -> 848, 8 of 1536 451 -> 433.)
__device__ __forceinline__ int row_chunk(int l) { return (l & 3) ^ ((l >> 4) & 3); }       // lane l loads this chunk of eight of row l >> 2
// N fragments at once (slots: 64 N of the wave's own), so that one waits for LDS under the next.
template <int N, typename X8>
__device__ __forceinline__ void to_operands(X8* slots, X8 (&x)[N]) {
    const int l = threadIdx.x & 63, c = l & 15, g = l >> 4;
#pragma unroll
    for (int i = 0; i < N; ++i) slots[64 * i + l] = x[i];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");          // (a wave's LDS accesses are in order: only the compiler is held back)
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = slots[64 * i + 4 * c + (g ^ ((c >> 2) & 3))];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One workgroup: 16 columns of the output, a share of the contraction given by blockIdx.y and, inside it, by the wave.
// MT: token tiles of 16.  Lane (c, g) has 16 bytes of weight row n0 + c and of token row 16 m + c: columns 32 k + 8 g .. +7.
// IN / OUT: x / y in the order of row_at.
template <int DT, int MT, bool IN, bool OUT, bool GELU, bool PART>
__global__ __launch_bounds__(512) void small_gemm_kernel(const void* xv, const void* wv, const void* bias, void* y, int M, int N, int K, int splits) {
    using E = Elem<DT>;
    using X8 = typename E::X8;
    using T = typename E::T;
    extern __shared__ __attribute__((aligned(16))) float red[];
    __shared__ X8 s_w[8 * 4 * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6, l = threadIdx.x & 63;
    const int c = l & 15, g = l >> 4, n0 = blockIdx.x * 16, steps = K / 32;
    const int parts = splits * waves, part = blockIdx.y * waves + wave;
    const int k0 = steps * part / parts, k1 = steps * (part + 1) / parts;
    const T* const w = static_cast<const T*>(wv) + int64_t(n0 + (l >> 2)) * K + 8 * row_chunk(l);
    const T* x[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) x[m] = static_cast<const T*>(xv) + (IN ? m * 512 + l * 8 : min(16 * m + (l >> 2), M - 1) * K + 8 * row_chunk(l));
    typedef __attribute__((ext_vector_type(4))) T T4;
    const int col = n0 + 4 * g;             // (of every element this thread sums up below)
    T4 b4;
    if (!PART) b4 = *reinterpret_cast<const T4*>(static_cast<const T*>(bias) + col);
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto run = [&](int k, auto count) {     // `count` steps from k: all requested before the first is used
        constexpr int U = decltype(count)::value;
        X8 a[U], b[U][MT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a[u] = *reinterpret_cast<const X8*>(w + 32 * (k + u));
#pragma unroll
            for (int m = 0; m < MT; ++m) b[u][m] = *reinterpret_cast<const X8*>(x[m] + (k + u) * (IN ? MT * 512 : 32));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (!IN) to_operands(s_w + wave * 256, b[u]);
        }
        to_operands(s_w + wave * 256, a);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = E::mfma(a[u], b[u][m], acc[m]);
    };
    int k = k0;
    for (; k + 3 <= k1; k += 3) run(k, std::integral_constant<int, 3>{});
    if (k + 2 == k1) run(k, std::integral_constant<int, 2>{});
    else if (k + 1 == k1) run(k, std::integral_constant<int, 1>{});
#pragma unroll
    for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(&red[((wave * MT + m) * 64 + l) * 4]) = acc[m];
    __syncthreads();
    for (int idx = threadIdx.x; idx < MT * 64; idx += blockDim.x) {
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int v = 0; v < waves; ++v) sum += *reinterpret_cast<const f32x4*>(&red[(v * MT * 64 + idx) * 4]);
        const int row = 16 * (idx >> 6) + (idx & 15);
        if (row >= M) continue;
        if (PART) {
            *reinterpret_cast<f32x4*>(static_cast<float*>(y) + (int64_t(blockIdx.y) * M + row) * N + col) = sum;
        } else {
            T4 out;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float v = sum[i] + float(b4[i]);
                if (GELU) v = tdb_gelu(v);
                out[i] = T(v);
            }
            *reinterpret_cast<T4*>(static_cast<T*>(y) + row_at(row, col >> 3, N, OUT ? MT : 0) + (col & 7)) = out;
        }
    }
}

// The two kinds of products of a short request, where a launch costs as much as what it does: the residual + LayerNorm between them
// is no launch of its own.  A product with a hidden-sized output adds the residual in its epilogue and writes the row before its LayerNorm in
// float32, with the mean and the sum of squared deviations of each 16 columns (`x`, `stats`); whoever reads the row joins these and normalises
// what it loads.  A workgroup takes 16 rows and 16 columns of the output, its waves share out the contraction.
// What bounds them: a launch (1.6 us even in a graph), one round trip for what the kernel before wrote, and what a CU reads, at some 30 bytes a clk: hence
// workgroups of few rows and as many columns as leave one workgroup to a CU.  12 layers of 768 as a graph, 7 launches a layer -> 5: 48 rows
// 351 -> 338 us, 64 rows 366 -> 346; as launches 13 % where the host is slow.  See FUSED_WIDTH.

// Sums of a row's blocks of 16 columns around the mean of the first one.
struct Moments {
    float shift, d, dd, q;                  // sums of (mean - shift), its square, and squared deviations
    __device__ __forceinline__ void join(float& mean, float& rstd, int hidden, float eps) const {
        const float blocks = float(hidden / 16);
        mean = shift + d / blocks;
        rstd = rsqrtf((q + 16.f * (dd - d * d / blocks)) / float(hidden) + eps);
    }
};
// This thread's share of row 16 m + (thread & 15), whose blocks the groups of 16 threads share out: requested, then summed up over the wave.
template <int GROUPS>
struct MomentLoads {
    static constexpr int AT_ONCE = 64 / GROUPS < 2 ? 2 : 64 / GROUPS;   // (all of a row of 1024)
    const float2* at;
    float2 first, v[AT_ONCE];
    int blocks, rows;
    __device__ __forceinline__ void request(const float2* stats, int hidden, int mt, int m) {
        blocks = hidden / 16, rows = 16 * mt, at = stats + 16 * m + (threadIdx.x & 15);
        first = at[0];
        more(0);
    }
    __device__ __forceinline__ void more(int from) {
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) v[i] = at[min(from + i * GROUPS + int(threadIdx.x >> 4), blocks - 1) * rows];
    }
    __device__ __forceinline__ Moments sums() {
        Moments s = {first.x, 0.f, 0.f, 0.f};
        for (int from = 0;;) {
#pragma unroll
            for (int i = 0; i < AT_ONCE; ++i)
                if (from + i * GROUPS + int(threadIdx.x >> 4) < blocks) {
                    const float d = v[i].x - s.shift;
                    s.d += d, s.dd += d * d, s.q += v[i].y;
                }
            from += AT_ONCE * GROUPS;
            if (from >= blocks) break;
            more(from);
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) s.d += __shfl_xor(s.d, o), s.dd += __shfl_xor(s.dd, o), s.q += __shfl_xor(s.q, o);
        return s;
    }
};
// (LDS: [wave][row] of three sums)
__device__ __forceinline__ void put_moments(float4* lds, const Moments& s) {
    if ((threadIdx.x & 63) < 16) lds[(threadIdx.x >> 6) * 16 + (threadIdx.x & 15)] = float4{s.d, s.dd, s.q, 0.f};
}
__device__ __forceinline__ void get_moments(const float4* lds, int waves, Moments s, int hidden, float eps, float& mean, float& rstd) {
    s.d = s.dd = s.q = 0.f;
    for (int w = 0; w < waves; ++w) {
        const float4 v = lds[w * 16 + (threadIdx.x & 15)];
        s.d += v.x, s.dd += v.y, s.q += v.z;
    }
    s.join(mean, rstd, hidden, eps);
}

// f(how many of the steps that are left come next, at most MOST)
template <int MOST, typename F>
__device__ __forceinline__ void with_steps(int left, F f) {
    if (left >= MOST) f(std::integral_constant<int, MOST>{});
    else if constexpr (MOST > 1) with_steps<MOST - 1>(left, f);
}

// Weights of the products to come, brought into the L2 of the XCD that will read them by workgroups of their own (blockIdx.y >= mt), beside the present
// product as far as there is room: chunk i, the rows of one workgroup of that product, by blocks whose number is i modulo 8, which go to the same XCD.  (12 layers of 768, 48 rows, weights in HBM: 414 -> 380 us; weights in the last-level cache 348 -> 343.
// The attention's table rows as well: no change.)
struct Ahead {
    static constexpr int MOST = 2;
    const char* w[MOST];
    int lines[MOST], chunks[MOST];          // 128-byte lines of a chunk
    __device__ __forceinline__ void fetch(int mt) const {
        const int id = blockIdx.y * gridDim.x + blockIdx.x, xcd = id & 7;
        const int thread = ((id - mt * gridDim.x) >> 3) * blockDim.x + threadIdx.x, threads = max((int(gridDim.y - mt) * int(gridDim.x)) >> 3, 1) * blockDim.x;
        uint32_t any = 0;
#pragma unroll
        for (int i = 0; i < MOST; ++i) {
            const int mine = (chunks[i] - xcd + 7) >> 3;        // chunks of this XCD
            for (int at = thread; at < mine * lines[i]; at += threads) {
                const int chunk = at / lines[i];
                any |= *reinterpret_cast<const uint32_t*>(w[i] + (int64_t(8 * chunk + xcd) * lines[i] + (at - chunk * lines[i])) * 128);
            }
        }
        asm volatile("" ::"v"(any));        // (loaded, though nobody wants to know)
    }
};

struct NormRows {                           // rows before their LayerNorm, and what it needs
    const float* x;
    const float2* stats;
    const void *gamma, *beta;
    float eps;
};

// y = LayerNorm(rows) w^T + bias; GELU: of that, and y in the order of row_at.  K: the rows' width; NB: blocks of 16 columns a workgroup.
template <int DT, int NB, bool GELU>
__global__ __launch_bounds__(512) void norm_gemm_kernel(NormRows in, const void* wv, const void* bias, void* y, int M, int N, int K, int mt, Ahead next) {
    if (int(blockIdx.y) >= mt) return next.fetch(mt);
    using E = Elem<DT>;
    using X8 = typename E::X8;
    using T = typename E::T;
    typedef __attribute__((ext_vector_type(4))) T T4;
    constexpr int WAVES = 8, U = 4;         // steps at a time
    __shared__ float4 s_moments[WAVES * 16];
    __shared__ f32x4 s_sum[WAVES * NB * 64];
    __shared__ X8 s_w[WAVES * NB * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int c = l & 15, g = l >> 4, n0 = blockIdx.x * 16 * NB, m = blockIdx.y, steps = K / 32;
    const int k0 = steps * wave / WAVES, k1 = steps * (wave + 1) / WAVES;
    const T* w[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) w[j] = static_cast<const T*>(wv) + int64_t(min(n0 + 16 * j, N - 16) + (l >> 2)) * K + 8 * row_chunk(l);
    const float* const x = in.x + (m * 2 * 64 + l) * 4;
    X8 a[U][NB], gamma[U], beta[U];
    f32x4 lo[U], hi[U];
    auto load = [&](int k, auto count) {
#pragma unroll
        for (int u = 0; u < decltype(count)::value; ++u) {
#pragma unroll
            for (int j = 0; j < NB; ++j) a[u][j] = *reinterpret_cast<const X8*>(w[j] + 32 * (k + u));
            lo[u] = *reinterpret_cast<const f32x4*>(x + int64_t(k + u) * mt * 512);
            hi[u] = *reinterpret_cast<const f32x4*>(x + int64_t(k + u) * mt * 512 + 256);
            gamma[u] = *reinterpret_cast<const X8*>(static_cast<const T*>(in.gamma) + 32 * (k + u) + 8 * g);
            beta[u] = *reinterpret_cast<const X8*>(static_cast<const T*>(in.beta) + 32 * (k + u) + 8 * g);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    float mean, rstd;
    f32x4 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto use = [&](auto count) {
#pragma unroll
        for (int u = 0; u < decltype(count)::value; ++u) {
            to_operands(s_w + wave * NB * 64, a[u]);
            X8 b;
#pragma unroll
            for (int i = 0; i < 8; ++i) b[i] = T(((i < 4 ? lo[u][i & 3] : hi[u][i & 3]) - mean) * rstd * float(gamma[u][i]) + float(beta[u][i]));
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[j] = E::mfma(a[u][j], b, acc[j]);
        }
    };
    MomentLoads<WAVES * 4> moments;
    moments.request(in.stats, K, mt, m);
    with_steps<U>(k1 - k0, [&](auto count) { load(k0, count); });
    const Moments part = moments.sums();
    put_moments(s_moments, part);
    __syncthreads();
    get_moments(s_moments, WAVES, part, K, in.eps, mean, rstd);
    with_steps<U>(k1 - k0, use);
    for (int k = k0 + U; k < k1; k += U)
        with_steps<U>(k1 - k, [&](auto count) {
            load(k, count);
            use(count);
#pragma unroll
            for (int j = 0; j < NB; ++j) acc[j] = tdb_settled(acc[j]);
        });
#pragma unroll
    for (int j = 0; j < NB; ++j) s_sum[(wave * NB + j) * 64 + l] = acc[j];
    __syncthreads();
    const int row = 16 * m + c, col = n0 + 16 * wave + 4 * g;          // (a wave for each block)
    if (wave >= NB || col >= N || row >= M) return;
    const T4 b4 = *reinterpret_cast<const T4*>(static_cast<const T*>(bias) + col);
    f32x4 sum = s_sum[wave * 64 + l];
#pragma unroll
    for (int v = 1; v < WAVES; ++v) sum += s_sum[(v * NB + wave) * 64 + l];
    T4 out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float v = sum[i] + float(b4[i]);
        if (GELU) v = tdb_gelu(v);
        out[i] = T(v);
    }
    *reinterpret_cast<T4*>(static_cast<T*>(y) + row_at(row, col >> 3, N, GELU ? mt : 0) + (col & 7)) = out;
}

// rows (x, stats) = in w^T + bias + LayerNorm(residual), the latter rounded to the type as a product reads it.  IN: in the order of row_at.
template <int DT, int WAVES, bool IN>
__global__ __launch_bounds__(WAVES * 64) void gemm_add_kernel(const void* inv, const void* wv, const void* bias, NormRows residual, float* x, float2* stats, int M,
                                                              int N, int K, int mt, Ahead next) {
    if (int(blockIdx.y) >= mt) return next.fetch(mt);
    using E = Elem<DT>;
    using X8 = typename E::X8;
    using T = typename E::T;
    typedef __attribute__((ext_vector_type(4))) T T4;
    __shared__ float4 s_moments[WAVES * 16];
    __shared__ f32x4 s_sum[WAVES * 64];
    __shared__ X8 s_w[WAVES * 8 * 64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
    const int c = l & 15, g = l >> 4, n0 = blockIdx.x * 16, m = blockIdx.y, steps = K / 32;
    const int k0 = steps * wave / WAVES, k1 = steps * (wave + 1) / WAVES;
    const T* const w = static_cast<const T*>(wv) + int64_t(n0 + (l >> 2)) * K + 8 * row_chunk(l);
    const T* const in = static_cast<const T*>(inv) + (IN ? (m * 64 + l) * 8 : int64_t(min(16 * m + (l >> 2), M - 1)) * K + 8 * row_chunk(l));
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto run = [&](int k, auto count) {     // `count` steps from k: all requested before the first is used
        constexpr int U = decltype(count)::value;
        X8 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a[u] = *reinterpret_cast<const X8*>(w + 32 * (k + u));
            b[u] = *reinterpret_cast<const X8*>(in + int64_t(k + u) * (IN ? mt * 512 : 32));
        }
        __builtin_amdgcn_sched_barrier(0);
        to_operands(s_w + wave * 512, a);
        if constexpr (!IN) to_operands(s_w + wave * 512, b);
#pragma unroll
        for (int u = 0; u < U; ++u) acc = E::mfma(a[u], b[u], acc);
    };
    const int row = 16 * m + c, col = n0 + 4 * g;
    MomentLoads<WAVES * 4> moments;
    moments.request(residual.stats, N, mt, m);
    f32x4 old;
    T4 b4, g4, s4;
    if (wave == 0) {                        // (what the epilogue needs: not another round trip behind the sums)
        old = *reinterpret_cast<const f32x4*>(residual.x + x_at(row, col >> 2, mt));
        b4 = *reinterpret_cast<const T4*>(static_cast<const T*>(bias) + col);
        g4 = *reinterpret_cast<const T4*>(static_cast<const T*>(residual.gamma) + col);
        s4 = *reinterpret_cast<const T4*>(static_cast<const T*>(residual.beta) + col);
    }
    for (int k = k0; k < k1; k += 8) with_steps<8>(k1 - k, [&](auto count) { run(k, count); });
    const Moments part = moments.sums();
    put_moments(s_moments, part);
    s_sum[wave * 64 + l] = acc;
    __syncthreads();
    if (wave > 0) return;
    float mean, rstd;
    get_moments(s_moments, WAVES, part, N, residual.eps, mean, rstd);
    f32x4 sum = acc;
#pragma unroll
    for (int v = 1; v < WAVES; ++v) sum += s_sum[v * 64 + l];
    float s1 = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sum[i] += float(b4[i]);
        sum[i] += float(T((old[i] - mean) * rstd * float(g4[i]) + float(s4[i])));
        s1 += sum[i];
    }
    s1 += __shfl_xor(s1, 16);
    s1 += __shfl_xor(s1, 32);
    const float mid = s1 * (1.f / 16.f);
    float dev = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) dev += (sum[i] - mid) * (sum[i] - mid);
    dev += __shfl_xor(dev, 16);
    dev += __shfl_xor(dev, 32);
    *reinterpret_cast<f32x4*>(x + x_at(row, col >> 2, mt)) = sum;       // (rows past M: there is room, and nothing looks at them)
    if (g == 0) stats[blockIdx.x * 16 * mt + row] = float2{mid, dev};
}

// out = LayerNorm(rows), row after row.
template <int DT, int CH>
__global__ __launch_bounds__(64) void norm_rows_kernel(NormRows in, int hidden, int mt, void* out) {
    const int t = blockIdx.x, l = threadIdx.x, chunks = hidden / 8;
    float v[CH][8], w[CH][8], b[CH][8];
    load_affine<DT, CH>(w, b, chunks, in.gamma, in.beta);
#pragma unroll
    for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if (l + 64 * c < chunks) x = *reinterpret_cast<const f32x4*>(in.x + x_at(t, 2 * (l + 64 * c) + h, mt));
#pragma unroll
            for (int i = 0; i < 4; ++i) v[c][4 * h + i] = x[i];
        }
    norm_row<DT, CH>(v, w, b, chunks, hidden, in.eps, out, t, 0);
}

struct ScanIds {
    const void* ids;                        // of the row, or nullptr
    int ids64;
    int64_t vocab;
    __device__ __forceinline__ bool in_table(int i) const {
        if (!ids) return true;
        const int64_t id = ids64 ? static_cast<const int64_t*>(ids)[i] : static_cast<const int32_t*>(ids)[i];
        return id >= 0 && id < vocab;
    }
};

template <typename T>
__device__ __forceinline__ void scan_row(const T* row, int64_t stride, int L, const ScanIds& ids, int& count, int& last, bool& ones, bool& known) {
    const int l = threadIdx.x & 63;
    for (int i = l; i < L; i += 64) {
        const T x = row[i * stride];
        const bool in = ids.in_table(i);
        if (x != T(0)) {
            ++count;
            last = i + 1;
            ones = ones && x == T(1);
            known = known && in;
        }
    }
}

__global__ __launch_bounds__(1024) void scan_mask_kernel(const void* mask, int type, int64_t sb, int64_t sl, int B, int L, ScanIds ids,
                                                         int32_t* lens, int32_t* cu, int32_t* flags, int ticket) {
    __shared__ int s_len[TDB_SCAN_MAX_BATCH], s_ok, s_ones, s_known;
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (threadIdx.x == 0) s_ok = s_ones = s_known = 1;
    __syncthreads();
    for (int b = wave; b < B; b += 16) {
        int count = 0, last = 0;
        bool ones = true, known = true;
        ScanIds row = ids;
        if (ids.ids) row.ids = static_cast<const char*>(ids.ids) + int64_t(b) * L * (ids.ids64 ? 8 : 4);
        switch (type) {
            case TDB_MASK_I64: scan_row(static_cast<const int64_t*>(mask) + b * sb, sl, L, row, count, last, ones, known); break;
            case TDB_MASK_I32: scan_row(static_cast<const int32_t*>(mask) + b * sb, sl, L, row, count, last, ones, known); break;
            case TDB_MASK_U8: scan_row(static_cast<const uint8_t*>(mask) + b * sb, sl, L, row, count, last, ones, known); break;
            case TDB_F32: scan_row(static_cast<const float*>(mask) + b * sb, sl, L, row, count, last, ones, known); break;
            case TDB_BF16: scan_row(static_cast<const __bf16*>(mask) + b * sb, sl, L, row, count, last, ones, known); break;
            default: scan_row(static_cast<const _Float16*>(mask) + b * sb, sl, L, row, count, last, ones, known); break;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            count += __shfl_xor(count, o);
            last = max(last, __shfl_xor(last, o));
        }
        const bool all_ones = __builtin_amdgcn_ballot_w64(!ones) == 0, all_known = __builtin_amdgcn_ballot_w64(!known) == 0;
        if (l == 0) {
            s_len[b] = count;
            if (last != count) s_ok = 0;    // (every writer writes the same)
            if (!all_ones) s_ones = 0;
            if (!all_known) s_known = 0;
        }
    }
    __syncthreads();
    if (wave == 0) {
        int before = 0;
        for (int b0 = 0; b0 < B; b0 += 64) {
            const int n = b0 + l < B ? s_len[b0 + l] : 0;
            int incl = n;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int up = __shfl_up(incl, d);
                if (l >= d) incl += up;
            }
            if (b0 + l < B) {
                lens[b0 + l] = n;
                cu[b0 + l + 1] = before + incl;
            }
            before += __shfl(incl, 63);
        }
        if (l == 0) {
            cu[0] = 0;
            flags[0] = s_ok;
            flags[1] = before;
            flags[2] = s_ones;
            flags[3] = s_known;
            __threadfence_system();
            __hip_atomic_store(flags + 4, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

__global__ __launch_bounds__(256) void unpack_kernel(const uint4* x, const int32_t* cu, int rows, int L, int T, int chunks, uint4* out) {
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (r >= rows) return;
    const int b = r / L, i = r - b * L, lo = cu[b];
    const bool in = i < cu[b + 1] - lo && lo >= 0 && lo < T - i;
    for (int c = l; c < chunks; c += 64) out[int64_t(r) * chunks + c] = in ? x[int64_t(lo + i) * chunks + c] : uint4{0, 0, 0, 0};
}

// hidden up to 4096 in chunks of eight, CH of them per lane
template <typename F>
void with_chunks(int hidden, F f) {
    if (hidden <= 512) f(std::integral_constant<int, 1>{});
    else if (hidden <= 1024) f(std::integral_constant<int, 2>{});
    else if (hidden <= 2048) f(std::integral_constant<int, 4>{});
    else f(std::integral_constant<int, 8>{});
}
template <typename F>
void with_type(int dtype, F f) {
    if (dtype == TDB_F32) f(std::integral_constant<int, TDB_F32>{});
    else if (dtype == TDB_BF16) f(std::integral_constant<int, TDB_BF16>{});
    else f(std::integral_constant<int, TDB_F16>{});
}

// Up to here a layer's four products take less here than in the tiles of gemm.hip (768 wide: 16.5 against 18.5 us at 64 rows,
// 20.2 against 19.1 at 80).
constexpr int SMALL_ROWS = 64;
// Each of the column blocks reads and normalises its rows anew, 64 bytes of float32 for each column of them: 24 layers of 1024 take 927 us that way and 848 with
// launches for residual + LayerNorm.  12 layers replayed as a graph, with such launches against without, 1, 16, 17..32, 33..48 and 49..64 rows: 128 wide
// 1.07, 1.12, 1.14, 1.15, 1.17x; 256 1.03, 1.06, 1.09; 384 0.98, 1.01, 1.04, 1.05, 1.06; 512 0.94, 0.97, 1.00, 1.00, 1.03; 640 0.99, 1.03, 1.03, 1.04, 1.00; 768 0.99,
// 1.02, 1.00, 1.02, 1.03; 832 0.98, 1.00, 0.97, 0.94, 0.98; 896 1.00, 1.02, 1.01, 0.98, 1.06; 960 0.99, 1.01, 0.97, 1.00, 0.95; 1024 0.98, 1.00, 1.01, 0.99, 0.94.
// At 448 and 512 wide with up to 16 rows the contraction shared out over 8 workgroups there is what is ahead.  That stays as it is: calls from a program are bound by
// the host's launches, 63 here and 86 there, where it is slow (512 wide, one row: 379 -> 271 us; on a faster host 258 -> 270).
constexpr int FUSED_WIDTH = 768;

// Blocks of 16 columns that a workgroup of norm_gemm_kernel takes: as few as give each compute unit one workgroup.
int norm_blocks(int N, int mt) {
    const int blocks = N / 16, units = tdb_compute_units(-1);
    int n = 1;
    while (n < 4 && (blocks + n - 1) / n * mt > units) ++n;
    return n;
}
Ahead ahead_of(const tdb_enc_next* next, int nexts, int mt) {
    Ahead a{};
    int n = 0;
    for (int i = 0; i < nexts; ++i) {
        const int rows = 16 * (next[i].norm ? norm_blocks(next[i].N, mt) : 1);
        const int64_t bytes = int64_t(rows) * next[i].K * 2;
        if (!next[i].w || bytes % 128 || next[i].N % rows) continue;
        a.w[n] = static_cast<const char*>(next[i].w), a.lines[n] = int(bytes / 128), a.chunks[n] = next[i].N / rows;
        ++n;
    }
    return a;
}

bool hidden_ok(int hidden) { return hidden > 0 && hidden % 8 == 0 && hidden <= 4096; }

}  // namespace

extern "C" {

int tdb_enc_scan_mask(const void* mask, int type, int64_t stride_b, int64_t stride_l, int B, int L, const void* ids, int ids64, int64_t vocab,
                      int32_t* lens, int32_t* cu, int32_t* flags, int ticket, void* stream) {
    if (B < 1 || B > TDB_SCAN_MAX_BATCH || L < 1) return int(hipErrorInvalidValue);
    hipLaunchKernelGGL(scan_mask_kernel, dim3(1), dim3(1024), 0, static_cast<hipStream_t>(stream), mask, type, stride_b, stride_l, B, L,
                       ScanIds{ids, ids64, vocab}, lens, cu, flags, ticket);
    return int(hipGetLastError());
}

int tdb_enc_embed(const void* ids, int ids64, const void* table, int64_t vocab, const void* gamma, const void* beta, float eps, const int32_t* cu,
                  int B, int L, int T, int hidden, int dtype, int mt, void* out, void* stream) {
    if (!hidden_ok(hidden) || T < 1) return int(hipErrorInvalidValue);
    with_type(dtype, [&](auto dt) {
        with_chunks(hidden, [&](auto ch) {
            hipLaunchKernelGGL((embed_kernel<decltype(dt)::value, decltype(ch)::value, false>), dim3((T + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream),
                               ids, ids64, table, vocab, gamma, beta, eps, cu, B, L, T, hidden, mt, out, nullptr);
        });
    });
    return int(hipGetLastError());
}

int tdb_enc_add_norm(const void* x, int splits, const void* bias, const void* residual, const void* gamma, const void* beta, float eps, int T,
                     int hidden, int dtype, int mt_in, int mt_out, void* out, void* stream) {
    if (!hidden_ok(hidden) || T < 1 || splits < 0 || splits > MAX_SPLITS) return int(hipErrorInvalidValue);
    with_type(dtype, [&](auto dt) {
        with_chunks(hidden, [&](auto ch) {
            constexpr int DT = decltype(dt)::value, CH = decltype(ch)::value;
            // (few rows: one to a CU -- 48 rows of 768 with five parts 4.0 -> 3.2 us, 512 5.2 -> 4.5, 1024 the same)
            const int waves = T <= 512 ? 1 : 4;
            const dim3 grid((T + waves - 1) / waves), block(64 * waves);
            hipStream_t s = static_cast<hipStream_t>(stream);
            auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, x, splits, bias, residual, gamma, beta, eps, T, hidden, mt_in, mt_out, out); };
            if (splits == 0) go(add_norm_kernel<DT, CH, 0>);
            else if (splits <= 2) go(add_norm_kernel<DT, CH, 2>);
            else if (splits <= 4) go(add_norm_kernel<DT, CH, 4>);
            else if (splits <= 6) go(add_norm_kernel<DT, CH, 6>);
            else go(add_norm_kernel<DT, CH, MAX_SPLITS>);
        });
    });
    return int(hipGetLastError());
}

int tdb_enc_small_tiles(int M, int N, int K, int dtype) {
    if ((dtype != TDB_BF16 && dtype != TDB_F16) || M < 1 || M > SMALL_ROWS || N < 1 || N % 32 || K < 1 || K % 32) return 0;
    return (M + 15) / 16;
}

// About one workgroup (of 16 columns) per CU.
int tdb_enc_small_splits(int N) { return std::max(1, std::min(MAX_SPLITS, tdb_compute_units(-1) * 16 / std::max(N, 1))); }

int tdb_enc_small_gemm(const void* x, const void* w, const void* bias, int flags, int splits, int M, int N, int K, int dtype, void* y, void* stream) {
    const int tiles = tdb_enc_small_tiles(M, N, K, dtype);
    if (tiles == 0 || splits < 0 || splits > MAX_SPLITS) return int(hipErrorInvalidValue);
    hipStream_t s = static_cast<hipStream_t>(stream);
    bool known = true;
    auto launch = [&](auto dt, auto mt) {
        constexpr int DT = decltype(dt)::value, MT = decltype(mt)::value;
        constexpr int waves = 8;
        const dim3 grid(N / 16, splits > 0 ? splits : 1), block(waves * 64);
        const size_t smem = size_t(waves) * MT * 1024;
        const int shape = splits > 0 ? 8 : 0;
        switch (shape | flags) {            // the four products of a layer
            case TDB_ENC_IN: hipLaunchKernelGGL((small_gemm_kernel<DT, MT, true, false, false, false>), grid, block, smem, s, x, w, bias, y, M, N, K, 1); break;
            case 8: hipLaunchKernelGGL((small_gemm_kernel<DT, MT, false, false, false, true>), grid, block, smem, s, x, w, bias, y, M, N, K, splits); break;
            case TDB_ENC_IN | TDB_ENC_OUT | TDB_ENC_GELU:
                hipLaunchKernelGGL((small_gemm_kernel<DT, MT, true, true, true, false>), grid, block, smem, s, x, w, bias, y, M, N, K, 1);
                break;
            case 8 | TDB_ENC_IN: hipLaunchKernelGGL((small_gemm_kernel<DT, MT, true, false, false, true>), grid, block, smem, s, x, w, bias, y, M, N, K, splits); break;
            default: known = false;
        }
    };
    auto rows = [&](auto dt) {
        switch (tiles) {
            case 1: launch(dt, std::integral_constant<int, 1>{}); break;
            case 2: launch(dt, std::integral_constant<int, 2>{}); break;
            case 3: launch(dt, std::integral_constant<int, 3>{}); break;
            default: launch(dt, std::integral_constant<int, 4>{});
        }
    };
    if (dtype == TDB_BF16) rows(std::integral_constant<int, TDB_BF16>{});
    else rows(std::integral_constant<int, TDB_F16>{});
    return known ? int(hipGetLastError()) : int(hipErrorInvalidValue);
}

int tdb_enc_rows_fused(int M, int hidden, int inner, int dtype) {
    return hidden % 32 == 0 && hidden <= FUSED_WIDTH && tdb_enc_small_tiles(M, 3 * hidden, hidden, dtype) && tdb_enc_small_tiles(M, inner, hidden, dtype)
               ? tdb_enc_small_tiles(M, hidden, inner, dtype)
               : 0;
}

int tdb_enc_embed_rows(const void* ids, int ids64, const void* table, int64_t vocab, const int32_t* cu, int B, int L, int T, int hidden, int dtype, int mt,
                       float* x, float* stats, void* stream) {
    if (!hidden_ok(hidden) || hidden % 32 || T < 1 || T > 16 * mt || dtype == TDB_F32) return int(hipErrorInvalidValue);
    auto go = [&](auto dt) {
        with_chunks(hidden, [&](auto ch) {
            hipLaunchKernelGGL((embed_kernel<decltype(dt)::value, decltype(ch)::value, true>), dim3((T + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream),
                               ids, ids64, table, vocab, nullptr, nullptr, 0.f, cu, B, L, T, hidden, mt, x, reinterpret_cast<float2*>(stats));
        });
    };
    if (dtype == TDB_BF16) go(std::integral_constant<int, TDB_BF16>{});
    else go(std::integral_constant<int, TDB_F16>{});
    return int(hipGetLastError());
}

int tdb_enc_norm_gemm(const tdb_enc_rows* in, const void* w, const void* bias, int gelu, int M, int N, int K, int dtype, const tdb_enc_next* next,
                      int nexts, void* y, void* stream) {
    const int mt = tdb_enc_small_tiles(M, N, K, dtype);
    if (!mt || K % 32 || nexts < 0 || nexts > Ahead::MOST) return int(hipErrorInvalidValue);
    const Ahead ahead = ahead_of(next, nexts, mt);
    const int extra = ahead.chunks[0] > 0;
    const NormRows r{in->x, reinterpret_cast<const float2*>(in->stats), in->gamma, in->beta, in->eps};
    const int blocks = N / 16;
    auto wide = [&](auto nb) {
        constexpr int NB = decltype(nb)::value;
        auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((blocks + NB - 1) / NB, mt + extra), dim3(512), 0, static_cast<hipStream_t>(stream), r, w, bias, y, M, N, K, mt, ahead); };
        if (dtype == TDB_BF16) gelu ? go(norm_gemm_kernel<TDB_BF16, NB, true>) : go(norm_gemm_kernel<TDB_BF16, NB, false>);
        else gelu ? go(norm_gemm_kernel<TDB_F16, NB, true>) : go(norm_gemm_kernel<TDB_F16, NB, false>);
    };
    const int nb = norm_blocks(N, mt);
    if (nb == 1) wide(std::integral_constant<int, 1>{});
    else if (nb == 2) wide(std::integral_constant<int, 2>{});
    else if (nb == 3) wide(std::integral_constant<int, 3>{});
    else wide(std::integral_constant<int, 4>{});
    return int(hipGetLastError());
}

int tdb_enc_gemm_add(const void* in, int ordered, const void* w, const void* bias, const tdb_enc_rows* residual, int M, int N, int K, int dtype, const tdb_enc_next* next,
                     int nexts, float* x, float* stats, void* stream) {
    const int mt = tdb_enc_small_tiles(M, N, K, dtype);
    if (!mt || N % 32 || nexts < 0 || nexts > Ahead::MOST) return int(hipErrorInvalidValue);
    const Ahead ahead = ahead_of(next, nexts, mt);
    // Two rows of workgroups to fetch ahead.  (12 layers of 768 as a graph, none, one and two: 16 rows 311, 310, 304 us, 32 325, 326, 319, 48 350, 352, 345; also where
    // they are more than one to a compute unit, 49 rows 358, 360, 356.  640 wide 300, 302, 294 to 358, 354, 355; 384 wide equal.)
    const int extra = ahead.chunks[0] > 0 ? 2 : 0;
    const NormRows r{residual->x, reinterpret_cast<const float2*>(residual->stats), residual->gamma, residual->beta, residual->eps};
    auto go = [&](auto kernel, int waves) {
        hipLaunchKernelGGL(kernel, dim3(N / 16, mt + extra), dim3(waves * 64), 0, static_cast<hipStream_t>(stream), in, w, bias, r, x,
                           reinterpret_cast<float2*>(stats), M, N, K, mt, ahead);
    };
    auto typed = [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if (K > 1536) ordered ? go(gemm_add_kernel<DT, 16, true>, 16) : go(gemm_add_kernel<DT, 16, false>, 16);
        else ordered ? go(gemm_add_kernel<DT, 8, true>, 8) : go(gemm_add_kernel<DT, 8, false>, 8);
    };
    if (dtype == TDB_BF16) typed(std::integral_constant<int, TDB_BF16>{});
    else typed(std::integral_constant<int, TDB_F16>{});
    return int(hipGetLastError());
}

int tdb_enc_norm_rows(const tdb_enc_rows* in, int T, int hidden, int dtype, void* out, void* stream) {
    const int mt = (T + 15) / 16;
    if (!hidden_ok(hidden) || hidden % 32 || T < 1 || dtype == TDB_F32) return int(hipErrorInvalidValue);
    const NormRows r{in->x, reinterpret_cast<const float2*>(in->stats), in->gamma, in->beta, in->eps};
    auto go = [&](auto dt) {
        with_chunks(hidden, [&](auto ch) {
            hipLaunchKernelGGL((norm_rows_kernel<decltype(dt)::value, decltype(ch)::value>), dim3(T), dim3(64), 0, static_cast<hipStream_t>(stream), r, hidden, mt, out);
        });
    };
    if (dtype == TDB_BF16) go(std::integral_constant<int, TDB_BF16>{});
    else go(std::integral_constant<int, TDB_F16>{});
    return int(hipGetLastError());
}

int tdb_enc_unpack(const void* x, const int32_t* cu, int B, int L, int T, int hidden, int dtype, void* out, void* stream) {
    const int bytes = hidden * (dtype == TDB_F32 ? 4 : 2);
    if (bytes % 16 || B < 1 || L < 1) return int(hipErrorInvalidValue);
    hipLaunchKernelGGL(unpack_kernel, dim3((B * L + 3) / 4), dim3(256), 0, static_cast<hipStream_t>(stream), static_cast<const uint4*>(x), cu, B * L, L, T,
                       bytes / 16, static_cast<uint4*>(out));
    return int(hipGetLastError());
}

}  // extern "C"
