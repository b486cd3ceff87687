// Launchers of the kernels around attention in an encoder layer (encoder.hip), called by the native encoder loop (host.cpp).
// All return a hipError_t as int and take a hipStream_t; nothing here allocates or synchronises.
#pragma once
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

// Element types as in tdb_attn.h; masks additionally: 3 = int64, 4 = int32, 5 = one byte.
enum { TDB_MASK_I64 = 3, TDB_MASK_I32 = 4, TDB_MASK_U8 = 5 };
enum { TDB_SCAN_MAX_BATCH = 1024 };

// lens[b] = number of nonzero entries of row b, cu = their running sum from 0; flags[0] = 1 if every row has its nonzero
// entries first, flags[1] = sum of lens, flags[2] = 1 if every nonzero entry is 1, flags[3] = 1 if the ids at nonzero entries
// (ids: [B, L] row after row, or NULL: not looked at) lie in [0, vocab); then flags[4] = ticket.  `flags` may be pinned host
// memory.
int tdb_enc_scan_mask(const void* mask, int type, int64_t stride_b, int64_t stride_l, int B, int L, const void* ids, int ids64, int64_t vocab,
                      int32_t* lens, int32_t* cu, int32_t* flags, int ticket, void* stream);

// Order of activation rows: mt = 0 row after row; mt > 0 (tdb_enc_small_tiles) the order in which the small products load
// them, 16 mt rows of room.

// out[t] = LayerNorm(table[ids of token t]), NaN for an id outside the table; cu != NULL: token t of the packed batch, cu == NULL: ids in order.
int tdb_enc_embed(const void* ids, int ids64, const void* table, int64_t vocab, const void* gamma, const void* beta, float eps,
                  const int32_t* cu, int B, int L, int T, int hidden, int dtype, int mt, void* out, void* stream);

// out = LayerNorm(x + residual); x: [T, hidden] of `dtype`, or (splits > 0, at most 8) [splits, T, hidden] float32 partial sums
// to which `bias` is added.  mt_in: order of the residual, mt_out: of the output.
int tdb_enc_add_norm(const void* x, int splits, const void* bias, const void* residual, const void* gamma, const void* beta, float eps,
                     int T, int hidden, int dtype, int mt_in, int mt_out, void* out, void* stream);

// Products with few rows, 16-bit: y[M, N] = x[M, K] w[N, K]^T + bias, or (splits > 0, at most 8) float32 partial sums
// [splits, M, N] without bias.  flags: x in the small products' order, y too, GELU (the erf form) applied.  Four combinations
// exist: IN; splits; IN | OUT | GELU; IN with splits.
enum { TDB_ENC_IN = 1, TDB_ENC_OUT = 2, TDB_ENC_GELU = 4 };
int tdb_enc_small_gemm(const void* x, const void* w, const void* bias, int flags, int splits, int M, int N, int K, int dtype, void* y,
                       void* stream);
// 16-row tiles (mt) of a product that the above takes, else 0
int tdb_enc_small_tiles(int M, int N, int K, int dtype);
// the number of partial sums of a product with N columns whose reader adds them up
int tdb_enc_small_splits(int N);

// The same products with the residual + LayerNorm between them in their own launches, 16-bit, up to 64 rows.  Rows before their LayerNorm are float32 in
// an order of their own ([16 mt, hidden] floats, mt = tdb_enc_rows_fused) with the mean and sum of squared deviations of each 16
// columns ([hidden / 16, 16 mt, 2] floats).
typedef struct tdb_enc_rows {
    const float *x, *stats;
    const void *gamma, *beta;               // of the LayerNorm
    float eps;
} tdb_enc_rows;
// A weight [N, K] that a product to come will read, a tdb_enc_norm_gemm (norm) or a tdb_enc_gemm_add: brought nearer meanwhile (w may be NULL).
typedef struct tdb_enc_next {
    const void* w;
    int N, K, norm;
} tdb_enc_next;
// mt where the four products of a layer are taken this way, else 0
int tdb_enc_rows_fused(int M, int hidden, int inner, int dtype);
// rows = table[ids of token t], NaN for an id outside the table; cu as above
int tdb_enc_embed_rows(const void* ids, int ids64, const void* table, int64_t vocab, const int32_t* cu, int B, int L, int T, int hidden, int dtype,
                       int mt, float* x, float* stats, void* stream);
// y[M, N] = LayerNorm(in)[M, K] w[N, K]^T + bias, row after row; gelu: GELU of that, in the small products' order.  next: up to 2.
int tdb_enc_norm_gemm(const tdb_enc_rows* in, const void* w, const void* bias, int gelu, int M, int N, int K, int dtype, const tdb_enc_next* next,
                      int nexts, void* y, void* stream);
// rows (x, stats) = in[M, K] w[N, K]^T + bias + LayerNorm(residual); ordered: `in` is in the small products' order.  Not in place.
int tdb_enc_gemm_add(const void* in, int ordered, const void* w, const void* bias, const tdb_enc_rows* residual, int M, int N, int K, int dtype,
                     const tdb_enc_next* next, int nexts, float* x, float* stats, void* stream);
// out[T, hidden] = LayerNorm(in), row after row
int tdb_enc_norm_rows(const tdb_enc_rows* in, int T, int hidden, int dtype, void* out, void* stream);

// Products of any size, 16-bit, rows in order: y[M, N] = x[M, K] w[N, K]^T + bias (flags: 0 or TDB_ENC_GELU), or (splits > 1)
// float32 partial sums [splits, M, N] without bias.  K a multiple of 64, N of 8; pointers 16-byte aligned.
// flags >> TDB_ENC_TILE_SHIFT: 1 + the number of a tile, for tests; 0: the kernel's choice.
enum { TDB_ENC_TILE_SHIFT = 8 };
int tdb_enc_gemm(const void* x, const void* w, const void* bias, int flags, int splits, int M, int N, int K, int dtype, void* y,
                 void* stream);
// the number of partial sums that is best for a product whose reader adds them up; 0: a product that the above does not take
int tdb_enc_gemm_splits(int M, int N, int K, int dtype);

// out[b, l] = x[cu[b] + l] for l < cu[b+1] - cu[b], zeros elsewhere (and for what does not lie in the T rows of x)
int tdb_enc_unpack(const void* x, const int32_t* cu, int B, int L, int T, int hidden, int dtype, void* out, void* stream);

#ifdef __cplusplus
}
#endif
