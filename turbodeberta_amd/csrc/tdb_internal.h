// Internal declarations shared by the C-ABI front end and the HIP kernels of libtdb_attn.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tdb_attn.h"

// One flattened description of a launch; fixed-length and packed calls both reduce to it.
// A sequence b starts at element offset  b*stride_b  (fixed)  or  cu_seqlens[b]*stride_l  (packed)
// and its row l, head h lives at  + l*stride_l + h*stride_h.
struct TdbKernelParams {
    const void *q, *k, *v;
    void* o;
    int64_t qs_b, qs_h, qs_l;
    int64_t ks_b, ks_h, ks_l;
    int64_t vs_b, vs_h, vs_l;
    int64_t os_b, os_h, os_l;
    const int32_t* seqlens;     // fixed: [B] valid lengths or nullptr
    const int32_t* cu_seqlens;  // packed: [B+1] or nullptr
    const int32_t* gap_cu;      // packed: the call's whole cu_seqlens if rows outside every sequence are to be zeroed, or nullptr
    int32_t gap_B;              // and its batch
    int32_t B, H, D, L;         // L: padded length (fixed) / max_seqlen (packed)
    int32_t total;              // packed: token count
    int32_t varlen;
    float scale;
    // position terms
    int32_t span, lut_half;
    const int32_t* lut;
    const void *pk, *pq;        // fused tables [H, 2*span, D]
    int64_t pks_h, pks_r, pqs_h, pqs_r;
    const void *c2p, *p2c;      // strips
    int64_t c2s_b, c2s_h, c2s_l;
    int64_t p2s_b, p2s_h, p2s_l;
};

// Compute units of a device (negative: the current one); 256, an MI355X, where there is none to ask.
extern "C" int tdb_compute_units(int device);

// tile heights (query rows per workgroup)
constexpr int TDB_GENERIC_TILE = 16;
constexpr int TDB_MFMA_TILE = 128;
constexpr int TDB_SHORT_TILE = 32;     // per wave

// true when the float32 matrix-core kernel can take this launch
bool tdb_f32_supported(const TdbKernelParams& p, int dtype);
// true when the float32 kernel that takes its operands apart once per workgroup can, and with how many sets of waves it is the
// faster one on the current device (0: it is not)
bool tdb_f32_split_supported(const TdbKernelParams& p, int dtype);
int tdb_f32_split_sets(const TdbKernelParams& p);
// true when the 16-bit matrix-core kernel can take this launch
bool tdb_mfma_supported(const TdbKernelParams& p, int dtype);

// true when the 16-bit kernel for short sequences can take this launch
bool tdb_short_supported(const TdbKernelParams& p, int dtype);

// true when the 16-bit kernel with position tables resident in LDS can take this launch
bool tdb_resident_supported(const TdbKernelParams& p, int dtype);

// launchers; return hipError_t of the launch
hipError_t tdb_launch_generic(const TdbKernelParams& p, int dtype, hipStream_t stream);
hipError_t tdb_zero_gaps(const TdbKernelParams& p, int dtype, hipStream_t stream);     // a launch of its own
hipError_t tdb_launch_short(const TdbKernelParams& p, int dtype, hipStream_t stream);
hipError_t tdb_launch_f32(const TdbKernelParams& p, hipStream_t stream);
hipError_t tdb_launch_f32_split(const TdbKernelParams& p, int sets, hipStream_t stream);
hipError_t tdb_launch_mfma(const TdbKernelParams& p, int dtype, hipStream_t stream);
// what the rules say of a launch on the current device: whether that kernel is the faster one, and whether its units have 32 query rows
bool tdb_resident_pays(const TdbKernelParams& p);
bool tdb_resident_wide(const TdbKernelParams& p);
hipError_t tdb_launch_resident(const TdbKernelParams& p, int dtype, hipStream_t stream);
// Cap on the persistent workgroups of a launch (multiple of 8, 0 = none); returns the cap in force.
int tdb_mfma_set_workgroup_limit(int workgroups);
int tdb_mfma_workgroup_limit();
constexpr int TDB_FAR_MIN_LEN = 1536;   // 16-bit launches of longer maxima keep the position terms of far steps in 32 bits

// Maps blockIdx.x to (sequence, first row of the tile, valid length).  Returns false when the
// block has no tile (packed launches are sized by an upper bound on the tile count).  Must be
// called by whole waves with identical arguments.  For packed input the wave scans cu_seqlens 64
// sequences at a time: one load per lane, a prefix sum of the per-sequence tile counts across the
// wave, and a ballot to pick the sequence that owns tile `block` -- no serial chain of dependent
// loads, and no work list built on the host.
__device__ __forceinline__ bool tdb_locate_tile(const TdbKernelParams& p, int tile_rows, int block,
                                                int& b, int& row0, int& len, int64_t& tok0) {
    if (!p.varlen) {
        const int tiles = (p.L + tile_rows - 1) / tile_rows;
        b = block / tiles;
        row0 = (block - b * tiles) * tile_rows;
        len = p.seqlens ? min(max(p.seqlens[b], 0), p.L) : p.L;
        tok0 = 0;
        return true;
    }
    const int lane = threadIdx.x & 63;
    int t = block;
    for (int b0 = 0; b0 < p.B; b0 += 64) {
        const int bb = b0 + lane;
        int s = 0, n = 0;
        if (bb < p.B) {
            s = p.cu_seqlens[bb];
            const int e = p.cu_seqlens[bb + 1];
            n = e - s;
            if (s < 0 || n < 0 || e > p.total) n = 0;   // malformed entry: no tiles
            n = min(n, p.L);
        }
        const int nt = (n + tile_rows - 1) / tile_rows;
        int incl = nt;                                   // inclusive prefix sum over the wave
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(incl, d);
            if (lane >= d) incl += up;
        }
        const int chunk_tiles = __builtin_amdgcn_readlane(incl, 63);
        if (t < chunk_tiles) {
            const unsigned long long owners = __builtin_amdgcn_ballot_w64(incl > t);
            const int ln = __builtin_amdgcn_readfirstlane(__builtin_ctzll(owners));
            const int before = __builtin_amdgcn_readlane(incl, ln) - __builtin_amdgcn_readlane(nt, ln);
            b = b0 + ln;
            row0 = (t - before) * tile_rows;
            len = __builtin_amdgcn_readlane(n, ln);
            tok0 = __builtin_amdgcn_readlane(s, ln);
            return true;
        }
        t -= chunk_tiles;
    }
    return false;
}

// The same map with the sequences taken in order of decreasing length, for up to 64 sequences of different lengths
// (packed, or a fixed layout with lengths; whole tiles of padding come last): workgroups start in block order, so the
// long ones start first and the short ones fill the gaps at the end.  A rank per lane (its sequence against every
// other), one push of the tile counts to their rank, a prefix sum and a ballot; all inside the wave.
__device__ __forceinline__ bool tdb_locate_tile_sorted(const TdbKernelParams& p, int tile_rows, int block,
                                                       int& b, int& row0, int& len, int64_t& tok0) {
    if (p.B > 64 || (!p.varlen && !p.seqlens)) return tdb_locate_tile(p, tile_rows, block, b, row0, len, tok0);
    const int lane = threadIdx.x & 63;
    int s = 0, n = 0;
    if (lane < p.B) {
        if (p.varlen) {
            s = p.cu_seqlens[lane];
            const int e = p.cu_seqlens[lane + 1];
            n = e - s;
            if (s < 0 || n < 0 || e > p.total) n = 0;   // malformed entry: no tiles
            n = min(n, p.L);
        } else {
            n = min(max(p.seqlens[lane], 0), p.L);
        }
    }
    int rank = lane >= p.B ? lane : 0;
    for (int o = 0; o < p.B; ++o) {
        const int other = __builtin_amdgcn_readlane(n, o);
        if (lane < p.B) rank += (other > n || (other == n && o < lane)) ? 1 : 0;
    }
    const int nt = (n + tile_rows - 1) / tile_rows;
    auto pick = [&](int count, int t, int& ln, int& within) {   // lane that owns element t of the lanes' counts
        int incl = count;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(incl, d);
            if (lane >= d) incl += up;
        }
        const unsigned long long owners = __builtin_amdgcn_ballot_w64(incl > t);
        if (owners == 0) {
            within = t - __builtin_amdgcn_readlane(incl, 63);   // (what is left of t beyond all counts)
            return false;
        }
        ln = __builtin_amdgcn_readfirstlane(__builtin_ctzll(owners));
        within = t - (__builtin_amdgcn_readlane(incl, ln) - __builtin_amdgcn_readlane(count, ln));
        return true;
    };
    int ln = 0, within = 0, first = 0;
    if (pick(__builtin_amdgcn_ds_permute(rank * 4, nt), block, ln, within)) {
        ln = __builtin_amdgcn_readlane(__builtin_amdgcn_ds_permute(rank * 4, lane), ln);
    } else {
        if (p.varlen) return false;
        const int all = (p.L + tile_rows - 1) / tile_rows;
        if (!pick(lane < p.B ? all - nt : 0, within, ln, within)) return false;
        first = __builtin_amdgcn_readlane(nt, ln);
    }
    b = ln;
    row0 = (first + within) * tile_rows;
    len = __builtin_amdgcn_readlane(n, ln);
    tok0 = p.varlen ? __builtin_amdgcn_readlane(s, ln) : 0;
    return true;
}

// A product's result as it is behind all wait states that a matrix instruction may need (12; 16 of them).  The compiler counts them, but where
// paths join behind a condition it follows one of them back to the product: on another, which jumps over what lies between, the result
// may be read, or its registers reused, too early (seen: 1 state of 8, and the score of the step before).  Not needed where a vector
// instruction reads the result ahead of the condition.  tests/test_wait_states_cpu.py follows every path of the built kernels.
template <typename T>
__device__ __forceinline__ T tdb_settled(T x) {
    asm volatile("s_nop 7\n\ts_nop 7" : "+v"(x));
    return x;
}

// v Phi(v) as v / (1 + 2^-(v r(v^2))), r a polynomial fitted here to the logarithm of Phi(v) / Phi(-v).  Error against 64 bits,
// evaluated in 32 (in brackets that of v (1 + erf) / 2 in 32 bits, which cancels below): relative 2.4e-6 on [-1, 0] and 3.1e-6
// (2.6e-6) on [-2.5, 0], 3.6e-6 (4.6e-4) to -4, 4.4e-6 (4.3e-3) to -4.5, 6e-6 (4.7e-2) to -5; below, where the result is under
// 1.5e-6 in size, 1e-10 absolute to -5.5 and 3e-10 beyond.  v r grows with v throughout, so the result goes to 0 and to v.
// 13 plain instructions and two quarter-rate ones per element; erff takes about 40.
__device__ __forceinline__ float tdb_gelu(float v) {
    const float u = v * v;
    float r = 1.8808817e-12f;
    r = fmaf(r, u, -2.7793998e-10f);
    r = fmaf(r, u, 1.7831045e-8f);
    r = fmaf(r, u, -6.4697991e-7f);
    r = fmaf(r, u, 1.4255226e-5f);
    r = fmaf(r, u, -1.751849e-4f);
    r = fmaf(r, u, -5.1022547e-5f);
    r = fmaf(r, u, 0.10478447f);
    r = fmaf(r, u, 2.3022261f);
    return v * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-(v * r)));
}

// Zeros for the rows of a packed output that belong to no sequence: in front of, between and behind them, and what
// max_seqlen cuts off.  One wave of each of `workers` workgroups runs this beside the attention itself (a fill of the whole
// output by a launch of its own took 12 us in front of a 91 us call).  Packings without gaps, all but a few, end after one
// look at the boundaries, 64 at a time.
__device__ __forceinline__ void tdb_fill_gaps(const int32_t* cu, int B, int L, int total, char* o, int64_t row_bytes,
                                              int64_t head_bytes, int heads, int head_dim_bytes, int worker, int workers) {
    const int lane = threadIdx.x & 63;
    bool exact = true;
    for (int b0 = 0; b0 < B; b0 += 64) {
        const int b = min(b0 + lane, B - 1);
        const int lo = cu[b], hi = cu[b + 1];
        exact = exact && lo >= 0 && hi >= lo && hi <= total && hi - lo <= L && (b > 0 || lo == 0) && (b < B - 1 || hi == total);
    }
    if (__builtin_amdgcn_ballot_w64(!exact) == 0) return;
    for (int row = worker; row < total; row += workers) {
        bool mine = false;
        for (int b0 = 0; b0 < B; b0 += 64) {
            const int b = min(b0 + lane, B - 1);
            const int lo = cu[b], hi = cu[b + 1];
            mine = mine || (lo >= 0 && hi >= lo && hi <= total && row >= lo && row < lo + min(hi - lo, L));
        }
        if (__builtin_amdgcn_ballot_w64(mine) != 0) continue;
        const int per_head = head_dim_bytes / 16;
        for (int idx = lane; idx < heads * per_head; idx += 64)
            *reinterpret_cast<uint4*>(o + row * row_bytes + (idx / per_head) * head_bytes + (idx % per_head) * 16) = uint4{0, 0, 0, 0};
    }
}
