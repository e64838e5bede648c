// xq_fa_common.h — definitions shared by the two flash-attention pass-1
// engines (VALU in xq_fa.hip, matrix cores in xq_fa_mma.hip) and the split
// reduce: launch arguments, the sinks/normalisation tail, helpers.
#pragma once

#include <math.h>

#include "xq_kernels.h"

namespace xq {

constexpr int kTile = 64;
constexpr int kThreads = 256;
constexpr int kMaxSplits = 256;

// LDS record stride: a multiple of 16 bytes with an odd number of 16-byte
// units, so 16 lanes reading 16 bytes from consecutive records hit distinct
// bank groups.
constexpr int pad_rec(int rec) {
    int u = (rec + 15) / 16;
    if ((u & 1) == 0) ++u;
    return u * 16;
}
constexpr int chunk_bytes(int rec) { return rec % 16 == 0 ? 16 : rec % 8 == 0 ? 8 : 4; }

template <int CH> struct ChunkT;
template <> struct ChunkT<16> { using T = uint4; };
template <> struct ChunkT<8> { using T = uint2; };
template <> struct ChunkT<4> { using T = uint32_t; };

// Division of numbers up to max_x by one the host knows: x / d = mulhi(x,
// floor(2^32 / d) + 1) for x below 2^32 / d (one multiply, against about 20
// instructions of the general division). m 0: d is 1; m 1: max_x lies beyond that,
// the general division.
struct UDiv {
    uint32_t d, m;
    UDiv() = default;
    UDiv(uint32_t n, uint64_t max_x)
        : d(n), m(n <= 1 ? 0u : max_x * n < ((uint64_t)1 << 32) ? (uint32_t)(((uint64_t)1 << 32) / n) + 1u : 1u) {}
    __host__ __device__ __forceinline__ uint32_t quot(uint32_t x) const {
        if (m == 0u) return x;
        if (m == 1u) return x / d;
        return (uint32_t)(((uint64_t)x * m) >> 32);
    }
};

// The same without branches, for numbers below 2^31: with l = ceil(log2 d) and
// m = ceil(2^(31 + l) / d), below 2^32, x / d = x m >> (31 + l), as mulhi(2x, m) >> l.
// (m d - 2^(31 + l) < d <= 2^l, so x m / 2^(31 + l) exceeds x / d by less than
// x / (2^31 d) < 1 / d.)
struct UDivFlat {
    uint32_t d, m;
    UDivFlat() = default;
    explicit UDivFlat(uint32_t n) : d(n), m((uint32_t)((((uint64_t)1 << (31 + log2_up(n))) + n - 1) / n)) {}
    static __host__ __device__ __forceinline__ int log2_up(uint32_t n) { return 31 - __builtin_clz(2u * n - 1u); }
    __host__ __device__ __forceinline__ uint32_t quot(uint32_t x) const {
        return (uint32_t)(((uint64_t)(2u * x) * m) >> 32) >> log2_up(d);
    }
};

struct FaArgs {
    const uint8_t* k;
    const uint8_t* v;
    int64_t k_nb1, k_nb2, k_nb3;
    int64_t v_nb1, v_nb2, v_nb3;
    const uint8_t* mask;
    int64_t m_nb1, m_nb2, m_nb3;
    int32_t m_ne2, m_ne3;
    const int32_t* positions;
    int32_t origin;
    const float* sinks;
    uint8_t* dst;
    int64_t d_nb1, d_nb2, d_nb3;
    float* lse;
    float* part_o;
    float2* part_ml;
    int64_t L;
    int64_t split_rows;
    int32_t interleave;  // fa_dec: split s takes the slice groups s, s + n_splits, ...
    int32_t H, Hkv, G, NQ, B, QT, n_qtiles, n_splits, rk3, rv3;
    float scale, softcap, max_bias, m0, m1;
    int32_t n_head_log2;
    // fa_dec
    uint32_t n_wg;
    int32_t tile_pairs;  // (query, head) pairs per tile
    UDiv d_tiles, d_hkv, d_splits, d_rk3, d_rv3, d_g;
    int32_t poison;
    // matrix-core engine: f32 Q rows (quantised inside the kernel), hi-only
    // f16 Q for the NATIVE policy
    const uint8_t* q;
    int64_t q_nb1, q_nb2, q_nb3;
    int32_t hi_only;
    // d_g's divisor (here, after the rest: between the arguments that the prologue loads at
    // once it cost a 377-row decode 0.1 us)
    UDivFlat d_gf;
};

XQ_DEV float alibi_slope(const FaArgs& a, int h) {
    if (!(a.max_bias > 0.0f)) return 1.0f;
    return h < a.n_head_log2 ? powf(a.m0, (float)(h + 1))
                             : powf(a.m1, (float)(2 * (h - a.n_head_log2) + 1));
}

// Sinks and 1/S exactly as ggml's tail of the one-chunk loop: a sink above the
// running maximum rescales the accumulator by exp(M - sink) and adds 1 to S,
// otherwise S += exp(sink - M); then out = acc * (S == 0 ? 0 : 1/S).
XQ_DEV void fa_finalize(float M, float S, bool has_sink, float sink, float& a1, float& inv,
                        float& lse) {
    a1 = 1.0f;
    float meff = M;
    if (has_sink) {
        if (sink > M) {
            const float ms = expf(M - sink);
            a1 = ms;
            S = fmaf(S, ms, 1.0f);
            meff = sink;
        } else {
            S = S + expf(sink - M);
        }
    }
    inv = S == 0.0f ? 0.0f : 1.0f / S;
    lse = S > 0.0f ? meff + logf(S) : -INFINITY;
}

// e^x through the hardware base-2 exponential (v_exp_f32, 1 ulp) on x*log2(e);
// exact 0 for x = -inf. Used for the online-softmax weights (arguments <= 0).
XQ_DEV float fast_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

XQ_DEV uint32_t lds_u32(const uint8_t* p) { return *(const uint32_t*)p; }
XQ_DEV uint32_t lds_u16(const uint8_t* p) { return *(const uint16_t*)p; }


struct FaLaunch;
hipError_t fa_mma_launch(FaArgs a, const FaLaunch& L, hipStream_t stream);
// The matrix-core engine's 32-bit row indices.
inline bool fa_mma_rows_ok(int64_t rows) { return rows < (int64_t)1 << 30; }
// Whether the matrix-core engine reads the mask where it lies (else its rows are
// re-laid on 4 bytes first).
bool fa_mma_mask_ok(const FaArgs& a, int kt, int d);
// Separate split-merge kernel (used when the merge cannot run inside pass 1).
hipError_t fa_reduce_launch(const FaArgs& a, int d, hipStream_t stream);

}  // namespace xq
