// xq_kv.hip — KV append: F32 rows -> KV cache records at row positions.
//
// The scatter of shaders/rkva/rkva_store_f16.hlsl:63-85 (F32 -> ggml F16 RNE at
// absolute positions) widened to every KV storage type of this path, with
// ggml's block quantizers reproduced bit for bit:
//   Q8_0  quantize_row_q8_0 (x86: id = 127/amax, round half to even) or
//         quantize_row_q8_0_ref (id = 1/d, roundf);
//   Q4_0  quantize_row_q4_0_ref (d = max/-8 with max the first element of
//         largest magnitude, q = min(15, (int8)(x*id + 8.5)));
//   E5M2  f16 RNE then E5M2 RNE with finite saturation (the Q/OUT wire codec of
//         shaders/rkva/rkva_range_bulk_f16.hlsl:156-167).
// Built with -ffp-contract=off so the q4_0 "x*id + 8.5" rounds twice, as the CPU
// reference does.
#include "xq_kernels.h"

namespace xq {

XQ_DEV uint32_t f16_to_e5m2(uint32_t h) {
    const uint32_t sign = (h >> 8) & 0x80u;
    if ((h & 0x7c00u) == 0x7c00u) {
        if (!(h & 0x03ffu)) return sign | 0x7cu;
        const uint32_t top = (h >> 8) & 3u;
        return sign | 0x7cu | (top ? top : 1u);
    }
    uint32_t mag = h & 0x7fffu;
    if (mag > 0x7b00u) mag = 0x7b00u;
    return sign | ((mag + 0x7fu + ((mag >> 8) & 1u)) >> 8);
}

XQ_DEV uint32_t f32_to_bf16_bits(float x) {
    const uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return ((u >> 16) | 64u) & 0xffffu;
    return ((u + (0x7fffu + ((u >> 16) & 1u))) >> 16) & 0xffffu;
}

// Unaligned-tolerant vectors: the caller's rows and planes need not be aligned
// beyond their elements (gfx950 global accesses take any alignment).
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32u __attribute__((aligned(1)));
typedef uint16_t u16u __attribute__((aligned(1)));
typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(1)));
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(1)));

// Bound by HBM: 5/4 of the f32 source for q8_0. One lane converts four
// consecutive elements: a wave's load is 1 KiB of contiguous source, and a
// 32-element block is eight lanes, whose maximum takes three DPP steps and no
// LDS. UN such 256-element units per wave, every load issued before the first is
// used. 8192 tokens x 4 heads x 256 to q8_0 (42.5 MB): 9.2 us per launch (4.6
// TB/s), against 30 us with one lane per 32-element block behind an LDS copy of
// the record (one record per wave, eight of its 64 lanes at work).
template <int KT, int D, int UN>
__global__ __launch_bounds__(256) void kv_store_kernel(const float* __restrict__ src,
                                                       const int32_t* __restrict__ positions,
                                                       uint32_t n_rec, uint32_t n_head_kv,
                                                       int32_t q8_variant, uint8_t* __restrict__ dst,
                                                       int32_t capacity) {
    constexpr int REC = KT == XQ_TYPE_BF16 ? 2 * D : rec_bytes(KT, D);
    constexpr uint32_t RPU = 256 / D;  // records per unit
    constexpr uint32_t LPR = D / 4;    // lanes per record
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t unit0 = (blockIdx.x * 4u + threadIdx.x / 64u) * UN;
    const uint32_t el = 4u * (lane % LPR);  // first element in the record
    f4u x[UN];
    int32_t pos[UN];
    uint32_t head[UN];
#pragma unroll
    for (int i = 0; i < UN; ++i) {
        const uint32_t rec = (unit0 + i) * RPU + lane / LPR;
        const bool ok = rec < n_rec;
        const uint32_t t = ok ? rec / n_head_kv : 0u;
        head[i] = ok ? rec - t * n_head_kv : 0u;
        x[i] = *(const f4u*)(src + (int64_t)(ok ? rec : 0u) * D + el);
        pos[i] = ok ? positions[t] : -1;
    }
#pragma unroll
    for (int i = 0; i < UN; ++i) {
        float amax = 0.0f, vmax = 0.0f;
        if constexpr (KT == XQ_TYPE_Q8_0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) amax = fabsf(x[i][j]) > amax ? fabsf(x[i][j]) : amax;  // skips every NaN
            amax = fmaxf(amax, dpp<0xB1>(amax));
            amax = fmaxf(amax, dpp<0x4E>(amax));
            amax = fmaxf(amax, dpp<0x141>(amax));
        } else if constexpr (KT == XQ_TYPE_Q4_0) {
            // the first element of the largest magnitude: of two halves the later
            // one wins only when it is strictly larger
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float m = fabsf(x[i][j]);
                if (amax < m) {
                    amax = m;
                    vmax = x[i][j];
                }
            }
            auto fold = [&](float oa, float ov, bool first) {  // first: this lane's half comes first
                const bool take = first ? amax < oa : !(oa < amax);
                amax = take ? oa : amax;
                vmax = take ? ov : vmax;
            };
            fold(dpp<0xB1>(amax), dpp<0xB1>(vmax), !(lane & 1u));
            fold(dpp<0x4E>(amax), dpp<0x4E>(vmax), !(lane & 2u));
            fold(dpp<0x141>(amax), dpp<0x141>(vmax), !(lane & 4u));
        }
        const bool live = pos[i] >= 0 && pos[i] < capacity;
        uint8_t* y = dst + ((int64_t)pos[i] * n_head_kv + head[i]) * REC;
        if constexpr (KT == XQ_TYPE_F32) {
            if (live) *(u32x4u*)(y + 4 * el) = __builtin_bit_cast(u32x4u, x[i]);
        } else if constexpr (KT == XQ_TYPE_F16 || KT == XQ_TYPE_BF16) {
            uint32_t h[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) h[j] = KT == XQ_TYPE_F16 ? f32_to_f16_bits(x[i][j]) : f32_to_bf16_bits(x[i][j]);
            if (live) *(u32x2u*)(y + 2 * el) = u32x2u{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
        } else if constexpr (KT == XQ_TYPE_E5M2) {
            uint32_t w = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) w |= f16_to_e5m2(f32_to_f16_bits(x[i][j])) << (8 * j);
            if (live) *(u32u*)(y + el) = w;
        } else if constexpr (KT == XQ_TYPE_Q8_0) {
            const float d = amax / 127.0f;
            float id;
            if (q8_variant == 0)
                id = amax != 0.0f ? 127.0f / amax : 0.0f;
            else
                id = d != 0.0f ? 1.0f / d : 0.0f;
            uint32_t w = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float tq = x[i][j] * id;
                const float r = q8_variant == 0 ? rintf(tq) : roundf(tq);
                w |= (uint32_t)(uint8_t)(int8_t)(int)r << (8 * j);
            }
            uint8_t* yb = y + el / kQK * 34;
            if (live) {
                *(u32u*)(yb + 2 + el % kQK) = w;
                if (!(lane & 7u)) *(u16u*)yb = (uint16_t)f32_to_f16_bits(d);
            }
        } else {
            const float d = vmax / -8.0f;
            const float id = d != 0.0f ? 1.0f / d : 0.0f;
            uint32_t w = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int n = (int8_t)(x[i][j] * id + 8.5f);
                n = n > 15 ? 15 : n;
                w |= (uint32_t)(uint8_t)n << (8 * j);
            }
            // byte j of the block holds element j low and element 16 + j high: lanes
            // 0..3 of a block take their partner's (lane + 4) nibbles
            const uint32_t hi = (uint32_t)__shfl_xor((int)w, 4);
            uint8_t* yb = y + el / kQK * 18;
            if (live && !(lane & 4u)) {
                *(u32u*)(yb + 2 + el % kQK) = w | ((hi & 0x0f0f0f0fu) << 4);
                if (!(lane & 7u)) *(u16u*)yb = (uint16_t)f32_to_f16_bits(d);
            }
        }
    }
}

template <int KT, int D>
static void kv_store_dispatch(const float* src, const int32_t* positions, int64_t n_rec, int32_t n_head_kv,
                              int32_t q8_variant, uint8_t* dst, int32_t capacity, hipStream_t stream) {
    const int64_t units = (n_rec + 256 / D - 1) / (256 / D);
    // Records of 16 and 32 bits per element: four units per wave once that still gives
    // every CU four workgroups. The narrower ones, whose conversion takes longer than
    // their loads, one unit whatever the size: more waves hide it better. us per append
    // of K and V, 4 heads x 256, with 1 / 2 / 4 units:
    //   tokens       f16               f32               e5m2              q8_0              q4_0
    //   3000    8.2  8.5  8.6   10.1 10.4 10.3    9.4  9.8 10.4    9.2  9.3 10.1    9.1  9.3  9.7
    //   6000   15.8 15.5 15.5   18.7 18.1 17.3   15.8 17.2 17.9   15.2 16.6 17.8   15.4 16.3 17.1
    //   8192   20.8 19.8 18.9   23.7 23.0 22.1   19.7 20.7 22.4   19.0 20.2 21.6   18.8 19.6 20.9
    //   16384  35.2 33.1 33.2   43.2 41.3 45.4   32.8 34.0 35.4   31.4 32.7 34.2   31.7 32.5 31.7
    constexpr bool wide = KT == XQ_TYPE_F32 || KT == XQ_TYPE_F16 || KT == XQ_TYPE_BF16;
    if constexpr (wide) {
        if (units >= 256 * 4 * 4 * 4) {
            launch("kv_store", kv_store_kernel<KT, D, 4>, dim3((uint32_t)((units + 15) / 16)), dim3(256), stream, src,
                   positions, (uint32_t)n_rec, (uint32_t)n_head_kv, q8_variant, dst, capacity);
            return;
        }
    }
    launch("kv_store", kv_store_kernel<KT, D, 1>, dim3((uint32_t)((units + 3) / 4)), dim3(256), stream, src,
           positions, (uint32_t)n_rec, (uint32_t)n_head_kv, q8_variant, dst, capacity);
}

template <int KT>
static hipError_t kv_store_type(int32_t head_dim, const float* src, const int32_t* positions, int64_t n_rec,
                                int32_t n_head_kv, int32_t q8_variant, uint8_t* dst, int32_t capacity,
                                hipStream_t stream) {
    switch (head_dim) {
    case 64: kv_store_dispatch<KT, 64>(src, positions, n_rec, n_head_kv, q8_variant, dst, capacity, stream); break;
    case 128: kv_store_dispatch<KT, 128>(src, positions, n_rec, n_head_kv, q8_variant, dst, capacity, stream); break;
    case 256: kv_store_dispatch<KT, 256>(src, positions, n_rec, n_head_kv, q8_variant, dst, capacity, stream); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t kv_store_launch(const float* src, const int32_t* positions, int32_t n_tokens,
                           int32_t n_head_kv, int32_t head_dim, int32_t kv_type,
                           int32_t q8_variant, void* dst, int32_t capacity, hipStream_t stream) {
    const int64_t n_rec = (int64_t)n_tokens * n_head_kv;
    if (n_rec == 0) return hipSuccess;
    uint8_t* y = (uint8_t*)dst;
    switch (kv_type) {
    case XQ_TYPE_F32: return kv_store_type<XQ_TYPE_F32>(head_dim, src, positions, n_rec, n_head_kv, q8_variant, y, capacity, stream);
    case XQ_TYPE_F16: return kv_store_type<XQ_TYPE_F16>(head_dim, src, positions, n_rec, n_head_kv, q8_variant, y, capacity, stream);
    case XQ_TYPE_BF16: return kv_store_type<XQ_TYPE_BF16>(head_dim, src, positions, n_rec, n_head_kv, q8_variant, y, capacity, stream);
    case XQ_TYPE_E5M2: return kv_store_type<XQ_TYPE_E5M2>(head_dim, src, positions, n_rec, n_head_kv, q8_variant, y, capacity, stream);
    case XQ_TYPE_Q8_0: return kv_store_type<XQ_TYPE_Q8_0>(head_dim, src, positions, n_rec, n_head_kv, q8_variant, y, capacity, stream);
    case XQ_TYPE_Q4_0: return kv_store_type<XQ_TYPE_Q4_0>(head_dim, src, positions, n_rec, n_head_kv, q8_variant, y, capacity, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace xq
