// Merging the partials of one query head, shared by the merge kernel
// (decode.hip) and the pair kernel (decode_mfma.hip).
#pragma once
#include "common.h"
#include "decode.h"

namespace kitty {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float wave_max(float v)
{
    for (int off = 32; off > 0; off >>= 1)
        v = fmaxf(v, __shfl_xor(v, off));
    return v;
}

__device__ __forceinline__ float wave_sum(float v)
{
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off);
    return v;
}

// An output value's bits: fp16, or the fp16 value converted to bf16.
__device__ __forceinline__ uint16_t out_bits(const DecodeParams &p, float v)
{
    const uint16_t h = f2h(v);
    return p.out_bf16 ? f2bf(h2f(h)) : h;
}

// Merge of NS <= 4 K partials of D = 128 channels in one round trip: lane
// group g = lane / 16 takes partials g, g + 4, g + 8, ... and lane c = lane
// % 16 of the group channels 8c .. 8c + 7, so one 16-byte load per lane
// covers four partial rows (two per row and lane), every (m, l) and O load
// issued together (indices past NS clamp to the last partial and weigh 0).
// The weighted sums of the four groups are added across lanes 16 and 32
// apart.  Configs 3 and 5 (17 and 66 partials per row) take 12 and 60 loads
// per lane where a float2 per lane and partial took 33 and 130.
template <int K>
__device__ __forceinline__ void merge_quads(const DecodeParams &p, int64_t row0, int64_t rstep, int NS, uint16_t *o)
{
    const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
    const float ninf = -__builtin_inff();
    float4 va[K], vb[K];
    float2 ml[K];
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const int64_t row = row0 + (int64_t)min(g + 4 * i, NS - 1) * rstep;
        const float *src = p.ws_o + row * 128 + 8 * c;
        va[i] = *(const float4 *)src;
        vb[i] = *(const float4 *)(src + 4);
        ml[i] = *(const float2 *)(p.ws_ml + 2 * row);
    }
    float mloc = ninf;
    bool nanl = false;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        if (g + 4 * i < NS) {
            mloc = fmaxf(mloc, ml[i].x);
            nanl |= ml[i].x != ml[i].x;
        }
    }
    const float M = wave_max(mloc);
    const bool nan = wave_max(nanl ? 1.0f : 0.0f) > 0.0f;
    float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, lsum = 0.0f;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const float w = g + 4 * i < NS && ml[i].x != ninf && M != ninf ? exp2f(ml[i].x - M) : 0.0f;
        lsum += w * ml[i].y;
        acc[0] += w * va[i].x;
        acc[1] += w * va[i].y;
        acc[2] += w * va[i].z;
        acc[3] += w * va[i].w;
        acc[4] += w * vb[i].x;
        acc[5] += w * vb[i].y;
        acc[6] += w * vb[i].z;
        acc[7] += w * vb[i].w;
    }
#pragma unroll
    for (int off = 16; off <= 32; off *= 2) {
        lsum += __shfl_xor(lsum, off);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            acc[e] += __shfl_xor(acc[e], off);
    }
    if (g != 0)
        return;
    const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;  // no tokens -> zeros (attention.py:180-182)
    uint16_t h[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        h[e] = out_bits(p, nan ? __builtin_nanf("") : acc[e] * inv);
    uint16_t *dst = o + 8 * c;
    if (((uintptr_t)dst & 15) == 0) {
        *(u32x4 *)dst = u32x4{(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16),
                              (uint32_t)h[4] | ((uint32_t)h[5] << 16), (uint32_t)h[6] | ((uint32_t)h[7] << 16)};
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            dst[e] = h[e];
    }
}

} // namespace kitty
