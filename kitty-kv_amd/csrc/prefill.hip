// Causal attention of a prompt (the T > 1 branch of KittyPagedAttention.forward,
// kitty/attention.py:179-191) at head_dim 128, fp16 or bf16, on gfx950.
//
// One wave takes 32 consecutive queries of one head; a 256-thread workgroup
// takes four waves of one (sequence, KV head) pair, ordered (query block,
// head of the group) with the head fastest, so at a GQA group of 4 the four
// heads of one query block share each key / value tile.  Tiles of 64 tokens
// stream HBM -> LDS with global_load_lds (two 32 KB stages, the next tile in
// flight while the current one is computed), chunk-swizzled so that neither
// the key reads nor the transposing value reads conflict.
//
//  S^T = K Q^T with 32x32x16 MFMAs (exact 16-bit products, fp32 sums): lane
//  (n = query l & 31, g = l / 32) ends with the scores of its one query for
//  tokens 8j + 4g + 0..3, so the softmax needs one exchange between lanes l
//  and l + 32 per tile and the rescale factor of the output is one number per
//  lane.
//  O^T += V^T P^T: the scores' registers are the B operand as they stand; the
//  reduction slots k = 8g + e of a 16-token step stand for tokens
//  4g + e (e < 4) and 8 + 4g + e - 4, and ds_read_b64_tr_b16 fetches the value
//  rows in that order (each 16-lane group transposes 4 tokens x 16 channels).
//
// Probabilities enter PV as two 16-bit terms (fp16: the rounded-to-zero value
// and its remainder, 21 bits; bf16: 16 bits) where fp32 has 24, the row's sum in
// fp32.  Error against float64, 17 to 1,801 tokens: 2.070e-4 fp16, 1.652e-3 bf16,
// the rounding of the output, and to four digits that of a float32 product
// (terms rounded to nearest, 23 bits in fp16: the same error, 6,001 tokens 1.5 %
// slower).  Each term has its own MFMA, in fp16 scaled by 2^7 (up to 2^15 while the running maximum lags)
// so that small probabilities stay clear of its subnormals; bf16 has fp32's
// exponents, and unscaled sums leave its values their range.  The running
// maximum is raised only when a tile passes it by 2^8, so most tiles skip
// the rescale of the 64 accumulator registers.
//
// Bound by the matrix cores plus the softmax's vector instructions: 48
// MFMAs of 32x32x16 (16 QK, 32 PV) and about 180 VALU per wave and 64-token
// tile.  Measured, 32 query / 8 KV heads: 6,001 tokens fp16 436 us (677 TFLOP/s
// of the plain causal product) where torch's float32 attention took 4,903 us;
// 2 x 517 tokens bf16 21 us against 147 us plus 60 us of float32 copies.
#include "common.h"

namespace kitty {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 32;            // queries per wave
constexpr int kTile = 64;            // tokens per LDS tile
constexpr int kWavesWg = 4;
constexpr int kRegion = kTile * 256; // bytes of the K or V half of a stage

struct PrefillParams {
    const uint16_t *q, *k, *v;
    uint16_t *out;
    int64_t q_s_seq, q_s_head, q_s_tok, k_s_seq, k_s_head, v_s_seq, v_s_head, o_s_seq, o_s_head, o_s_tok;
    uint32_t k_row, v_row;           // token strides in bytes
    int T, Hkv, gq, pairs, n_wg;     // n_wg: workgroups per pair
    float c;                         // sm_scale * log2(e)
};

template <bool BF16>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c)
{
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}

// (a, b) as packed 16-bit terms hi + lo.
template <bool BF16>
__device__ __forceinline__ void split2(float a, float b, unsigned &hi, unsigned &lo)
{
    if constexpr (BF16) {
        bf16x2 h;
        h[0] = (__bf16)a, h[1] = (__bf16)b;
        hi = __builtin_bit_cast(unsigned, h);
        bf16x2 r;
        r[0] = (__bf16)(a - __builtin_bit_cast(float, hi << 16));
        r[1] = (__bf16)(b - __builtin_bit_cast(float, hi & 0xffff0000u));
        lo = __builtin_bit_cast(unsigned, r);
    } else {
        const auto h = __builtin_amdgcn_cvt_pkrtz(a, b);
        hi = __builtin_bit_cast(unsigned, h);
        lo = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(a - (float)h[0], b - (float)h[1]));
    }
}

// max / sum of a value with the lane 32 apart
__device__ __forceinline__ float other_max(float v)
{
    const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    return fmaxf(__builtin_bit_cast(float, (int)s[0]), __builtin_bit_cast(float, (int)s[1]));
}
__device__ __forceinline__ float other_sum(float v)
{
    const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), false, false);
    return __builtin_bit_cast(float, (int)s[0]) + __builtin_bit_cast(float, (int)s[1]);
}

// 16 bytes per lane HBM -> LDS at lds_base + 16 * lane
__device__ __forceinline__ void to_lds16(const unsigned char *src, unsigned char *lds_base)
{
    __builtin_amdgcn_global_load_lds((const void *)src, (__attribute__((address_space(3))) void *)lds_base, 16, 0, 0);
}

// Every wave's loads into LDS have landed.  The wait is explicit: the compiler
// orders the direct-to-LDS loads with the issuing wave's own LDS reads only,
// and a barrier without it lets the other waves read a tile still in flight.
__device__ __forceinline__ void tile_barrier()
{
    __builtin_amdgcn_s_waitcnt((0x7 << 4));   // vmcnt(0) lgkmcnt(0), expcnt not waited for
    __syncthreads();
}

struct WaveQ {
    u32x4 q[8];        // the query's 128 channels: k-step s holds channels 16s + 8g .. + 7
    f32x16 O[4];       // O^T: channels 32dt + 8 (i / 4) + 4g + i % 4
    float m, l;        // running maximum (scaled scores) and this lane's half of the sum
    int qi, q_lo;      // this lane's query (clamped), first query of the wave
    int k_base, k_x;   // LDS offset of the lane's key row, chunk XOR
    int v_base[4];     // LDS offsets of the lane's value reads per 32-channel tile
};

// Tokens t0 .. t0 + 63 in stage (kst, vst) folded into the wave's state.
template <bool BF16>
__device__ __forceinline__ void tile_step(WaveQ &W, const unsigned char *kst, const unsigned char *vst, int t0, float c, int g)
{
    f32x16 S[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            S[mt][i] = 0.0f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const int off = W.k_base + ((W.k_x ^ (2 * s)) << 4);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
            S[mt] = mfma32<BF16>(*(const u32x4 *)(kst + off + 8192 * mt), W.q[s], S[mt]);
    }
    if (t0 + kTile - 1 > W.q_lo) {   // the diagonal: tokens after the query
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int tok = t0 + 32 * mt + 8 * (i >> 2) + 4 * g + (i & 3);
                S[mt][i] = tok > W.qi ? -__builtin_inff() : S[mt][i];
            }
    }
    float mx = S[0][0];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            mx = fmaxf(mx, S[mt][i]);
    mx = other_max(mx) * c;
    const bool raise = mx > W.m + 8.0f;
    if (__ballot(raise)) {
        const float mn = raise ? mx : W.m;
        const float alpha = __builtin_amdgcn_exp2f(W.m - mn);
        W.m = mn;
        W.l *= alpha;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                W.O[dt][i] *= alpha;
    }
    const float sub = BF16 ? W.m : W.m - 7.0f;
    unsigned hi[2][8], lo[2][8];
    float ls[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float a = __builtin_amdgcn_exp2f(__builtin_fmaf(S[mt][2 * i], c, -sub));
            const float b = __builtin_amdgcn_exp2f(__builtin_fmaf(S[mt][2 * i + 1], c, -sub));
            ls[(2 * i) & 3] += a;
            ls[(2 * i + 1) & 3] += b;
            split2<BF16>(a, b, hi[mt][i], lo[mt][i]);
        }
    W.l += (ls[0] + ls[1]) + (ls[2] + ls[3]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int mt = s >> 1, r = 4 * (s & 1);
        const u32x4 ph = {hi[mt][r], hi[mt][r + 1], hi[mt][r + 2], hi[mt][r + 3]};
        const u32x4 pl = {lo[mt][r], lo[mt][r + 1], lo[mt][r + 2], lo[mt][r + 3]};
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
            const unsigned char *src = vst + W.v_base[dt] + 4096 * s;
            const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)src);
            const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(src + 2048));
            const uint2 a = __builtin_bit_cast(uint2, v0), b = __builtin_bit_cast(uint2, v1);
            const u32x4 vf = {a.x, a.y, b.x, b.y};
            W.O[dt] = mfma32<BF16>(vf, ph, W.O[dt]);
            W.O[dt] = mfma32<BF16>(vf, pl, W.O[dt]);
        }
    }
}

template <bool BF16>
__global__ __launch_bounds__(64 * kWavesWg) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_attention_kernel(PrefillParams p)
{
    // stages in arrays of their own, so that reads of one do not wait for the loads into the other
    __shared__ __attribute__((aligned(16))) unsigned char k0[kRegion], v0[kRegion], k1[kRegion], v1[kRegion];
    const int lane = threadIdx.x & 63, g = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroup i runs on XCD i % 8: pairs vary fastest, so with a multiple of
    // eight pairs a pair's keys and values stay in one XCD's L2.  The last
    // query blocks, with the most tokens, start first.
    const int pair = blockIdx.x % p.pairs, item = p.n_wg - 1 - (int)(blockIdx.x / p.pairs);
    const int b = pair / p.Hkv, kh = pair - b * p.Hkv;
    const int n_qb = (p.T + kRows - 1) / kRows, n_w = n_qb * p.gq;
    const int w_last = min(n_w, (item + 1) * kWavesWg) - 1;
    const int q_end = min(p.T, (w_last / p.gq + 1) * kRows);   // queries below this in the workgroup
    const int nt = (q_end + kTile - 1) / kTile;
    const int w = min(n_w - 1, item * kWavesWg + wave);        // a wave past the end repeats the last one's work
    const bool active = item * kWavesWg + wave < n_w;
    const int qb = w / p.gq, h = kh * p.gq + (w - qb * p.gq);

    // ---- loads of tile t: wave w brings rows 16w .. 16w + 15 of K and of V,
    // four rows per instruction; slot (row, s) of K holds chunk s ^ (row & 15),
    // of V chunk s ^ 4 (row & 3).  Rows past the prompt repeat its last one.
    const unsigned char *kp = (const unsigned char *)(p.k + b * p.k_s_seq + kh * p.k_s_head);
    const unsigned char *vp = (const unsigned char *)(p.v + b * p.v_s_seq + kh * p.v_s_head);
    const uint32_t k_last = (uint32_t)(p.T - 1) * p.k_row, v_last = (uint32_t)(p.T - 1) * p.v_row;
    const int lr = lane >> 4, ls = lane & 15;
    auto issue = [&](int t, unsigned char *kst, unsigned char *vst) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 16 * wave + 4 * i + lr;
            const uint32_t ko = min((uint32_t)(t * kTile + row) * p.k_row, k_last) + 16u * (uint32_t)(ls ^ (row & 15));
            const uint32_t vo = min((uint32_t)(t * kTile + row) * p.v_row, v_last) + 16u * (uint32_t)(ls ^ (4 * (row & 3)));
            to_lds16(kp + ko, kst + 4096 * wave + 1024 * i);
            to_lds16(vp + vo, vst + 4096 * wave + 1024 * i);
        }
    };
    issue(0, k0, v0);

    WaveQ W;
    W.q_lo = qb * kRows;
    W.qi = min(W.q_lo + n, p.T - 1);
    {
        const uint16_t *qrow = p.q + b * p.q_s_seq + h * p.q_s_head + W.qi * p.q_s_tok;
#pragma unroll
        for (int s = 0; s < 8; ++s)
            W.q[s] = *(const u32x4 *)(qrow + 16 * s + 8 * g);
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            W.O[dt][i] = 0.0f;
    W.m = -3.402823466e38f;   // the lowest finite value: a row of -inf scores keeps it
    W.l = 0.0f;
    W.k_base = n * 256;
    W.k_x = g ^ (n & 15);
    {
        const int i = lane & 15, hs = (lane >> 4) & 1;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
            W.v_base[dt] = (4 * g + (i >> 2)) * 256 + 64 * (dt ^ (i >> 2)) + 32 * hs + 8 * (i & 3);
    }
    const int wave_nt = min(nt, (W.q_lo + kRows - 1) / kTile + 1);   // tiles this wave's queries see

    for (int t = 0; t < nt; t += 2) {
        tile_barrier();    // tile t has landed; every wave is done with the other stage
        if (t + 1 < nt)
            issue(t + 1, k1, v1);
        if (t < wave_nt)
            tile_step<BF16>(W, k0, v0, t * kTile, p.c, g);
        if (t + 1 >= nt)
            break;
        tile_barrier();
        if (t + 2 < nt)
            issue(t + 2, k0, v0);
        if (t + 1 < wave_nt)
            tile_step<BF16>(W, k1, v1, (t + 1) * kTile, p.c, g);
    }

    const float lsum = other_sum(W.l), inv = 1.0f / lsum;
    const bool row = active && W.q_lo + n < p.T;
    uint16_t *o = p.out + b * p.o_s_seq + h * p.o_s_head + W.qi * p.o_s_tok;
    bool odd = false;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint16_t r[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                r[e] = f2x(W.O[dt][4 * j + e] * inv, BF16);
                odd |= !(__builtin_fabsf(W.O[dt][4 * j + e]) < __builtin_inff());
            }
            if (row)
                *(uint2 *)(o + 32 * dt + 8 * j + 4 * g) =
                    make_uint2((uint32_t)r[0] | ((uint32_t)r[1] << 16), (uint32_t)r[2] | ((uint32_t)r[3] << 16));
        }

    // Infinite values: the second term of a weight is 0 or negative where the
    // weight is not, and times infinity makes the sum NaN (as does the weight 0
    // of a later token in the tile).  A wave that met one sums the infinities and
    // NaNs of the value rows its queries see, and writes those sums; rows whose
    // softmax is itself NaN stay as they are.
    odd = odd && row && lsum > 0.0f && lsum < __builtin_inff();
    if (!__ballot(odd))
        return;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            W.O[dt][i] = 0.0f;
    for (int t = 0; t <= min(W.q_lo + kRows, p.T) - 1; ++t) {
        const unsigned char *vrow = vp + (uint32_t)t * p.v_row + 8 * g;
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint2 v = *(const uint2 *)(vrow + 64 * dt + 16 * j);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = x2f((uint16_t)((e < 2 ? v.x : v.y) >> (16 * (e & 1))), BF16);
                    if (t <= W.qi && !(__builtin_fabsf(x) < __builtin_inff()))
                        W.O[dt][4 * j + e] += x;
                }
            }
    }
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (odd && !(__builtin_fabsf(W.O[dt][i]) < __builtin_inff()))
                o[32 * dt + 8 * (i >> 2) + 4 * g + (i & 3)] = f2x(W.O[dt][i], BF16);
}

static bool al(const void *p, unsigned a) { return ((uintptr_t)p & (a - 1)) == 0; }

} // namespace kitty

using namespace kitty;

extern "C" int kitty_prefill_attention(const kitty_prefill_args *args, kitty_stream_t stream)
{
    if (!args)
        return fail(KITTY_E_INVALID, "args is NULL");
    const kitty_prefill_args &a = *args;
    if (a.batch < 0 || a.tokens < 0 || a.num_kv_heads <= 0 || a.num_q_heads <= 0 || a.num_q_heads % a.num_kv_heads)
        return fail(KITTY_E_INVALID, "num_q_heads must be a positive multiple of num_kv_heads");
    if (a.dtype != KITTY_DTYPE_F16 && a.dtype != KITTY_DTYPE_BF16)
        return fail(KITTY_E_INVALID, "dtype must be KITTY_DTYPE_F16 or KITTY_DTYPE_BF16");
    if (!(a.sm_scale > 0.0f) || a.sm_scale > 1e30f)
        return fail(KITTY_E_INVALID, "sm_scale must be positive and finite");
    if (a.head_dim != 128)
        return fail(KITTY_E_UNSUPPORTED, "prefill attention is built for head_dim 128");
    if (a.batch == 0 || a.tokens == 0)
        return KITTY_OK;
    if (!a.q || !a.k || !a.v || !a.out)
        return fail(KITTY_E_INVALID, "NULL q, k, v or out");
    const int64_t s16[] = {a.q_s_seq, a.q_s_head, a.q_s_tok, a.k_s_seq, a.k_s_head, a.k_s_tok,
                           a.v_s_seq, a.v_s_head, a.v_s_tok};
    for (int64_t s : s16)
        if (s % 8)
            return fail(KITTY_E_UNSUPPORTED, "q, k and v strides must be multiples of 8 elements (16-byte rows)");
    if (!al(a.q, 16) || !al(a.k, 16) || !al(a.v, 16) || !al(a.out, 8) || a.o_s_seq % 4 || a.o_s_head % 4 || a.o_s_tok % 4)
        return fail(KITTY_E_UNSUPPORTED, "q, k and v must be 16-byte aligned, out 8-byte aligned");
    // a head's rows are addressed with 32-bit byte offsets (one tile past the end before clamping)
    for (int64_t s : {a.k_s_tok, a.v_s_tok})
        if (s < 0 || ((int64_t)a.tokens + kTile) * s * 2 + 256 >= (int64_t)1 << 31)
            return fail(KITTY_E_UNSUPPORTED, "k and v token strides must be non-negative and a head's rows span less than 2 GiB");
    PrefillParams p;
    p.q = a.q, p.k = a.k, p.v = a.v, p.out = a.out;
    p.q_s_seq = a.q_s_seq, p.q_s_head = a.q_s_head, p.q_s_tok = a.q_s_tok;
    p.k_s_seq = a.k_s_seq, p.k_s_head = a.k_s_head, p.v_s_seq = a.v_s_seq, p.v_s_head = a.v_s_head;
    p.o_s_seq = a.o_s_seq, p.o_s_head = a.o_s_head, p.o_s_tok = a.o_s_tok;
    p.k_row = (uint32_t)(2 * a.k_s_tok), p.v_row = (uint32_t)(2 * a.v_s_tok);
    p.T = a.tokens, p.Hkv = a.num_kv_heads, p.gq = a.num_q_heads / a.num_kv_heads;
    const int64_t pairs = (int64_t)a.batch * a.num_kv_heads;
    const int64_t n_w = ((int64_t)a.tokens + kRows - 1) / kRows * p.gq;
    const int64_t n_wg = (n_w + kWavesWg - 1) / kWavesWg;
    if (n_w > 0x7fffffff || pairs * n_wg > 0x7fffffff)
        return fail(KITTY_E_UNSUPPORTED, "too many query blocks for one launch");
    p.pairs = (int)pairs, p.n_wg = (int)n_wg;
    p.c = a.sm_scale * kLog2e;
    const dim3 grid((unsigned)(pairs * n_wg)), block(64 * kWavesWg);
    if (a.dtype == KITTY_DTYPE_BF16)
        hipLaunchKernelGGL(prefill_attention_kernel<true>, grid, block, 0, (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL(prefill_attention_kernel<false>, grid, block, 0, (hipStream_t)stream, p);
    return check_launch("prefill_attention_kernel");
}
