// MFMA split-K paged decode for the production shape (D = G = 128,
// D_boost <= 32, GQA group 4, 8 or 16; smaller groups run as the next of
// these, whose extra members repeat the first head) on gfx950.
//
// One wave (64 lanes) takes an equal share of the batch's work units (the
// pages of every (sequence b, KV head kh) pair, then a weighted share of its
// FP16 sink + tail tokens; see the unit-balanced plan in decode.h), one
// segment per pair it touches.  Per page it streams the 9.5-10 KB
// (page, head) record from HBM into a 10 KB LDS stage one page ahead, and:
//
//  QK   S[h][t] = sum_k A[h][k] * B[k][t] with v_mfma_f32_16x16x32_f16.
//       B: 2-bit codes as fp16 subnormals: the code of token slot a (bits
//       2a, 2a+1 of a byte) masked in place is c 4^a 2^-24 exactly, one
//       v_and_b32 per two codes, the odd bytes of each word after one shift
//       by 8.  ds_read_b64_tr_b8 transposes the channel-major page in LDS so
//       each lane holds 8 channels of one byte column (4 tokens, one per
//       slot a).
//       A: q * scale_k[d] on two MFMA rows per head, the fp16-rounded
//       product and its exact residual (qk_residual), so the scores keep
//       fp32 accuracy; sm_scale * log2(e) multiplies the scores.
//       Every MFMA of slot a accumulates 4^a 2^-24 sum_k A[k] c; the softmax
//       scales it by 2^24 4^-a and subtracts Y = sum_k A[k] z_k (bias tile Y,
//       4-5 MFMAs).  High 2 bits of boosted channels are 16-32 extra
//       reduction rows with A = 4 q[channel(rank)] scale_k.
//  softmax  online, base 2, one DPP row reduction per page.
//  PV, GQA 4: v_mfma_f32_16x16x128_f8f6f4 with the value codes as fp4 B
//       operands (ds_read_b64_tr_b4 + one mask per 8 codes) and P' as three
//       fp8 terms on the three spare rows of each head (see pv_fp8_fp4):
//       8 MFMAs per page instead of 32.
//  PV, GQA 8 / 16: O[h][d] = sum_t P'[h][t] * B[t][d], P' = p * s_t (fp16) staged
//       through a 1-2 KB LDS buffer; value codes get the same tr8 + mask
//       treatment, so output tile a (channel slot a) accumulates
//       4^a 2^-24 sum_t P' c; the per-token zero points are subtracted in
//       those units at each page, and 2^24 4^-a is applied when the
//       segment's partial is written.
//
// bf16 (q, sinks, tails and metadata all bf16): an instance of the same kernel
// whose error stays within 0.1 % of that of the generic fp32 kernel it replaces
// at this shape (page_qk, qk_setup, pv_split say how).  8 sequences of 3,000-9,000
// tokens, 32 query / 8 KV heads: the whole decode 23.3 us (in a trace 19.6 split
// and 4.3 merge) against 115.9, both 2.1e-4 off float64 (the output rounding).
//
// Reduction index k of every MFMA follows the natural channel / token order
// within a 32-wide step (the tr8 row order puts even and odd bytes of a
// word on consecutive k).
#include <utility>
#include "common.h"
#include "decode.h"
#include "merge.h"
#include "qk_exact.h"

namespace kitty {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// LDS stage of one (page, head) record, byte offsets.
constexpr int kKlo = 0;       // key low bits   (128 rows x 32 B), chunk-swizzled
constexpr int kVal = 4096;    // value codes    (128 rows x 32 B), chunk-swizzled
constexpr int kKhi = 8192;    // key high bits  (<= 32 rows x 32 B), chunk-swizzled
constexpr int kMeta = 9216;   // key scale (256 B), key zero (256 B), value (scale, zero) (512 B)
constexpr int kStage = 10240;

// 16-byte chunk λ of a 128 x 32 B region lives at LDS slot λ; it holds row
// λ/2, chunk (λ & 1) ^ ((row >> 3) & 1) of the page.  The XOR keeps the 32
// rows read by one ds_read_b64_tr_b8 spread over all LDS banks.
__device__ __forceinline__ int chunk_global_offset(int slot)
{
    const int row = slot >> 1;
    return row * 32 + (((slot & 1) ^ ((row >> 3) & 1)) << 4);
}

__device__ __forceinline__ i32x2 tr8(const unsigned char *lds)
{
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) i32x2 *)lds);
}

// A tr8 result and its odd bytes moved down: {w0, w1, w0 >> 8, w1 >> 8}.
struct RawCodes {
    unsigned w[4];
};

__device__ __forceinline__ RawCodes raw_codes(i32x2 raw)
{
    return RawCodes{{(unsigned)raw[0], (unsigned)raw[1], (unsigned)raw[0] >> 8, (unsigned)raw[1] >> 8}};
}

// Slot `a` (token 4j+a of a key byte, or channel 4j+a of a value byte) of
// the 8 transposed bytes -> 8 fp16 MFMA inputs: the code masked in place is
// the fp16 subnormal c 4^a 2^-24, exactly, one v_and_b32 per two codes (the
// odd bytes of each word after one shift by 8, shared by the four slots).
// The MFMA sums then hold only the signal, 4^a 2^-24 sum A c, which keeps
// full fp32 accuracy (an offset would cancel in the accumulator); the
// consumers scale slot a by 2^24 / 4^a.
constexpr float kSub = 16777216.0f;  // 2^24

// q enters the page path's QK operand times 2^-3 (exact: a power of two),
// and the scores are multiplied back by 2^3.
constexpr float kQPre = 0.125f, kQInv = 8.0f;

template <int A>
__device__ __forceinline__ half8 codes_to_half8(const RawCodes &r)
{
    constexpr unsigned m = 0x00030003u << (2 * A);
    u32x4 v;
    v[0] = r.w[0] & m;
    v[1] = r.w[2] & m;
    v[2] = r.w[1] & m;
    v[3] = r.w[3] & m;
    return __builtin_bit_cast(half8, v);
}

__device__ __forceinline__ half8 slot_codes(const RawCodes &r, int a)
{
    return a == 0 ? codes_to_half8<0>(r) : a == 1 ? codes_to_half8<1>(r) : a == 2 ? codes_to_half8<2>(r)
                                                                                  : codes_to_half8<3>(r);
}

// The bf16 instances' codes: even slots moved to bits 8-9 of their half (code
// 4^4 2^-24, a place above slot 3's), odd ones to bits 6-7 (slot 3's place), one
// shift more per word.  The matrix core aligns a block's products by the
// exponents of their operands before it adds, and a subnormal counts with the
// smallest normal exponent: a code of slot 0 sits ten bits below that, and its
// sums keep 14 bits where slot 3's keep 20 and bits 8-9 keep 22 (measured score
// errors: 1e-4, 2.5e-5, 5e-6 and 1e-6 for slots 0 to 3).  With the even slots in
// slot 2's place the output of 1 x 30,000 tokens was 1.05 % further from float64
// than the fp32 kernel's, in theirs 0.06 %.
constexpr int bf_slot(int a) { return 4 - (a & 1); }

struct RawCodesUp {
    unsigned w[2], l4[2], l8[2], r4[2], r8[2];
};

__device__ __forceinline__ RawCodesUp raw_codes_up(i32x2 raw)
{
    const unsigned a = (unsigned)raw[0], b = (unsigned)raw[1];
    return RawCodesUp{{a, b}, {a << 4, b << 4}, {a << 8, b << 8}, {a >> 4, b >> 4}, {a >> 8, b >> 8}};
}

// Slot a from the shifted words that hold it in place for the even and the odd bytes.
__device__ __forceinline__ half8 slot_codes(const RawCodesUp &c, int a)
{
    const unsigned m = 0x00030003u << (2 * bf_slot(a));
    const unsigned *even = a == 0 ? c.l8 : a == 3 ? c.w : c.l4;
    const unsigned *odd = a == 0 ? c.w : a == 3 ? c.r8 : c.r4;
    return __builtin_bit_cast(half8, u32x4{even[0] & m, odd[0] & m, even[1] & m, odd[1] & m});
}

// Codes of the production (fp16) and the bf16 instances, and 4^slot of their scale.
template <bool BF>
__device__ __forceinline__ auto page_codes(i32x2 raw)
{
    if constexpr (BF)
        return raw_codes_up(raw);
    else
        return raw_codes(raw);
}
template <bool BF>
__device__ __forceinline__ constexpr float slot_weight(int a)
{
    return (float)(1 << (2 * (BF ? bf_slot(a) : a)));
}

// PV operands of the GQA-4 path (v_mfma_f32_16x16x128_f8f6f4, A fp8 e4m3,
// B fp4 e2m1).  A 2-bit value code in the low bits of a nibble whose top
// two bits are clear is the e2m1 number code / 2, so value codes become B
// operands with one mask per 8 codes.  K order of the instruction: fp4 B
// nibble i of lane group g is K = 32 g + i; fp8 A byte i of lane group g is
// K = 16 g + i for i < 16 and 64 + 16 g + (i - 16) above.
__device__ __forceinline__ i32x2 tr4(const unsigned char *lds)
{
    return __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) i32x2 *)lds);
}

__device__ __forceinline__ f32x4 mfma_fp8_fp4(i32x8 a, u32x4 b)
{
    const i32x8 b8 = {(int)b[0], (int)b[1], (int)b[2], (int)b[3], 0, 0, 0, 0};  // fp4 reads the first 4 registers
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b8, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 4, 0, 0, 0, 0);
}

// Four fp32 values / scale -> four fp8 e4m3 (round to nearest even) in one
// dword, byte i = value i.  The caller keeps |value / scale| <= 448.
__device__ __forceinline__ unsigned fp8x4(float a, float b, float c, float d, float scale)
{
    s16x2 v = __builtin_bit_cast(s16x2, a);  // both halves are overwritten
    v = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(v, a, b, scale, false);
    v = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(v, c, d, scale, true);
    return __builtin_bit_cast(unsigned, v);
}

// x[i] -= (fp8 byte i of w) * scale: the residual the next fp8 term encodes.
__device__ __forceinline__ void fp8_residual(float *x, unsigned w, float scale)
{
    const f32x2 lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, scale, false);
    const f32x2 hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(w, scale, true);
    x[0] -= lo[0];
    x[1] -= lo[1];
    x[2] -= hi[0];
    x[3] -= hi[1];
}

__device__ __forceinline__ f32x4 mfma(half8 a, half8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 mfma_bf(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The two halves of a word of bf16 values as fp32 (exact).
__device__ __forceinline__ float bf_lo(unsigned w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf_hi(unsigned w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// Two fp32 values as packed fp16, rounded toward zero.
__device__ __forceinline__ unsigned pack_rtz(float a, float b)
{
    return __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_pkrtz(a, b));
}

template <int CTRL>
__device__ __forceinline__ float dpp(float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Reductions over the 16 lanes of a DPP row (one lane group = one head).
// Max over the 16 lanes of a DPP row: one v_max_f32 with a row rotation per
// step (fmaxf would add a DPP move and an input canonicalisation per step).
// The s_nop 1 ahead of each step covers the two wait states a DPP read needs
// after a VALU write of the same VGPR.  Scores are never NaN.
__device__ __forceinline__ float row_max16(float v)
{
    asm volatile("s_nop 1\n\t"
                 "v_max_f32_dpp %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 1\n\t"
                 "v_max_f32_dpp %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 1\n\t"
                 "v_max_f32_dpp %0, %0, %0 row_ror:2 row_mask:0xf bank_mask:0xf\n\t"
                 "s_nop 1\n\t"
                 "v_max_f32_dpp %0, %0, %0 row_ror:1 row_mask:0xf bank_mask:0xf"
                 : "+v"(v));
    return v;
}

__device__ __forceinline__ float row_sum16(float v)
{
    v += dpp<0x128>(v);
    v += dpp<0x124>(v);
    v += dpp<0x122>(v);
    v += dpp<0x121>(v);
    return v;
}

__device__ __forceinline__ unsigned pack_h2(float a, float b)
{
    half2v h;
    h[0] = (_Float16)a;
    h[1] = (_Float16)b;
    return __builtin_bit_cast(unsigned, h);
}

__device__ __forceinline__ half2v as_h2(unsigned u) { return __builtin_bit_cast(half2v, u); }
__device__ __forceinline__ unsigned as_u(half2v h) { return __builtin_bit_cast(unsigned, h); }


// Lane of the wave (single-wave workgroups and the waves of a pair workgroup alike).
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// The wave's LDS accesses so far are done before the ones that follow.  A
// workgroup of one wave uses its barrier; the waves of a pair workgroup
// (decode_pair_kernel) run on their own stages and wait only for themselves.
template <bool PAIR>
__device__ __forceinline__ void wave_sync()
{
    if constexpr (PAIR) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

struct PageSrc {
    const unsigned char *klo, *val, *khi, *kmeta, *vmeta;
};

__device__ __forceinline__ PageSrc page_src(const DecodeParams &p, int64_t ph)
{
    PageSrc s;
    s.klo = p.key_low + ph * 4096;
    s.val = p.value + ph * 4096;
    s.khi = p.key_high + ph * (int64_t)p.Dk * 32;
    s.kmeta = (const unsigned char *)p.key_meta + ph * 512;
    s.vmeta = (const unsigned char *)p.value_meta + ph * 512;
    return s;
}

// global_load_lds_dwordx4: lane l's 16 bytes land at lds_base + 16 l.  The
// pages are streamed once, so the loads carry the non-temporal hint.
constexpr int kLoadAux = 2;
__device__ __forceinline__ void gll16(const unsigned char *src, unsigned char *lds_base)
{
    __builtin_amdgcn_global_load_lds((const void *)src, (__attribute__((address_space(3))) void *)lds_base, 16, 0,
                                     kLoadAux);
}
// The same with an immediate offset, which the instruction adds to the
// global and the LDS address alike.
template <int OFF>
__device__ __forceinline__ void gll16_at(const unsigned char *src, unsigned char *lds_base)
{
    __builtin_amdgcn_global_load_lds((const void *)src, (__attribute__((address_space(3))) void *)lds_base, 16, OFF,
                                     kLoadAux);
}

// Ten direct-to-LDS loads of one (page, head) record; lane l fetches the
// chunk that belongs in LDS slot l (chunk_global_offset), which applies the
// bank swizzle without extra instructions.  Lanes past 2*Dk re-read the
// first K-high chunk (the first key-metadata chunk when Dk = 0) into unused
// K-high slots, so every page issues exactly kLoadsPerPage loads.  Slot
// 64 j + l of a 4 KB region is chunk_global_offset(l) + 1024 j, so nine of
// the loads are a wave-uniform base plus one 32-bit lane offset plus a
// constant: the SGPR-base form, with no 64-bit address arithmetic per lane.
constexpr int kLoadsPerPage = 10;

__device__ __forceinline__ void issue_page(unsigned char *st, const PageSrc &s, int lane, int Dk)
{
    uint32_t off = (uint32_t)chunk_global_offset(lane), hoff = lane < 2 * Dk ? off : 0u;
    // Fresh 32-bit values in the caller's block: a page loop would otherwise
    // hoist their 64-bit extensions, and the loads would fall back to 64-bit
    // per-lane addresses.
    asm volatile("" : "+v"(off), "+v"(hoff));
    gll16_at<0>(s.klo + off, st + kKlo);
    gll16_at<0>(s.val + off, st + kVal);
    gll16_at<1024>(s.klo + off, st + kKlo);
    gll16_at<1024>(s.val + off, st + kVal);
    gll16_at<2048>(s.klo + off, st + kKlo);
    gll16_at<2048>(s.val + off, st + kVal);
    gll16_at<3072>(s.klo + off, st + kKlo);
    gll16_at<3072>(s.val + off, st + kVal);
    gll16((Dk > 0 ? s.khi : s.kmeta) + hoff, st + kKhi);
    gll16((lane < 32 ? s.kmeta : s.vmeta) + 16u * (uint32_t)(lane & 31), st + kMeta);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
    // s_waitcnt vmcnt(N) expcnt(7) lgkmcnt(15)
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// Running state of one wave across its pages.
template <int GQ, bool BF>
struct WaveState {
    static constexpr int HPL = GQ / 4;      // heads per lane group
    u32x4 qv[4], qvh;                        // static halves of the QK A operand (fp16 q)
    float qk_c[BF ? HPL : 1];                // sm_scale * log2(e): scores in log2 units (bf16: times the head's 2^E)
    int hch[8];                              // channel of high-bit row 8q + i
    int tr_base0, tr_base1;                  // tr8 source offsets (byte columns 0-15 / 16-31)
    int prow;                                // head row whose P' this lane reads for PV
    float m_run[HPL], l_run[HPL];
    f32x4 O[2][4];                           // GQA 8 / 16: output tiles (4^a O of channels 64cb + 4r + a)
    float ob[2][4][HPL];                     // bf16: O of head slot j, channels 64cb + 4r + a
    float o4[4][2];                          // GQA 4: O of head q, channels 32ch + 2r + e
    int trv[2][2];                           // GQA 4: tr4 offsets of value rows 32q + 16k + r, 16-byte chunk c
};

// GQA 4: online softmax and PV of one page with fp8 x fp4 MFMAs.  Lane
// (q, r) holds head q's scores of tokens 64cb + 4r + a (S[cb][a] register 0,
// scaled by 4^a, zero-point term Y not yet subtracted).
//  P' = p * s_t (value scale of token t) is written to LDS as three fp8
//  terms on MFMA rows 4h + t: term 0 = fp8(P' / sig), term t encodes the
//  remaining residual with scale sig / 64^t (12 significant bits in all, or
//  2^-24 of s_max).  sig = 2^(e - 4) with s_max < 2^e, the page's largest value
//  scale, so P' / sig < 16 (p <= 1), and the residuals stay below 64 of their
//  scales (fp8 ends at 448).
//  The matrix core aligns a row's products to the largest and drops what lies
//  below its window, so a term 0 that spans fp8's range loses the low bits of
//  all but a page's top tokens, the more the more pages start a chunk (p = 1 in
//  each).  Below 2^-6 fp8 is fixed-point, whose sums lose nothing; what a smaller
//  term 0 leaves is the other terms', which need the wide step for it.  Error
//  against float64, 1 x 1,024 tokens of 8 heads / 1 x 30,000 of 32 / 16 x 32K / 1 x
//  30,000 in chunks of 64 pages: sig 2^(e - 8), steps of 16, 4.6e-4 / 9.5e-4 / 6.8e-4 /
//  6.3e-4; 2^(e - 4), 16: 2.14e-4 / 2.10e-4 / 2.57e-4 / 5.2e-4; 2^(e - 4), 64: 2.14e-4 /
//  2.07e-4 / 2.02e-4 / 2.08e-4, the rounding of the output.
//  Value codes: two tr4 reads per 8-byte chunk ch give each lane the nibble
//  of channels 32ch + 2r, +1 for tokens 32q + 0..31; the nibble masked with
//  0x3 (even channel) or shifted down by 2 (odd) is the fp4 operand.
//  O[h][d] += 2 sig (C0 + C1 / 64 + C2 / 64^2) - sum_t P'_t z_t, C_t = row
//  4h + t of the MFMA output (fp4 value = code / 2).
constexpr float kTermStep = 1.0f / 64.0f;

template <int GQ>
__device__ __forceinline__ void pv_fp8_fp4(WaveState<GQ, false> &W, unsigned char *st, const f32x4 (&S)[2][4],
                                           const f32x4 &Yt, int lane)
{
    const int q = lane >> 4, r = lane & 15;
    i32x2 vr[4][2];  // [chunk][read]: tokens 32q + 16k + 0..15
#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
#pragma unroll
        for (int k = 0; k < 2; ++k)
            vr[ch][k] = tr4(st + kVal + W.trv[k][ch >> 1] + 8 * (ch & 1));

    const u32x4 vm0 = *(const u32x4 *)(st + kMeta + 512 + 4 * (4 * r));
    const u32x4 vm1 = *(const u32x4 *)(st + kMeta + 512 + 4 * (64 + 4 * r));
    // head q's score: rows 4q (rounded product) + 4q + 1 (residual), times
    // sm_scale log2(e) 2^24 / 4^a
    float sv[2][4];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            sv[cb][a] = (S[cb][a][0] + S[cb][a][1]) * (W.qk_c[0] * (kSub / (float)(1 << (2 * a))));
    float mx = sv[0][0];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            mx = fmaxf(mx, sv[cb][a]);
    const float yk = (Yt[0] + Yt[1]) * W.qk_c[0];
    mx = row_max16(mx) - yk;
    const float mn = fmaxf(W.m_run[0], mx);
    const float alpha = __builtin_amdgcn_exp2f(W.m_run[0] - mn);
    W.m_run[0] = mn;
    const float mny = mn + yk;

    float x[2][4], lsum = 0.0f, ysum = 0.0f, smax = 0.0f;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        const u32x4 vm = cb ? vm1 : vm0;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const half2v sz = as_h2(vm[a]);  // (scale, zero) of token 64cb + 4r + a
            const float sc = (float)sz[0], zp = (float)sz[1];
            const float pr = __builtin_amdgcn_exp2f(sv[cb][a] - mny);
            lsum += pr;
            x[cb][a] = pr * sc;
            ysum = __builtin_fmaf(x[cb][a], zp, ysum);
            smax = fmaxf(smax, sc);
        }
    }
    W.l_run[0] = W.l_run[0] * alpha + lsum;
    const float yv = row_sum16(ysum);
    smax = row_max16(smax);
    const float sig = __builtin_amdgcn_ldexpf(1.0f, __builtin_amdgcn_frexp_expf(smax) - 4);

    unsigned char *pb = st + kKlo;  // 16 rows x 128 fp8, over the consumed key codes
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        float *xc = x[cb];
        unsigned w0 = fp8x4(xc[0], xc[1], xc[2], xc[3], sig);
        fp8_residual(xc, w0, sig);
        unsigned w1 = fp8x4(xc[0], xc[1], xc[2], xc[3], sig * kTermStep);
        fp8_residual(xc, w1, sig * kTermStep);
        unsigned w2 = fp8x4(xc[0], xc[1], xc[2], xc[3], sig * (kTermStep * kTermStep));
        unsigned char *row = pb + 128 * (4 * q) + 64 * cb + 4 * r;
        *(unsigned *)(row) = w0;
        *(unsigned *)(row + 128) = w1;
        *(unsigned *)(row + 256) = w2;
    }

    // A operand: row r of the P' terms (row 4h + 3 is never written; its
    // output row is ignored).  Inline asm for the reason given in
    // compute_page (no wait for the other stage's prefetch).
    __builtin_amdgcn_s_setprio(1);
    i32x8 Ap;
    {
        u32x4 a0, a1;
        const unsigned addr = (unsigned)(uintptr_t)(pb + 128 * r + 16 * q);
        asm volatile("ds_read_b128 %0, %2\n\t"
                     "ds_read_b128 %1, %2 offset:64\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=v"(a0), "=v"(a1)
                     : "v"(addr)
                     : "memory");
        Ap = i32x8{(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
    }
    const float s2 = 2.0f * sig;
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
        const unsigned m = 0x33333333u;
        const u32x4 ev = {(unsigned)vr[ch][0][0] & m, (unsigned)vr[ch][0][1] & m, (unsigned)vr[ch][1][0] & m,
                          (unsigned)vr[ch][1][1] & m};
        const u32x4 od = {((unsigned)vr[ch][0][0] >> 2) & m, ((unsigned)vr[ch][0][1] >> 2) & m,
                          ((unsigned)vr[ch][1][0] >> 2) & m, ((unsigned)vr[ch][1][1] >> 2) & m};
        const f32x4 ce = mfma_fp8_fp4(Ap, ev);
        const f32x4 co = mfma_fp8_fp4(Ap, od);
        const float ve = __builtin_fmaf(ce[2], kTermStep * kTermStep, __builtin_fmaf(ce[1], kTermStep, ce[0]));
        const float vo = __builtin_fmaf(co[2], kTermStep * kTermStep, __builtin_fmaf(co[1], kTermStep, co[0]));
        W.o4[ch][0] = __builtin_fmaf(W.o4[ch][0], alpha, __builtin_fmaf(ve, s2, -yv));
        W.o4[ch][1] = __builtin_fmaf(W.o4[ch][1], alpha, __builtin_fmaf(vo, s2, -yv));
    }
    __builtin_amdgcn_s_setprio(0);
}

// One (page, head) record in LDS stage `st` -> QK, online softmax, PV.
// QK of the (page, head) record in stage `st`: S[cb][a] holds 4^a 2^-24
// sum_k A c for tokens 64 cb + 4 r + a on the head rows (rounded product and
// residual rows, or one row and a second chain at GQA 16), Yt the
// zero-point term Y per head row.
//
// bf16 metadata: the page's 128 scales and 128 zero points are converted to
// fp16 in the stage first, two of each pair of channels per lane (converted
// where they are read, each of the 16 lanes of a group would redo its
// 40 words: 120 VALU against 12).  q enters times 2^9 (qk_setup), so that the
// products and their residuals stay clear of fp16's subnormals.  A page
// whose largest scale is 16 or more, or below 2^-6, is brought to [8, 16) by a
// power of two, 1 / kmul, which the scores take back: scales decode with all
// their bits down to 2^-12 of 2^-6 or of the page's largest (fp16 subnormals
// below).
template <int GQ, bool BF>
__device__ __forceinline__ void page_qk(const WaveState<GQ, BF> &W, unsigned char *st, int lane, int Dk,
                                        f32x4 (&S)[2][4], f32x4 &Yt, float &kmul)
{
    kmul = 1.0f;
    if constexpr (BF) {
        // lanes 0-31: scales of channels 4 lane .. + 3, lanes 32-63: zero
        // points (inline asm: see compute_page)
        unsigned w0, w1;
        {
            uint64_t w;
            const unsigned addr = (unsigned)(uintptr_t)(st + kMeta + 8 * lane);
            asm volatile("ds_read_b64 %0, %1\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=v"(w)
                         : "v"(addr)
                         : "memory");
            w0 = (unsigned)w, w1 = (unsigned)(w >> 32);
        }
        const unsigned mag = max(max(w0 << 16 & 0x7fffffffu, w0 & 0x7fff0000u), max(w1 << 16 & 0x7fffffffu, w1 & 0x7fff0000u));
        float f0 = bf_lo(w0), f1 = bf_hi(w0), f2 = bf_lo(w1), f3 = bf_hi(w1);
        const uint64_t big = __ballot(lane < 32 && mag >= 0x41800000u), mid = __ballot(lane < 32 && mag >= 0x3c800000u);
        if (__builtin_expect(big != 0 || mid == 0, 0)) {
            int e = lane < 32 ? (int)(mag >> 23) : 0;   // biased exponent
            for (int off = 1; off < 64; off <<= 1)
                e = max(e, __shfl_xor(e, off));
            const int k = max(e - 130, -126);           // the largest scale in [2^3, 2^4)
            kmul = __builtin_amdgcn_ldexpf(1.0f, k);
            if (lane < 32) {
                f0 = __builtin_amdgcn_ldexpf(f0, -k), f1 = __builtin_amdgcn_ldexpf(f1, -k);
                f2 = __builtin_amdgcn_ldexpf(f2, -k), f3 = __builtin_amdgcn_ldexpf(f3, -k);
            }
        }
        *(uint2 *)(st + kMeta + 8 * lane) = make_uint2(pack_rtz(f0, f1), pack_rtz(f2, f3));
    }
    const int q = lane >> 4;

    // ---------------- operands from LDS, issued together
    u32x4 ks[4], kz[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        ks[s] = *(const u32x4 *)(st + kMeta + 2 * (32 * s + 8 * q));
        kz[s] = *(const u32x4 *)(st + kMeta + 256 + 2 * (32 * s + 8 * q));
    }
    i32x2 kraw[4][2], hraw[2];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        kraw[s][0] = tr8(st + kKlo + 1024 * s + W.tr_base0);
        kraw[s][1] = tr8(st + kKlo + 1024 * s + W.tr_base1);
    }
    _Float16 ksh[8];
    if (Dk > 0) {
        hraw[0] = tr8(st + kKhi + W.tr_base0);
        hraw[1] = tr8(st + kKhi + W.tr_base1);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            ksh[i] = *(const _Float16 *)(st + kMeta + 2 * W.hch[i]);
    }

    // ---------------- QK A operands q s_k (rounded product and residual
    // rows, qk_residual; GQA 16: residual operands Al for a second chain)
    // and the bias tile Y = sum A z (per head row, broadcast over token
    // columns)
    half8 A[4], Ahi, Al[4], Alhi;
    Yt = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        u32x4 av;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            av[j] = as_u(as_h2(W.qv[s][j]) * as_h2(ks[s][j]));
        if constexpr (GQ == 16) {
            u32x4 lo = av;
            qk_residual(lo, W.qv[s], ks[s], ~0ull);
            Al[s] = __builtin_bit_cast(half8, lo);
            Yt = mfma(Al[s], __builtin_bit_cast(half8, kz[s]), Yt);
        } else {
            qk_residual(av, W.qv[s], ks[s], kResidualLanes<GQ>);
        }
        A[s] = __builtin_bit_cast(half8, av);
        Yt = mfma(A[s], __builtin_bit_cast(half8, kz[s]), Yt);
    }
    if (Dk > 0) {
        u32x4 av, sh;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            half2v h;
            h[0] = ksh[2 * j];
            h[1] = ksh[2 * j + 1];
            sh[j] = as_u(h);
            av[j] = as_u(as_h2(W.qvh[j]) * h);
        }
        if constexpr (GQ == 16) {
            u32x4 lo = av;
            qk_residual(lo, W.qvh, sh, ~0ull);
            Alhi = __builtin_bit_cast(half8, lo);
        } else {
            qk_residual(av, W.qvh, sh, kResidualLanes<GQ>);
        }
        Ahi = __builtin_bit_cast(half8, av);
    }

    // The MFMA blocks run at raised wave priority: the other wave of the SIMD
    // is then most often in its VALU / memory phase, and the matrix core
    // stays fed (measured: 1.5-2 us less per launch at config 3).
    __builtin_amdgcn_s_setprio(1);
    // ---------------- QK token tiles: S[cb][a] covers tokens 64cb + 4r + a.
    // S[cb][a] ends at 4^a 2^-24 sum_k A c; the softmax scales it back and
    // subtracts the zero-point term Y.
#pragma unroll
    for (int a = 0; a < 4; ++a)
        S[0][a] = S[1][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const auto rc = page_codes<BF>(kraw[s][cb]);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const half8 kc = slot_codes(rc, a);
                S[cb][a] = mfma(A[s], kc, S[cb][a]);
                if constexpr (GQ == 16)
                    S[cb][a] = mfma(Al[s], kc, S[cb][a]);
            }
        }
    if (Dk > 0) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const auto rc = page_codes<BF>(hraw[cb]);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const half8 kc = slot_codes(rc, a);
                S[cb][a] = mfma(Ahi, kc, S[cb][a]);
                if constexpr (GQ == 16)
                    S[cb][a] = mfma(Alhi, kc, S[cb][a]);
            }
        }
    }

    __builtin_amdgcn_s_setprio(0);
}

// bf16: online softmax and PV of one page with fp16 MFMAs and P'
// = p * s_t in two fp16 terms, the rounded value and its rounded remainder: 23
// bits of the 24 that the generic kernel's fp32 probabilities have.  (Rounded
// toward zero, all terms lean the same way, and where a flat softmax cancels
// sum P' c against the zero points' sum P' z the output moved: 25,600 tokens at a
// fifth of the usual scores 0.58 % further from float64 than the generic
// kernel, 0.0006 % so.)  P' enters scaled by 2^(15 - e), s_max < 2^e the page's largest value scale, so
// it stays below 2^15 whatever range bf16 scales have.  GQA 4 and 8 put the
// terms on the first two MFMA rows of each head, GQA 16 runs a second chain; a
// page's output tiles start at zero and are folded into O in fp32.  (GQA 4 on
// the fp8 x fp4 MFMAs of the fp16 instance, with a fourth term, kept errors of
// 4-6e-4 where the generic kernel has 2e-4: those sums hold too few bits.)
template <int GQ>
__device__ __forceinline__ void pv_split(WaveState<GQ, true> &W, unsigned char *st, const f32x4 (&S)[2][4],
                                         const f32x4 &Yt, float kmul, int lane)
{
    constexpr int HPL = GQ / 4;
    constexpr int RSTEP = 4 / HPL;
    const int q = lane >> 4, r = lane & 15;
    i32x2 vraw[4][2];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        vraw[s][0] = tr8(st + kVal + 1024 * s + W.tr_base0);
        vraw[s][1] = tr8(st + kVal + 1024 * s + W.tr_base1);
    }
    const u32x4 vm0 = *(const u32x4 *)(st + kMeta + 512 + 4 * (4 * r));
    const u32x4 vm1 = *(const u32x4 *)(st + kMeta + 512 + 4 * (64 + 4 * r));
    float smax = 0.0f;
#pragma unroll
    for (int a = 0; a < 4; ++a)
        smax = fmaxf(smax, fmaxf(bf_lo(vm0[a]), bf_lo(vm1[a])));
    const int e15 = __builtin_amdgcn_frexp_expf(row_max16(smax)) - 15;
    const float down = __builtin_amdgcn_ldexpf(1.0f, -e15);
    float alpha[HPL], yv[HPL];
#pragma unroll
    for (int j = 0; j < HPL; ++j) {
        const int ri = j * RSTEP;
        const float qk_c = W.qk_c[j] * kmul;
        float sv[2][4];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                sv[cb][a] = (GQ == 16 ? S[cb][a][ri] : S[cb][a][ri] + S[cb][a][ri + 1]) *
                            (qk_c * (kSub / slot_weight<true>(a)));
        float mx = sv[0][0];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                mx = fmaxf(mx, sv[cb][a]);
        const float yk = (GQ == 16 ? Yt[ri] : Yt[ri] + Yt[ri + 1]) * qk_c;
        mx = row_max16(mx) - yk;
        const float mn = fmaxf(W.m_run[j], mx);
        alpha[j] = __builtin_amdgcn_exp2f(W.m_run[j] - mn);
        W.m_run[j] = mn;
        const float mny = mn + yk;
        float lsum = 0.0f, ysum = 0.0f;
        const int h = q * HPL + j;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const u32x4 vm = cb ? vm1 : vm0;
            float x[4];
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const float pr = __builtin_amdgcn_exp2f(sv[cb][a] - mny);
                lsum += pr;
                x[a] = pr * bf_lo(vm[a]);
                ysum = __builtin_fmaf(x[a], bf_hi(vm[a]), ysum);
                x[a] *= down;
            }
            const unsigned h0 = pack_h2(x[0], x[1]), h1 = pack_h2(x[2], x[3]);
            const unsigned l0 = pack_h2(x[0] - (float)as_h2(h0)[0], x[1] - (float)as_h2(h0)[1]);
            const unsigned l1 = pack_h2(x[2] - (float)as_h2(h1)[0], x[3] - (float)as_h2(h1)[1]);
            // rows over the consumed key codes (GQA 16: the second terms over the value codes, read above)
            unsigned char *hi = st + kKlo + 256 * (16 / GQ * h) + 2 * (64 * cb + 4 * r);
            *(uint2 *)hi = make_uint2(h0, h1);
            *(uint2 *)(GQ == 16 ? hi + (kVal - kKlo) : hi + 256) = make_uint2(l0, l1);
        }
        W.l_run[j] = W.l_run[j] * alpha[j] + lsum;
        yv[j] = row_sum16(ysum);
    }
    // A operand: row r of the terms (inline asm for the reason given in compute_page)
    __builtin_amdgcn_s_setprio(1);
    half8 Ap[4], Al[GQ == 16 ? 4 : 1];
    {
        const unsigned addr = (unsigned)(uintptr_t)(st + kKlo + 256 * r + 16 * q);
        asm volatile("ds_read_b128 %0, %4\n\t"
                     "ds_read_b128 %1, %4 offset:64\n\t"
                     "ds_read_b128 %2, %4 offset:128\n\t"
                     "ds_read_b128 %3, %4 offset:192\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=&v"(Ap[0]), "=&v"(Ap[1]), "=&v"(Ap[2]), "=&v"(Ap[3])
                     : "v"(addr)
                     : "memory");
        if constexpr (GQ == 16) {
            const unsigned addr_l = addr + (kVal - kKlo);
            asm volatile("ds_read_b128 %0, %4\n\t"
                         "ds_read_b128 %1, %4 offset:64\n\t"
                         "ds_read_b128 %2, %4 offset:128\n\t"
                         "ds_read_b128 %3, %4 offset:192\n\t"
                         "s_waitcnt lgkmcnt(0)"
                         : "=&v"(Al[0]), "=&v"(Al[1]), "=&v"(Al[2]), "=&v"(Al[3])
                         : "v"(addr_l)
                         : "memory");
        }
    }
    const float up = __builtin_amdgcn_ldexpf(kSub, e15);  // tile a holds slot_weight(a) 2^-24 2^-e15 sum P' c
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        f32x4 T[4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
            T[a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const auto rc = page_codes<true>(vraw[s][cb]);
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const half8 vc = slot_codes(rc, a);
                T[a] = mfma(Ap[s], vc, T[a]);
                if constexpr (GQ == 16)
                    T[a] = mfma(Al[s], vc, T[a]);
            }
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int j = 0; j < HPL; ++j) {
                const float t = GQ == 16 ? T[a][j * RSTEP] : T[a][j * RSTEP] + T[a][j * RSTEP + 1];
                W.ob[cb][a][j] = __builtin_fmaf(W.ob[cb][a][j], alpha[j],
                                                __builtin_fmaf(t, up * (1.0f / slot_weight<true>(a)), -yv[j]));
            }
    }
    __builtin_amdgcn_s_setprio(0);
}

template <int GQ, bool BF>
__device__ __forceinline__ void compute_page(WaveState<GQ, BF> &W, unsigned char *st, int lane, int Dk)
{
    constexpr int HPL = GQ / 4;
    constexpr int RSTEP = 4 / HPL;  // accumulator register of head slot j = j * RSTEP
    const int q = lane >> 4, r = lane & 15;
    f32x4 S[2][4], Yt;
    float kmul;
    page_qk<GQ, BF>(W, st, lane, Dk, S, Yt, kmul);
    if constexpr (BF) {
        pv_split<GQ>(W, st, S, Yt, kmul, lane);
        return;
    } else if constexpr (GQ == 4) {
        pv_fp8_fp4(W, st, S, Yt, lane);
        return;
    }
    // value codes for PV, issued before the softmax so they arrive meanwhile
    i32x2 vraw[4][2];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        vraw[s][0] = tr8(st + kVal + 1024 * s + W.tr_base0);
        vraw[s][1] = tr8(st + kVal + 1024 * s + W.tr_base1);
    }

    // ---------------- online softmax and P' = p * s_t (fp16) with the PV bias.
    // P' goes to the key-low region of this stage, whose codes are consumed.
    _Float16 *pbuf = (_Float16 *)(st + kKlo);
    const u32x4 vm0 = *(const u32x4 *)(st + kMeta + 512 + 4 * (4 * r));
    const u32x4 vm1 = *(const u32x4 *)(st + kMeta + 512 + 4 * (64 + 4 * r));
    float alpha[HPL], yv[HPL];
#pragma unroll
    for (int j = 0; j < HPL; ++j) {
        const int ri = j * RSTEP;
        // the head's score: its rounded-product row plus (GQA 8) its residual
        // row, times sm_scale log2(e) 2^24 / 4^a
        float sv[2][4];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                sv[cb][a] = (GQ == 16 ? S[cb][a][ri] : S[cb][a][ri] + S[cb][a][ri + 1]) *
                            (W.qk_c[0] * (kSub / (float)(1 << (2 * a))));
        float mx = sv[0][0];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                mx = fmaxf(mx, sv[cb][a]);
        // scores are sv - Y: the max over the row and the exponents absorb Y
        const float yk = (GQ == 16 ? Yt[ri] : Yt[ri] + Yt[ri + 1]) * W.qk_c[0];
        mx = row_max16(mx) - yk;
        const float mn = fmaxf(W.m_run[j], mx);
        alpha[j] = __builtin_amdgcn_exp2f(W.m_run[j] - mn);
        W.m_run[j] = mn;
        const float mny = mn + yk;
        float lsum = 0.0f, ysum = 0.0f;
        const int h = q * HPL + j;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const u32x4 vm = cb ? vm1 : vm0;
            const float p0v = __builtin_amdgcn_exp2f(sv[cb][0] - mny);
            const float p1v = __builtin_amdgcn_exp2f(sv[cb][1] - mny);
            const float p2v = __builtin_amdgcn_exp2f(sv[cb][2] - mny);
            const float p3v = __builtin_amdgcn_exp2f(sv[cb][3] - mny);
            lsum += (p0v + p1v) + (p2v + p3v);
            // (scale, zero) pairs of tokens 64cb + 4r + {0..3}
            const half2v sv01 = as_h2(__builtin_amdgcn_perm(vm[1], vm[0], 0x05040100u));
            const half2v zv01 = as_h2(__builtin_amdgcn_perm(vm[1], vm[0], 0x07060302u));
            const half2v sv23 = as_h2(__builtin_amdgcn_perm(vm[3], vm[2], 0x05040100u));
            const half2v zv23 = as_h2(__builtin_amdgcn_perm(vm[3], vm[2], 0x07060302u));
            const half2v a01 = as_h2(pack_h2(p0v, p1v)) * sv01;
            const half2v a23 = as_h2(pack_h2(p2v, p3v)) * sv23;
            ysum = __builtin_amdgcn_fdot2(a01, zv01, ysum, false);
            ysum = __builtin_amdgcn_fdot2(a23, zv23, ysum, false);
            *(uint2 *)(pbuf + h * 128 + 64 * cb + 4 * r) = make_uint2(as_u(a01), as_u(a23));
        }
        W.l_run[j] = W.l_run[j] * alpha[j] + lsum;
        yv[j] = row_sum16(ysum);
    }

    // ---------------- PV, in the subnormal codes' units 4^a 2^-24:
    // O_a = O_a * alpha - 4^a 2^-24 sum P' z + P' C_a
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int j = 0; j < HPL; ++j)
                W.O[cb][a][j * RSTEP] =
                    W.O[cb][a][j * RSTEP] * alpha[j] - yv[j] * ((float)(1 << (2 * a)) / kSub);
    // P' rows are read with inline asm: the compiler cannot tell this stage
    // apart from the one the next page is streaming into and would otherwise
    // wait for that prefetch (vmcnt(0)) here.  LDS executes a wave's
    // operations in order, so the reads see the writes above; lgkmcnt(0)
    // makes their results available.
    __builtin_amdgcn_s_setprio(1);
    half8 Ap[4];
    {
        const unsigned addr = (unsigned)(uintptr_t)(pbuf + W.prow * 128 + 8 * q);
        asm volatile("ds_read_b128 %0, %4\n\t"
                     "ds_read_b128 %1, %4 offset:64\n\t"
                     "ds_read_b128 %2, %4 offset:128\n\t"
                     "ds_read_b128 %3, %4 offset:192\n\t"
                     "s_waitcnt lgkmcnt(0)"
                     : "=v"(Ap[0]), "=v"(Ap[1]), "=v"(Ap[2]), "=v"(Ap[3])
                     : "v"(addr)
                     : "memory");
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
            const RawCodes rc = raw_codes(vraw[s][cb]);
            W.O[cb][0] = mfma(Ap[s], codes_to_half8<0>(rc), W.O[cb][0]);
            W.O[cb][1] = mfma(Ap[s], codes_to_half8<1>(rc), W.O[cb][1]);
            W.O[cb][2] = mfma(Ap[s], codes_to_half8<2>(rc), W.O[cb][2]);
            W.O[cb][3] = mfma(Ap[s], codes_to_half8<3>(rc), W.O[cb][3]);
        }
    __builtin_amdgcn_s_setprio(0);
}

// Global loads that start a page segment of pair (b, kh): boost_idx of the
// lane's two channels, the lane's slice of the q rows and the ids of pages
// p0 .. p0 + 63 (below p1).  Issued by the caller, so the kernel can start
// them for its first segment before its plan is known.
struct SegSetup {
    int bi0, bi1;
    u32x4 qraw[4];
    int ids;
};

template <int GQ>
__device__ __forceinline__ SegSetup load_setup(const DecodeParams &p, int b, int kh, int p0, int p1)
{
    constexpr int ROWS_PER_HEAD = 16 / GQ;
    const int lane = lane_id(), q = lane >> 4, r = lane & 15;
    SegSetup s;
    s.bi0 = p.boost_idx[kh * 128 + lane];
    s.bi1 = p.boost_idx[kh * 128 + 64 + lane];
    const uint16_t *qrow = p.q + b * p.q_s_seq + q_head(p, kh, r / ROWS_PER_HEAD) * p.q_s_head;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        s.qraw[i] = *(const u32x4 *)(qrow + 32 * i + 8 * q);
    s.ids = p0 + lane < min(p1, p.max_pages) ? p.block_table[b * p.bt_stride + p0 + lane] : 0;
    return s;
}

// QK operand state of pair (b, kh) for its pages (page_qk): the static fp16
// q halves, the high-bit rows' q values and channels, the tr8 offsets and
// the score scale.  scratch: LDS the wave may overwrite (256 + GQ * 256 B),
// free again on return.
//
// bf16: q of a head enters as q 2^(9 - E) in fp16, 2^E the power of two just
// above its largest |q| (exact for every channel within 2^-23 of that), and
// the scores take 2^(E - 9) back: with page scales below 16 the operands stay
// below 2^13, 2^15 on the high-bit rows.
template <int GQ, bool BF, bool PAIR = false>
__device__ __forceinline__ void qk_setup(WaveState<GQ, BF> &W, const DecodeParams &p, int b, int kh, const SegSetup &su,
                                         unsigned char *scratch, int lane, int Dk)
{
    constexpr int ROWS_PER_HEAD = 16 / GQ;
    const int q = lane >> 4, r = lane & 15;
    // rank -> channel map of this KV head (inverse of boost_idx) and the q
    // rows of the group, staged in scratch before any page lands there; the
    // boosted channels' q values are then read from LDS, not by a global load
    // that would wait on the map (one memory round trip before the first
    // page's loads).
    const bool head_row = (r % ROWS_PER_HEAD) == 0;
    const int hr = r / ROWS_PER_HEAD;  // head of MFMA row r
    int *rank_chan = (int *)scratch;
    _Float16 *q_lds = (_Float16 *)(scratch + 256);  // [GQ][128]
    if (lane < 32)
        rank_chan[lane] = 0;
    wave_sync<PAIR>();
    if (su.bi0 < Dk)
        rank_chan[su.bi0] = lane;
    if (su.bi1 < Dk)
        rank_chan[su.bi1] = 64 + lane;
    if (GQ <= 8 && head_row) {  // (GQA 16 keeps the global loads: staged, its page loop waited on the prefetch)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            *(u32x4 *)(q_lds + hr * 128 + 32 * s + 8 * q) = su.qraw[s];
    }

    wave_sync<PAIR>();

    // Static half of the QK A operand: 2^-3 q (fp16) of the lane's 8 channels
    // of every K-step on the two rows of each head (the product with the key
    // scale and its residual, qk_residual), zero on the other rows.
    // 2^3 sm_scale log2(e) scales the scores, so A stays exact; the 2^-3
    // keeps fp16 products finite up to |q s_k| < 2^19 (2^17 on the high-bit
    // rows, whose q is also multiplied by 4).
    W.prow = hr;
    const bool qk_row = GQ == 16 || (r % ROWS_PER_HEAD) < 2;
    if constexpr (BF) {
        unsigned mag = 0;   // largest |q| of MFMA row r's head, as bits
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                mag = max(mag, max(su.qraw[s][j] << 16 & 0x7fffffffu, su.qraw[s][j] & 0x7fff0000u));
        mag = max(mag, (unsigned)__shfl_xor((int)mag, 16));
        mag = max(mag, (unsigned)__shfl_xor((int)mag, 32));
        const int E = (int)(mag >> 23) - 126;
#pragma unroll
        for (int j = 0; j < GQ / 4; ++j)   // head slot j of this lane: MFMA row (q HPL + j) ROWS_PER_HEAD
            W.qk_c[j] = __builtin_amdgcn_ldexpf(p.sm_scale * kLog2e, __shfl(E, (q * (GQ / 4) + j) * ROWS_PER_HEAD) - 9);
#pragma unroll
        for (int i = 0; i < 8; ++i)
            W.hch[i] = rank_chan[8 * q + i];
        const uint16_t *qrow = p.q + b * p.q_s_seq + q_head(p, kh, hr) * p.q_s_head;
        const uint16_t *q16 = (const uint16_t *)q_lds;
        const int pre = 9 - E;
        float qh[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
            qh[i] = __builtin_amdgcn_ldexpf(bf2f(GQ <= 8 ? q16[hr * 128 + W.hch[i]] : qrow[W.hch[i]]), pre + 2);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                W.qv[s][j] = qk_row ? pack_h2(__builtin_amdgcn_ldexpf(bf_lo(su.qraw[s][j]), pre),
                                              __builtin_amdgcn_ldexpf(bf_hi(su.qraw[s][j]), pre)) : 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r0 = 8 * q + 2 * j;
            W.qvh[j] = qk_row ? pack_h2(r0 < Dk ? qh[2 * j] : 0.0f, r0 + 1 < Dk ? qh[2 * j + 1] : 0.0f) : 0u;
        }
    } else {
        W.qk_c[0] = p.sm_scale * kLog2e * kQInv;
        const u32x4 *qraw = su.qraw;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            W.hch[i] = rank_chan[8 * q + i];
        _Float16 qh[8];
        const uint16_t *qrow = p.q + b * p.q_s_seq + q_head(p, kh, hr) * p.q_s_head;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            qh[i] = GQ <= 8 ? q_lds[hr * 128 + W.hch[i]] : *(const _Float16 *)(qrow + W.hch[i]);
        const half2v pre = {(_Float16)kQPre, (_Float16)kQPre};
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                W.qv[s][j] = qk_row ? as_u(as_h2(qraw[s][j]) * pre) : 0u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float inv = qk_row ? 4.0f * kQPre : 0.0f;  // high bits weigh 4 (exact in fp16)
            const int r0 = 8 * q + 2 * j;
            W.qvh[j] = pack_h2(r0 < Dk ? (float)qh[2 * j] * inv : 0.0f,
                               r0 + 1 < Dk ? (float)qh[2 * j + 1] * inv : 0.0f);
        }
    }
    // tr8 source address of this lane inside a 128 x 32 B region: rows
    // 8q + rho(r/2) (rho swaps the middle pair so extracted halves come out in
    // natural order), byte column 8 (r & 1) of chunk cb ^ (q & 1).
    {
        const int i = r >> 1;
        const int rho = (i & 4) | ((i & 1) << 1) | ((i >> 1) & 1);
        const int tr_row = 8 * q + rho;
        W.tr_base0 = 32 * tr_row + 16 * (0 ^ (q & 1)) + 8 * (r & 1);
        W.tr_base1 = 32 * tr_row + 16 * (1 ^ (q & 1)) + 8 * (r & 1);
    }
}

// Pages [p0, p1) of pair (b, kh) folded into partial t: row t * GQ + h
// holds query head kh * GQ + h.  A page count outside [0, max_pages] or a
// page id outside the pool makes the partial NaN; no pages leave an empty
// partial (m = -inf, l = 0, O = 0).
// PAIR: su.ids holds the block table's first 64 entries instead of those from p0.
template <int GQ, bool BF, bool PAIR = false>
__device__ __forceinline__ void page_segment(const DecodeParams &p, unsigned char *stage0, unsigned char *stage1,
                                             int b, int kh, int np_raw, int p0, int p1, int64_t t, const SegSetup &su)
{
    constexpr int HPL = GQ / 4;
    constexpr int RSTEP = 4 / HPL;
    // lane-derived offsets are rebuilt per segment (the asm hides the lane
    // id): kept across the caller's segment loop they would be spilled
    int lane = lane_id();
    asm volatile("" : "+v"(lane));
    const int q = lane >> 4, r = lane & 15;
    const int Dk = p.Dk;
    // segment bounds come out of VALU divisions: keep the loop control scalar
    b = __builtin_amdgcn_readfirstlane(b);
    kh = __builtin_amdgcn_readfirstlane(kh);
    np_raw = __builtin_amdgcn_readfirstlane(np_raw);
    p0 = __builtin_amdgcn_readfirstlane(p0);
    p1 = __builtin_amdgcn_readfirstlane(p1);
    bool poison = np_raw < 0 || np_raw > p.max_pages;
    if (poison)
        p1 = p0;
    else if (p1 > np_raw)
        p1 = np_raw;

    WaveState<GQ, BF> W;
    qk_setup<GQ, BF, PAIR>(W, p, b, kh, su, stage1, lane, Dk);
    // tr4 offsets of value rows R = 32q + 16k + r (GQA 4): 16-byte chunk c of
    // row R sits at 32 R + 16 (c ^ ((R >> 3) & 1)) in the stage.
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int R = 32 * q + 16 * k + r;
            W.trv[k][c] = 32 * R + 16 * (c ^ ((R >> 3) & 1));
        }
#pragma unroll
    for (int j = 0; j < HPL; ++j) {
        W.m_run[j] = -__builtin_inff();
        W.l_run[j] = 0.0f;
    }
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int a = 0; a < 4; ++a)
            W.O[cb][a] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (BF) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int j = 0; j < HPL; ++j)
                    W.ob[cb][a][j] = 0.0f;
    }
#pragma unroll
    for (int ch = 0; ch < 4; ++ch)
        W.o4[ch][0] = W.o4[ch][1] = 0.0f;
    wave_sync<PAIR>();  // stage1 reads done before the next page lands there

    // Page ids, 64 at a time (one per lane), read back with v_readlane so no
    // page waits on a dependent global load; pages are asked for in order,
    // so the next 64 ids are fetched when the first page past them is.  That
    // fetch waits for itself at once (and for the page in flight, once per 64
    // pages): left pending, it would make the compiler wait for every
    // outstanding load before each page's v_readlane.
    const int32_t *bt = p.block_table + b * p.bt_stride;
    int chunk0 = PAIR ? 0 : p0;
    int ids = su.ids;
    auto page_ok = [&](int32_t page) { return page >= 0 && page < p.num_pool_pages; };
    auto page_at = [&](int pi) -> int32_t {
        while (PAIR && pi - chunk0 >= 128)
            chunk0 += 64;
        if (pi - chunk0 >= 64) {
            chunk0 += 64;
            ids = chunk0 + lane < p1 ? bt[chunk0 + lane] : 0;
            wait_vmcnt<0>();
        }
        return __builtin_amdgcn_readlane(ids, pi - chunk0);
    };

    if (p0 < p1) {
        const int32_t page = page_at(p0);
        if (!page_ok(page))
            poison = true;
        else
            issue_page(stage0, page_src(p, (int64_t)page * p.Hkv + kh), lane, Dk);
    }
    // Pages alternate between the stages; each step prefetches the next page
    // into the other stage, waits for its own page's loads, and computes.
    for (int pi = p0; pi < p1 && !poison; pi += 2) {
        {
            bool next = false;
            if (pi + 1 < p1) {
                const int32_t page = page_at(pi + 1);
                if (!page_ok(page))
                    poison = true;
                else {
                    issue_page(stage1, page_src(p, (int64_t)page * p.Hkv + kh), lane, Dk);
                    next = true;
                }
            }
            if (next)
                wait_vmcnt<kLoadsPerPage>();
            else
                wait_vmcnt<0>();
            compute_page<GQ, BF>(W, stage0, lane, Dk);
            if (!next)
                break;
        }
        {
            bool next = false;
            if (pi + 2 < p1) {
                const int32_t page = page_at(pi + 2);
                if (!page_ok(page))
                    poison = true;
                else {
                    issue_page(stage0, page_src(p, (int64_t)page * p.Hkv + kh), lane, Dk);
                    next = true;
                }
            }
            if (next)
                wait_vmcnt<kLoadsPerPage>();
            else
                wait_vmcnt<0>();
            compute_page<GQ, BF>(W, stage1, lane, Dk);
        }
    }
    if (poison)
        wait_vmcnt<0>();  // no load may still be writing LDS when the wave retires

    // ---------------------------------------------------- write partial
#pragma unroll
    for (int j = 0; j < HPL; ++j) {
        const float l = row_sum16(W.l_run[j]);
        const int h = q * HPL + j;
        const int64_t row = t * GQ + h;
        float *o = p.ws_o + row * 128;
        if constexpr (GQ == 4 && !BF) {
            // o4[ch][e] is O of channel 32ch + 2r + e
#pragma unroll
            for (int ch = 0; ch < 4; ++ch) {
                float2 v = make_float2(W.o4[ch][0], W.o4[ch][1]);
                if (poison)
                    v = make_float2(__builtin_nanf(""), __builtin_nanf(""));
                *(float2 *)(o + 32 * ch + 2 * r) = v;
            }
        } else {
#pragma unroll
            for (int cb = 0; cb < 2; ++cb) {
                // output tile a holds 4^a 2^-24 O for channels 64cb + 4r + a
                float4 v = make_float4(W.O[cb][0][j * RSTEP] * kSub, W.O[cb][1][j * RSTEP] * (kSub * 0.25f),
                                       W.O[cb][2][j * RSTEP] * (kSub * 0.0625f),
                                       W.O[cb][3][j * RSTEP] * (kSub * 0.015625f));
                if constexpr (BF)
                    v = make_float4(W.ob[cb][0][j], W.ob[cb][1][j], W.ob[cb][2][j], W.ob[cb][3][j]);
                if (poison)
                    v = make_float4(__builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""), __builtin_nanf(""));
                *(float4 *)(o + 64 * cb + 4 * r) = v;
            }
        }
        if (r == 0) {
            p.ws_ml[2 * row] = poison ? __builtin_nanf("") : W.m_run[j];
            p.ws_ml[2 * row + 1] = l;
        }
    }
}

// Empty partial t (m = -inf, l = 0, O = 0) for the slot between a pair's
// pages and its FP16 tokens when a wave boundary falls exactly there.
template <int GQ>
__device__ __forceinline__ void empty_partial(const DecodeParams &p, int64_t t)
{
    const int lane = lane_id();
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
        const int64_t row = t * GQ + g;
        *(float2 *)(p.ws_o + row * 128 + 2 * lane) = make_float2(0.0f, 0.0f);
        if (lane == 0) {
            p.ws_ml[2 * row] = -__builtin_inff();
            p.ws_ml[2 * row + 1] = 0.0f;
        }
    }
}

// Inclusive prefix sum over the 64 lanes.
__device__ __forceinline__ int wave_incl_scan(int v, int lane)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(v, off);
        if (lane >= off)
            v += y;
    }
    return v;
}

__device__ __forceinline__ int64_t uniform64(int64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}

// FP16-region tokens of sequence b: sinks and the value tail (the key-only
// pages' tokens and the key tail); none for a bad sequence.
__device__ __forceinline__ int seq_tokens(const DecodeParams &p, int b)
{
    const SeqLens L = seq_lens(p, b);
    return L.ns + L.nv;
}

// Sequence b as the unit plan sees it (all fields wave-uniform).
struct SeqUnits {
    int b, np_raw, npu, fu;  // raw page count, page units, FP16 units (per pair)
    int64_t base;            // first unit of pair (b, 0)
};

// Units [u0, u1) of wave w: floor(w U / W) = w Q + (w R) / W with Q = U / W,
// R = U % W (w R < W^2 < 2^32); one 32-bit division when U fits.
__device__ __forceinline__ void wave_units(int64_t U, int W, int w, int64_t &u0, int64_t &u1)
{
    uint64_t Q;
    uint32_t R;
    if (U <= 0xffffffffll) {
        Q = (uint32_t)U / (uint32_t)W;
        R = (uint32_t)U - (uint32_t)Q * (uint32_t)W;
    } else {
        Q = (uint64_t)U / (uint64_t)W;
        R = (uint32_t)((uint64_t)U - Q * (uint64_t)W);
    }
    u0 = (int64_t)(Q * (uint64_t)w + ((uint32_t)w * R) / (uint32_t)W);
    u1 = (int64_t)(Q * (uint64_t)(w + 1) + ((uint32_t)(w + 1) * R) / (uint32_t)W);
}

// The kernel's parameters read again from the kernarg segment (pp: the
// kernel's own __builtin_amdgcn_kernarg_segment_ptr(), which is only defined
// inside the kernel and so is passed to functions that are not inlined).  The
// segment loop below calls this in each branch so that only the plan state
// stays live from one segment to the next; the empty asm hides the pointer's
// value so the loads cannot be hoisted out of the loop.
typedef const __attribute__((address_space(4))) DecodeParams *KernargParams;
__device__ __forceinline__ DecodeParams kernel_params(KernargParams pp)
{
    asm volatile("" : "+s"(pp));
    DecodeParams r;
    __builtin_memcpy(&r, (const void *)pp, sizeof(r));
    return r;
}

// FP16-region tokens [lo, hi) of pair (b, kh), 32 per step, as partial t.  The
// region is the sinks, then the tokens of the key-only pages P_v .. P_k - 1 (an
// independent value stream: their keys are quantised, their values are the
// first (P_k - P_v) G rows of the value tail), then the key tail, whose
// values follow in the value tail; with one stream the middle part is empty.
// A step's rows stream into the two LDS stages with global_load_lds (no
// registers hold data in flight): K chunk c of token row n is stored at
// chunk c ^ (n & 15), so the 16 rows one MFMA B read touches hit 16
// different bank groups; V rows lie as they are.  QK: f16 or bf16 MFMAs
// with head h on rows 16 / GQ h .. (A = q, B = K rows, exact products; scores
// times sm_scale log2(e) in fp32), so a lane holds the scores of its group's
// GQ / 4 heads; for a key-only page the page path's exact QK (page_qk) writes
// the page's scores to kst once and its steps read them back.  Base-2 online
// softmax per head with DPP row reductions.  PV: fp32 MFMAs of 4 heads x 1 token
// x 4 channels in 16 blocks, whose columns are the lanes in order: a lane holds a
// channel pair, one MFMA does a token, 4 heads and one channel of every pair.
// One register holds P of 16 tokens x 4 heads, a token's block broadcast to all.
// (16-bit terms of P in 16 x 16 x 32 MFMAs were as fast, but their products are
// aligned to the largest and truncated: rms error of the output against 64 bits
// 8e-8 where fp32 has 2.4e-8.)
// Steps do not cross from sinks into key-only pages, nor out of one.  The
// partial's m is NaN if a key-only page id lies outside the pool.
// Bound by its chain of loads, MFMAs and softmax per step, not by the units:
// PV on the VALU (lane = channel pair, fp32 P) and four scores per lane for
// every group took 13.8 us where this takes 12.6 (1 x 1,024 tokens, split and
// merge) and 24.6 against 23.3 (8 x 3-9K tokens, bf16).  q is loaded
// again by every step: kept, with 16-bit terms, the split kernel spilled 25-43
// registers (16 x 32K tokens: 80 us instead of 66), and even 8 spilled ones cost
// 4 x 128K tokens, groups of 8, 2 us of 76.
//
// L: the sequence's lengths.  Token nt.last (PAIR only) is the one this step
// appends: its rows are read from the step's inputs.
struct NewToken {
    const uint16_t *k, *v;
    int last;  // its index in the region, -1: none
};

// O += P V of 16 tokens: the lane's channel pair of each in x, P of head group
// g at pb + 128 g.
template <int GQ, bool BF, int... T>
__device__ __forceinline__ void pv16(f32x4 (&O)[GQ / 4][2], const float *pb, const uint32_t *x, int lane,
                                     std::integer_sequence<int, T...>)
{
    float pr[GQ / 4];
#pragma unroll
    for (int g = 0; g < GQ / 4; ++g)
        pr[g] = pb[128 * g + lane];
    auto token = [&](auto tc) {
        constexpr int tok = decltype(tc)::value;
        const float v0 = BF ? bf2f((uint16_t)x[tok]) : h2f((uint16_t)x[tok]);
        const float v1 = BF ? bf2f((uint16_t)(x[tok] >> 16)) : h2f((uint16_t)(x[tok] >> 16));
#pragma unroll
        for (int g = 0; g < GQ / 4; ++g) {
            O[g][0] = __builtin_amdgcn_mfma_f32_4x4x1f32(pr[g], v0, O[g][0], 4, tok, 0);
            O[g][1] = __builtin_amdgcn_mfma_f32_4x4x1f32(pr[g], v1, O[g][1], 4, tok, 0);
        }
    };
    (token(std::integral_constant<int, T>{}), ...);
}

template <int GQ, bool BF, bool PAIR>
__device__ void fp16_segments(const DecodeParams &p, int b, int kh, int lo, int hi, int64_t t, const SeqLens &L,
                              const NewToken &nt, unsigned char *kst, unsigned char *vst)
{
    constexpr int kTok = 32;
    constexpr int HPL = GQ / 4;              // heads per lane group
    constexpr int RSTEP = 4 / HPL;           // accumulator register of head slot j = j * RSTEP
    constexpr int RPH = 16 / GQ;             // MFMA rows per head
    constexpr int NG = GQ / 4;               // groups of 4 heads
    const int lane = lane_id(), r = lane & 15, kq = lane >> 4;
    static_assert(kTok * 256 + GQ * kTok * 4 <= kStage, "P does not fit behind the value rows");
    float *pbuf = (float *)(vst + kTok * 256);  // P[head / 4][token][head % 4]
    // A operand: row r = head r / RPH, k = 8 kq + i of each 32-channel step
    // (q as is: q k is exact in the fp32 accumulator, and the scores
    // are scaled by sm_scale log2(e) afterwards)
    const uint16_t *qrow = p.q + b * p.q_s_seq + q_head(p, kh, r / RPH) * p.q_s_head + 8 * kq;
    const float qk_c = p.sm_scale * kLog2e;
    float m[HPL], l[HPL];  // head kq HPL + j; l: this lane's tokens
#pragma unroll
    for (int j = 0; j < HPL; ++j) {
        m[j] = -__builtin_inff();
        l[j] = 0.0f;
    }
    f32x4 O[NG][2];        // heads 4 g + i, channels 2 lane + c
#pragma unroll
    for (int g = 0; g < NG; ++g)
        O[g][0] = O[g][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int ns = L.ns, kbeg = L.ns, kend = L.ns + L.nmix;  // key-only tokens [kbeg, kend)
    const uint16_t *sk = p.sink_k.ptr + b * p.sink_k.s_seq + kh * p.sink_k.s_head;
    const uint16_t *sv = p.sink_v.ptr + b * p.sink_v.s_seq + kh * p.sink_v.s_head;
    const uint16_t *tk = p.tail_k.ptr + b * p.tail_k.s_seq + kh * p.tail_k.s_head;
    const uint16_t *tv = p.tail_v.ptr + b * p.tail_v.s_seq + kh * p.tail_v.s_head;
    const float *sc = (const float *)kst;  // [GQ][128] scores of the key-only page in hand
    int page_in_kst = -1;
    bool poison = false;
    for (int c0 = lo; c0 < hi;) {
        int end = min(hi, c0 + kTok);
        const bool konly = c0 >= kbeg && c0 < kend;
        const int pg = konly ? (c0 - kbeg) >> 7 : 0;  // key-only page of this step
        if (konly)
            end = min(end, kbeg + 128 * (pg + 1));
        else if (c0 < kbeg && kend > kbeg)
            end = min(end, kbeg);
        const int cnt = end - c0;
        float S[2][HPL];
        if (konly) {
            if (pg != page_in_kst) {
                // scores of key page P_v + pg: the page path's QK into kst
                const int32_t page = p.block_table[(int64_t)b * p.bt_stride + L.npv + pg];
                if (page < 0 || page >= p.num_pool_pages) {
                    poison = true;
                    c0 = min(hi, kbeg + 128 * (pg + 1));
                    continue;
                }
                WaveState<GQ, BF> W;
                const SegSetup su = load_setup<GQ>(p, b, kh, L.npv + pg, L.npv + pg + 1);
                qk_setup<GQ, BF, PAIR>(W, p, b, kh, su, vst, lane, p.Dk);
                issue_page(kst, page_src(p, (int64_t)page * p.Hkv + kh), lane, p.Dk);
                wait_vmcnt<0>();
                f32x4 Sp[2][4], Yt;
                float kmul;
                page_qk<GQ, BF>(W, kst, lane, p.Dk, Sp, Yt, kmul);
                float *scw = (float *)kst;
#pragma unroll
                for (int j = 0; j < HPL; ++j) {
                    const int ri = j * RSTEP;
                    // the page path's scale (its operand carries 2^-3 q)
                    const float page_c = BF ? W.qk_c[BF ? j : 0] * kmul : W.qk_c[0];
                    const float yk = (GQ == 16 ? Yt[ri] : Yt[ri] + Yt[ri + 1]) * page_c;
#pragma unroll
                    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                        for (int a = 0; a < 4; ++a)
                            scw[(kq * HPL + j) * 128 + 64 * cb + 4 * r + a] =
                                (GQ == 16 ? Sp[cb][a][ri] : Sp[cb][a][ri] + Sp[cb][a][ri + 1]) *
                                    (page_c * (kSub / slot_weight<BF>(a))) - yk;
                }
                wave_sync<PAIR>();  // scores in kst before they are read back
                page_in_kst = pg;
            }
            // ---- value rows of the step: value-tail rows c0 - ns ..
#pragma unroll
            for (int i = 0; i < kTok / 4; ++i) {
                const int n = 4 * i + kq;
                const int tt = c0 + min(n, cnt - 1);
                gll16((const unsigned char *)(tv + (int64_t)(tt - ns) * p.tail_v.s_tok + 8 * r), vst + 1024 * i);
            }
            wait_vmcnt<0>();
            const int t0 = c0 - kbeg - 128 * pg;  // page token of the step's first token
#pragma unroll
            for (int tg = 0; tg < 2; ++tg)
#pragma unroll
                for (int j = 0; j < HPL; ++j) {
                    const int tok = 16 * tg + r;
                    S[tg][j] = tok < cnt ? sc[(kq * HPL + j) * 128 + t0 + tok] : -__builtin_inff();
                }
        } else {
            u32x4 qa[4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
                qa[s] = *(const u32x4 *)(qrow + 32 * s);
            // ---- 16 direct-to-LDS loads: instruction i covers rows 4i .. 4i+3
#pragma unroll
            for (int i = 0; i < kTok / 4; ++i) {
                const int n = 4 * i + kq;                 // token row of this lane's slot
                const int tt = c0 + min(n, cnt - 1);      // rows past cnt repeat the last token
                const bool sink = tt < ns;
                const uint16_t *krow = sink ? sk + (int64_t)tt * p.sink_k.s_tok
                                            : tk + (int64_t)(tt - kend) * p.tail_k.s_tok;
                const uint16_t *vrow = sink ? sv + (int64_t)tt * p.sink_v.s_tok
                                            : tv + (int64_t)(tt - ns) * p.tail_v.s_tok;
                if (PAIR && tt == nt.last) {
                    krow = nt.k;
                    vrow = nt.v;
                }
                gll16((const unsigned char *)(krow + 8 * (r ^ (n & 15))), kst + 1024 * i);
                gll16((const unsigned char *)(vrow + 8 * r), vst + 1024 * i);
            }
            wait_vmcnt<0>();
            // ---- QK: tile tg covers tokens 16 tg + r
#pragma unroll
            for (int tg = 0; tg < 2; ++tg) {
                f32x4 acc = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                const int n = 16 * tg + r;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const u32x4 kb = *(const u32x4 *)(kst + 256 * n + 16 * ((4 * s + kq) ^ r));
                    if constexpr (BF)
                        acc = mfma_bf(__builtin_bit_cast(bf16x8, qa[s]), __builtin_bit_cast(bf16x8, kb), acc);
                    else
                        acc = mfma(__builtin_bit_cast(half8, qa[s]), __builtin_bit_cast(half8, kb), acc);
                }
#pragma unroll
                for (int j = 0; j < HPL; ++j)
                    S[tg][j] = n < cnt ? acc[j * RSTEP] * qk_c : -__builtin_inff();
            }
            page_in_kst = -1;  // K rows went over any page scores
        }
        // the step's values, ahead of the softmax: read two at a time between the
        // MFMAs they cost an LDS round trip each
        uint32_t x[kTok];
#pragma unroll
        for (int n = 0; n < kTok; ++n)
            x[n] = *(const uint32_t *)(vst + 256 * n + 4 * lane);
        __builtin_amdgcn_sched_barrier(0);
        // ---- online softmax per head (tokens past cnt masked), P to LDS
        float alpha[HPL];
#pragma unroll
        for (int j = 0; j < HPL; ++j) {
            const float mn = fmaxf(m[j], row_max16(fmaxf(S[0][j], S[1][j])));
            alpha[j] = __builtin_amdgcn_exp2f(m[j] - mn);
            m[j] = mn;
            const float p0 = __builtin_amdgcn_exp2f(S[0][j] - mn), p1 = __builtin_amdgcn_exp2f(S[1][j] - mn);
            l[j] = l[j] * alpha[j] + (p0 + p1);
            const int h = kq * HPL + j;
            float *ph = pbuf + (h >> 2) * (4 * kTok) + (h & 3);
            ph[4 * r] = p0;
            ph[4 * (16 + r)] = p1;
        }
#pragma unroll
        for (int h = 0; h < GQ; ++h) {  // the head's alpha from its lane group
            const float x = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, alpha[h % HPL]), 16 * (h / HPL)));
            O[h / 4][0][h % 4] *= x;
            O[h / 4][1][h % 4] *= x;
        }
        wave_sync<PAIR>();
        // ---- PV, 16 tokens per P register
        pv16<GQ, BF>(O, pbuf, x, lane, std::make_integer_sequence<int, 16>{});
        if (cnt > 16)
            pv16<GQ, BF>(O, pbuf + 64, x + 16, lane, std::make_integer_sequence<int, 16>{});
        wave_sync<PAIR>();  // LDS reads done before the next step's loads land
        c0 = end;
    }
#pragma unroll
    for (int j = 0; j < HPL; ++j) {
        const float lsum = row_sum16(l[j]);
        if (r == 0) {
            const int64_t row = t * GQ + kq * HPL + j;
            p.ws_ml[2 * row] = poison ? __builtin_nanf("") : m[j];
            p.ws_ml[2 * row + 1] = lsum;
        }
    }
#pragma unroll
    for (int h = 0; h < GQ; ++h)
        *(float2 *)(p.ws_o + (t * GQ + h) * 128 + 2 * lane) = make_float2(O[h / 4][0][h % 4], O[h / 4][1][h % 4]);
}

// FP16 tokens [lo, hi) of pair (b, kh) as partial t.
template <int GQ, bool BF>
__device__ __forceinline__ void fp16_partial(KernargParams kp, int b, int kh, int lo, int hi, int64_t t,
                                          unsigned char *stage0, unsigned char *stage1)
{
    // arguments arrive in vector registers: the pointer is the same in every lane
    const uint64_t a = (uint64_t)kp;
    const uint32_t lo32 = __builtin_amdgcn_readfirstlane((uint32_t)a), hi32 = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const DecodeParams P = kernel_params((KernargParams)(((uint64_t)hi32 << 32) | lo32));
    b = __builtin_amdgcn_readfirstlane(b);
    kh = __builtin_amdgcn_readfirstlane(kh);
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    fp16_segments<GQ, BF, false>(P, b, kh, lo, hi, t, seq_lens(P, b), NewToken{nullptr, nullptr, -1}, stage0, stage1);
    __syncthreads();  // stage reads done before the next segment reuses them
}

// Occupancy target (waves per SIMD): two waves for GQA groups of 4 and 8
// (256 registers each, measured faster than one wave with no register cap),
// one for 16 heads, whose accumulators do not fit in 256.
//
// Wave w works through units [w U / W, (w + 1) U / W) of the unit-balanced
// plan: a run of pages or of FP16 tokens of one pair per segment, one
// partial per segment.  w is the workgroup's XCD-local order
// (plan_wave_of), so the consecutive waves of a pair share an XCD and its L2.
template <int GQ, bool BF>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(GQ <= 8 ? 2 : 1)))
void decode_mfma_kernel(DecodeParams p)
{
    // Two LDS stages: the wave computes on one while the next page streams
    // into the other with global_load_lds.
    __shared__ __attribute__((aligned(16))) unsigned char stage0[kStage];
    __shared__ __attribute__((aligned(16))) unsigned char stage1[kStage];

    const int lane = threadIdx.x;
    const KernargParams kp = (KernargParams)__builtin_amdgcn_kernarg_segment_ptr();
    const int F = p.fp16_units;
    // ---- the plan's input, page counts 64 sequences per step (issued first)
    int np_l = 0, units_l = 0;  // sequence b0 + lane of the current step
    auto load_step = [&](int b0) {
        const int b = b0 + lane;
        np_l = b < p.B ? seq_np_raw(p, b) : 0;
        units_l = b < p.B ? seq_page_units(np_l, p.max_pages, F) + F : 0;
    };
    load_step(0);
    // ---- static plan: every sequence at max_pages.  Its first page segment
    // is loaded while the page counts are in flight; when the batch turns out
    // to be that uniform, it is the plan and no scan is needed.
    const int units_s = seq_page_units(p.max_pages, p.max_pages, F) + F;
    const int npu_s = units_s - F;
    const int64_t U_s = (int64_t)p.B * p.Hkv * units_s;
    const int W_s = p.static_waves;
    int w = plan_wave_of(blockIdx.x, gridDim.x, W_s);
    int64_t s0 = 0, s1 = 0;
    int g_j = 0;
    bool g_page = false;
    if (w < W_s) {
        wave_units(U_s, W_s, w, s0, s1);
        g_j = U_s <= 0xffffffffll ? (int)((uint32_t)s0 / (uint32_t)units_s) : (int)((uint64_t)s0 / (uint32_t)units_s);
        g_page = s0 - (int64_t)g_j * units_s < npu_s;
    }
    const int g_b = g_j / p.Hkv, g_kh = g_j - g_b * p.Hkv;
    const int g_p0 = (int)(s0 - (int64_t)g_j * units_s);
    const int g_p1 = (int)min((int64_t)npu_s, s1 - (int64_t)g_j * units_s);
    SegSetup spec;
    if (g_page)
        spec = load_setup<GQ>(p, g_b, g_kh, g_p0, g_p1);
    bool uniform = __ballot(lane < p.B && units_l != units_s) == 0;
    for (int b0 = 64; b0 < p.B && uniform; b0 += 64) {
        load_step(b0);
        uniform = __ballot(b0 + lane < p.B && units_l != units_s) == 0;
    }
    int64_t U, u, u_last;
    int W;
    SeqUnits sq;
    sq.fu = F;
    if (uniform) {
        if (w >= W_s)
            return;
        U = U_s;
        W = W_s;
        u = uniform64(s0);
        u_last = uniform64(s1);
        sq.b = g_b;
        sq.base = (int64_t)g_b * p.Hkv * units_s;
        sq.np_raw = p.B <= 64 ? __builtin_amdgcn_readlane(np_l, g_b) : seq_np_raw(p, g_b);
        sq.npu = seq_page_units(sq.np_raw, p.max_pages, F);
    } else {
        // ---- plan for U: prefix sums of the units, 64 sequences per step
        if (p.B > 64)
            load_step(0);  // the uniformity check moved on to later steps
        int incl = wave_incl_scan(units_l, lane);
        int64_t tot = __builtin_amdgcn_readlane(incl, 63);
        for (int b0 = 64; b0 < p.B; b0 += 64) {
            load_step(b0);
            tot += __builtin_amdgcn_readlane(wave_incl_scan(units_l, lane), 63);
        }
        U = tot * p.Hkv;
        W = plan_waves(U, p.page_waves, p.simd_waves, p.chunk_lo, p.min_chunk);
        w = plan_wave_of(blockIdx.x, gridDim.x, W);
        if (w >= W)
            return;
        int64_t u_end;
        wave_units(U, W, w, u, u_end);
        u = uniform64(u);
        u_last = uniform64(u_end);
        // ---- the sequence holding unit u (with more than 64 sequences the
        // total above moved the step registers on: start again from step 0)
        int64_t base = 0;
        for (int b0 = 0;; b0 += 64) {
            if (b0 > 0 || p.B > 64) {
                load_step(b0);
                incl = wave_incl_scan(units_l, lane);
            }
            const unsigned long long hit = __ballot(b0 + lane < p.B && base + (int64_t)p.Hkv * incl > u);
            if (hit || b0 + 64 >= p.B) {
                const int lb = hit ? __builtin_ctzll(hit) : min(63, p.B - 1 - b0);  // second case not reached for u < U
                sq.b = b0 + lb;
                sq.base = base + (int64_t)p.Hkv * __builtin_amdgcn_readlane(incl - units_l, lb);
                sq.np_raw = __builtin_amdgcn_readlane(np_l, lb);
                sq.npu = seq_page_units(sq.np_raw, p.max_pages, F);
                break;
            }
            base += (int64_t)p.Hkv * __builtin_amdgcn_readlane(incl, 63);
        }
    }
    bool use_spec = uniform && g_page;  // the first segment is the one loaded above
    int kh = uniform ? g_kh : (int)((uint32_t)(u - sq.base) / (uint32_t)(sq.npu + F));
    const int Hkv = p.Hkv;
    if (sq.b < 0 || sq.b >= p.B || kh < 0 || kh >= Hkv || u < sq.base)
        return;  // not reached: the plan places every unit in a pair of the batch
#pragma clang loop unroll(disable)
    for (;;) {
        const int64_t u_end = u_last;
        const int64_t per_pair = sq.npu + F;
        const int64_t s_j = sq.base + kh * per_pair;
        const int j = sq.b * Hkv + kh;
        if (u == s_j && lane == 0)  // this wave starts the pair: its first partial
            kernel_params(kp).ws_pair[2 * j] = w + 2 * j + (sq.npu > 0 ? 0 : 1);
        const int64_t off = u - s_j;
        if (off < sq.npu) {
            const DecodeParams P = kernel_params(kp);
            const int64_t e = min(u_end, s_j + sq.npu);
            const int p0 = (int)off, p1 = (int)(e - s_j);
            SegSetup su;
            if (use_spec)
                su = spec;
            else
                su = load_setup<GQ>(P, sq.b, kh, p0, p1);
            use_spec = false;
            page_segment<GQ, BF>(P, stage0, stage1, sq.b, kh, sq.np_raw, p0, p1, (int64_t)w + 2 * j, su);
            if (e == u_end && F > 0 && e == s_j + sq.npu)
                empty_partial<GQ>(P, (int64_t)w + 2 * j + 1);
            u = e;
        } else {
            use_spec = false;
            const int64_t e = min(u_end, s_j + per_pair);
            const int fa = (int)(off - sq.npu), fc = (int)(e - s_j - sq.npu);
            const int ntok = seq_tokens(kernel_params(kp), sq.b);  // the tokens the F units share
            fp16_partial<GQ, BF>(kp, sq.b, kh, fa * ntok / F, fc * ntok / F, (int64_t)w + 2 * j + 1, stage0, stage1);
            u = e;
        }
        spec = SegSetup{};  // dead from here: its registers are the walk's
        if (u == s_j + per_pair && lane == 0)  // this wave ends the pair: its last partial
            kernel_params(kp).ws_pair[2 * j + 1] = w + 2 * j + (F > 0 ? 1 : 0);
        if (u >= u_end)
            break;
        if (u == s_j + per_pair && ++kh == Hkv) {
            kh = 0;
            const DecodeParams P = kernel_params(kp);
            sq.b += 1;
            sq.base += Hkv * per_pair;
            sq.np_raw = seq_np_raw(P, sq.b);
            sq.npu = seq_page_units(sq.np_raw, P.max_pages, F);
        }
    }
}

// Decode of batches with few pairs of few units in one launch: one workgroup
// per (sequence, KV head) pair, whose waves each take an equal run of the
// pair's units (pages, then FP16 units) on stages of their own, write their
// partials, and after one barrier merge them, a head per wave.  With `step`
// the launch also appends the step's token: its rows are stored to the buffers
// and attended from the inputs, and the last workgroup of a sequence to finish
// (step.tickets) advances its counters, which every workgroup has read by then.
//
// Such a decode is bound by its chain of launches and dependent loads, not by
// the chip: a split launch (plan over all sequences, then the first segment),
// a merge launch, and the append launch before them.  The lengths, q, ranks and
// page ids are one round trip here.  1 x 512 tokens, 8 KV heads: 12.5 us against
// 12.9 of the split and merge launches, 32 x 512 tokens 15.8 against 21.3; a
// module step of 1 x 1,000 tokens 16.7 us against 22.6, of 16 x 1,000 tokens and 8
// KV heads 22.3 against 27.5.
template <int GQ, bool BF>
__global__ __launch_bounds__(64 * kPairWaves) __attribute__((amdgpu_waves_per_eu(2)))
void decode_pair_kernel(DecodeParams p, StepParams step)
{
    constexpr int NW = kPairWaves;
    __shared__ __attribute__((aligned(16))) unsigned char stage0[NW][kStage];
    __shared__ __attribute__((aligned(16))) unsigned char stage1[NW][kStage];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int pair = blockIdx.x, b = pair / p.Hkv, kh = pair - b * p.Hkv;

    // ---- lengths as they stand, then (with a step) as this token leaves them
    int ns = p.sink_len[b], nk = p.tail_len[b], npk = p.num_pages[b];
    int npv = p.num_pages_v ? p.num_pages_v[b] : npk, nv = p.tail_len_v ? p.tail_len_v[b] : nk;
    const SegSetup su = load_setup<GQ>(p, b, kh, 0, p.max_pages);
    bool fresh = false, to_sink = false;
    int slot = 0;
    if (step.tickets) {
        const kitty_append_args &a = step.append;
        slot = a.slots[b];
        to_sink = ns < a.sink_size;
        fresh = slot == step.slot0 + b && (to_sink || !(nk >= a.buf_tokens || (a.val_len && nv >= a.val_tokens)));
    }
    const int ns0 = ns, nk0 = nk, nv0 = nv;
    if (fresh) {
        ns += to_sink ? 1 : 0;
        nk += to_sink ? 0 : 1;
        nv += to_sink ? 0 : 1;
    }
    const SeqLens L = check_lens(p, ns, npk, npv, nk, nv);
    NewToken nt{nullptr, nullptr, -1};
    if (fresh) {
        const kitty_append_args &a = step.append;
        nt.k = a.key + b * a.key_s_seq + kh * a.key_s_head;
        nt.v = a.value + b * a.value_s_seq + kh * a.value_s_head;
        nt.last = to_sink ? L.ns - 1 : L.ns + L.nv - 1;
        if (wave == 0 && lane < 32) {   // its rows into the buffers: lanes 0-15 the key, 16-31 the value
            const bool v = lane >= 16;
            const kitty_slot_layout KL = to_sink ? a.sink_layout : (v && a.val_len ? a.val_layout : a.buf_layout);
            uint16_t *dst = to_sink ? (v ? a.sink_v : a.sink_k) : (v ? (a.val_len ? a.val_buf : a.buf_v) : a.buf_k);
            const int row = to_sink ? ns0 : (v && a.val_len ? nv0 : nk0);
            *(u32x4 *)(dst + slot * KL.s_slot + kh * KL.s_head + row * KL.s_tok + 8 * (lane & 15)) =
                *(const u32x4 *)((v ? nt.v : nt.k) + 8 * (lane & 15));
        }
    }
    // ---- wave w takes units [w U / NW, (w + 1) U / NW) of the pair (none where
    // the two meet); waves [0, wp) start in the pages, waves [wf, NW) end past them
    const int F = p.fp16_units;
    const int npu = __builtin_amdgcn_readfirstlane(L.npv);
    const unsigned U = npu + F;
    const int ua = wave * U / NW, ue = (wave + 1) * U / NW;
    int wp = 0, wf = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        wp += (int)(w * U / NW) < npu ? 1 : 0;
        wf += (int)((w + 1) * U / NW) <= npu ? 1 : 0;
    }
    const int64_t t0 = (int64_t)pair * (2 * NW);
    if (ua < npu && !L.bad)
        page_segment<GQ, BF, true>(p, stage0[wave], stage1[wave], b, kh, npu, ua, ue < npu ? ue : npu, t0 + wave, su);
    if (wave >= wf) {
        const int fa = (ua > npu ? ua : npu) - npu, fc = ue - npu;
        const unsigned ntok = __builtin_amdgcn_readfirstlane(L.ns + L.nv);  // F is a few dozen here
        wave_sync<true>();
        fp16_segments<GQ, BF, true>(p, b, kh, (int)(fa * ntok / (unsigned)F), (int)(fc * ntok / (unsigned)F),
                                    t0 + wp + (wave - wf), L, nt, stage0[wave], stage1[wave]);
    }
    __syncthreads();
    for (int g = wave; g < p.gq; g += NW) {
        uint16_t *o = p.out + b * p.out_s_seq + ((int64_t)kh * p.gq_stride + g) * p.out_s_head;
        if (L.bad) {
            o[2 * lane] = o[2 * lane + 1] = out_bits(p, __builtin_nanf(""));
            continue;
        }
        merge_quads<3>(p, t0 * GQ + g, GQ, wp + NW - wf, o);
    }
    if (step.tickets && threadIdx.x == 0) {
        const kitty_append_args &a = step.append;
        // the last of the sequence's Hkv workgroups; the ticket wraps to 0 with it
        if (atomicInc((unsigned *)step.tickets + step.slot0 + b, (unsigned)p.Hkv - 1) == (unsigned)p.Hkv - 1) {
            if (!fresh) {   // a full buffer, or a slot that is not the row the decode reads
                if (slot >= 0 && slot < a.num_slots)
                    a.overflow[b] = 1;
            } else if (to_sink) {
                a.sink_fill[slot] = ns0 + 1;
            } else {
                a.buf_len[slot] = nk0 + 1;
                if (a.val_len)
                    a.val_len[slot] = nv0 + 1;
            }
        }
    }
}

static bool seg_aligned(const kitty_fp16_seg &s)
{
    return ((uintptr_t)s.ptr & 15) == 0 && s.s_seq % 8 == 0 && s.s_head % 8 == 0 && s.s_tok % 8 == 0;
}

bool mfma_shape_supported(const DecodeParams &p)
{
    return p.D == 128 && p.G == 128 && p.Dk >= 0 && p.Dk <= 32 && (p.GQ == 4 || p.GQ == 8 || p.GQ == 16) &&
           p.meta_bf16 == p.act_bf16;
}

bool mfma_path_supported(const DecodeParams &p)
{
    return mfma_shape_supported(p) &&
           (p.flags & KITTY_DECODE_UNIQUE_BOOST_ROWS) && seg_aligned(p.sink_k) && seg_aligned(p.sink_v) &&
           seg_aligned(p.tail_k) && seg_aligned(p.tail_v) && ((uintptr_t)p.key_low & 15) == 0 &&
           ((uintptr_t)p.key_high & 15) == 0 && ((uintptr_t)p.key_meta & 15) == 0 &&
           ((uintptr_t)p.value & 15) == 0 && ((uintptr_t)p.value_meta & 15) == 0;
}

template <int GQ>
static void launch_group(const DecodeParams &p, hipStream_t stream)
{
    const dim3 grid((unsigned)p.page_waves);
    if (p.act_bf16)
        hipLaunchKernelGGL((decode_mfma_kernel<GQ, true>), grid, dim3(64), 0, stream, p);
    else
        hipLaunchKernelGGL((decode_mfma_kernel<GQ, false>), grid, dim3(64), 0, stream, p);
}

template <int GQ>
static void launch_pair_group(const DecodeParams &p, const StepParams &step, hipStream_t stream)
{
    const dim3 grid((unsigned)(p.B * p.Hkv)), block(64 * kPairWaves);
    if (p.act_bf16)
        hipLaunchKernelGGL((decode_pair_kernel<GQ, true>), grid, block, 0, stream, p, step);
    else
        hipLaunchKernelGGL((decode_pair_kernel<GQ, false>), grid, block, 0, stream, p, step);
}

int launch_pair(const DecodeParams &p, const StepParams &step, hipStream_t stream)
{
    switch (p.GQ) {
    case 4: launch_pair_group<4>(p, step, stream); break;
    case 8: launch_pair_group<8>(p, step, stream); break;
    default: return fail(KITTY_E_UNSUPPORTED, "the pair kernel needs a GQA group of 4 or 8");
    }
    return check_launch("decode_pair_kernel");
}

int launch_mfma(const DecodeParams &p, hipStream_t stream)
{
    switch (p.GQ) {
    case 4: launch_group<4>(p, stream); break;
    case 8: launch_group<8>(p, stream); break;
    case 16: launch_group<16>(p, stream); break;
    default: return fail(KITTY_E_UNSUPPORTED, "MFMA decode needs a GQA group of 4, 8 or 16");
    }
    return check_launch("decode_mfma_kernel");
}

} // namespace kitty
