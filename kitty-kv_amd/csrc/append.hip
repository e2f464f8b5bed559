// Token append of the Kitty pipeline on the device: one launch per
// layer-step writes the new FP16 key / value of every sequence of a batch
// into its sink buffer (while it holds fewer than S tokens) or its key /
// value buffer, and advances the sequence's device-side counters.
// Replaces the FP16 part of KittyInferencePipeline.push_token
// (kitty/pipeline.py:115-181); spilling a full buffer into a page stays with
// the caller (kitty_quantize_kv_blocks).
#include "common.h"

#include <algorithm>

namespace kitty {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// One workgroup per sequence, 64 threads; H x D 16-bit values of K and of V
// (fp16 or bf16: rows are copied bit for bit).  The kernel is one basic block
// up to its last stores, so the token's first kAppendRows x 64 16-byte
// vectors (all of them at H x D = 8 x 128), the slot id, and then the
// counters are loaded back to back: a launch costs two memory round trips.
// The row loads are unconditional (a lane past the end reloads the last
// vector and writes it back to its own place), and the row stores go through
// buffer descriptors whose record count is 0 when nothing may be written, so
// the hardware drops them; a store under a branch would let the compiler sink
// the loads feeding it behind the counter loads.
constexpr int kAppendRows = 2;
constexpr int kBufferWord3 = 0x00020000;  // raw (untyped) buffer, gfx9 family

__global__ __launch_bounds__(64) void append_tokens_kernel(kitty_append_args a)
{
    const int b = blockIdx.x;
    const int vec = a.head_dim / 8;  // 16-byte vectors per head row
    const int n = a.num_kv_heads * vec;
    u32x4 kr[kAppendRows], vr[kAppendRows];
    int hd[kAppendRows], ch[kAppendRows];
#pragma unroll
    for (int i = 0; i < kAppendRows; ++i) {
        const int e = min((int)threadIdx.x + i * 64, n - 1);
        hd[i] = e / vec;
        ch[i] = (e - hd[i] * vec) * 8;
        kr[i] = *(const u32x4 *)(a.key + b * a.key_s_seq + hd[i] * a.key_s_head + ch[i]);
        vr[i] = *(const u32x4 *)(a.value + b * a.value_s_seq + hd[i] * a.value_s_head + ch[i]);
    }
    const int slot = a.slots[b];
    const bool valid = slot >= 0 && slot < a.num_slots;
    const int s = valid ? slot : 0;
    const bool own_values = a.val_len != nullptr;
    const int fill = a.sink_fill[s], qlen = a.buf_len[s];
    const int vlen = (own_values ? a.val_len : a.buf_len)[s];
    const bool to_sink = fill < a.sink_size;
    // the caller did not spill a full buffer: flag it, write nothing
    const bool full = !to_sink && (qlen >= a.buf_tokens || (own_values && vlen >= a.val_tokens));
    const bool write = valid && !full;
    const kitty_slot_layout KL = to_sink ? a.sink_layout : a.buf_layout;
    const kitty_slot_layout VL = to_sink ? a.sink_layout : (own_values ? a.val_layout : a.buf_layout);
    uint16_t *dk = (to_sink ? a.sink_k : a.buf_k) + s * KL.s_slot + (to_sink ? fill : qlen) * KL.s_tok;
    uint16_t *dv = (to_sink ? a.sink_v : (own_values ? a.val_buf : a.buf_v)) + s * VL.s_slot +
                   (to_sink ? fill : vlen) * VL.s_tok;
    const int records = __builtin_amdgcn_readfirstlane(write ? -1 : 0);  // uniform: keep the descriptor in SGPRs
    const auto rk = __builtin_amdgcn_make_buffer_rsrc(dk, 0, records, kBufferWord3);
    const auto rv = __builtin_amdgcn_make_buffer_rsrc(dv, 0, records, kBufferWord3);
#pragma unroll
    for (int i = 0; i < kAppendRows; ++i) {
        // byte offsets below 2^31: the host checks (H - 1) * s_head + D
        __builtin_amdgcn_raw_buffer_store_b128(kr[i], rk, (int)(hd[i] * KL.s_head + ch[i]) * 2, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b128(vr[i], rv, (int)(hd[i] * VL.s_head + ch[i]) * 2, 0, 0);
    }
    if (write) {
        for (int e = threadIdx.x + kAppendRows * 64; e < n; e += blockDim.x) {   // H x D past 8 x 128
            const int h = e / vec, c = (e - h * vec) * 8;
            *(u32x4 *)(dk + h * KL.s_head + c) = *(const u32x4 *)(a.key + b * a.key_s_seq + h * a.key_s_head + c);
            *(u32x4 *)(dv + h * VL.s_head + c) =
                *(const u32x4 *)(a.value + b * a.value_s_seq + h * a.value_s_head + c);
        }
    }
    if (threadIdx.x == 0 && valid) {
        if (full) {
            a.overflow[b] = 1;
        } else if (to_sink) {
            a.sink_fill[s] = fill + 1;
        } else {
            a.buf_len[s] = qlen + 1;
            if (own_values)
                a.val_len[s] = vlen + 1;
        }
    }
}

static bool al16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

// Spill bookkeeping: a list that travels in the kernel arguments (at most
// 4 KB), so the host's page-table and counter updates need no staging copy.
struct StoreI32Args {
    int32_t n;
    int32_t value[KITTY_STORE_I32_MAX];
    int32_t *addr[KITTY_STORE_I32_MAX];
};
static_assert(sizeof(StoreI32Args) <= 4096, "kernel arguments above 4 KB");

__global__ __launch_bounds__(256) void store_i32_kernel(StoreI32Args a)
{
    for (int i = threadIdx.x; i < a.n; i += 256)
        *a.addr[i] = a.value[i];
}

// A prompt's FP16 rows, block-table entries and counters (kitty_store_prompt).
// Workgroup (x, b): 256 threads copy 16-byte vectors of sequence b's rows, all
// four row kinds laid end to end; workgroup (0, b) also writes the table row
// and the counters.  Launch-bound: 5-8 us (8 MB read and written for 16 prompts
// of 4,096 tokens) for what took four strided torch copies of 3-9 us, two index
// copies and a staged counter copy, each with its gap.
constexpr int kPromptThreads = 256;

__global__ __launch_bounds__(kPromptThreads) void store_prompt_kernel(kitty_prompt_args a)
{
    const int b = blockIdx.y, vec = a.head_dim / 8;
    const int nk0 = a.n_sink + a.key_pages * a.page_tokens, nv0 = a.n_sink + a.value_pages * a.page_tokens;
    const int krem = a.tokens - nk0, vrem = a.tokens - nv0;
    // rows per head: sink keys, sink values, key tail, value tail
    const int rows = 2 * a.n_sink + krem + vrem;
    const int64_t n = (int64_t)a.num_kv_heads * rows * vec;
    const uint16_t *key = a.key + b * a.key_s_seq, *value = a.value + b * a.value_s_seq;
    for (int64_t e = (int64_t)blockIdx.x * kPromptThreads + threadIdx.x; e < n; e += (int64_t)gridDim.x * kPromptThreads) {
        const int hr = (int)(e / vec), c = 8 * (int)(e - (int64_t)hr * vec);
        const int h = hr / rows;
        int r = hr - h * rows;
        const uint16_t *src;
        uint16_t *dst;
        if (r < 2 * a.n_sink) {
            const bool v = r >= a.n_sink;
            r -= v ? a.n_sink : 0;
            src = v ? value + h * a.value_s_head + r * a.value_s_tok : key + h * a.key_s_head + r * a.key_s_tok;
            dst = (v ? a.sink_v : a.sink_k) + b * a.sink_layout.s_slot + h * a.sink_layout.s_head + r * a.sink_layout.s_tok;
        } else if ((r -= 2 * a.n_sink) < krem) {
            src = key + h * a.key_s_head + (int64_t)(nk0 + r) * a.key_s_tok;
            dst = a.key_buf + b * a.key_layout.s_slot + h * a.key_layout.s_head + r * a.key_layout.s_tok;
        } else {
            r -= krem;
            src = value + h * a.value_s_head + (int64_t)(nv0 + r) * a.value_s_tok;
            dst = a.value_buf + b * a.value_layout.s_slot + h * a.value_layout.s_head + r * a.value_layout.s_tok;
        }
        *(u32x4 *)(dst + c) = *(const u32x4 *)(src + c);
    }
    if (blockIdx.x == 0) {
        for (int p = threadIdx.x; p < a.key_pages; p += kPromptThreads)
            a.block_table[b * a.bt_stride + p] = a.pages[(int64_t)b * a.key_pages + p];
        if (threadIdx.x < 5) {
            const int counts[5] = {a.n_sink, krem, a.key_pages, a.value_pages, vrem};
            int v = counts[0];
#pragma unroll
            for (int i = 1; i < 5; ++i)
                v = threadIdx.x == i ? counts[i] : v;
            a.counters[threadIdx.x * a.counters_stride + b] = v;
        }
    }
}

// Zero regions of one launch: workgroup (x, region) walks the region's rows;
// 16-byte stores where base, row and stride allow them.  2.7 us for a slot at 8
// KV heads, where six torch fills took 2 us each and their launches: 16 resets
// and the prompts' arrival, 16 x 4,096 tokens, 866 -> 345 us.
struct ZeroArgs {
    kitty_zero_region r[KITTY_ZERO_MAX];
};

__global__ __launch_bounds__(256) void zero_regions_kernel(ZeroArgs a)
{
    const kitty_zero_region r = a.r[blockIdx.y];
    const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
    if ((((uintptr_t)r.ptr | (uintptr_t)r.row_bytes | (uintptr_t)r.row_stride) & 15u) == 0) {
        const int64_t per = r.row_bytes / 16, n = r.rows * per;
        for (int64_t i = i0; i < n; i += step)
            *(u32x4 *)((char *)r.ptr + i / per * r.row_stride + i % per * 16) = u32x4{0u, 0u, 0u, 0u};
    } else {
        const int64_t per = r.row_bytes / 4, n = r.rows * per;
        for (int64_t i = i0; i < n; i += step)
            *(uint32_t *)((char *)r.ptr + i / per * r.row_stride + i % per * 4) = 0u;
    }
}

} // namespace kitty

using namespace kitty;

int kitty::check_append(const kitty_append_args *args)
{
    if (!args)
        return fail(KITTY_E_INVALID, "args is NULL");
    const kitty_append_args &a = *args;
    if (a.batch < 0 || a.num_kv_heads <= 0 || a.head_dim <= 0 || a.head_dim % 8 || a.sink_size < 0 ||
        a.buf_tokens <= 0 || a.num_slots <= 0)
        return fail(KITTY_E_INVALID, "bad append shape (head_dim must be a positive multiple of 8)");
    if (a.batch == 0)
        return KITTY_OK;
    const bool own_values = a.val_len != nullptr;
    if (!a.key || !a.value || !a.slots || !a.sink_fill || !a.buf_len || !a.overflow || !a.buf_k ||
        (own_values ? !a.val_buf : !a.buf_v) || (a.sink_size > 0 && (!a.sink_k || !a.sink_v)))
        return fail(KITTY_E_INVALID, "NULL pointer in append args");
    if (own_values && a.val_tokens <= 0)
        return fail(KITTY_E_INVALID, "val_tokens must be positive with a value buffer");
    const int64_t strides[] = {a.key_s_seq, a.key_s_head, a.value_s_seq, a.value_s_head, a.sink_layout.s_slot,
                               a.sink_layout.s_head, a.sink_layout.s_tok, a.buf_layout.s_slot,
                               a.buf_layout.s_head, a.buf_layout.s_tok, own_values ? a.val_layout.s_slot : 0,
                               own_values ? a.val_layout.s_head : 0, own_values ? a.val_layout.s_tok : 0};
    for (int64_t s : strides)
        if (s % 8)
            return fail(KITTY_E_INVALID, "append strides must be multiples of 8 elements (16-byte rows)");
    // the kernel addresses a token's H x D block of a buffer with 32-bit byte offsets
    const int64_t head_strides[] = {a.sink_layout.s_head, a.buf_layout.s_head, own_values ? a.val_layout.s_head : 0};
    for (int64_t s : head_strides)
        if (s < 0 || (a.num_kv_heads - 1) * s + a.head_dim >= (int64_t(1) << 30))
            return fail(KITTY_E_INVALID, "append buffer head stride must be non-negative with (H-1)*s_head+D < 2^30");
    if (!al16(a.key) || !al16(a.value) || !al16(a.buf_k) || !al16(own_values ? a.val_buf : a.buf_v) ||
        (a.sink_size > 0 && (!al16(a.sink_k) || !al16(a.sink_v))))
        return fail(KITTY_E_INVALID, "append buffers must be 16-byte aligned");
    return KITTY_OK;
}

extern "C" int kitty_append_tokens(const kitty_append_args *args, kitty_stream_t stream)
{
    const int rc = check_append(args);
    if (rc || args->batch == 0)
        return rc;
    hipLaunchKernelGGL(append_tokens_kernel, dim3(args->batch), dim3(64), 0, (hipStream_t)stream, *args);
    return check_launch("append_tokens_kernel");
}

extern "C" int kitty_store_i32(int32_t *const *addrs, const int32_t *values, int32_t n, kitty_stream_t stream)
{
    if (n < 0 || (n > 0 && (!addrs || !values)))
        return fail(KITTY_E_INVALID, "kitty_store_i32: n < 0 or NULL list");
    for (int32_t i = 0; i < n; ++i)
        if (!addrs[i] || ((uintptr_t)addrs[i] & 3u))
            return fail(KITTY_E_INVALID, "kitty_store_i32: NULL or misaligned address");
    for (int32_t i0 = 0; i0 < n; i0 += KITTY_STORE_I32_MAX) {
        StoreI32Args a;
        a.n = std::min<int32_t>(KITTY_STORE_I32_MAX, n - i0);
        for (int32_t i = 0; i < a.n; ++i) {
            a.addr[i] = addrs[i0 + i];
            a.value[i] = values[i0 + i];
        }
        hipLaunchKernelGGL(store_i32_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream, a);
        const int rc = check_launch("store_i32_kernel");
        if (rc != KITTY_OK)
            return rc;
    }
    return KITTY_OK;
}

extern "C" int kitty_store_prompt(const kitty_prompt_args *args, kitty_stream_t stream)
{
    if (!args)
        return fail(KITTY_E_INVALID, "args is NULL");
    const kitty_prompt_args &a = *args;
    if (a.batch < 0 || a.num_kv_heads <= 0 || a.head_dim <= 0 || a.head_dim % 8 || a.tokens < 0 || a.page_tokens <= 0 ||
        a.n_sink < 0 || a.key_pages < 0 || a.value_pages < 0 || a.value_pages > a.key_pages ||
        (int64_t)a.n_sink + (int64_t)a.key_pages * a.page_tokens > a.tokens)
        return fail(KITTY_E_INVALID, "kitty_store_prompt: bad shape (head_dim must be a positive multiple of 8)");
    if (a.batch == 0)
        return KITTY_OK;
    const int64_t krem = a.tokens - a.n_sink - (int64_t)a.key_pages * a.page_tokens;
    const int64_t vrem = a.tokens - a.n_sink - (int64_t)a.value_pages * a.page_tokens;
    if (!a.counters || (a.tokens > 0 && (!a.key || !a.value)) || (a.n_sink > 0 && (!a.sink_k || !a.sink_v)) ||
        (krem > 0 && !a.key_buf) || (vrem > 0 && !a.value_buf) || (a.key_pages > 0 && (!a.block_table || !a.pages)))
        return fail(KITTY_E_INVALID, "kitty_store_prompt: NULL pointer");
    const int64_t strides[] = {a.key_s_seq, a.key_s_head, a.key_s_tok, a.value_s_seq, a.value_s_head, a.value_s_tok,
                               a.sink_layout.s_slot, a.sink_layout.s_head, a.sink_layout.s_tok, a.key_layout.s_slot,
                               a.key_layout.s_head, a.key_layout.s_tok, a.value_layout.s_slot, a.value_layout.s_head,
                               a.value_layout.s_tok};
    for (int64_t s : strides)
        if (s % 8)
            return fail(KITTY_E_INVALID, "kitty_store_prompt: strides must be multiples of 8 elements (16-byte rows)");
    if (!al16(a.key) || !al16(a.value) || !al16(a.sink_k) || !al16(a.sink_v) || !al16(a.key_buf) || !al16(a.value_buf))
        return fail(KITTY_E_INVALID, "kitty_store_prompt: rows must be 16-byte aligned");
    if ((2 * (int64_t)a.n_sink + krem + vrem) * a.num_kv_heads > 0x7fffffff || a.batch > 65535)
        return fail(KITTY_E_UNSUPPORTED, "kitty_store_prompt: too many rows for one launch");
    const int64_t n = (2 * (int64_t)a.n_sink + krem + vrem) * a.num_kv_heads * (a.head_dim / 8);
    const int64_t want = (n + 4 * kPromptThreads - 1) / (4 * kPromptThreads);   // four vectors per thread
    const unsigned x = (unsigned)std::max<int64_t>(1, std::min<int64_t>(want, 256));
    hipLaunchKernelGGL(store_prompt_kernel, dim3(x, (unsigned)a.batch), dim3(kPromptThreads), 0, (hipStream_t)stream, a);
    return check_launch("store_prompt_kernel");
}

extern "C" int kitty_zero_regions(const kitty_zero_region *regions, int32_t n, kitty_stream_t stream)
{
    if (n < 0 || (n > 0 && !regions))
        return fail(KITTY_E_INVALID, "kitty_zero_regions: n < 0 or NULL list");
    for (int32_t i = 0; i < n; ++i) {
        const kitty_zero_region &r = regions[i];
        if (r.rows < 0 || r.row_bytes < 0 || r.row_bytes % 4 || r.row_stride % 4 || ((uintptr_t)r.ptr & 3u) ||
            (!r.ptr && r.rows * r.row_bytes > 0))
            return fail(KITTY_E_INVALID, "kitty_zero_regions: regions must be 4-byte aligned and sized");
    }
    for (int32_t i0 = 0; i0 < n; i0 += KITTY_ZERO_MAX) {
        ZeroArgs a{};
        int m = 0;
        int64_t most = 0;
        for (int32_t i = i0; i < n && i < i0 + KITTY_ZERO_MAX; ++i) {
            if (regions[i].rows == 0 || regions[i].row_bytes == 0)
                continue;
            most = std::max(most, regions[i].rows * regions[i].row_bytes);
            a.r[m++] = regions[i];
        }
        if (m == 0)
            continue;
        const int64_t want = (most / 16 + 4 * 256 - 1) / (4 * 256);
        const unsigned x = (unsigned)std::max<int64_t>(1, std::min<int64_t>(want, 512));
        hipLaunchKernelGGL(zero_regions_kernel, dim3(x, (unsigned)m), dim3(256), 0, (hipStream_t)stream, a);
        const int rc = check_launch("zero_regions_kernel");
        if (rc != KITTY_OK)
            return rc;
    }
    return KITTY_OK;
}
