// append_body.h - device bodies of the KV append kernels (gfx950): the f32 /
// f16 row copy through the block table or a slot mapping, the FP8
// quantize-on-append per physical block, and the mixed step's batched copy.
// Included by append.hip (the library's kernels) and by the code-object
// entries (module_entry.hip), which wrap the same bodies.
#pragma once
#include "kernels.h"
#include "pam_device.h"

namespace pam {

template <typename CH>
__device__ __forceinline__ void append_body(const AppendParams &p, int64_t chunks_per_row, int64_t total) {
    if (p.length_patch && blockIdx.x == 0 && threadIdx.x == 0) {
        if (p.table_patch) p.table_patch[p.patch_index] = p.patch_block;
        *p.length_patch = p.length_value;
    }
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t t = i / chunks_per_row, c = i % chunks_per_row;
        int64_t slot;
        if (p.slot_mapping) {
            slot = p.slot_mapping[t];
            if (slot < 0) continue;  // padding token
        } else if (p.fixed_slot >= 0) {
            slot = p.fixed_slot;  // one token
        } else {
            const int64_t pos = (int64_t)p.token_offset + t;
            slot = (int64_t)p.block_table[pos / p.block_size] * p.block_size + pos % p.block_size;
        }
        const CH *ks = static_cast<const CH *>(p.keys) + t * chunks_per_row + c;
        const CH *vs = static_cast<const CH *>(p.values) + t * chunks_per_row + c;
        static_cast<CH *>(p.k_pool)[slot * chunks_per_row + c] = *ks;
        static_cast<CH *>(p.v_pool)[slot * chunks_per_row + c] = *vs;
    }
}

// 8 halves as e4m3 codes by a finite positive scale, bit for bit fp8_quantize's.
// `inv` is 1 / scale raised by 2^-20.  A quotient of two halves that is not exactly
// half way between two codes is at least 2^-16 of itself away from there, and one
// that is exactly half way goes to the larger magnitude; raising every quotient by
// 2^-20 therefore leaves the nearest code as it is, ties included, and the IEEE
// division with its case analysis becomes a product, an add and a shift.
// (test_fp8_fast_quantiser checks all 2^31 pairs of halves on the CPU; contraction is off,
// as the device would otherwise fuse the product with the sum below it.)
__host__ __device__ __forceinline__ uint32_t fp8_code(float v, float inv) {
#pragma clang fp contract(off)
    const float x = __builtin_fabsf(v) * inv;
    const uint32_t b = __builtin_bit_cast(uint32_t, x);
    uint32_t normal = ((b + 0x80000u) >> 20) - (120u << 3);  // 3-bit mantissa, half away from zero
    normal = normal < 0x7Eu ? normal : 0x7Eu;
    // multiples of 2^-9 below 2^-6: 1.5 2^14 + x keeps exactly those bits
    uint32_t low = __builtin_bit_cast(uint32_t, x + 24576.0f) - 0x46C00000u;
    low = low < 7u ? low : 7u;
    const uint32_t m = x < 0x1p-6f ? low : normal;
    return v >= 0.0f ? m : m | 0x80u;  // -0 is +0; NaN saturates negative
}
__device__ __forceinline__ uint2 fp8_codes8(const f16x8 a, float inv) {
    uint32_t w[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; i++) w[i >> 2] |= fp8_code((float)a[i], inv) << (8 * (i & 3));
    return make_uint2(w[0], w[1]);
}

constexpr int kFp8Threads = 512;  // threads of a quantise-on-append workgroup
constexpr int kFp8Keep = 4;       // 8-element pieces a thread keeps between the passes

// One workgroup per touched (sequence, logical block) and pool (blockIdx.y: K, V).
// The block's new tokens are consecutive rows of the input and consecutive slots of
// the physical block, so both passes (the max for the scale rule, then the
// quantisation) stream one contiguous range: 8 halves in, 8 codes out per thread and
// step when the rows are 16-byte multiples, one element at a time otherwise.  The
// first kFp8Keep pieces of a thread stay in registers between the passes (all of a
// block of 16 tokens of 8 heads of 128).
// What bounds it: the latency of one block's loads, reduction and stores (a few
// hundred workgroups, one round); before, the quantiser's division and case analysis
// and half the workgroups.  2000 tokens of 8 heads of 128 (12.3 MB) on gfx950: 28.1
// -> 6.7 µs per call (1.8 TB/s).
__device__ __forceinline__ void append_fp8_body(const AppendBatchParams &p, int32_t first_lb,
                                                int32_t single_offset) {
    int seq, lb;
    if (p.work) {
        const int4 w = p.work[blockIdx.x];
        seq = w.x;
        lb = w.y;
    } else {
        seq = 0;
        lb = first_lb + blockIdx.x;
    }
    const bool is_v = blockIdx.y != 0;
    const int64_t row = (int64_t)p.num_kv_heads * p.head_dim;  // elements per token
    const int64_t tok_base = p.cu_tokens ? p.cu_tokens[seq] : 0;
    const int64_t n_tok = p.cu_tokens ? p.cu_tokens[seq + 1] - tok_base : p.total_tokens;
    const int64_t off = p.token_offsets ? p.token_offsets[seq] : single_offset;
    const int bs = p.block_size;
    int64_t t0 = (int64_t)lb * bs - off, t1 = t0 + bs;
    if (t0 < 0) t0 = 0;
    if (t1 > n_tok) t1 = n_tok;
    const int32_t phys = p.block_tables[(int64_t)seq * p.bt_stride + lb];
    uint16_t *scale = (is_v ? p.v_scale : p.k_scale) + phys;
    const uint16_t old_scale = *scale;
    // input elements [t0 * row, t1 * row) -> pool elements from the slot of t0
    const int64_t n = (t1 - t0) * row;
    const f16 *in = static_cast<const f16 *>(is_v ? p.values : p.keys) + (tok_base + t0) * row;
    uint8_t *out = static_cast<uint8_t *>(is_v ? p.v_pool : p.k_pool) +
                   ((int64_t)phys * bs + (off + t0 - (int64_t)lb * bs)) * row;
    // 16-byte input rows and aligned buffers: every token row keeps the alignment
    const bool vec = (row % 8) == 0 && (((uintptr_t)p.keys | (uintptr_t)p.values) & 15) == 0 &&
                     (((uintptr_t)p.k_pool | (uintptr_t)p.v_pool) & 7) == 0;
    const int64_t step = (int64_t)blockDim.x * 8;

    f16x8 keep[kFp8Keep];
    float mx = 0.0f;
    if (vec) {
        f16x8 m8 = (f16x8)(f16)0.0f;
        const int64_t e0 = (int64_t)threadIdx.x * 8;
#pragma unroll
        for (int i = 0; i < kFp8Keep; i++)
            if (e0 + i * step < n) keep[i] = *reinterpret_cast<const f16x8 *>(in + e0 + i * step);
#pragma unroll
        for (int i = 0; i < kFp8Keep; i++)
            if (e0 + i * step < n) m8 = __builtin_elementwise_max(m8, __builtin_elementwise_abs(keep[i]));
        for (int64_t e = e0 + kFp8Keep * step; e < n; e += step)
            m8 = __builtin_elementwise_max(m8, __builtin_elementwise_abs(*reinterpret_cast<const f16x8 *>(in + e)));
#pragma unroll
        for (int i = 0; i < 8; i++) mx = fmaxf(mx, (float)m8[i]);
    } else {
        for (int64_t e = threadIdx.x; e < n; e += blockDim.x) mx = fmaxf(mx, fabsf((float)in[e]));
    }
    mx = wave_max_xor(mx, 1, 64);
    __shared__ float red[kFp8Threads / 64];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kFp8Threads / 64; w++) mx = fmaxf(mx, red[w]);
    const f16 s = fp8_scale_rule(mx, bits_to_f16(old_scale));
    if (vec && (float)s > 0.0f && __builtin_isfinite((float)s)) {
        const float inv = (1.0f / (float)s) * (1.0f + 0x1p-20f);
        const int64_t e0 = (int64_t)threadIdx.x * 8;
#pragma unroll
        for (int i = 0; i < kFp8Keep; i++)
            if (e0 + i * step < n) *reinterpret_cast<uint2 *>(out + e0 + i * step) = fp8_codes8(keep[i], inv);
        for (int64_t e = e0 + kFp8Keep * step; e < n; e += step)
            *reinterpret_cast<uint2 *>(out + e) = fp8_codes8(*reinterpret_cast<const f16x8 *>(in + e), inv);
    } else {
        for (int64_t e = threadIdx.x; e < n; e += blockDim.x) out[e] = (uint8_t)fp8_quantize(in[e], s);
    }
    if (threadIdx.x == 0) *scale = f16_to_bits(s);
}

template <typename CH>
__device__ __forceinline__ void append_batch_body(const AppendBatchParams &p, int64_t chunks_per_row,
                                                  int64_t total) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int64_t t = i / chunks_per_row, c = i % chunks_per_row;
        const int2 tp = p.token_pos[t];
        const int64_t slot =
            (int64_t)p.block_tables[(int64_t)tp.x * p.bt_stride + tp.y / p.block_size] * p.block_size +
            tp.y % p.block_size;
        static_cast<CH *>(p.k_pool)[slot * chunks_per_row + c] = static_cast<const CH *>(p.keys)[i];
        static_cast<CH *>(p.v_pool)[slot * chunks_per_row + c] = static_cast<const CH *>(p.values)[i];
    }
}

// Copy-on-write of one physical block: its K and V bytes (n16 16-byte pieces
// each) from block `src` to block `dst` of the pools, and its FP8 half scales
// when the pools have them.
__device__ __forceinline__ void block_copy_body(uint4 *k_pool, uint4 *v_pool, uint16_t *k_scale, uint16_t *v_scale,
                                                int64_t n16, int32_t src, int32_t dst) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n16) {
        k_pool[(int64_t)dst * n16 + i] = k_pool[(int64_t)src * n16 + i];
        v_pool[(int64_t)dst * n16 + i] = v_pool[(int64_t)src * n16 + i];
    }
    if (i == 0 && k_scale) {
        k_scale[dst] = k_scale[src];
        v_scale[dst] = v_scale[src];
    }
}

}  // namespace pam
