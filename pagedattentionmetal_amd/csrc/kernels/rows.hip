// rows.hip - attention over blocks of query rows with f32 probabilities on the
// matrix units (gfx950): prefill and decode kernels and their launchers.  The
// bodies are in rows_body.h.
#include "rows_body.h"

#include <algorithm>
#include <cmath>

namespace pam {

template <typename KV, typename QT, int NT>
__global__ __launch_bounds__(64 * kRowsWaves, (NT <= 4 ? 2 : 1)) void prefill_rows_kernel(AttnParams p) {
    __shared__ __attribute__((aligned(16))) float lds[kRowsLds<NT, kPrefillRowsRB<KV, NT>>];
    prefill_rows_body<KV, QT, NT>(p, lds);
}

template <typename KV, typename QT, int NT>
__global__ __launch_bounds__(64 * kRowsWaves, (NT <= 4 ? 2 : 1)) void decode_rows_kernel(AttnParams p) {
    __shared__ __attribute__((aligned(16))) float lds[kRowsLds<NT, 1>];
    decode_rows_body<KV, QT, NT>(p, lds);
}

// the instantiation (NT = 1, 2, 3, 4, 8 tiles of 32 dims) that takes a head size
static int dim_slot(int32_t head_dim) {
    const int nt = (head_dim + 31) / 32;
    return nt <= 4 ? nt - 1 : 4;
}

// Whole pieces of a head's row (16 bytes of Q and of f32 / f16 K, 8 of e4m3) and
// their alignment; every row keeps the buffers' alignment then.
bool rows_supported(const AttnParams &p, int32_t dtype) {
    if (p.head_dim <= 0 || p.head_dim > 256 || p.head_dim % (dtype == kF32 ? 4 : 8) != 0) return false;
    const uintptr_t kv = (uintptr_t)p.k_pool | (uintptr_t)p.v_pool, io = (uintptr_t)p.q | (uintptr_t)p.out;
    return (kv & (dtype == kFP8 ? 7 : 15)) == 0 && (io & 15) == 0;
}

// query rows of a prefill block (kPrefillRowsRB)
static int64_t block_rows(int32_t head_dim, int32_t dtype) { return dtype == kF32 && head_dim > 128 ? 16 : 32; }

// Partition length of a prefill of p.rows rows over its keys: the candidate whose
// estimate is least.  Two workgroups fit a CU, two waves a SIMD.  The launch takes
// the larger of its whole work over those places and its longest workgroup, half of
// that again when the workgroups need several rounds, and partitions cost the
// reduce.  The constants are fits to calls measured on gfx950 (µs, estimate /
// measured: f32 8/8 d = 128, 777 tokens after 391 in partitions of 24 tiles 49 / 51,
// of 12 65 / 61; 17 after 2000 in partitions of 4 17 / 17; 64 in one 11 / 8; f32 32/8
// 2048 tokens in one 457 / 378, of 32 505 / 468).
int32_t prefill_rows_part_tokens(const AttnParams &p, int32_t dtype, int32_t cus) {
    constexpr double kStartUs = 8.0, kReduceUs = 4.0, kReduceGBs = 3000.0, kCyclesPerUs = 2400.0;
    const int64_t G = p.num_heads / p.num_kv_heads;
    const int64_t kv_len = (int64_t)p.q_offset + p.rows;
    const int64_t k_lo = p.window > 0 && kv_len > p.window ? (kv_len - p.window) / 16 * 16 : 0;
    const int64_t R = block_rows(p.head_dim, dtype), nblocks = (p.rows * G + R - 1) / R, nt = (p.head_dim + 31) / 32;
    const int64_t longest = (kv_len - k_lo + 15) / 16;
    const int64_t first = p.q_offset + (R + G - 1) / G;  // keys of the first block's last row
    const int64_t shortest = p.causal ? std::max<int64_t>(0, (std::min(first, kv_len) - k_lo + 15) / 16) : longest;
    // a tile's matrix cycles (f32: scores and outputs; else the outputs) and the rest of its work
    const double tile_us = 1.4 * (R / 16) * (dtype == kF32 ? 512.0 : 280.0) * nt / kCyclesPerUs + 0.2;
    const double tiles = 0.5 * (shortest + longest) * nblocks * p.num_kv_heads, places = 2.0 * (cus > 0 ? cus : 1);
    double best = 1e300;
    int64_t best_per = longest;
    for (int64_t w = 1;; w = w < 8 ? w + 1 : w + w / 4) {  // tiles per wave
        const int64_t per = w * kRowsWaves;
        double groups = 0.0;
        const int64_t samples = std::min<int64_t>(nblocks, 64);
        for (int64_t i = 0; i < samples; i++) {
            const int64_t t = samples > 1 ? shortest + (longest - shortest) * i / (samples - 1) : longest;
            groups += (double)std::max<int64_t>(1, (t + per - 1) / per);
        }
        groups *= (double)nblocks / samples * p.num_kv_heads;
        const double share = 2.0 * groups <= places ? 1.0 : 2.0;  // waves a SIMD
        const double one = kStartUs + share * tile_us * (double)std::min(w, (longest + kRowsWaves - 1) / kRowsWaves);
        double us = std::max(one, (groups * kStartUs + tiles / kRowsWaves * share * tile_us) / places);
        if (groups > places) us += 0.5 * one;
        if (per < longest) us += kReduceUs + 8.0 * groups * R * p.head_dim / (kReduceGBs * 1e3);
        if (us < best) best = us, best_per = per;
        if (per >= longest) break;
    }
    return (int32_t)(best_per >= longest ? (longest + 1) * 16 : best_per * 16);
}

#define PAM_ROWS_SWITCH(KERNEL)                                                                        \
    switch (dim_slot(p.head_dim)) {                                                                    \
        case 0: hipLaunchKernelGGL((KERNEL<KV, QT, 1>), grid, block, 0, stream, p); break;             \
        case 1: hipLaunchKernelGGL((KERNEL<KV, QT, 2>), grid, block, 0, stream, p); break;             \
        case 2: hipLaunchKernelGGL((KERNEL<KV, QT, 3>), grid, block, 0, stream, p); break;             \
        case 3: hipLaunchKernelGGL((KERNEL<KV, QT, 4>), grid, block, 0, stream, p); break;             \
        default: hipLaunchKernelGGL((KERNEL<KV, QT, 8>), grid, block, 0, stream, p); break;            \
    }

template <typename KV, typename QT>
static hipError_t launch_rows(const AttnParams &p, hipStream_t stream, const KernelTable *kt) {
    const dim3 block(64 * kRowsWaves);
    const int kvi = sizeof(KV) == 4 ? 0 : (sizeof(KV) == 2 ? 1 : 2);
    const int64_t G = p.num_heads / p.num_kv_heads;
    const int64_t parts = p.max_parts > 1 ? p.max_parts : 1;
    hipError_t me;
    if (p.mode == kRowPrefill) {
        const int64_t R = block_rows(p.head_dim, kvi == 0 ? kF32 : kF16), nblocks = ((int64_t)p.rows * G + R - 1) / R;
        if (nblocks * p.num_kv_heads >= ((int64_t)1 << 31) || p.rows * G >= ((int64_t)1 << 31) - 32 || parts > kMaxGridYZ)
            return hipErrorInvalidValue;
        const dim3 grid((unsigned)(nblocks * p.num_kv_heads), (unsigned)parts);
        if (via_module(kt, kt ? kt->prefill_rows[kvi][dim_slot(p.head_dim)] : nullptr, &me, grid, block, stream, p)) return me;
        PAM_ROWS_SWITCH(prefill_rows_kernel)
        return hipGetLastError();
    }
    const int64_t slots = p.num_kv_heads * ((G + 15) / 16);
    if (p.rows > kMaxGridYZ || parts > kMaxGridYZ) return hipErrorInvalidValue;
    const dim3 grid((unsigned)slots, (unsigned)p.rows, (unsigned)parts);
    if (via_module(kt, kt ? kt->decode_rows[kvi][dim_slot(p.head_dim)] : nullptr, &me, grid, block, stream, p)) return me;
    PAM_ROWS_SWITCH(decode_rows_kernel)
    return hipGetLastError();
}

hipError_t launch_rows(const AttnParams &p, int32_t dtype, hipStream_t stream, hipEvent_t after_main,
                       const KernelTable *kt) {
    if (p.rows <= 0) return hipSuccess;
    if (!rows_supported(p, dtype) || !p.row_blocks || p.part_tokens <= 0 || p.part_tokens % 16 != 0 ||
        p.zero_page == nullptr || (p.max_parts > 1 && (p.part_o == nullptr || p.part_ml == nullptr)))
        return hipErrorInvalidValue;
    hipError_t e;
    switch (dtype) {
        case kF32: e = launch_rows<float, float>(p, stream, kt); break;
        case kF16: e = launch_rows<f16, f16>(p, stream, kt); break;
        case kFP8: e = launch_rows<uint8_t, f16>(p, stream, kt); break;
        default: return hipErrorInvalidValue;
    }
    if (e != hipSuccess) return e;
    if (after_main) (void)hipEventRecord(after_main, stream);
    return p.max_parts > 1 ? launch_reduce(p, dtype, stream, kt) : e;
}

}  // namespace pam
