// rows_body.h - attention over blocks of query rows with f32 probabilities on
// the matrix units (gfx950): the prefill of f32 caches and of the f16 / e4m3
// head sizes and block sizes the dense prefill does not take, and the decode of
// f32 caches, small head groups and those same sizes.  Included by rows.hip
// (the library's kernels) and by the code-object entries.
//
// A wave owns RB blocks of 16 query rows (token, head) of one kv head and walks
// 16-key tiles.  S^T = K Q^T runs on v_mfma_f32_16x16x4_f32 (f32 caches) or
// v_mfma_f32_16x16x32_f16 (f16 and dequantised e4m3: exact products, f32 sums);
// lane (n, g) = (lane % 16, lane / 16) then holds keys 4g .. 4g + 3 of row n, and
// accumulator register r is, as it stands, the B operand of
// O^T += V^T P^T over the keys {r, 4 + r, 8 + r, 12 + r} on
// v_mfma_f32_16x16x4_f32.  Probabilities, sums and outputs stay in f32 registers.
//
// Sums of f32 caches: a score adds up in a tree (dot_tree), a tile's outputs by
// themselves before they join the row's.  Error norms against 64 bits over those of
// the VALU rows (which add a lane's 4 products and then lanes, pairwise), geometric
// mean and largest of 30 to 60 calls a head size: decode 0.87-0.93 and 1.05-1.16 (a few
// outputs of one row), prefill 0.66-0.90 and 1.03; d > 128 0.83 and 0.98, 0.76 and 0.94.
// With one chain of a tile's outputs and two to eight chains of a score: 0.96-1.06 and
// 1.23, 0.80-1.07 and 1.40.  Time against that: prefills of 2048 tokens 2-5% more, short
// ones 4-16%, decodes 2-5%, short ones up to 9%; d > 128 3-10%, 5-20% with trees of 4
// dims there (ragged 264 rows of 16/16 d = 256 654 us, 722 and 787).  Trees of 8 dims
// up to d = 128: decode 0.96-1.02 and 1.10, prefill 0.92-1.00 and 1.05.
//
// Operands come straight from the pools: a lane loads its K operand in 16-byte
// pieces (a key's 64 bytes per instruction) and its V operand as VW consecutive
// dims of one key (whole 256-byte rows per instruction at d = 128), one tile
// ahead.  The 16-key tiles were chosen for the first of these: with 32-key tiles
// a K instruction takes 32 bytes from each of 32 rows, and the waves' open lines
// no longer fit the first-level cache.
//
// What bounds it: a prefill of f32 caches, the f32 matrix rate (a 16-key tile of
// 32 rows is 4096 matrix cycles at d = 128); a decode, the pools' bytes (a tile
// is 2048 matrix cycles for 16 KB in f32, 1150 for 8 KB in f16), and, for e4m3,
// the f32 matrix time of O^T.  Measured on gfx950 against the VALU rows that
// served these calls before (µs per call): f32 8/8 d = 128, 777 tokens after 391
// 784 -> 55 (44 TFLOP/s); f32 32/8 d = 128, 2048 tokens 399 (86 TFLOP/s); f16
// 32/8 d = 96, 2048 tokens 162 (159 TFLOP/s); f16 16/16 d = 64 decode of 24 rows
// of up to 3000 tokens 162 -> 48 (3.4 TB/s); f32 8/8 d = 128 64 rows of up to
// 2000 130 -> 124; f32 32/8 d = 128 one row of 5598 646 -> 22; e4m3 12/4 d = 128
// 205 rows of up to 4000 2617 -> 175.
#pragma once
#include "valu_body.h"

namespace pam {

constexpr int kRowsWaves = 4;  // waves of a workgroup

// 8 e4m3 codes as binary16, dequantised as fp8_dequant does.  The hardware
// conversion and one product differ from it for the codes 0x7F / 0xFF and for
// scales that are not finite; those take it.
__device__ __forceinline__ f16x8 e4m3x8_dequant(uint32_t w0, uint32_t w1, f16 scale) {
    auto top = [](uint32_t w) { return ((w & 0x7F7F7F7Fu) + 0x01010101u) & 0x80808080u; };
    f16x8 v;
    if (__builtin_expect((top(w0) | top(w1)) != 0u || !__builtin_isfinite((float)scale), 0)) {
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = fp8_dequant(((i < 4 ? w0 : w1) >> (8 * (i & 3))) & 0xFFu, scale);
    } else {
        v = e4m3x8_to_f16x8(w0, w1) * scale;
    }
    return v;
}

// N consecutive elements of a V row as they lie in the pool (a load in flight),
// and their values as floats
template <typename KV, int N>
struct RawVec {
    typedef KV V __attribute__((ext_vector_type(N)));
    V v;
    __device__ __forceinline__ void load(const void *ptr) { v = *static_cast<const V *>(ptr); }
    __device__ __forceinline__ void floats(uint16_t scale, float *out) const {
        if constexpr (sizeof(KV) == 1) {
            uint32_t w[2] = {0u, 0u};
            __builtin_memcpy(w, &v, N);
            const f16x8 x = e4m3x8_dequant(w[0], w[1], bits_to_f16(scale));
#pragma unroll
            for (int i = 0; i < N; i++) out[i] = (float)x[i];
        } else {
#pragma unroll
            for (int i = 0; i < N; i++) out[i] = (float)v[i];
        }
    }
};

template <typename KV>
struct KPiece;
template <>
struct KPiece<float> {
    typedef f32x4 K;
    typedef f32x4 Q;
};
template <>
struct KPiece<f16> {
    typedef f16x8 K;
    typedef f16x8 Q;
};
template <>
struct KPiece<uint8_t> {
    typedef uint32_t K __attribute__((ext_vector_type(2)));
    typedef f16x8 Q;
};

// A pool's token slot of token `slot` of a block: 64 bits, as a pool of narrow rows
// holds more than 2^31 of them (tests/native/pool_slot_check.cpp)
__host__ __device__ __forceinline__ int64_t pool_slot(int32_t block, int block_size, int slot) {
    return (int64_t)block * block_size + slot;
}

__host__ __device__ __forceinline__ int block_shift(int bs) { return (bs & (bs - 1)) == 0 ? __builtin_ctz((unsigned)bs) : -1; }

// Pool slots of a backward's sequence (-1 outside its keys)
struct KeySlots {
    const int32_t *bt;
    int lo, hi, bs, shift;
    __host__ __device__ __forceinline__ KeySlots(const BackwardParams &p)
        : bt(p.block_table), lo(p.window_start), hi(p.seq_len), bs(p.block_size), shift(block_shift(p.block_size)) {}
    __host__ __device__ __forceinline__ int64_t at(int j) const {
        if (j < lo || j >= hi) return -1;
        const int b = shift >= 0 ? j >> shift : j / bs;
        return pool_slot(bt[b], bs, j - b * bs);
    }
};

// The keys of a workgroup: tile t holds keys key0 + 16 t .. + 15 of the block
// table's sequence.  Loads stay inside [lo, hi).
struct TileKeys {
    const int32_t *bt;
    int key0, lo, hi;   // keys any row of the wave sees: lo .. hi - 1
    int hi_all;         // keys below it (from lo on) are seen by every row
    int block_size, shift;  // shift: log2(block_size), or -1
};

// The compiler otherwise moves additions whose results are read later down to there,
// and every product summed by them holds its registers until then.
__device__ __forceinline__ void keep_here(f32x4 &x) { asm volatile("" : "+v"(x)); }

// f32 products of 16 rows a and 16 columns b over KC pieces of 16 dims (4 a lane).
// The matrix unit sums LEAF dims, and these sums add up in a tree, as the VALU kernels
// add a lane's 4 products and then the lanes.  The additions of a piece follow the
// products of the next, which hide them.
template <int LEAF, int KC>
__device__ __forceinline__ f32x4 dot_tree(const f32x4 (&a)[KC], const f32x4 (&b)[KC]) {
    constexpr int T = 16 / LEAF;  // leaves of a piece
    f32x4 t[2][T], level[8];
    // the additions of piece c, in the order in which its products end
    auto add = [&](int c, int step) {
        f32x4 *x = t[c & 1];
        if (T == 4 && step < 2) {
            x[step] += x[step + 2];
            keep_here(x[step]);
        } else if (step == 2) {
            x[0] += x[1];
            keep_here(x[0]);
        } else if (step == 3) {
            int l = 0;
#pragma unroll
            for (; (c >> l) & 1; l++) x[0] += level[l];
            level[l] = x[0];
            keep_here(level[l]);
        }
    };
#pragma unroll
    for (int c = 0; c < KC; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            f32x4 &x = t[c & 1][e % T];
            x = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][e], b[c][e], e < T ? (f32x4)0.0f : x, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (c) add(c - 1, e);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
    for (int e = 0; e < 4; e++) add(KC - 1, e);
    f32x4 s = (f32x4)0.0f;
    bool any = false;
#pragma unroll
    for (int l = 0; l < 8; l++)
        if ((KC >> l) & 1) s = any ? s + level[l] : level[l], any = true;
    keep_here(s);
    return s;
}

template <typename KV, typename QT, int NT, int RB>
struct RowTiles {
    static constexpr bool F32 = sizeof(KV) == 4;
    static constexpr int KC = F32 ? 2 * NT : NT;     // K loads of a tile
    static constexpr int KD = F32 ? 4 : 8;           // dims per lane and K load
    // V: A row m of dim tile t = u VW + w is dim 16 VW u + VW m + w
    static constexpr int VW = F32 ? (NT % 2 == 0 ? 4 : 2) : (NT % 4 == 0 ? 8 : (NT == 2 ? 4 : 2));
    static constexpr int NU = 2 * NT / VW;
    static constexpr int LS = 32 * NT + 4;           // LDS row stride (floats)
    // dot_tree's: 8 where the registers hold no more, and where the sums are no further
    // from 64 bits than the VALU rows' all the same (d > 128)
    static constexpr int LEAF = NT > 4 || (RB > 1 && NT > 3) ? 8 : 4;
    typedef typename KPiece<KV>::K KOp;
    typedef typename KPiece<KV>::Q QOp;

    QOp q[RB][KC];
    f32x4 o[RB][2 * NT];
    float m[RB], l[RB];  // reference max (log2 units) and this lane's share of the sum
    KOp k[KC];
    RawVec<KV, VW> v[4][NU];
    uint16_t ks, vs[4];
    bool odd;            // a V row outside some row's keys was not finite

    int n, g;
    const char *kbase, *vbase, *zero;
    int64_t row_bytes;
    int d;

    __device__ __forceinline__ void init(const AttnParams &p, int kvh) {
        const int lane = threadIdx.x & 63;
        n = lane & 15, g = lane >> 4;
        d = p.head_dim;
        row_bytes = (int64_t)p.num_kv_heads * d * (int)sizeof(KV);
        kbase = static_cast<const char *>(p.k_pool) + (int64_t)kvh * d * (int)sizeof(KV);
        vbase = static_cast<const char *>(p.v_pool) + (int64_t)kvh * d * (int)sizeof(KV);
        zero = static_cast<const char *>(p.zero_page);
        odd = false;
        ks = 0;
#pragma unroll
        for (int b = 0; b < RB; b++) {
            m[b] = -INFINITY;
            l[b] = 0.0f;
#pragma unroll
            for (int t = 0; t < 2 * NT; t++) o[b][t] = (f32x4)0.0f;
        }
    }
    // dims of piece c in this lane; pieces past head_dim are zeros (zero page)
    __device__ __forceinline__ int k_dim(int c) const { return 4 * KD * c + KD * g; }
    __device__ __forceinline__ void load_q(int b, const QT *row) {
#pragma unroll
        for (int c = 0; c < KC; c++)
            q[b][c] = *reinterpret_cast<const QOp *>(k_dim(c) < d ? (const char *)(row + k_dim(c)) : zero);
    }
    __device__ __forceinline__ void issue_k(const AttnParams &p, int64_t row, int block) {
        const char *ptr = kbase + row * row_bytes;
        if constexpr (sizeof(KV) == 1) ks = p.k_scale[block];
#pragma unroll
        for (int c = 0; c < KC; c++)
            k[c] = *reinterpret_cast<const KOp *>(k_dim(c) < d ? ptr + k_dim(c) * (int)sizeof(KV) : zero);
    }
    __device__ __forceinline__ void issue_v(const AttnParams &p, int64_t row, int block) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const char *ptr = vbase + __shfl(row, 4 * g + r, 64) * row_bytes;
            if constexpr (sizeof(KV) == 1) vs[r] = p.v_scale[__shfl(block, 4 * g + r, 64)];
#pragma unroll
            for (int u = 0; u < NU; u++) {
                const int e0 = 16 * VW * u + VW * n;
                v[r][u].load(e0 < d ? ptr + e0 * (int)sizeof(KV) : zero);
            }
        }
    }

    // Tiles t0, t0 + step, .. below t1.  k_hi[b]: end of the keys of row n of block b.
    __device__ __forceinline__ void run(const AttnParams &p, const TileKeys &keys, const int (&k_hi)[RB], int t0, int t1,
                                        int step) {
        if (t0 >= t1) return;
        const int bs = keys.block_size;
        auto lookup = [&](int t, int &slot) {
            int j = keys.key0 + 16 * t + n;
            j = j < keys.lo ? keys.lo : (j < keys.hi ? j : keys.hi - 1);
            const int b = keys.shift >= 0 ? j >> keys.shift : j / bs;
            slot = j - b * bs;
            return keys.bt[b];
        };
        int slot, block = lookup(t0, slot), slot_n = 0, block_n = 0;
        if (t0 + step < t1) block_n = lookup(t0 + step, slot_n);
        issue_k(p, pool_slot(block, bs, slot), block);
        issue_v(p, pool_slot(block, bs, slot), block);
        for (int t = t0; t < t1; t += step) {
            const int kb = keys.key0 + 16 * t;
            const bool more = t + step < t1;
            f32x4 s[RB];
            if constexpr (F32) {
#pragma unroll
                for (int b = 0; b < RB; b++) s[b] = dot_tree<LEAF, KC>(k, q[b]);
            } else {
#pragma unroll
                for (int b = 0; b < RB; b++) s[b] = (f32x4)0.0f;
#pragma unroll
                for (int c = 0; c < KC; c++) {
                    f16x8 a;
                    if constexpr (sizeof(KV) == 1)
                        a = e4m3x8_dequant(k[c][0], k[c][1], bits_to_f16(ks));
                    else
                        a = k[c];
#pragma unroll
                    for (int b = 0; b < RB; b++) s[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, q[b][c], s[b], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            // the next tile's K, and the block-table entry of the one after
            const int64_t row_n = pool_slot(block_n, bs, slot_n);
            const int blk_n = block_n;
            if (more) {
                if (t + 2 * step < t1) block_n = lookup(t + 2 * step, slot_n);
                issue_k(p, row_n, blk_n);
            }
            __builtin_amdgcn_sched_barrier(0);
            // Online softmax.  The reference max of a row moves only when a score
            // passes it by 8, a factor of 2^8 (or the row has none yet): the probabilities
            // are f32, so their scale is free, and most tiles need no reduction across
            // lanes.
            const bool full = kb >= keys.lo && kb + 16 <= keys.hi_all;
            bool grow = false;
#pragma unroll
            for (int b = 0; b < RB; b++) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float x = s[b][r] * p.scale_log2;
                    if (!full) {
                        const int j = kb + 4 * g + r;
                        x = j >= keys.lo && j < keys.hi && j < k_hi[b] ? x : -INFINITY;
                    }
                    s[b][r] = x;
                    grow |= x > m[b] + 8.0f;
                }
            }
            if (__any(grow)) {
#pragma unroll
                for (int b = 0; b < RB; b++) {
                    float mt = fmaxf(fmaxf(s[b][0], s[b][1]), fmaxf(s[b][2], s[b][3]));
                    mt = fmaxf(mt, shfl_xor(mt, 16));
                    mt = fmaxf(mt, shfl_xor(mt, 32));
                    const float m_new = fmaxf(m[b], mt);
                    const float corr = m[b] == -INFINITY ? 0.0f : exp2f(m[b] - m_new);
                    if (m_new > m[b]) l[b] *= corr;
#pragma unroll
                    for (int i = 0; i < 2 * NT; i++) o[b][i] = m_new > m[b] ? o[b][i] * corr : o[b][i];
                    m[b] = m_new;
                }
            }
#pragma unroll
            for (int b = 0; b < RB; b++) {
                const float m_use = m[b] == -INFINITY ? 0.0f : m[b];  // a row without keys so far
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    s[b][r] = exp2f(s[b][r] - m_use);
                    l[b] += s[b][r];
                }
            }
            // O^T.  In an edge tile a V element of a key that some row must not see
            // enters only if it is finite (0 * Inf would reach the rows that mask
            // it); add_odd gives the others to the rows that do see the key.
            auto hide = [&](int r, float &x) {
                const int j = kb + 4 * g + r;
                const bool bad = !(j >= keys.lo && j < keys.hi_all) && !__builtin_isfinite(x);
                odd |= bad;
                x = bad ? 0.0f : x;
            };
            if constexpr (F32) {
                if (!full)
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int i = 0; i < 2 * NT; i++) {
                            float x = v[r][i / VW].v[i % VW];
                            hide(r, x);
                            v[r][i / VW].v[i % VW] = x;
                        }
                // A tile's sum by itself, in two chains of 8 keys, then added; the additions
                // follow the next sum's products, as in dot_tree.
                constexpr int N = 2 * NT * RB;
                f32x4 t[2][2];
                auto add = [&](int x, int step) {
                    f32x4 *y = t[x & 1], &sum = o[x % RB][x / RB];
                    if (step == 2) y[0] += y[1], keep_here(y[0]);
                    if (step == 3) sum += y[0], keep_here(sum);
                };
#pragma unroll
                for (int x = 0; x < N; x++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int i = x / RB;
                        f32x4 &y = t[x & 1][r & 1];
                        y = __builtin_amdgcn_mfma_f32_16x16x4f32(v[r][i / VW].v[i % VW], s[x % RB][r],
                                                                 r < 2 ? (f32x4)0.0f : y, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (x) add(x - 1, r);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                add(N - 1, 2), add(N - 1, 3);
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    float a[2 * NT];
#pragma unroll
                    for (int u = 0; u < NU; u++) v[r][u].floats(sizeof(KV) == 1 ? vs[r] : (uint16_t)0, a + VW * u);
                    if (!full)
#pragma unroll
                        for (int i = 0; i < 2 * NT; i++) hide(r, a[i]);
#pragma unroll
                    for (int i = 0; i < 2 * NT; i++)
#pragma unroll
                        for (int b = 0; b < RB; b++)
                            o[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], s[b][r], o[b][i], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (more) issue_v(p, row_n, blk_n);
        }
#pragma unroll
        for (int b = 0; b < RB; b++) {
            l[b] += shfl_xor(l[b], 16);
            l[b] += shfl_xor(l[b], 32);
        }
    }

    // O^T of block b times f into the LDS row of row n
    __device__ __forceinline__ void put(int b, float f, float *row) const {
#pragma unroll
        for (int u = 0; u < NU; u++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float *dst = row + 16 * VW * u + VW * (4 * g + r);
#pragma unroll
                for (int w = 0; w < VW; w++) dst[w] = o[b][VW * u + w][r] * f;
            }
    }
};

// floats of LDS: every wave's O^T and (m, l) of its rows
template <int NT, int RB>
constexpr int kRowsLds = kRowsWaves * 16 * RB * (32 * NT + 4 + 2);

// 4 dims of a row's output and its denominator, from the waves' O^T scaled to the
// common maximum M.
struct RowSum {
    float a[4], den, M;
};
__device__ __forceinline__ RowSum row_sum(const float *o, int o_stride, const float *ml, int ml_stride) {
    RowSum s{{0.f, 0.f, 0.f, 0.f}, 0.0f, -INFINITY};
    for (int w = 0; w < kRowsWaves; w++) s.M = fmaxf(s.M, ml[w * ml_stride]);
    for (int w = 0; w < kRowsWaves; w++) {
        const float mw = ml[w * ml_stride];
        s.den += mw == -INFINITY ? 0.0f : exp2f(mw - s.M) * ml[w * ml_stride + 1];
        const float4 v = *reinterpret_cast<const float4 *>(o + w * o_stride);
        s.a[0] += v.x, s.a[1] += v.y, s.a[2] += v.z, s.a[3] += v.w;
    }
    // a row whose scores are all NaN keeps no maximum: its sum is NaN all the same
    for (int w = 0; w < kRowsWaves; w++)
        if (__builtin_isnan(ml[w * ml_stride + 1])) s.den = ml[w * ml_stride + 1];
    return s;
}

// The V elements RowTiles::run left out: not finite, at keys [j0, j1) that the
// row sees and some other row of its block does not.  Adds p v to a's 4 dims at e0.
template <typename KV, typename QT>
__device__ __forceinline__ void add_odd(const AttnParams &p, const int32_t *bt, const QT *qr, int kvh, int e0, int j0,
                                        int j1, float M, float *a) {
    const int d = p.head_dim, bs = p.block_size;
    const float m_use = M == -INFINITY ? 0.0f : M;
    for (int j = j0; j < j1; j++) {
        const int blk = bt[j / bs];
        const int64_t off = (pool_slot(blk, bs, j % bs) * p.num_kv_heads + kvh) * d;
        f16 ks = (f16)1.0f, vs = (f16)1.0f;
        if constexpr (sizeof(KV) == 1) ks = bits_to_f16(p.k_scale[blk]), vs = bits_to_f16(p.v_scale[blk]);
        float v[4];
        load_kv4<KV>(static_cast<const KV *>(p.v_pool) + off + e0, vs, v);
        if (__builtin_isfinite(v[0]) && __builtin_isfinite(v[1]) && __builtin_isfinite(v[2]) && __builtin_isfinite(v[3]))
            continue;
        float sd = 0.0f;
        for (int e = 0; e < d; e += 4) {
            float kv[4], qv[4];
            load_kv4<KV>(static_cast<const KV *>(p.k_pool) + off + e, ks, kv);
            load4<QT>(qr + e, qv);
            sd += qv[0] * kv[0] + qv[1] * kv[1] + qv[2] * kv[2] + qv[3] * kv[3];
        }
        const float pj = exp2f(sd * p.scale_log2 - m_use);
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (!__builtin_isfinite(v[e])) a[e] += pj * v[e];
    }
}

// 4 dims of a row: the result, or the row's partial for attn_reduce_kernel
template <typename QT>
__device__ __forceinline__ void write_row(const AttnParams &p, int64_t out_row, int64_t row, int head, int part, int np,
                                          int e0, RowSum &s) {
    if (np <= 1) {
        const float inv = 1.0f / s.den;
#pragma unroll
        for (int e = 0; e < 4; e++) s.a[e] *= inv;
        store4<QT>(static_cast<QT *>(p.out) + (out_row * p.num_heads + head) * (int64_t)p.head_dim + e0, s.a);
    } else {
        const int64_t slot = (row * p.num_heads + head) * p.max_parts + part;
        store4<float>(p.part_o + slot * p.head_dim + e0, s.a);
        if (e0 == 0) {
            p.part_ml[slot * 2] = s.M;
            p.part_ml[slot * 2 + 1] = s.den;
        }
    }
}

// 16-row blocks of a prefill wave: two share every K and V operand (one where
// the registers hold no more)
template <typename KV, int NT>
constexpr int kPrefillRowsRB = sizeof(KV) == 4 && NT > 4 ? 1 : 2;

// Prefill: a workgroup runs one block of 16 RB query rows over one partition of its
// keys, its waves taking the tiles in turn.  grid: x = kv head + Hkv * block
// (blocks from the last to the first: the longest causal ones start first; a kv
// head's blocks fall on one XCD when Hkv is a multiple of 8), y = partition.
template <typename KV, typename QT, int NT>
__device__ __forceinline__ void prefill_rows_body(const AttnParams &p, float *lds) {
    constexpr int RB = kPrefillRowsRB<KV, NT>, RN = 16 * RB;
    typedef RowTiles<KV, QT, NT, RB> Tiles;
    constexpr int LS = Tiles::LS;
    const int tid = threadIdx.x, wave = tid >> 6;
    const int Hkv = p.num_kv_heads, H = p.num_heads, G = H / Hkv, d = p.head_dim;
    const int nrows = p.rows * G, nblocks = (nrows + RN - 1) / RN;
    const int kvh = blockIdx.x % Hkv, row0 = (nblocks - 1 - (int)(blockIdx.x / Hkv)) * RN, part = blockIdx.y;
    const int last = row0 + RN - 1 < nrows ? row0 + RN - 1 : nrows - 1;
    const int kv_len = p.q_offset + p.rows;
    const int k_lo = p.window > 0 && kv_len > p.window ? kv_len - p.window : 0;
    const int tile0 = k_lo / 16, tpp = p.part_tokens / 16;
    TileKeys keys;
    keys.bt = p.block_tables;
    keys.block_size = p.block_size;
    keys.shift = block_shift(p.block_size);
    keys.key0 = (tile0 + part * tpp) * 16;
    keys.lo = k_lo;
    keys.hi = p.causal ? p.q_offset + last / G + 1 : kv_len;
    keys.hi_all = p.causal ? p.q_offset + row0 / G + 1 : kv_len;
    if (part > 0 && keys.key0 >= keys.hi) return;
    int ntiles = keys.hi > k_lo ? (keys.hi - keys.key0 + 15) / 16 : 0;
    ntiles = ntiles < tpp ? ntiles : tpp;

    Tiles x;
    x.init(p, kvh);
    int k_hi[RB];
#pragma unroll
    for (int b = 0; b < RB; b++) {
        const int rho = row0 + 16 * b + x.n <= last ? row0 + 16 * b + x.n : last;
        const int tok = rho / G;
        k_hi[b] = p.causal ? p.q_offset + tok + 1 : kv_len;
        x.load_q(b, static_cast<const QT *>(p.q) + ((int64_t)tok * H + kvh * G + rho % G) * d);
    }
    x.run(p, keys, k_hi, wave, ntiles, kRowsWaves);

    // merge the waves: O^T scaled to the row maxima, summed by all threads
    float *ml = lds + kRowsWaves * RN * LS;  // [wave][row][2]
    const bool any_odd = __syncthreads_or(x.odd);
    if (x.g == 0) {
#pragma unroll
        for (int b = 0; b < RB; b++) {
            ml[(wave * RN + 16 * b + x.n) * 2] = x.m[b];
            ml[(wave * RN + 16 * b + x.n) * 2 + 1] = x.l[b];
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < RB; b++) {
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kRowsWaves; w++) M = fmaxf(M, ml[(w * RN + 16 * b + x.n) * 2]);
        x.put(b, x.m[b] == -INFINITY ? 0.0f : exp2f(x.m[b] - M), lds + (wave * RN + 16 * b + x.n) * LS);
    }
    __syncthreads();
    for (int i = tid; i < RN * (d / 4); i += 64 * kRowsWaves) {
        const int rn = i / (d / 4), e0 = i % (d / 4) * 4, rho = row0 + rn;
        if (rho > last) continue;
        const int rt = rho / G, head = kvh * G + rho % G;
        const int rhi = p.causal ? p.q_offset + rt + 1 : kv_len;
        const int np = rhi > k_lo ? ((rhi + 15) / 16 - tile0 + tpp - 1) / tpp : 0;
        if (part >= np && part > 0) continue;  // part 0 writes the rows without keys (0 / 0)
        RowSum s = row_sum(lds + rn * LS + e0, RN * LS, ml + rn * 2, RN * 2);
        if (any_odd) {
            const int j0 = keys.hi_all > keys.lo ? keys.hi_all : keys.lo, j1 = keys.key0 + 16 * ntiles;
            add_odd<KV, QT>(p, p.block_tables, static_cast<const QT *>(p.q) + ((int64_t)rt * H + head) * d, kvh, e0,
                            j0 > keys.key0 ? j0 : keys.key0, j1 < rhi ? j1 : rhi, s.M, s.a);
        }
        write_row<QT>(p, rt, rt, head, part, np, e0, s);
    }
}

// Decode and ragged rows: a workgroup runs one (row, slot) over one partition,
// its waves taking the tiles in turn.  A slot is up to 16 query heads of one kv
// head.  grid: x = slot, y = row, z = partition.
template <typename KV, typename QT, int NT>
__device__ __forceinline__ void decode_rows_body(const AttnParams &p, float *lds) {
    typedef RowTiles<KV, QT, NT, 1> Tiles;
    constexpr int LS = Tiles::LS;
    const int tid = threadIdx.x, wave = tid >> 6;
    const int H = p.num_heads, G = H / p.num_kv_heads, d = p.head_dim;
    const int sub = (G + 15) / 16, r = blockIdx.y, part = blockIdx.z;
    const int kvh = blockIdx.x / sub, h0 = blockIdx.x % sub * 16;
    const int nh = G - h0 < 16 ? G - h0 : 16;  // query heads of the slot
    const RowCtx c = row_ctx(p, r);
    const PartRange pr = part_range(c, part, p.part_tokens);
    if (part >= (pr.nparts > 1 ? pr.nparts : 1)) return;
    TileKeys keys;
    keys.bt = c.bt;
    keys.block_size = p.block_size;
    keys.shift = block_shift(p.block_size);
    keys.key0 = pr.t_begin * 16;
    keys.lo = c.k_lo;
    keys.hi = keys.hi_all = c.k_hi;

    Tiles x;
    x.init(p, kvh);
    x.load_q(0, static_cast<const QT *>(p.q) + ((int64_t)c.out_row * H + kvh * G + h0 + (x.n < nh ? x.n : nh - 1)) * d);
    const int k_hi[1] = {c.k_hi};
    x.run(p, keys, k_hi, wave, pr.nparts > 0 ? pr.t_end - pr.t_begin : 0, kRowsWaves);

    float *ml = lds + kRowsWaves * 16 * LS;
    if (x.g == 0) {
        ml[(wave * 16 + x.n) * 2] = x.m[0];
        ml[(wave * 16 + x.n) * 2 + 1] = x.l[0];
    }
    __syncthreads();
    float M = -INFINITY;
    #pragma unroll
    for (int w = 0; w < kRowsWaves; w++) M = fmaxf(M, ml[(w * 16 + x.n) * 2]);
    if (x.n < nh) x.put(0, x.m[0] == -INFINITY ? 0.0f : exp2f(x.m[0] - M), lds + (wave * 16 + x.n) * LS);
    __syncthreads();
    for (int i = tid; i < nh * (d / 4); i += 64 * kRowsWaves) {
        const int hn = i / (d / 4), e0 = i % (d / 4) * 4;
        RowSum s = row_sum(lds + hn * LS + e0, 16 * LS, ml + hn * 2, 16 * 2);
        write_row<QT>(p, c.out_row, r, kvh * G + h0 + hn, part, pr.nparts, e0, s);
    }
}

}  // namespace pam
