// backward_rows.hip - gradients of paged attention with f32 probabilities on the
// matrix units (gfx950): f32 caches, and f16 caches that backward.hip's f16
// matrix kernels do not take (other head sizes, groups that are no power of two).
//
// The semantics and the split of the work are backward.hip's, without atomics:
//   * bwd_d_rows: a workgroup owns one or two blocks of 16 query rows (token, head)
//     of one kv head; its waves take the 16-key tiles in turn for
//     D_i = sum_j P_ij dP_ij and sum in LDS;
//   * bwd_grads_rows: workgroups of such row blocks, whose waves take the key tiles
//     in turn for dQ^T += K^T dS^T, and workgroups of key blocks, each with one
//     share of the group's query rows, whose waves take the 16-row tiles in turn for
//     dV^T += dO^T P and dK^T += Q^T dS.  Shares of one key block go through f32
//     partials that bwd_dkv_sum adds to the gradient pools in order.
// The arrangement is rows_body.h's: S and dP on v_mfma_f32_16x16x4_f32 (f16:
// v_mfma_f32_16x16x32_f16, exact products), whose accumulator registers are the
// B operands of the gradient products on v_mfma_f32_16x16x4_f32; P, dS and the
// gradients stay in f32 registers.  Operands come straight from memory, 16 bytes a
// lane, in two forms: as rows (lane n's row, a piece of its dims) for S and dP,
// and by dims (VW dims of one row) for the gradients.
//
// Sums of f32 caches: S and dP add up in a tree (dot_tree).  Error norms of the
// gradients against 64 bits over the VALU kernels', geometric mean of 45 to 57 calls a
// head size: 0.45-0.63, largest 1.02.  With two chains over the head: 0.48-0.74, and up to
// 1.84 for a few tokens; the tree costs 2-4% of a call up to d = 128 (MFMA results in VGPRs
// take 10% off at d = 256).
//
// What bounds it: the f32 matrix rate (nine products over the (row, key) pairs
// where five are needed: S and dP are formed for D, for dQ and for dK / dV); a
// short sequence, its few workgroups and the latency of its tiles' loads.  Measured
// on gfx950 against the VALU kernels, which served these shapes before (µs per
// call): f32 8/2 d = 64, 600 tokens 2500 -> 80; f32 16/4 d = 64, 1000 tokens 7160 -> 235;
// f16 8/8 d = 64, 1000 tokens 3700 -> 77; f16 32/8 d = 64, 2000 tokens 50300 -> 847 (97
// TFLOP/s of the five products).  One block of rows or keys a wave in place of two:
// 322, 106 and 1124 for the last three; D alone with one: 259, 83 and 940.  dQ (with D)
// and dK / dV in launches of their own, where each leaves CUs idle: 94, 246, 76 and 858;
// 12/4 d = 96, 200 tokens 50 against 40.  f32 32/8 d = 128, 1000 tokens: 1091 (38 TFLOP/s).
#include "rows_body.h"

namespace pam {

// Shape of the kernels for one type and NT 32-dim tiles (32 NT >= head_dim).  A
// wave owns B blocks of 16 rows (dQ) or keys (dK / dV): two share the other
// side's operands, addresses and conversions, where the registers hold them.
// EX: head_dim is 32 NT, so no load reaches past a row.
template <typename T, int NT_, bool EX_>
struct BwdShape {
    static constexpr int NT = NT_;
    static constexpr bool EX = EX_;
    static constexpr int W = NT <= 4 ? 8 : 4;  // waves of a workgroup
    static constexpr int BQ = NT > 4 || (sizeof(T) == 4 && NT > 2) ? 1 : 2;
    static constexpr int BK = NT > 3 || (sizeof(T) == 4 && NT > 2) ? 1 : 2;
    static constexpr int KC = sizeof(T) == 4 ? 2 * NT : NT, KD = sizeof(T) == 4 ? 4 : 8;  // row operand: pieces, their dims
    // dims operand: VW dims in each of NU groups (rows_body.h's V)
    static constexpr int VW = sizeof(T) == 4 ? (NT % 2 == 0 ? 4 : 2) : (NT % 4 == 0 ? 8 : (NT == 2 ? 4 : 2));
    static constexpr int NU = 2 * NT / VW;
    static constexpr int LS = 32 * NT + 4;  // LDS row stride (floats)
};

// Row-layout operand: the pieces of one row held by lane (n, g).  Rows outside
// the sequence and dims past head_dim are zeros from the zero page.
template <typename T, class S>
struct RowOp {
    typedef typename KPiece<T>::Q V;
    V v[S::KC];
    // row: its first byte, or the zero page
    __device__ __forceinline__ void load(const char *row, int g, int d, const char *zero) {
#pragma unroll
        for (int c = 0; c < S::KC; c++) {
            const int e = 4 * S::KD * c + S::KD * g;
            v[c] = *reinterpret_cast<const V *>(S::EX || e < d ? row + e * (int)sizeof(T) : zero);
        }
    }
    // 16x16 products of rows a (the result's rows) and b (its columns)
    __device__ __forceinline__ static f32x4 dot(const RowOp &a, const RowOp &b) {
        if constexpr (sizeof(T) == 4) {
            return dot_tree<8, S::KC>(a.v, b.v);
        } else {
            f32x4 s = (f32x4)0.0f;
#pragma unroll
            for (int c = 0; c < S::KC; c++) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(a.v[c], b.v[c], s, 0, 0, 0);
            return s;
        }
    }
};

// Dims-layout operand of one row
template <typename T, class S>
struct DimOp {
    RawVec<T, S::VW> x[S::NU];
    __device__ __forceinline__ void load(const char *row, int n, int d, const char *zero) {
#pragma unroll
        for (int u = 0; u < S::NU; u++) {
            const int e = 16 * S::VW * u + S::VW * n;
            x[u].load(S::EX || e < d ? row + e * (int)sizeof(T) : zero);
        }
    }
    // acc[b]^T (dims x columns) += row^T w[b]
    template <int B>
    __device__ __forceinline__ void add(const float (&w)[B], f32x4 (&acc)[B][2 * S::NT]) const {
        float a[2 * S::NT];
#pragma unroll
        for (int u = 0; u < S::NU; u++) x[u].floats(0, a + S::VW * u);
#pragma unroll
        for (int i = 0; i < 2 * S::NT; i++)
#pragma unroll
            for (int b = 0; b < B; b++) acc[b][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], w[b], acc[b][i], 0, 0, 0);
    }
    __device__ __forceinline__ static void put(const f32x4 (&acc)[2 * S::NT], int g, float *row) {
#pragma unroll
        for (int u = 0; u < S::NU; u++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int w = 0; w < S::VW; w++) row[16 * S::VW * u + S::VW * (4 * g + r) + w] = acc[S::VW * u + w][r];
    }
};

// a row of one kv head by its pool slot (negative: the zero page)
__device__ __forceinline__ const char *at_row(const char *base, int64_t i, int64_t row_bytes, const char *zero) {
    return i < 0 ? zero : base + i * row_bytes;
}

// the rows' {m, 1 / l, D, 0}, [kv head][row of the head's group]
__device__ __forceinline__ float4 *row_terms(const BackwardParams &p, int kvh) {
    return reinterpret_cast<float4 *>(p.row_d) + (int64_t)kvh * p.seq_len * (p.num_heads / p.num_kv_heads);
}
__device__ __forceinline__ float prob(float s, float scale, float m, float inv_l) {
    return exp2f(fmaf(s, scale, -m) * kLog2e) * inv_l;
}

// 4 dims at e0 of row rn summed over the waves' LDS blocks
template <class S>
__device__ __forceinline__ void lds_sum(const float *lds, int rn, int e0, float *a) {
    a[0] = a[1] = a[2] = a[3] = 0.0f;
#pragma unroll
    for (int w = 0; w < S::W; w++) {
        const float4 x = *reinterpret_cast<const float4 *>(lds + (w * 16 + rn) * S::LS + e0);
        a[0] += x.x, a[1] += x.y, a[2] += x.z, a[3] += x.w;
    }
}

// row of q and d_out of the group's row rho (-1: past the end)
__device__ __forceinline__ int query_row(const BackwardParams &p, int kvh, int rho) {
    const int H = p.num_heads, G = H / p.num_kv_heads;
    return rho < p.seq_len * G ? rho / G * H + kvh * G + rho % G : -1;
}

// The row terms, D among them.  grid: kv head + Hkv * (16 B rows).
template <typename T, class S, int B>
__global__ __launch_bounds__(64 * S::W, (S::NT <= 4 ? 2 : 1)) void bwd_d_rows(BackwardParams p) {
    constexpr int W = S::W;
    __shared__ float d_lds[W][16 * B];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int Hkv = p.num_kv_heads, d = p.head_dim;
    const int kvh = blockIdx.x % Hkv, row0 = (int)(blockIdx.x / Hkv) * 16 * B, rows = p.seq_len * (p.num_heads / Hkv);
    const char *zero = static_cast<const char *>(p.zero_page);
    const int64_t q_bytes = (int64_t)d * (int)sizeof(T), kv_bytes = Hkv * q_bytes;
    const char *kbase = static_cast<const char *>(p.k_pool) + kvh * q_bytes, *vbase = static_cast<const char *>(p.v_pool) + kvh * q_bytes;
    RowOp<T, S> q[B], go[B];
    float m[B], inv_l[B], D[B];
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int so = query_row(p, kvh, row0 + 16 * b + n);
        q[b].load(at_row(static_cast<const char *>(p.q), so, q_bytes, zero), g, d, zero);
        go[b].load(at_row(static_cast<const char *>(p.d_out), so, q_bytes, zero), g, d, zero);
        m[b] = p.m[so < 0 ? 0 : so];
        inv_l[b] = 1.0f / p.l[so < 0 ? 0 : so];
        D[b] = 0.0f;
    }
    const KeySlots keys(p);
    const int t1 = (p.seq_len + 15) / 16, first = p.window_start / 16 + wave;
    auto slot_of = [&](int t) { return t < t1 ? keys.at(16 * t + n) : (int64_t)-1; };
    RowOp<T, S> k, v;
    int64_t slot = slot_of(first), ahead = slot_of(first + W);
    if (first < t1) {
        k.load(at_row(kbase, slot, kv_bytes, zero), g, d, zero);
        v.load(at_row(vbase, slot, kv_bytes, zero), g, d, zero);
    }
    for (int t = first; t < t1; t += W) {
        f32x4 s[B], dp[B];
#pragma unroll
        for (int b = 0; b < B; b++) s[b] = RowOp<T, S>::dot(k, q[b]);
        __builtin_amdgcn_sched_barrier(0);
        const bool more = t + W < t1;
        slot = ahead;
        if (more) {
            ahead = slot_of(t + 2 * W);
            k.load(at_row(kbase, slot, kv_bytes, zero), g, d, zero);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < B; b++) dp[b] = RowOp<T, S>::dot(v, go[b]);
        __builtin_amdgcn_sched_barrier(0);
        if (more) v.load(at_row(vbase, slot, kv_bytes, zero), g, d, zero);
        __builtin_amdgcn_sched_barrier(0);
        const bool edge = 16 * t < p.window_start || 16 * t + 16 > p.seq_len;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = 16 * t + 4 * g + r;
#pragma unroll
            for (int b = 0; b < B; b++) {
                float P = prob(s[b][r], p.scale, m[b], inv_l[b]);
                if (edge) P = j >= p.window_start && j < p.seq_len ? P : 0.0f;
                D[b] = fmaf(P, dp[b][r], D[b]);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < B; b++) {
        D[b] += shfl_xor(D[b], 16);
        D[b] += shfl_xor(D[b], 32);
        if (g == 0) d_lds[wave][16 * b + n] = D[b];
    }
    __syncthreads();
    if (wave != 0 || g != 0) return;
#pragma unroll
    for (int b = 0; b < B; b++) {
        D[b] = 0.0f;
#pragma unroll
        for (int w = 0; w < W; w++) D[b] += d_lds[w][16 * b + n];
        const int rho = row0 + 16 * b + n;
        if (rho < rows) row_terms(p, kvh)[rho] = make_float4(m[b], inv_l[b], D[b], 0.0f);
    }
}

// dQ of workgroup id: kv head + Hkv * (16 BQ rows)
template <typename T, class S>
__device__ __forceinline__ void dq_rows_body(const BackwardParams &p, int id, float *lds) {
    constexpr int B = S::BQ, W = S::W, LS = S::LS;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int H = p.num_heads, Hkv = p.num_kv_heads, G = H / Hkv, d = p.head_dim;
    const int kvh = id % Hkv, row0 = id / Hkv * 16 * B, rows = p.seq_len * G;
    const char *zero = static_cast<const char *>(p.zero_page);
    const int64_t q_bytes = (int64_t)d * (int)sizeof(T), kv_bytes = Hkv * q_bytes;
    const char *kbase = static_cast<const char *>(p.k_pool) + kvh * q_bytes, *vbase = static_cast<const char *>(p.v_pool) + kvh * q_bytes;
    RowOp<T, S> q[B], go[B];
    float4 rt[B];
    f32x4 dq[B][2 * S::NT];
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int rho = row0 + 16 * b + n, so = query_row(p, kvh, rho);
        q[b].load(at_row(static_cast<const char *>(p.q), so, q_bytes, zero), g, d, zero);
        go[b].load(at_row(static_cast<const char *>(p.d_out), so, q_bytes, zero), g, d, zero);
        rt[b] = row_terms(p, kvh)[rho < rows ? rho : rows - 1];
#pragma unroll
        for (int i = 0; i < 2 * S::NT; i++) dq[b][i] = (f32x4)0.0f;
    }
    const KeySlots keys(p);
    const int t1 = (p.seq_len + 15) / 16, first = p.window_start / 16 + wave;
    auto slot_of = [&](int t) { return t < t1 ? keys.at(16 * t + n) : (int64_t)-1; };
    RowOp<T, S> k, v;
    int64_t slot = slot_of(first), ahead = slot_of(first + W);
    if (first < t1) {
        k.load(at_row(kbase, slot, kv_bytes, zero), g, d, zero);
        v.load(at_row(vbase, slot, kv_bytes, zero), g, d, zero);
    }
    for (int t = first; t < t1; t += W) {
        DimOp<T, S> kd[4];
#pragma unroll
        for (int r = 0; r < 4; r++) kd[r].load(at_row(kbase, __shfl(slot, 4 * g + r, 64), kv_bytes, zero), n, d, zero);
        f32x4 s[B], dp[B];
#pragma unroll
        for (int b = 0; b < B; b++) s[b] = RowOp<T, S>::dot(k, q[b]);
        __builtin_amdgcn_sched_barrier(0);
        const bool more = t + W < t1;
        slot = ahead;
        if (more) {
            ahead = slot_of(t + 2 * W);
            k.load(at_row(kbase, slot, kv_bytes, zero), g, d, zero);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < B; b++) dp[b] = RowOp<T, S>::dot(v, go[b]);
        __builtin_amdgcn_sched_barrier(0);
        if (more) v.load(at_row(vbase, slot, kv_bytes, zero), g, d, zero);
        __builtin_amdgcn_sched_barrier(0);
        const bool edge = 16 * t < p.window_start || 16 * t + 16 > p.seq_len;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = 16 * t + 4 * g + r;
            float dS[B];
#pragma unroll
            for (int b = 0; b < B; b++) {
                float P = prob(s[b][r], p.scale, rt[b].x, rt[b].y);
                if (edge) P = j >= p.window_start && j < p.seq_len ? P : 0.0f;
                dS[b] = P * (dp[b][r] - rt[b].z);
            }
            kd[r].add(dS, dq);
        }
    }
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int rb = row0 + 16 * b;
        if (b) __syncthreads();
        DimOp<T, S>::put(dq[b], g, lds + (wave * 16 + n) * LS);
        __syncthreads();
        for (int i = tid; i < 16 * (d / 4); i += 64 * W) {
            const int rn = i / (d / 4), e0 = i % (d / 4) * 4, r = rb + rn;
            if (r >= rows) continue;
            float a[4];
            lds_sum<S>(lds, rn, e0, a);
#pragma unroll
            for (int e = 0; e < 4; e++) a[e] *= p.scale;
            store4<T>(static_cast<T *>(p.d_q) + ((int64_t)(r / G) * H + kvh * G + r % G) * d + e0, a);
        }
    }
}

// add 4 dims to key j's row of a gradient pool
template <typename T>
__device__ __forceinline__ void pool_add(void *pool, const BackwardParams &p, const KeySlots &keys, int j, int kvh, int e0,
                                         const float *a) {
    T *row = static_cast<T *>(pool) + (keys.at(j) * p.num_kv_heads + kvh) * p.head_dim + e0;
    float x[4];
    load4<T>(row, x);
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] += a[e];
    store4<T>(row, x);
}

// dK / dV of workgroup id: kv head + Hkv * (16 BK keys), and a share of the rows
template <typename T, class S>
__device__ __forceinline__ void dkv_rows_body(const BackwardParams &p, int id, int share, float *lds) {
    constexpr int B = S::BK, W = S::W, LS = S::LS;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int H = p.num_heads, Hkv = p.num_kv_heads, G = H / Hkv, d = p.head_dim;
    const int kvh = id % Hkv, key0 = p.window_start + id / Hkv * 16 * B, rows = p.seq_len * G;
    const char *zero = static_cast<const char *>(p.zero_page), *Q = static_cast<const char *>(p.q),
               *dO = static_cast<const char *>(p.d_out);
    const int64_t q_bytes = (int64_t)d * (int)sizeof(T), kv_bytes = Hkv * q_bytes;
    const KeySlots keys(p);
    RowOp<T, S> k[B], v[B];
    f32x4 dk[B][2 * S::NT], dv[B][2 * S::NT];
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int64_t slot = keys.at(key0 + 16 * b + n);
        k[b].load(at_row(static_cast<const char *>(p.k_pool) + kvh * q_bytes, slot, kv_bytes, zero), g, d, zero);
        v[b].load(at_row(static_cast<const char *>(p.v_pool) + kvh * q_bytes, slot, kv_bytes, zero), g, d, zero);
#pragma unroll
        for (int i = 0; i < 2 * S::NT; i++) dk[b][i] = dv[b][i] = (f32x4)0.0f;
    }
    const float4 *terms = row_terms(p, kvh);
    const int tiles = (rows + 15) / 16, per = (tiles + p.shares - 1) / p.shares;
    const int t0 = share * per, t1 = t0 + per < tiles ? t0 + per : tiles;
    // row of q and d_out of the group's row rho (-1: past the end)
    const int gs = block_shift(G);
    auto row_of = [&](int rho) {
        const int tok = gs >= 0 ? rho >> gs : rho / G;
        return rho < rows ? tok * (H - G) + kvh * G + rho : -1;
    };
    RowOp<T, S> q, go;
    int off = row_of(16 * (t0 + wave) + n);
    if (t0 + wave < t1) {
        q.load(at_row(Q, off, q_bytes, zero), g, d, zero);
        go.load(at_row(dO, off, q_bytes, zero), g, d, zero);
    }
    for (int t = t0 + wave; t < t1; t += W) {
        // the dims-layout operands of the tile, dO rows then Q rows, RING loads ahead
        constexpr int RING = sizeof(T) == 4 && S::NT > 3 ? 2 : 8;
        DimOp<T, S> x[RING];
        int offs[4];
#pragma unroll
        for (int r = 0; r < 4; r++) offs[r] = __shfl(off, 4 * g + r, 64);
        auto issue = [&](int i) { x[i % RING].load(at_row(i < 4 ? dO : Q, offs[i & 3], q_bytes, zero), n, d, zero); };
        float4 rt[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int rho = 16 * t + 4 * g + r;
            rt[r] = terms[rho < rows ? rho : rows - 1];
        }
#pragma unroll
        for (int i = 0; i < RING; i++) issue(i);
        const bool more = t + W < t1;
        off = row_of(16 * (t + W) + n);
        f32x4 s[B], dp[B];
#pragma unroll
        for (int b = 0; b < B; b++) {
            s[b] = RowOp<T, S>::dot(q, k[b]);
            dp[b] = RowOp<T, S>::dot(go, v[b]);
        }
        __builtin_amdgcn_sched_barrier(0);
        const bool edge = 16 * t + 16 > rows;
        float P[4][B], dS[4][B];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int b = 0; b < B; b++) {
                P[r][b] = prob(s[b][r], p.scale, rt[r].x, rt[r].y);
                if (edge) P[r][b] = 16 * t + 4 * g + r < rows ? P[r][b] : 0.0f;
                dS[r][b] = P[r][b] * (dp[b][r] - rt[r].z);
            }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (i < 4)
                x[i % RING].add(P[i & 3], dv);
            else
                x[i % RING].add(dS[i & 3], dk);
            if (i + RING < 8) issue(i + RING);
            if (i == 3 && more) {  // the next tile's rows
                q.load(at_row(Q, off, q_bytes, zero), g, d, zero);
                go.load(at_row(dO, off, q_bytes, zero), g, d, zero);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int which = 0; which < 2; which++)
#pragma unroll
        for (int b = 0; b < B; b++) {
            if (which || b) __syncthreads();
            DimOp<T, S>::put(which ? dv[b] : dk[b], g, lds + (wave * 16 + n) * LS);
            __syncthreads();
            for (int i = tid; i < 16 * (d / 4); i += 64 * W) {
                const int kn = i / (d / 4), e0 = i % (d / 4) * 4, j = key0 + 16 * b + kn;
                if (j >= p.seq_len) continue;
                float a[4];
                lds_sum<S>(lds, kn, e0, a);
                if (!which)
#pragma unroll
                    for (int e = 0; e < 4; e++) a[e] *= p.scale;
                if (p.shares > 1) {
                    const int64_t nk = p.seq_len - p.window_start, row = (int64_t)(j - p.window_start) * Hkv + kvh;
                    store4<float>(p.partial + ((int64_t)(2 * share + which) * nk * Hkv + row) * d + e0, a);
                } else {
                    pool_add<T>(which ? p.d_v_pool : p.d_k_pool, p, keys, j, kvh, e0, a);
                }
            }
        }
}

// Both sides of the gradients in one launch, so that neither waits for the other's
// last workgroups: the first n_dq workgroups take dQ, the others dK / dV.
template <typename T, class S>
__global__ __launch_bounds__(64 * S::W, (S::NT <= 4 ? 2 : 1)) void bwd_grads_rows(BackwardParams p, int n_dq) {
    __shared__ __attribute__((aligned(16))) float lds[S::W * 16 * S::LS];
    const int id = blockIdx.x;
    if (id < n_dq)
        dq_rows_body<T, S>(p, id, lds);
    else
        dkv_rows_body<T, S>(p, (id - n_dq) / p.shares, (id - n_dq) % p.shares, lds);
}

// the shares' partials, summed in order, into the gradient pools
template <typename T>
__global__ __launch_bounds__(256) void bwd_dkv_sum(BackwardParams p) {
    const int d4 = p.head_dim / 4, Hkv = p.num_kv_heads;
    const int64_t n = (int64_t)(p.seq_len - p.window_start) * Hkv * d4, i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int which = blockIdx.y;
    float a[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < p.shares; s++) {
        const float4 x = reinterpret_cast<const float4 *>(p.partial)[(2 * s + which) * n + i];
        a[0] += x.x, a[1] += x.y, a[2] += x.z, a[3] += x.w;
    }
    pool_add<T>(which ? p.d_v_pool : p.d_k_pool, p, KeySlots(p), p.window_start + (int)(i / d4 / Hkv), (int)(i / d4 % Hkv),
                (int)(i % d4) * 4, a);
}

bool backward_rows_supported(const BackwardParams &p, int32_t dtype) {
    if (p.head_dim <= 0 || p.head_dim > 256 || p.head_dim % (dtype == kF32 ? 4 : 8) != 0) return false;
    if ((int64_t)p.seq_len * p.num_heads >= ((int64_t)1 << 31) - 512) return false;
    const uintptr_t all = (uintptr_t)p.q | (uintptr_t)p.k_pool | (uintptr_t)p.v_pool | (uintptr_t)p.d_out |
                          (uintptr_t)p.d_q | (uintptr_t)p.d_k_pool | (uintptr_t)p.d_v_pool;
    return (all & 15) == 0;
}

// The kernels' shape for p: f(S{}) for the instantiation that takes it.
template <typename T, typename F>
static auto with_shape(const BackwardParams &p, F &&f) {
    const bool ex = p.head_dim % 32 == 0;
    switch ((p.head_dim + 31) / 32) {
        case 1: return ex ? f(BwdShape<T, 1, true>{}) : f(BwdShape<T, 1, false>{});
        case 2: return ex ? f(BwdShape<T, 2, true>{}) : f(BwdShape<T, 2, false>{});
        case 3: return ex ? f(BwdShape<T, 3, true>{}) : f(BwdShape<T, 3, false>{});
        case 4: return ex ? f(BwdShape<T, 4, true>{}) : f(BwdShape<T, 4, false>{});
        default: return f(BwdShape<T, 8, false>{});
    }
}

// Shares of the query rows of a dK / dV block: a workgroup per CU, of no fewer
// than two row tiles a wave.
template <typename T>
static int32_t shares_of(const BackwardParams &p, int32_t cus) {
    return with_shape<T>(p, [&](auto shape) {
        typedef decltype(shape) S;
        const int64_t keys = p.seq_len - p.window_start, span = 16 * S::BK;
        const int64_t blocks = (keys + span - 1) / span * p.num_kv_heads;
        const int64_t tiles = ((int64_t)p.seq_len * (p.num_heads / p.num_kv_heads) + 15) / 16;
        int64_t s = blocks > 0 ? (cus + blocks - 1) / blocks : 1;
        s = s < tiles / (2 * S::W) ? s : tiles / (2 * S::W);
        return (int32_t)(s < 1 ? 1 : (s > 64 ? 64 : s));
    });
}

int32_t backward_rows_shares(const BackwardParams &p, int32_t dtype, int32_t cus) {
    return dtype == kF32 ? shares_of<float>(p, cus) : shares_of<f16>(p, cus);
}

hipError_t launch_backward_sum(const BackwardParams &p, int32_t dtype, hipStream_t stream) {
    const int64_t n = (int64_t)(p.seq_len - p.window_start) * p.num_kv_heads * (p.head_dim / 4);
    const dim3 grid((unsigned)((n + 255) / 256), 2);
    if (dtype == kF32)
        hipLaunchKernelGGL(bwd_dkv_sum<float>, grid, dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL(bwd_dkv_sum<f16>, grid, dim3(256), 0, stream, p);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_type(const BackwardParams &p, hipStream_t stream) {
    return with_shape<T>(p, [&](auto shape) {
        typedef decltype(shape) S;
        const int64_t rows = (int64_t)p.seq_len * (p.num_heads / p.num_kv_heads), keys = p.seq_len - p.window_start;
        const int64_t rspan = 16 * S::BQ, kspan = 16 * S::BK;
        const dim3 block(64 * S::W);
        const int64_t n_dq = (rows + rspan - 1) / rspan * p.num_kv_heads;
        const int64_t n_dkv = (keys + kspan - 1) / kspan * p.num_kv_heads * p.shares;
        if (n_dq + n_dkv >= ((int64_t)1 << 31)) return hipErrorInvalidValue;
        hipLaunchKernelGGL((bwd_d_rows<T, S, S::BQ>), dim3((unsigned)n_dq), block, 0, stream, p);
        hipLaunchKernelGGL((bwd_grads_rows<T, S>), dim3((unsigned)(n_dq + n_dkv)), block, 0, stream, p, (int)n_dq);
        if (keys > 0 && p.shares > 1) return launch_backward_sum(p, sizeof(T) == 4 ? kF32 : kF16, stream);
        return hipGetLastError();
    });
}

hipError_t launch_backward_rows(const BackwardParams &p, int32_t dtype, hipStream_t stream) {
    if (!backward_rows_supported(p, dtype) || p.zero_page == nullptr || p.shares < 1 || (p.shares > 1 && !p.partial))
        return hipErrorInvalidValue;
    return dtype == kF32 ? launch_type<float>(p, stream) : launch_type<f16>(p, stream);
}

}  // namespace pam
