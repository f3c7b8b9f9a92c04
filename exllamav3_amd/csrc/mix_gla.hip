// Gated linear attention with a decay per key channel: the token-by-token form (decode, and the exact float32 prefill) and the
// output stage (per-head RMS norm, silu gate).  State, decays, logarithms and every product that enters the recurrence are float32.
//
// Work split of the scan: one workgroup of 4 waves per (sequence, head, block of 64 value columns).  Lane = value column; wave w
// owns the key channels w, w + 4, w + 8, ... (DR of them per lane, in registers).  A chunk of SCAN_TC (16 or 8) tokens is staged in LDS
// (q, k, alpha as float32; alpha computed here from the low-rank decay input), the waves run the recurrence over the chunk without
// a barrier, and the partial outputs of the four waves are added through LDS at the end of the chunk.
#include "mix_common.cuh"

#define SCAN_WAVES 4

// MODE 0: a whole sequence per workgroup, state from / to its slot.
// Long prompts are cut into segments of `seg_len` rows that run in parallel (blockIdx.x = sequence * segs + segment):
// MODE 1: a segment from a zero state, no outputs; leaves its local state and the product of its decays in `seg_state` / `seg_decay`;
// MODE 2: a segment from the state that gla_combine_kernel put into `seg_state`, writes outputs, leaves the slot alone.
#define GLA_WHOLE 0
#define GLA_SEG_LOCAL 1
#define GLA_SEG_FINAL 2

template <typename T, int DR, int MODE>
__global__ __launch_bounds__(256) void gla_scan_kernel(float* __restrict__ o, float* __restrict__ state, const T* __restrict__ q, int64_t q_ld,
                                                       const T* __restrict__ k, int64_t k_ld, const T* __restrict__ v, int64_t v_ld,
                                                       const T* __restrict__ lr, int64_t lr_ld, const T* __restrict__ a2, const float* __restrict__ a2_bias,
                                                       const int32_t* __restrict__ cu, const int32_t* __restrict__ slots, const int32_t* __restrict__ pos0,
                                                       int heads, int dim, int vdim, int rank, float inv_tau, float q_scale, int SCAN_TC,
                                                       int segs, int seg_len, float* __restrict__ seg_state, float* __restrict__ seg_decay)
{
    extern __shared__ float smem[];
    float* qs = smem;                                  // [SCAN_TC][dim]
    float* ks = qs + SCAN_TC * dim;
    float* as = ks + SCAN_TC * dim;
    float* vs = as + SCAN_TC * dim;                    // [SCAN_TC][64]
    float* part = vs + SCAN_TC * 64;                   // [SCAN_TC][SCAN_WAVES][64]
    const int b = (MODE == GLA_WHOLE) ? blockIdx.x : blockIdx.x / segs, h = blockIdx.y, vt = blockIdx.z;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int col = vt * 64 + lane;
    const bool col_ok = col < vdim;
    int first = cu[b], last = cu[b + 1];
    float* st = state + ((int64_t) slots[b] * heads + h) * dim * vdim;
    bool resume = pos0[b] > 0;
    float D[DR];                                       // MODE 1: product of the segment's decays (the same in every lane of a wave)
    if (MODE != GLA_WHOLE)
    {
        const int sg = blockIdx.x - b * segs;
        first += sg * seg_len;
        last = min(last, first + seg_len);
        st = seg_state + ((int64_t) blockIdx.x * heads + h) * dim * vdim;
        resume = (MODE == GLA_SEG_FINAL);
    }

    float S[DR];
    #pragma unroll
    for (int i = 0; i < DR; ++i) D[i] = 1.f;
    #pragma unroll
    for (int i = 0; i < DR; ++i)
    {
        const int r = w + SCAN_WAVES * i;
        S[i] = (resume && col_ok && r < dim) ? st[(int64_t) r * vdim + col] : 0.f;
    }

    for (int n0 = first; n0 < last; n0 += SCAN_TC)
    {
        const int tc = min(SCAN_TC, last - n0);
        __syncthreads();                               // the previous chunk's LDS reads are over
        for (int idx = threadIdx.x; idx < tc * dim; idx += 256)
        {
            const int t = idx / dim, c = idx - t * dim;
            const int64_t n = n0 + t;
            const int hc = h * dim + c;
            if (MODE != GLA_SEG_LOCAL) qs[idx] = to_f(q[n * q_ld + hc]) * q_scale;
            ks[idx] = to_f(k[n * k_ld + hc]);
            float z = a2_bias ? a2_bias[hc] : 0.f;
            const T* lrow = lr + n * lr_ld;
            const T* arow = a2 + (int64_t) hc * rank;
            int r = 0;
            for (; r + 8 <= rank; r += 8)                   // eight loads in flight, then the sums (a rolled loop waits for every load in turn)
            {
                float a[8], bb[8];
                #pragma unroll
                for (int e = 0; e < 8; ++e) { a[e] = to_f(lrow[r + e]); bb[e] = to_f(arow[r + e]); }
                #pragma unroll
                for (int e = 0; e < 8; ++e) z += a[e] * bb[e];
            }
            for (; r < rank; ++r) z += to_f(lrow[r]) * to_f(arow[r]);
            as[idx] = expf(log_sigmoid_f(z) * inv_tau);
        }
        for (int idx = threadIdx.x; idx < tc * 64; idx += 256)
        {
            const int t = idx >> 6, c = vt * 64 + (idx & 63);
            vs[idx] = (c < vdim) ? to_f(v[(int64_t) (n0 + t) * v_ld + h * vdim + c]) : 0.f;
        }
        __syncthreads();
        for (int t = 0; t < tc; ++t)
        {
            const float vv = vs[t * 64 + lane];
            float po = 0.f;
            #pragma unroll
            for (int i = 0; i < DR; ++i)
            {
                const int r = w + SCAN_WAVES * i;
                if (r < dim)
                {
                    const float a = as[t * dim + r];
                    S[i] = a * S[i] + ks[t * dim + r] * vv;
                    if (MODE == GLA_SEG_LOCAL) D[i] *= a; else po += qs[t * dim + r] * S[i];
                }
            }
            if (MODE != GLA_SEG_LOCAL) part[(t * SCAN_WAVES + w) * 64 + lane] = po;
        }
        if (MODE == GLA_SEG_LOCAL) continue;
        __syncthreads();
        for (int idx = threadIdx.x; idx < tc * 64; idx += 256)
        {
            const int t = idx >> 6, l = idx & 63, c = vt * 64 + l;
            if (c < vdim)
            {
                float s = 0.f;
                #pragma unroll
                for (int ww = 0; ww < SCAN_WAVES; ++ww) s += part[(t * SCAN_WAVES + ww) * 64 + l];
                o[((int64_t) (n0 + t) * heads + h) * vdim + c] = s;
            }
        }
    }
    if (MODE == GLA_SEG_FINAL) return;
    #pragma unroll
    for (int i = 0; i < DR; ++i)
    {
        const int r = w + SCAN_WAVES * i;
        if (col_ok && r < dim) st[(int64_t) r * vdim + col] = S[i];
        if (MODE == GLA_SEG_LOCAL && vt == 0 && lane == 0 && r < dim) seg_decay[((int64_t) blockIdx.x * heads + h) * dim + r] = D[i];
    }
}

// Between the two segment passes: walks a sequence's segments in order.  seg_state[s] (the segment's local state) is replaced by the state the
// segment starts from, S_start[s+1] = diag(decay[s]) S_start[s] + local[s]; the state after the last segment goes to the sequence's slot.
__global__ __launch_bounds__(256) void gla_combine_kernel(float* __restrict__ state, float* __restrict__ seg_state, const float* __restrict__ seg_decay,
                                                          const int32_t* __restrict__ cu, const int32_t* __restrict__ slots, const int32_t* __restrict__ pos0,
                                                          int heads, int dim, int vdim, int segs, int seg_len)
{
    const int b = blockIdx.x, h = blockIdx.y;
    const int64_t per = (int64_t) dim * vdim;
    const int used = min(segs, (cu[b + 1] - cu[b] + seg_len - 1) / seg_len);
    float* st = state + ((int64_t) slots[b] * heads + h) * per;
    const bool resume = pos0[b] > 0;
    for (int64_t e = (int64_t) blockIdx.z * 256 + threadIdx.x; e < per; e += (int64_t) gridDim.z * 256)
    {
        const int r = (int) (e / vdim);
        float S = resume ? st[e] : 0.f;
        for (int sg = 0; sg < used; ++sg)
        {
            const int64_t blk = ((int64_t) b * segs + sg) * heads + h;
            const float local = seg_state[blk * per + e];
            seg_state[blk * per + e] = S;
            S = seg_decay[blk * dim + r] * S + local;
        }
        st[e] = S;
    }
}

// V elements per lane and access (4 where strides and addresses allow; else 1), 32 lanes per (row, head): a head of 128 columns is one piece per lane, read once.
// HBM-bound at prompt sizes: 4096 rows of 32 heads x 128 (bfloat16) 52 -> 33 us with wider accesses.
template <typename T, int V>
__global__ __launch_bounds__(256) void gla_out_kernel(T* __restrict__ out, const float* __restrict__ o, const float* __restrict__ w, const T* __restrict__ g,
                                                      int64_t g_ld, float eps, int64_t items, int heads, int vdim)
{
    const int lane = threadIdx.x & 31;
    const int64_t item = (int64_t) blockIdx.x * 8 + (threadIdx.x >> 5), it = item < items ? item : items - 1;
    const int64_t n = it / heads;
    const int h = (int) (it - n * heads);
    const float* orow = o + it * vdim;
    const T* gr = g + n * g_ld + (int64_t) h * vdim;
    T* dst = out + it * vdim;
    float x[V], gv[V];
    const int c0 = lane * V;
    #pragma unroll
    for (int e = 0; e < V; ++e) x[e] = gv[e] = 0.f;
    if (c0 < vdim) { load_n<float, V>(orow + c0, x); load_n<T, V>(gr + c0, gv); }
    float ss = 0.f;
    #pragma unroll
    for (int e = 0; e < V; ++e) ss += x[e] * x[e];
    for (int i = c0 + 32 * V; i < vdim; i += 32 * V)
    {
        float t[V];
        load_n<float, V>(orow + i, t);
        #pragma unroll
        for (int e = 0; e < V; ++e) ss += t[e] * t[e];
    }
    #pragma unroll
    for (int d = 16; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 32);
    if (item >= items) return;
    const float inv = 1.0f / sqrtf(ss / (float) vdim + eps);
    for (int i = c0; i < vdim; i += 32 * V)
    {
        float wv[V];
        if (i != c0) { load_n<float, V>(orow + i, x); load_n<T, V>(gr + i, gv); }
        load_n<float, V>(w + i, wv);
        #pragma unroll
        for (int e = 0; e < V; ++e) x[e] = x[e] * inv * wv[e] * silu_f(gv[e]);
        store_n<T, V>(dst + i, x);
    }
}

// ------------------------------------------------------------------------------------------------
// The two segment passes in chunks of 16 tokens on the float32 matrix instructions (v_mfma_f32_16x16x4_f32: exact products, float32 sums), for key dimensions of 64 and 128.
//
// Token by token the recurrence is bounded by LDS: three broadcast values per state row and token.  Over a chunk, with a_t the decays, P_t their product up to t, R_s the product behind
// s and G the whole product,
//     o_t = (q_t P_t) S + sum_{s <= t} A_ts v_s,    A_ts = sum_d q_td k_sd prod_{s < u <= t} a_ud,    S <- G S + sum_s (k_s R_s) v_s^T.
// No quotient of products is formed (P_t / P_s is lost where the decays underflow): every factor is a product of decays, at most one.  A is put together from four levels of
// blocks: for t in the upper and s in the lower half of a block of 16, 8, 4, 2 tokens with m the last token of the lower half, prod_{s < u <= t} = prod_{s < u <= m} prod_{m < u <= t};
// wave w forms level w as one 16 x 16 product of a matrix with itself (q rows in the upper halves, k rows in the lower ones) and keeps its blocks; the diagonal is a plain q . k.
//
// One workgroup of 4 waves per (segment, head, 128 value columns), wave = 32 columns; the state is the accumulator of the update and, register for register, the second operand of
// the output product (row 16 T + 4 g + i of lane group g is element g of contraction step (T, i)).  Three sequences of 4096 rows in all,
// 32 heads of 64 x 128, both passes: 907 us token by token -> 215 (the products alone: 55 us; the rest is the chain of a chunk, four barriers and the vector work between them).
// Relative error of float32 outputs against 64 bits at 500 .. 900 rows: 2.0e-7, 1.7e-7, 1.3e-7 token by token, 1.9e-7, 1.6e-7, 1.3e-7 here.
// ------------------------------------------------------------------------------------------------
#define GC_MAX_RANK 64
template <int V> struct gc_int { static constexpr int value = V; };

static size_t gla_chunk_lds(int dim, int rank, bool local)
{
    const size_t buf = (size_t) 16 * (dim + 4), pad = (size_t) (rank + 3) / 4 * 4;
    return sizeof(float) * (local ? 3 * buf + dim + pad * (16 + dim) : 9 * buf + dim + 4 * 16 * 20);
}

// exp(log_sigmoid(z) / tau).  log(1 + u) of u = exp(-|z|) in (0, 1] as 2 atanh(u / (2 + u)) by its series to s^17 (s <= 1/3: the rest is below 4e-9), a quarter of log1pf's instructions;
// this and the low-rank product are what the first pass spends its vector instructions on
__device__ __forceinline__ float gla_decay(float z, float inv_tau)
{
    const float u = expf(-fabsf(z)), s = u / (2.0f + u), q = s * s;
    float p = 1.0f / 17.0f;
    p = __builtin_fmaf(p, q, 1.0f / 15.0f); p = __builtin_fmaf(p, q, 1.0f / 13.0f); p = __builtin_fmaf(p, q, 1.0f / 11.0f); p = __builtin_fmaf(p, q, 1.0f / 9.0f);
    p = __builtin_fmaf(p, q, 1.0f / 7.0f); p = __builtin_fmaf(p, q, 1.0f / 5.0f); p = __builtin_fmaf(p, q, 1.0f / 3.0f); p = __builtin_fmaf(p, q, 1.0f);
    return expf((fminf(z, 0.f) - 2.0f * s * p) * inv_tau);
}

template <typename T, int DIM, bool LOCAL>
__global__ __launch_bounds__(256) void gla_chunk_kernel(float* __restrict__ o, const T* __restrict__ q, int64_t q_ld, const T* __restrict__ k, int64_t k_ld,
                                                        const T* __restrict__ v, int64_t v_ld, const T* __restrict__ lr, int64_t lr_ld, const T* __restrict__ a2,
                                                        const float* __restrict__ a2_bias, const int32_t* __restrict__ cu, int heads, int vdim, int rank, float inv_tau,
                                                        float q_scale, int segs, int seg_len, float* __restrict__ seg_state, float* __restrict__ seg_decay,
                                                        float* __restrict__ decay)
{
    typedef float f4 __attribute__((ext_vector_type(4)));
    constexpr int ND = DIM / 64, DT = DIM / 16, PITCH = DIM + 4, BUF = 16 * PITCH, LR = GC_MAX_RANK * 16 / 256;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    float* as = smem;                                  // [16][PITCH] each: decays, k, k R; then q P, q, one per level
    float* ks = as + BUF;
    float* kr = ks + BUF;
    float* gs = kr + BUF;                              // [DIM]
    float* lt = gs + DIM;                              // LOCAL: [rank, to fours][16]
    float* a2s = lt + (rank + 3) / 4 * 64;             //        [rank, to fours][DIM]
    float* qp = gs + DIM;                              // !LOCAL
    float* qs = qp + BUF;
    float* lv = qs + BUF;                              // [4][16][PITCH]
    float* ap = lv + 4 * BUF;                          // [4][16][20]: every wave's part of A
    const int k_behind_q = (int) (ks - qs);

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, r16 = lane & 15;
    const int b = blockIdx.x / segs, sg = blockIdx.x - b * segs, h = blockIdx.y;
    const int first = cu[b] + sg * seg_len, last = min(cu[b + 1], first + seg_len);
    const int col0 = blockIdx.z * 128 + 32 * w + r16;
    float* st = seg_state + ((int64_t) blockIdx.x * heads + h) * DIM * vdim;

    const int rank4 = (rank + 3) / 4;
    float bias[DT / 4], dec[ND];                       // bias: of the decays this lane forms, columns 16 (w + 4 u) + r16
    if (LOCAL)
    {
        for (int i = threadIdx.x; i < 4 * rank4 * DIM; i += 256) { const int d = i % DIM, r = i / DIM; a2s[i] = r < rank ? to_f(a2[(int64_t) (h * DIM + d) * rank + r]) : 0.f; }
        #pragma unroll
        for (int u = 0; u < DT / 4; ++u) bias[u] = a2_bias ? a2_bias[h * DIM + 16 * (w + 4 * u) + r16] : 0.f;
    }
    #pragma unroll
    for (int c = 0; c < ND; ++c) dec[c] = 1.f;

    f4 S[DT][2];
    #pragma unroll
    for (int t = 0; t < DT; ++t)
        #pragma unroll
        for (int c = 0; c < 2; ++c)
            #pragma unroll
            for (int i = 0; i < 4; ++i) S[t][c][i] = (!LOCAL && first < last && col0 + 16 * c < vdim) ? st[(int64_t) (16 * t + 4 * g + i) * vdim + col0 + 16 * c] : 0.f;

    // the next chunk's inputs: requested a chunk ahead.  Rows behind the end count as q = k = v = 0, decay 1
    T qn[ND][4], kn[ND][4], vn[2][4], ln[LR];
    float an[ND][4];
    auto request = [&] (int n0)
    {
        #pragma unroll
        for (int j = 0; j < 4; ++j)
        {
            const int64_t n = min(n0 + 4 * w + j, last - 1), nv = min(n0 + 4 * g + j, last - 1);
            #pragma unroll
            for (int c = 0; c < ND; ++c)
            {
                if (!LOCAL) { qn[c][j] = q[n * q_ld + h * DIM + 64 * c + lane]; an[c][j] = decay[(n * heads + h) * DIM + 64 * c + lane]; }
                kn[c][j] = k[n * k_ld + h * DIM + 64 * c + lane];
            }
            #pragma unroll
            for (int c = 0; c < 2; ++c) vn[c][j] = v[nv * v_ld + (int64_t) h * vdim + min(col0 + 16 * c, vdim - 1)];
        }
        if (!LOCAL) return;
        #pragma unroll
        for (int u = 0; u < LR; ++u)
        {
            const int i = u * 256 + threadIdx.x, r = i >> 4;
            if (r < rank) ln[u] = lr[(int64_t) min(n0 + (i & 15), last - 1) * lr_ld + r];
        }
    };
    if (first < last) request(first);

    for (int n0 = first; n0 < last; n0 += 16)
    {
        if (LOCAL)
        {
            #pragma unroll
            for (int u = 0; u < LR; ++u) { const int i = u * 256 + threadIdx.x; if ((i >> 4) < 4 * rank4) lt[i] = (i >> 4) < rank ? to_f(ln[u]) : 0.f; }
        }
        __syncthreads();                               // (also: the previous chunk's reads of everything below are over)
        if (LOCAL)
        {
            #pragma unroll
            for (int u = 0; u < DT / 4; ++u)
            {
                const int d = 16 * (w + 4 * u) + r16;
                f4 z = { bias[u], bias[u], bias[u], bias[u] };
                #pragma unroll 4
                for (int r = 0; r < rank4; ++r) z = __builtin_amdgcn_mfma_f32_16x16x4f32(lt[(4 * r + g) * 16 + r16], a2s[(4 * r + g) * DIM + d], z, 0, 0, 0);
                #pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    const int t = 4 * g + i;
                    const float al = gla_decay(z[i], inv_tau);
                    as[t * PITCH + d] = n0 + t < last ? al : 1.f;
                    if (blockIdx.z == 0 && n0 + t < last) decay[((int64_t) (n0 + t) * heads + h) * DIM + d] = al;
                }
            }
        }
        #pragma unroll
        for (int c = 0; c < ND; ++c)
        {
            #pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const int t = 4 * w + j, d = 64 * c + lane;
                const bool in = n0 + t < last;
                ks[t * PITCH + d] = in ? to_f(kn[c][j]) : 0.f;
                if (!LOCAL) { as[t * PITCH + d] = in ? an[c][j] : 1.f; qs[t * PITCH + d] = in ? to_f(qn[c][j]) * q_scale : 0.f; }
            }
        }
        float vv[2][4];
        #pragma unroll
        for (int c = 0; c < 2; ++c)
            #pragma unroll
            for (int j = 0; j < 4; ++j) vv[c][j] = (n0 + 4 * g + j < last && col0 + 16 * c < vdim) ? to_f(vn[c][j]) : 0.f;
        if (n0 + 16 < last) request(n0 + 16);
        __syncthreads();

        // lane = key dimension: the products of decays, four tokens of q P and k R and one level per wave.  All LDS reads come first: one chain of 16 products, not of 16 reads
        #pragma unroll
        for (int c = 0; c < ND; ++c)
        {
            const int d = 64 * c + lane, half = 8 >> w;
            float a[16], aw[4], qw[4], kw[4], x[16];
            #pragma unroll
            for (int t = 0; t < 16; ++t) a[t] = as[t * PITCH + d];
            #pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                aw[j] = as[(4 * w + j) * PITCH + d];
                kw[j] = ks[(4 * w + j) * PITCH + d];
                if (!LOCAL) qw[j] = qs[(4 * w + j) * PITCH + d];
            }
            if (!LOCAL)
            {
                #pragma unroll
                for (int t = 0; t < 16; ++t) x[t] = qs[((t & half) ? 0 : k_behind_q) + t * PITCH + d];
            }
            float c4[4];
            #pragma unroll
            for (int u = 0; u < 4; ++u) c4[u] = (a[4 * u] * a[4 * u + 1]) * (a[4 * u + 2] * a[4 * u + 3]);
            const float all = (c4[0] * c4[1]) * (c4[2] * c4[3]);
            if (w == 0) gs[d] = all;
            dec[c] *= all;
            float p = (w > 0 ? c4[0] : 1.f) * (w > 1 ? c4[1] : 1.f) * (w > 2 ? c4[2] : 1.f);
            if (!LOCAL)
            {
                #pragma unroll
                for (int j = 0; j < 4; ++j) { p *= aw[j]; qp[(4 * w + j) * PITCH + d] = qw[j] * p; }
            }
            p = (w < 3 ? c4[3] : 1.f) * (w < 2 ? c4[2] : 1.f) * (w < 1 ? c4[1] : 1.f);
            #pragma unroll
            for (int j = 3; j >= 0; --j) { kr[(4 * w + j) * PITCH + d] = kw[j] * p; p *= aw[j]; }
            if (!LOCAL)
            {
                float* dst = lv + w * BUF + d;
                auto level = [&] (auto hc) __attribute__((always_inline))
                {
                    constexpr int HALF = decltype(hc)::value;
                    float f = 1.f;
                    #pragma unroll
                    for (int t = 0; t < 16; ++t)
                        if (t & HALF) { f = (t & (HALF - 1)) ? f * a[t] : a[t]; dst[t * PITCH] = x[t] * f; }
                    #pragma unroll
                    for (int t = 15; t >= 0; --t)
                        if (!(t & HALF)) { f = (t & (HALF - 1)) == HALF - 1 ? 1.f : f * a[t + 1]; dst[t * PITCH] = x[t] * f; }
                };
                if (w == 0) level(gc_int<8>()); else if (w == 1) level(gc_int<4>()); else if (w == 2) level(gc_int<2>()); else level(gc_int<1>());
            }
        }
        __syncthreads();

        // sums over the key dimensions in four parts (every fourth tile each): four independent chains of matrix instructions, and sums as short as the token-by-token form's
        f4 O[4][2];
        #pragma unroll
        for (int u = 0; u < 4; ++u)
            #pragma unroll
            for (int c = 0; c < 2; ++c) O[u][c] = f4{ 0.f, 0.f, 0.f, 0.f };
        if (!LOCAL)
        {
            f4 A[4], dg = { 0.f, 0.f, 0.f, 0.f };
            #pragma unroll
            for (int u = 0; u < 4; ++u) A[u] = f4{ 0.f, 0.f, 0.f, 0.f };
            f4 x[DT];
            #pragma unroll
            for (int t = 0; t < DT; ++t) x[t] = *(const f4*) (lv + w * BUF + r16 * PITCH + 16 * t + 4 * g);
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                #pragma unroll
                for (int t = 0; t < DT; ++t) A[t & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t][i], x[t][i], A[t & 3], 0, 0, 0);
            #pragma unroll
            for (int u = 0; u < DT / 4; ++u)
            {
                const int t = w * (DT / 4) + u;
                const f4 xq = *(const f4*) (qs + r16 * PITCH + 16 * t + 4 * g), xk = *(const f4*) (ks + r16 * PITCH + 16 * t + 4 * g);
                #pragma unroll
                for (int i = 0; i < 4; ++i) dg = __builtin_amdgcn_mfma_f32_16x16x4f32(xq[i], xk[i], dg, 0, 0, 0);
            }
            A[0] = (A[0] + A[1]) + (A[2] + A[3]);
            const int half = 8 >> w;
            #pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                const int t = 4 * g + i, s = r16;
                const float lvl = ((t & half) && !(s & half) && (t ^ s) < 2 * half) ? A[0][i] : 0.f;
                ap[(w * 16 + t) * 20 + s] = lvl + (t == s ? dg[i] : 0.f);
            }
            #pragma unroll
            for (int t = 0; t < DT; ++t) x[t] = *(const f4*) (qp + r16 * PITCH + 16 * t + 4 * g);
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                #pragma unroll
                for (int t = 0; t < DT; ++t)
                    #pragma unroll
                    for (int c = 0; c < 2; ++c) O[t & 3][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t][i], S[t][c][i], O[t & 3][c], 0, 0, 0);
        }
        #pragma unroll
        for (int t = 0; t < DT; ++t)
        {
            const f4 gd = *(const f4*) (gs + 16 * t + 4 * g);
            #pragma unroll
            for (int c = 0; c < 2; ++c) S[t][c] *= gd;
            #pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const float x = kr[(4 * g + j) * PITCH + 16 * t + r16];
                #pragma unroll
                for (int c = 0; c < 2; ++c) S[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, vv[c][j], S[t][c], 0, 0, 0);
            }
        }
        if (!LOCAL)
        {
            __syncthreads();
            f4 A = *(const f4*) (ap + r16 * 20 + 4 * g), P[2] = { f4{ 0.f, 0.f, 0.f, 0.f }, f4{ 0.f, 0.f, 0.f, 0.f } };
            #pragma unroll
            for (int u = 1; u < 4; ++u) A += *(const f4*) (ap + (u * 16 + r16) * 20 + 4 * g);
            // A row of v that is not finite must not reach the rows in front of it, whose entries of A are zero (0 times infinity is NaN): such an entry counts as zero in the
            // product, and its column is NaN from its own row on
            int bad[2] = { 16, 16 };
            bool odd = false;
            #pragma unroll
            for (int c = 0; c < 2; ++c)
                #pragma unroll
                for (int j = 0; j < 4; ++j) odd |= !(fabsf(vv[c][j]) < INFINITY);
            const bool any_odd = __any(odd);
            if (any_odd)
            {
                #pragma unroll
                for (int c = 0; c < 2; ++c)
                {
                    #pragma unroll
                    for (int j = 3; j >= 0; --j) if (!(fabsf(vv[c][j]) < INFINITY)) { bad[c] = 4 * g + j; vv[c][j] = 0.f; }
                    bad[c] = min(bad[c], __shfl_xor(bad[c], 16, 64));
                    bad[c] = min(bad[c], __shfl_xor(bad[c], 32, 64));
                }
            }
            #pragma unroll
            for (int j = 0; j < 4; ++j)
                #pragma unroll
                for (int c = 0; c < 2; ++c) P[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[j], vv[c][j], P[c], 0, 0, 0);
            #pragma unroll
            for (int c = 0; c < 2; ++c) P[c] += (O[0][c] + O[1][c]) + (O[2][c] + O[3][c]);
            if (any_odd)
            {
                #pragma unroll
                for (int c = 0; c < 2; ++c)
                    #pragma unroll
                    for (int i = 0; i < 4; ++i) if (4 * g + i >= bad[c]) P[c][i] = NAN;
            }
            #pragma unroll
            for (int c = 0; c < 2; ++c)
                #pragma unroll
                for (int i = 0; i < 4; ++i)
                {
                    const int t = 4 * g + i;
                    if (n0 + t < last && col0 + 16 * c < vdim) o[((int64_t) (n0 + t) * heads + h) * vdim + col0 + 16 * c] = P[c][i];
                }
        }
    }
    if (!LOCAL) return;
    #pragma unroll
    for (int t = 0; t < DT; ++t)
        #pragma unroll
        for (int c = 0; c < 2; ++c)
            #pragma unroll
            for (int i = 0; i < 4; ++i) if (col0 + 16 * c < vdim) st[(int64_t) (16 * t + 4 * g + i) * vdim + col0 + 16 * c] = S[t][c][i];
    if (blockIdx.z == 0 && w == 0)
    {
        #pragma unroll
        for (int c = 0; c < ND; ++c) seg_decay[((int64_t) blockIdx.x * heads + h) * DIM + 64 * c + lane] = dec[c];
    }
}

template <bool LOCAL>
static int gla_chunk_launch(float* o, const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld, const void* lr, int64_t lr_ld, const void* a2,
                            const float* a2_bias, const int32_t* cu, int batch, int heads, int dim, int vdim, int rank, float tau, float q_scale, int dtype, void* stream,
                            int segs, int seg_len, float* seg_state, float* seg_decay, float* decay)
{
    const dim3 grid(batch * segs, heads, (vdim + 127) / 128);
    const size_t lds = gla_chunk_lds(dim, rank, LOCAL);
    #define GLA_CHUNK(DD) \
        if (lds > 65536) (void) hipFuncSetAttribute((const void*) gla_chunk_kernel<T, DD, LOCAL>, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds); \
        hipLaunchKernelGGL((gla_chunk_kernel<T, DD, LOCAL>), grid, dim3(256), lds, (hipStream_t) stream, o, (const T*) q, q_ld, (const T*) k, k_ld, (const T*) v, v_ld, \
                                             (const T*) lr, lr_ld, (const T*) a2, a2_bias, cu, heads, vdim, rank, 1.0f / tau, q_scale, segs, seg_len, seg_state, seg_decay, decay)
    MIX_DISPATCH_T(dtype, if (dim == 64) { GLA_CHUNK(64); } else { GLA_CHUNK(128); });
    #undef GLA_CHUNK
    return mix_check_launch("mix_gla_chunked");
}

template <int MODEV>
static int gla_launch(float* o, float* state, const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld,
                      const void* lr, int64_t lr_ld, const void* a2, const float* a2_bias, const int32_t* cu, const int32_t* slots, const int32_t* pos0,
                      int batch, int heads, int dim, int vdim, int rank, float tau, float q_scale, int dtype, void* stream,
                      int segs, int seg_len, float* seg_state, float* seg_decay)
{
    MIX_CHECK(o && state && q && k && v && lr && a2 && cu && slots && pos0, "mix_gla_scan: null pointer");
    MIX_CHECK(batch >= 0 && heads > 0 && dim > 0 && dim <= 256 && vdim > 0 && rank > 0 && tau > 0.f, "mix_gla_scan: sizes out of range (dim %d <= 256)", dim);
    MIX_CHECK(q_ld >= (int64_t) heads * dim && k_ld >= (int64_t) heads * dim && v_ld >= (int64_t) heads * vdim && lr_ld >= rank, "mix_gla_scan: bad row strides");
    if (batch == 0) return EXL3_MIX_OK;
    const dim3 grid(batch * segs, heads, (vdim + 63) / 64);
    const int SCAN_TC = dim > 128 ? 8 : 16;               // tokens staged per chunk: the LDS stays under 64 KB
    const size_t sm = (size_t) (3 * SCAN_TC * dim + SCAN_TC * 64 + SCAN_TC * SCAN_WAVES * 64) * sizeof(float);
    const int dr = (dim + SCAN_WAVES - 1) / SCAN_WAVES;
    #define GLA_SCAN(DRV) hipLaunchKernelGGL((gla_scan_kernel<T, DRV, MODEV>), grid, dim3(256), sm, (hipStream_t) stream, o, state, (const T*) q, q_ld, (const T*) k, k_ld, \
                                             (const T*) v, v_ld, (const T*) lr, lr_ld, (const T*) a2, a2_bias, cu, slots, pos0, heads, dim, vdim, rank, 1.0f / tau, q_scale, SCAN_TC, \
                                             segs, seg_len, seg_state, seg_decay)
    MIX_DISPATCH_T(dtype,
        if (dr <= 8) GLA_SCAN(8); else if (dr <= 16) GLA_SCAN(16); else if (dr <= 32) GLA_SCAN(32); else GLA_SCAN(64));
    #undef GLA_SCAN
    return mix_check_launch("mix_gla_scan");
}

extern "C" int exl3_mix_gla_scan(float* o, float* state, const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld,
                                 const void* lr, int64_t lr_ld, const void* a2, const float* a2_bias, const int32_t* cu, const int32_t* slots, const int32_t* pos0,
                                 int batch, int heads, int dim, int vdim, int rank, float tau, float q_scale, int dtype, void* stream)
{
    return gla_launch<GLA_WHOLE>(o, state, q, q_ld, k, k_ld, v, v_ld, lr, lr_ld, a2, a2_bias, cu, slots, pos0, batch, heads, dim, vdim, rank, tau, q_scale, dtype, stream,
                                 1, 0, nullptr, nullptr);
}

static int gla_combine_launch(float* state, float* seg_state, const float* seg_decay, const int32_t* cu, const int32_t* slots, const int32_t* pos0, int batch, int heads, int dim, int vdim,
                              int segs, int seg_len, void* stream)
{
    const int64_t per = (int64_t) dim * vdim;
    hipLaunchKernelGGL(gla_combine_kernel, dim3(batch, heads, (unsigned) ((per + 1023) / 1024)), dim3(256), 0, (hipStream_t) stream, state, seg_state, seg_decay, cu, slots, pos0,
                       heads, dim, vdim, segs, seg_len);
    return mix_check_launch("mix_gla (combine)");
}

extern "C" int exl3_mix_gla_segmented(float* o, float* state, const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld,
                                      const void* lr, int64_t lr_ld, const void* a2, const float* a2_bias, const int32_t* cu, const int32_t* slots, const int32_t* pos0,
                                      int batch, int heads, int dim, int vdim, int rank, float tau, float q_scale, int segs, int seg_len,
                                      float* seg_state, float* seg_decay, int dtype, void* stream)
{
    MIX_CHECK(segs >= 1 && seg_len >= 1 && seg_state && seg_decay, "mix_gla_segmented: bad segment arguments");
    int rc = gla_launch<GLA_SEG_LOCAL>(o, state, q, q_ld, k, k_ld, v, v_ld, lr, lr_ld, a2, a2_bias, cu, slots, pos0, batch, heads, dim, vdim, rank, tau, q_scale, dtype,
                                       stream, segs, seg_len, seg_state, seg_decay);
    if (rc || batch == 0) return rc;
    if ((rc = gla_combine_launch(state, seg_state, seg_decay, cu, slots, pos0, batch, heads, dim, vdim, segs, seg_len, stream))) return rc;
    return gla_launch<GLA_SEG_FINAL>(o, state, q, q_ld, k, k_ld, v, v_ld, lr, lr_ld, a2, a2_bias, cu, slots, pos0, batch, heads, dim, vdim, rank, tau, q_scale, dtype,
                                     stream, segs, seg_len, seg_state, seg_decay);
}

// its shapes: key dimensions that are whole matrix tiles of one or two values per lane, a low-rank input that fits LDS; there the chunk form wins from the first segment on
extern "C" int exl3_mix_gla_chunked(float* o, float* state, const void* q, int64_t q_ld, const void* k, int64_t k_ld, const void* v, int64_t v_ld,
                                    const void* lr, int64_t lr_ld, const void* a2, const float* a2_bias, const int32_t* cu, const int32_t* slots, const int32_t* pos0,
                                    int batch, int heads, int dim, int vdim, int rank, float tau, float q_scale, int segs, int seg_len,
                                    float* seg_state, float* seg_decay, float* decay, int dtype, void* stream)
{
    MIX_CHECK(segs >= 1 && seg_len >= 1 && seg_state && seg_decay && decay, "mix_gla_chunked: bad segment arguments");
    MIX_CHECK((dim == 64 || dim == 128) && rank <= GC_MAX_RANK, "mix_gla_chunked: key dimension 64 or 128, rank at most %d", GC_MAX_RANK);
    MIX_CHECK(o && state && q && k && v && lr && a2 && cu && slots && pos0 && batch >= 0 && heads > 0 && vdim > 0 && rank > 0 && tau > 0.f, "mix_gla_chunked: null pointer or sizes out of range");
    MIX_CHECK(q_ld >= (int64_t) heads * dim && k_ld >= (int64_t) heads * dim && v_ld >= (int64_t) heads * vdim && lr_ld >= rank, "mix_gla_chunked: bad row strides");
    if (batch == 0) return EXL3_MIX_OK;
    int rc = gla_chunk_launch<true>(o, q, q_ld, k, k_ld, v, v_ld, lr, lr_ld, a2, a2_bias, cu, batch, heads, dim, vdim, rank, tau, q_scale, dtype, stream, segs, seg_len,
                                    seg_state, seg_decay, decay);
    if (rc || (rc = gla_combine_launch(state, seg_state, seg_decay, cu, slots, pos0, batch, heads, dim, vdim, segs, seg_len, stream))) return rc;
    return gla_chunk_launch<false>(o, q, q_ld, k, k_ld, v, v_ld, lr, lr_ld, a2, a2_bias, cu, batch, heads, dim, vdim, rank, tau, q_scale, dtype, stream, segs, seg_len,
                                   seg_state, seg_decay, decay);
}

extern "C" int exl3_mix_gla_out(void* out, const float* o, const float* w, const void* g, int64_t g_ld, float eps, int n, int heads, int vdim, int dtype, void* stream)
{
    MIX_CHECK(out && o && w && g && n >= 0 && heads > 0 && vdim > 0 && g_ld >= (int64_t) heads * vdim, "mix_gla_out: bad arguments");
    if (n == 0) return EXL3_MIX_OK;
    const int64_t items = (int64_t) n * heads;
    const bool by4 = vdim % 4 == 0 && g_ld % 4 == 0 && (((uintptr_t) out | (uintptr_t) o | (uintptr_t) w | (uintptr_t) g) & 15) == 0;
    #define GLA_OUT(VV) hipLaunchKernelGGL((gla_out_kernel<T, VV>), dim3((unsigned) ((items + 7) / 8)), dim3(256), 0, (hipStream_t) stream, (T*) out, o, w, (const T*) g, g_ld, eps, \
                                           items, heads, vdim)
    MIX_DISPATCH_T(dtype, if (by4) GLA_OUT(4); else GLA_OUT(1));
    #undef GLA_OUT
    return mix_check_launch("mix_gla_out");
}
