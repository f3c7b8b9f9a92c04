// The row worker of the lane-per-key attention kernels (exact float32 scores and softmax): shared by the sliding-window kernels of mix_attn.hip
// and the latent-cache decode kernel of mix_latent.hip.
#pragma once
#include "mix_common.cuh"

// One workgroup of NW waves (AT_WAVES unless the caller asks for more: few rows, long caches) per (row, query head).  Keys kb + j * k_step, values vb + j * v_step, j < count: wave w takes the 64-key chunks
// w, w + NW, ... (one key per lane, its row read in 16-byte pieces when the layout allows), keeps its own running maximum, sum and
// value accumulators (MAXV = ceil(vdim / 64) per lane), and the waves are merged through LDS at the end.  Wave 0 starts from the sink.
// The query's first dim1 elements are read from q, the rest from q2 (dim1 = dim: one part).  softcap > 0: score <- softcap tanh(score / softcap).
// RowMap: where key j lies.  row_linear: row j.  row_jump: row j, and row j + jump from j = at on (the kept first tokens ahead of a window).  row_paged: through a
// page table.  gate_row (optional): vdim gate values before their sigmoid, multiplied element by element with the result (`gate` is one factor for all).
// TO: the element type of the result (float keeps the weighted sum unrounded for a caller that combines several maps).
#define AT_WAVES 4

// Whether bfloat16 rows take the form that reads whole 128-byte lines: rows of 64, 128, .. elements at addresses of 16 bytes, values of at most 256 (the accumulators fit)
static inline bool rows_of_lines(const void* k, int64_t k_step, const void* v, int64_t v_step, int dim, int vdim)
{
    return dim % 64 == 0 && vdim % 64 == 0 && vdim <= 256 && (((uintptr_t) k | (uintptr_t) v) & 15) == 0 && k_step % 8 == 0 && v_step % 8 == 0 && k_step < (1 << 27) && v_step < (1 << 27);
}

template <typename T> struct kvec;
template <> struct kvec<bf16_t> { static constexpr int N = 8; };
template <> struct kvec<float> { static constexpr int N = 4; };

struct row_linear
{
    static constexpr bool linear = true;
    __device__ __forceinline__ int64_t operator()(int j) const { return j; }
};
struct row_jump
{
    static constexpr bool linear = false;
    int at; int64_t jump;
    __device__ __forceinline__ int64_t operator()(int j) const { return j < at ? (int64_t) j : j + jump; }
};
struct row_paged
{
    static constexpr bool linear = false;
    const int32_t* table; int page;
    __device__ __forceinline__ int64_t operator()(int j) const { return (int64_t) table[j / page] * page + (j % page); }
};

// the waves' parts (maximum, sum, accumulators in LDS) to the row's result: wave 0 rescales them to the common maximum
template <typename T, int MAXV, typename TO, int NW>
__device__ __forceinline__ void attn_row_merge(TO* __restrict__ out, int vdim, float gate, const float* mg, const T* gate_row)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    float acc[MAXV];
    __syncthreads();
    if (w != 0) return;
    float mt = -INFINITY;
    #pragma unroll
    for (int ww = 0; ww < NW; ++ww) mt = fmaxf(mt, mg[ww * (2 + MAXV * 64)]);
    float lt = 0.f;
    #pragma unroll
    for (int i = 0; i < MAXV; ++i) acc[i] = 0.f;
    #pragma unroll
    for (int ww = 0; ww < NW; ++ww)
    {
        const float* o = mg + ww * (2 + MAXV * 64);
        const float f = (o[0] == -INFINITY) ? 0.f : expf(o[0] - mt);
        lt += o[1] * f;
        #pragma unroll
        for (int i = 0; i < MAXV; ++i) acc[i] += o[2 + i * 64 + lane] * f;
    }
    const float f = (lt > 0.f ? 1.0f / lt : 0.f) * gate;
    #pragma unroll
    for (int i = 0; i < MAXV; ++i)
    {
        const int c = lane + 64 * i;
        if (c < vdim) out[c] = from_f<TO>(acc[i] * f * (gate_row ? sigmoid_f(to_f(gate_row[c])) : 1.0f));
    }
}

template <typename T, int MAXV, bool LINES, typename TO = T, int NW = AT_WAVES, typename RowMap = row_linear>
__device__ __forceinline__ void attn_row(TO* __restrict__ out, const T* __restrict__ q, const T* q2, int dim1, const T* __restrict__ kb, int64_t k_step, const T* __restrict__ vb,
                                         int64_t v_step, int count, int dim, int vdim, float scale, bool has_sink, float sink, float gate, bool k_vec,
                                         float* smem, float softcap = 0.f, RowMap map = RowMap(), const T* gate_row = nullptr)
{
    float* qs = smem;                                   // [dim]
    float* ps = qs + dim;                               // [NW][64]
    float* mg = ps + NW * 64;                     // [NW][2 + MAXV * 64]: m, l, accumulators
    // the wave's index as a scalar helps the forms below whose loads leave registers (float32 of up to 256 values: 0.91 of the time) and costs one key per lane in bfloat16 2 to 10 %, in float32 over
    // 256 values up to 80 % (8 heads of 320, 1 key: 8.0 us, 14.6)
    constexpr bool SCALAR_WAVE = LINES || (sizeof(T) == 4 && MAXV <= 4);
    const int lane = threadIdx.x & 63, w = SCALAR_WAVE ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : (int) (threadIdx.x >> 6);
    for (int i = threadIdx.x; i < dim; i += 64 * NW) qs[i] = to_f(i < dim1 ? q[i] : q2[i - dim1]);      // the query may come in two parts
    __syncthreads();
    const bool seeded = has_sink && w == 0;
    float m = seeded ? sink : -INFINITY, l = seeded ? 1.0f : 0.0f;
    float acc[MAXV];
    #pragma unroll
    for (int i = 0; i < MAXV; ++i) acc[i] = 0.f;
    float* pw = ps + w * 64;
    constexpr int VN = kvec<T>::N;
    // LINES (rows_of_lines above): eight lanes share a row, 16 bytes each, so a load instruction reads eight rows as they lie in memory -- one key per lane fetches every
    // line eight times, and value rows two bytes at a time take 64 instructions -- and a chunk's key rows and value rows are all in flight at once.  Scores are added over
    // the eight lanes, outputs over the eight rows at the end.  Decode only: a kernel that held both forms spilled and ran short rows up to 1.5 times longer, and prompt
    // rows, whose neighbours read the same keys from the caches, are faster one key per lane (200 rows of 32 heads, 128 dimensions: 45 us against 77).
    // 8 rows of 32 heads, one key per lane / here: 1000 keys of 64 dimensions 13.6 / 10.9 us, of 128 21.0 / 15.5, of 256 66.7 / 27.1; 64 keys of 128 10.2 / 8.6;
    // 1 key of 128 7.5 / 7.7, and of 64 with values of 128 6.8 / 7.4 (the only sizes tried that lose more than 0.3 us).
    if constexpr (LINES)
    {
        constexpr bool AHEAD = MAXV == 1 || NW <= 8;                 // registers for the values next to the keys; else the values follow the scores and keys come four at a time
        constexpr int KR = AHEAD ? 8 : 4;
        const int kg = lane >> 3, kp = lane & 7;
        float va[MAXV][8];
        #pragma unroll
        for (int i = 0; i < MAXV; ++i)
            #pragma unroll
            for (int e = 0; e < 8; ++e) va[i][e] = 0.f;
        union piece { uint4 v; T e[8]; };
        // the eight rows from j on (past the end: the last one): where they lie in a line, a scalar base and a 32-bit offset per lane -- 16 waves leave 128 registers each
        auto rows = [&] (const T* base, int64_t step, int j, int c) __attribute__((always_inline)) -> uint4
        {
            const int first = min(j, count - 1);
            if constexpr (RowMap::linear) return *(const uint4*) (base + first * step + c + (min(kg, count - 1 - first) * (int) step + 8 * kp));
            else return *(const uint4*) (base + map(min(j + kg, count - 1)) * step + c + 8 * kp);
        };
        // chunks of 8 .. 64 keys: a row too short for 64 to every wave is shared by more of them, each with a shorter chain of loads (64 keys of 128 dimensions: 12.4 us in one chunk, 8.6)
        const int chunk = min(64, (count + 8 * NW - 1) / (8 * NW) * 8);
        for (int j0 = w * chunk; j0 < count; j0 += chunk * NW)
        {
            const int here = min(chunk, count - j0);                // keys of this chunk: eight rows at a time are skipped behind the last
            float d[8];
            piece tv[8];
            auto values = [&] (int c)
            {
                #pragma unroll
                for (int i = 0; i < 8; ++i) { if (8 * i >= here) break; tv[i].v = rows(vb, v_step, j0 + 8 * i, c); }
            };
            #pragma unroll
            for (int i = 0; i < 8; ++i) d[i] = 0.f;
            for (int c = 0; c < dim; c += 64)
            {
                float qv[8];
                #pragma unroll
                for (int e = 0; e < 8; ++e) qv[e] = qs[c + 8 * kp + e];
                #pragma unroll
                for (int i0 = 0; i0 < 8; i0 += KR)
                {
                    piece tk[KR];
                    #pragma unroll
                    for (int i = 0; i < KR; ++i) { if (8 * (i0 + i) >= here) break; tk[i].v = rows(kb, k_step, j0 + 8 * (i0 + i), c); }
                    if (AHEAD && c == 0 && i0 + KR == 8) values(0);
                    #pragma unroll
                    for (int i = 0; i < KR; ++i)
                    {
                        if (8 * (i0 + i) >= here) break;
                        #pragma unroll
                        for (int e = 0; e < 8; ++e) d[i0 + i] += qv[e] * to_f(tk[i].e[e]);
                    }
                }
            }
            #pragma unroll
            for (int i = 0; i < 8; ++i) d[i] = row8_sum(d[i]);
            if (kp == 0)
            {
                #pragma unroll
                for (int i = 0; i < 8; ++i) pw[8 * i + kg] = d[i];
            }
            __builtin_amdgcn_wave_barrier();
            float s = pw[lane] * scale;
            if (softcap > 0.f) s = softcap * tanhf(s / softcap);
            if (lane >= here) s = -INFINITY;
            const float m_new = fmaxf(m, wave_max(s));
            const float p = lane < here ? expf(s - m_new) : 0.f, corr = expf(m - m_new);
            l = l * corr + wave_sum(p);
            m = m_new;
            __builtin_amdgcn_wave_barrier();
            pw[lane] = p;
            __builtin_amdgcn_wave_barrier();
            #pragma unroll
            for (int i = 0; i < MAXV; ++i)
            {
                if (64 * i >= vdim) continue;
                if (i > 0 || !AHEAD) values(64 * i);
                #pragma unroll
                for (int e = 0; e < 8; ++e) va[i][e] *= corr;
                #pragma unroll
                for (int r = 0; r < 8; ++r)
                {
                    if (8 * r >= here) break;
                    const bool in = 8 * r + kg < here;
                    const float pr = pw[8 * r + kg];
                    #pragma unroll
                    for (int e = 0; e < 8; ++e) va[i][e] += in ? pr * to_f(tv[r].e[e]) : 0.f;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        float* part = mg + w * (2 + MAXV * 64);
        if (lane == 0) { part[0] = m; part[1] = l; }
        if (w * chunk < count)
        {
            #pragma unroll
            for (int i = 0; i < MAXV; ++i)
                #pragma unroll
                for (int e = 0; e < 8; ++e) va[i][e] = sum_of_8th_lanes(va[i][e]);
        }
        if (kg == 0)
        {
            #pragma unroll
            for (int i = 0; i < MAXV; ++i)
                #pragma unroll
                for (int e = 0; e < 8; ++e) part[2 + 64 * i + 8 * kp + e] = va[i][e];
        }
        attn_row_merge<T, MAXV, TO, NW>(out, vdim, gate, mg, gate_row);
        return;
    }
    for (int j0 = w * 64; j0 < count; j0 += 64 * NW)
    {
        const int j = j0 + lane;
        float s = -INFINITY;
        if (j < count)
        {
            const T* kr = kb + map(j) * k_step;
            float d = 0.f;
            if (k_vec)
            {
                for (int c = 0; c < dim; c += VN)
                {
                    union { uint4 v; T e[VN]; } t;
                    t.v = *(const uint4*) (kr + c);
                    #pragma unroll
                    for (int e = 0; e < VN; ++e) d += qs[c + e] * to_f(t.e[e]);
                }
            }
            else
                for (int c = 0; c < dim; ++c) d += qs[c] * to_f(kr[c]);
            s = d * scale;
            if (softcap > 0.f) s = softcap * tanhf(s / softcap);
        }
        const float m_new = fmaxf(m, wave_max(s));          // finite: j0 < count, so lane 0 of the chunk holds a score
        const float p = (j < count) ? expf(s - m_new) : 0.f;
        const float corr = expf(m - m_new);                 // m = -inf (nothing yet): 0
        l = l * corr + wave_sum(p);
        m = m_new;
        pw[lane] = p;
        __builtin_amdgcn_wave_barrier();                    // LDS serves a wave's accesses in order: its own stores are visible to the reads below
        const int cnt = min(64, count - j0);
        #pragma unroll
        for (int i = 0; i < MAXV; ++i)
        {
            const int c = lane + 64 * i;
            float a = acc[i] * corr;
            if (c < vdim)
            {
                int jj = 0;
                for (; jj + 8 <= cnt; jj += 8)                // eight value rows in flight, then the sums
                {
                    float vv[8];
                    #pragma unroll
                    for (int e = 0; e < 8; ++e) vv[e] = to_f(vb[map(j0 + jj + e) * v_step + c]);
                    #pragma unroll
                    for (int e = 0; e < 8; ++e) a += pw[jj + e] * vv[e];
                }
                for (; jj < cnt; ++jj) a += pw[jj] * to_f(vb[map(j0 + jj) * v_step + c]);
            }
            acc[i] = a;
        }
        __builtin_amdgcn_wave_barrier();
    }
    float* mine = mg + w * (2 + MAXV * 64);
    if (lane == 0) { mine[0] = m; mine[1] = l; }
    #pragma unroll
    for (int i = 0; i < MAXV; ++i) mine[2 + i * 64 + lane] = acc[i];
    attn_row_merge<T, MAXV, TO, NW>(out, vdim, gate, mg, gate_row);
}

template <typename T>
__device__ __forceinline__ bool rows_are_16_byte(const T* base, int64_t step, int dim)
{
    return ((uintptr_t) base % 16 == 0) && ((step * (int64_t) sizeof(T)) % 16 == 0) && (dim % kvec<T>::N == 0);
}

