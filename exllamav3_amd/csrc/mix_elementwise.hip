// Row-wise kernels over a float32 residual stream: embedding, RMS norm, gated residual (+ the next norm), PolyNorm, the router's
// top-k softmax.  One workgroup per row; every reduction is float32.
#include "mix_common.cuh"

static thread_local char g_mix_err[512] = "";
void mix_set_error(const char* fmt, ...)
{
    va_list ap; va_start(ap, fmt); vsnprintf(g_mix_err, sizeof(g_mix_err), fmt, ap); va_end(ap);
}
int mix_check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { mix_set_error("%s: launch failed: %s", what, hipGetErrorString(e)); return EXL3_MIX_ERR_HIP; }
    return EXL3_MIX_OK;
}
extern "C" const char* exl3_mix_last_error(void) { return g_mix_err; }
extern "C" int exl3_mix_abi_version(void) { return EXL3_MIX_ABI_VERSION; }

#define ROW_THREADS 256
#define ROW_WAVES 4

// The row kernels below are bounded by HBM at prompt sizes and by the latency of their one pass at decode sizes, so both want few, wide accesses that are all in flight at
// once: V elements per thread and access (V: 16 bytes of the activation type, where row strides and addresses allow; else 1), the first HELD pieces of a thread in
// registers between the sums and the write (a wider row reads its remaining pieces twice).
// Measured (us, one element per access and the row read again -> now; bfloat16): 4096 rows: polynorm of 14336 104 -> 47, embedding of 4096 56 -> 34, gated residual 51 -> 42, the
// first and last at the rate of a large copy (5 TB/s); 8 rows: polynorm of 8192 13.9 -> 4.7, embedding of 2048 9.4 -> 4.2, gated residual 6.8 -> 4.5.
template <typename T> __host__ __device__ constexpr int wide_n() { return 16 / (int) sizeof(T); }

#define ROW_HELD 4

// h = x inv w for the row whose first pieces are in `held`; the others come from x, which the same thread wrote or read
template <typename T, int V, int NT = ROW_THREADS, int HELD = ROW_HELD>
__device__ __forceinline__ void row_norm_write(T* __restrict__ hr, const float* xr, const float* __restrict__ w, const float (&held)[HELD][V], float inv, int width)
{
    auto write = [&] (int i, const float (&v)[V]) __attribute__((always_inline))
    {
        float wv[V];
        load_n<float, V>(w + i, wv);
        #pragma unroll
        for (int e = 0; e < V; ++e) wv[e] = v[e] * inv * wv[e];
        store_n<T, V>(hr + i, wv);
    };
    #pragma unroll
    for (int u = 0; u < HELD; ++u) { const int i = (u * NT + threadIdx.x) * V; if (i < width) write(i, held[u]); }
    for (int i = (HELD * NT + threadIdx.x) * V; i < width; i += NT * V) { float t[V]; load_n<float, V>(xr + i, t); write(i, t); }
}

template <typename T, int V>
__global__ __launch_bounds__(ROW_THREADS) void embed_kernel(float* __restrict__ x, T* __restrict__ h, const T* __restrict__ table,
                                                            const int32_t* __restrict__ tokens, float scale, const float* __restrict__ norm_w,
                                                            float eps, int width, int vocab)
{
    __shared__ float red[ROW_WAVES];
    const int n = blockIdx.x;
    int tok = tokens[n];
    tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);
    const T* src = table + (int64_t) tok * width;
    float* xr = x + (int64_t) n * width;
    float held[ROW_HELD][V];
    float ss = 0.f;
    auto form = [&] (int i, float (&t)[V]) __attribute__((always_inline))
    {
        #pragma unroll
        for (int e = 0; e < V; ++e) { t[e] *= scale; ss += t[e] * t[e]; }
        store_n<float, V>(xr + i, t);
    };
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u) { const int i = (u * ROW_THREADS + threadIdx.x) * V; if (i < width) load_n<T, V>(src + i, held[u]); }
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u) { const int i = (u * ROW_THREADS + threadIdx.x) * V; if (i < width) form(i, held[u]); }
    for (int i = (ROW_HELD * ROW_THREADS + threadIdx.x) * V; i < width; i += ROW_THREADS * V) { float t[V]; load_n<T, V>(src + i, t); form(i, t); }
    if (!norm_w) return;
    ss = block_sum<ROW_WAVES>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float) width + eps);
    row_norm_write<T, V>(h + (int64_t) n * width, xr, norm_w, held, inv, width);
}

template <typename T, int V>
__global__ __launch_bounds__(ROW_THREADS) void rms_norm_rows_kernel(T* __restrict__ h, const float* __restrict__ x, const int32_t* __restrict__ rows,
                                                                    const float* __restrict__ w, float eps, int width)
{
    __shared__ float red[ROW_WAVES];
    const int n = blockIdx.x;
    const float* xr = x + (int64_t) (rows ? rows[n] : n) * width;
    float held[ROW_HELD][V];
    float ss = 0.f;
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u) { const int i = (u * ROW_THREADS + threadIdx.x) * V; if (i < width) load_n<float, V>(xr + i, held[u]); }
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u)
    {
        if ((u * ROW_THREADS + (int) threadIdx.x) * V >= width) continue;
        #pragma unroll
        for (int e = 0; e < V; ++e) ss += held[u][e] * held[u][e];
    }
    for (int i = (ROW_HELD * ROW_THREADS + threadIdx.x) * V; i < width; i += ROW_THREADS * V)
    {
        float t[V];
        load_n<float, V>(xr + i, t);
        #pragma unroll
        for (int e = 0; e < V; ++e) ss += t[e] * t[e];
    }
    ss = block_sum<ROW_WAVES>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float) width + eps);
    row_norm_write<T, V>(h + (int64_t) n * width, xr, w, held, inv, width);
}

template <typename T, int V, int NW, int HELD>
__global__ __launch_bounds__(64 * NW) void gated_residual_kernel(float* __restrict__ x, const T* __restrict__ y, int64_t y_ld, const T* __restrict__ r,
                                                                     int64_t r_ld, const float* __restrict__ norm_w, T* __restrict__ h, float eps, int width)
{
    constexpr int NT = 64 * NW;
    __shared__ float red[NW];
    const int n = blockIdx.x;
    float* xr = x + (int64_t) n * width;
    const T* yr = y + (int64_t) n * y_ld;
    const T* rr = r + (int64_t) n * r_ld;
    float held[HELD][V], yv[HELD][V], rv[HELD][V];
    float ss = 0.f;
    auto form = [&] (int i, float (&v)[V], const float (&a)[V], const float (&g)[V]) __attribute__((always_inline))
    {
        #pragma unroll
        for (int e = 0; e < V; ++e) { v[e] = v[e] + a[e] * sigmoid_f(g[e]); ss += v[e] * v[e]; }
        store_n<float, V>(xr + i, v);
    };
    #pragma unroll
    for (int u = 0; u < HELD; ++u)
    {
        const int i = (u * NT + threadIdx.x) * V;
        if (i < width) { load_n<float, V>(xr + i, held[u]); load_n<T, V>(yr + i, yv[u]); load_n<T, V>(rr + i, rv[u]); }
    }
    #pragma unroll
    for (int u = 0; u < HELD; ++u) { const int i = (u * NT + threadIdx.x) * V; if (i < width) form(i, held[u], yv[u], rv[u]); }
    for (int i = (HELD * NT + threadIdx.x) * V; i < width; i += NT * V)
    {
        float v[V], a[V], g[V];
        load_n<float, V>(xr + i, v); load_n<T, V>(yr + i, a); load_n<T, V>(rr + i, g);
        form(i, v, a, g);
    }
    if (!norm_w) return;
    ss = block_sum<NW>(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float) width + eps);
    row_norm_write<T, V, NT, HELD>(h + (int64_t) n * width, xr, norm_w, held, inv, width);
}

template <typename T, int V, int NW>
__global__ __launch_bounds__(64 * NW) void polynorm_kernel(T* __restrict__ out, const T* __restrict__ z, int64_t z_ld, const float* __restrict__ coef,
                                                                   float eps, int ff)
{
    constexpr int NT = 64 * NW;
    __shared__ float red[3][NW];
    const int n = blockIdx.x;
    const T* zr = z + (int64_t) n * z_ld;
    float held[ROW_HELD][V];
    float s1 = 0.f, s2 = 0.f, s3 = 0.f;
    auto add = [&] (const float (&t)[V]) __attribute__((always_inline))
    {
        #pragma unroll
        for (int e = 0; e < V; ++e)
        {
            const float v = t[e], v2 = v * v, v3 = v2 * v;
            s1 += v2; s2 += v2 * v2; s3 += v3 * v3;
        }
    };
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u) { const int i = (u * NT + threadIdx.x) * V; if (i < ff) load_n<T, V>(zr + i, held[u]); }
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u) if ((u * NT + (int) threadIdx.x) * V < ff) add(held[u]);
    for (int i = (ROW_HELD * NT + threadIdx.x) * V; i < ff; i += NT * V) { float t[V]; load_n<T, V>(zr + i, t); add(t); }
    s1 = wave_sum(s1); s2 = wave_sum(s2); s3 = wave_sum(s3);
    if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = s1; red[1][threadIdx.x >> 6] = s2; red[2][threadIdx.x >> 6] = s3; }
    __syncthreads();
    s1 = s2 = s3 = 0.f;
    #pragma unroll
    for (int i = 0; i < NW; ++i) { s1 += red[0][i]; s2 += red[1][i]; s3 += red[2][i]; }
    const float i1 = 1.0f / sqrtf(s1 / (float) ff + eps), i2 = 1.0f / sqrtf(s2 / (float) ff + eps), i3 = 1.0f / sqrtf(s3 / (float) ff + eps);
    const float a = coef[0], b = coef[1], c = coef[2], k = coef[3];
    T* o = out + (int64_t) n * ff;
    auto write = [&] (int i, float (&t)[V]) __attribute__((always_inline))
    {
        #pragma unroll
        for (int e = 0; e < V; ++e) { const float v = t[e], v2 = v * v; t[e] = a * (v * i1) + b * (v2 * i2) + c * (v2 * v * i3) + k; }
        store_n<T, V>(o + i, t);
    };
    #pragma unroll
    for (int u = 0; u < ROW_HELD; ++u) { const int i = (u * NT + threadIdx.x) * V; if (i < ff) write(i, held[u]); }
    for (int i = (ROW_HELD * NT + threadIdx.x) * V; i < ff; i += NT * V) { float t[V]; load_n<T, V>(zr + i, t); write(i, t); }
}

__global__ void topk_softmax_kernel(int32_t* __restrict__ idx, float* __restrict__ wts, const float* __restrict__ logits, int n, int experts, int top)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float* l = logits + (int64_t) t * experts;
    int32_t* id = idx + (int64_t) t * top;
    float* w = wts + (int64_t) t * top;
    for (int r = 0; r < top; ++r)
    {
        int best = -1; float bv = 0.f;
        for (int e = 0; e < experts; ++e)
        {
            bool taken = false;
            for (int p = 0; p < r; ++p) taken |= (id[p] == e);
            if (taken) continue;
            float v = l[e];
            if (best < 0 || v > bv) { best = e; bv = v; }
        }
        id[r] = best; w[r] = bv;
    }
    const float m = w[0];
    float s = 0.f;
    for (int r = 0; r < top; ++r) { float e = expf(w[r] - m); w[r] = e; s += e; }
    for (int r = 0; r < top; ++r) w[r] = w[r] / s;
}

// whether rows of `width` elements, `ld` apart, can be walked in pieces of 16 bytes (addresses: aligned16)
template <typename T> static bool row_wide(int64_t width, int64_t ld) { return width % wide_n<T>() == 0 && ld % wide_n<T>() == 0; }
static bool aligned16(const void* a, const void* b, const void* c, const void* d) { return (((uintptr_t) a | (uintptr_t) b | (uintptr_t) c | (uintptr_t) d) & 15) == 0; }

extern "C" int exl3_mix_embed(float* x, void* h, const void* table, const int32_t* tokens, float scale, const float* norm_w, float eps,
                              int n, int width, int vocab, int dtype, void* stream)
{
    MIX_CHECK(x && table && tokens && n >= 0 && width > 0 && vocab > 0 && (!norm_w || h), "mix_embed: bad arguments");
    if (n == 0) return EXL3_MIX_OK;
    #define EMBED(VV) hipLaunchKernelGGL((embed_kernel<T, VV>), dim3(n), dim3(ROW_THREADS), 0, (hipStream_t) stream, x, (T*) h, (const T*) table, tokens, scale, norm_w, eps, width, vocab)
    // (up to 256 wide 16 bytes a lane leave most lanes idle: 128 wide, 4096 rows 5.1 us, 4.5 with one element)
    MIX_DISPATCH_T(dtype, if (width > 256 && row_wide<T>(width, width) && aligned16(x, h, table, norm_w)) EMBED(wide_n<T>()); else EMBED(1));
    #undef EMBED
    return mix_check_launch("mix_embed");
}

extern "C" int exl3_mix_rms_norm_rows(void* h, const float* x, const int32_t* rows, const float* w, float eps, int n, int width, int dtype, void* stream)
{
    MIX_CHECK(h && x && w && n >= 0 && width > 0, "mix_rms_norm_rows: bad arguments");
    if (n == 0) return EXL3_MIX_OK;
    #define NORM(VV) hipLaunchKernelGGL((rms_norm_rows_kernel<T, VV>), dim3(n), dim3(ROW_THREADS), 0, (hipStream_t) stream, (T*) h, x, rows, w, eps, width)
    MIX_DISPATCH_T(dtype, if (row_wide<T>(width, width) && aligned16(x, h, w, nullptr)) NORM(wide_n<T>()); else NORM(1));
    #undef NORM
    return mix_check_launch("mix_rms_norm_rows");
}

extern "C" int exl3_mix_gated_residual(float* x, const void* y, int64_t y_ld, const void* r, int64_t r_ld, const float* norm_w, void* h, float eps,
                                       int n, int width, int dtype, void* stream)
{
    MIX_CHECK(x && y && r && n >= 0 && width > 0 && y_ld >= width && r_ld >= width && (!norm_w || h), "mix_gated_residual: bad arguments");
    if (n == 0) return EXL3_MIX_OK;
    // 1000 wide, 4096 rows of bfloat16: 14.4 us with four waves, 11.6 with the two that the row keeps busy.  Short rows leave most lanes idle at 16 bytes each (8 rows, us with
    // one element a lane: 96 wide 3.0 / 2.3, 512 wide 2.8 / 2.6; 4096 rows of 512 10.1 / 11.2).  Single elements: one piece held -- four make long rows wait for more than they hide (2050 wide, 4096 rows 33.6 us with four, 30.7 with one) -- and, while the rows are too few to fill the
    // chip, eight waves (2050 wide, us of four / eight: 1 row 4.7 / 3.4, 1024 rows 12.2 / 10.2, 4096 rows 30.7 / 35.6).
    #define GATED(VV, NW, H) hipLaunchKernelGGL((gated_residual_kernel<T, VV, NW, H>), dim3(n), dim3(64 * NW), 0, (hipStream_t) stream, x, (const T*) y, y_ld, (const T*) r, r_ld, norm_w, (T*) h, eps, width)
    MIX_DISPATCH_T(dtype, constexpr int V = wide_n<T>();
                          const bool wide = width > (n <= 1024 ? 512 : 256) && row_wide<T>(width, y_ld) && row_wide<T>(width, r_ld) && aligned16(x, y, r, norm_w) && aligned16(h, nullptr, nullptr, nullptr);
                          if (wide && width <= 128 * V) GATED(V, 2, ROW_HELD); else if (wide) GATED(V, 4, ROW_HELD);
                          else if (width > 512 && n <= 1024) GATED(1, 8, 1); else GATED(1, 4, 1));
    #undef GATED
    return mix_check_launch("mix_gated_residual");
}

extern "C" int exl3_mix_polynorm(void* out, const void* z, int64_t z_ld, const float* coef, float eps, int n, int ff, int dtype, void* stream)
{
    MIX_CHECK(out && z && coef && n >= 0 && ff > 0 && z_ld >= ff, "mix_polynorm: bad arguments");
    if (n == 0) return EXL3_MIX_OK;
    // waves that a row keeps busy (bfloat16, 4096 rows, us with 8 waves / here: 1000 wide 14.9 / 7.3, 2048 wide 17.4 / 11.6; single elements, 2050 wide 17.6 / 14.7; 96 wide, 8 rows 2.6
    // with 16 bytes a lane, 2.4 with one element, 4096 rows 5.0 / 6.5)
    #define POLY(VV, NW) hipLaunchKernelGGL((polynorm_kernel<T, VV, NW>), dim3(n), dim3(64 * NW), 0, (hipStream_t) stream, (T*) out, (const T*) z, z_ld, coef, eps, ff)
    MIX_DISPATCH_T(dtype, constexpr int V = wide_n<T>(); if (!row_wide<T>(ff, z_ld) || !aligned16(out, z, nullptr, nullptr) || (ff <= 256 && n <= 1024)) POLY(1, 4); else if (ff <= 128 * V) POLY(V, 2);
                          else if (ff <= 256 * V) POLY(V, 4); else POLY(V, 8));
    #undef POLY
    return mix_check_launch("mix_polynorm");
}

extern "C" int exl3_mix_topk_softmax(int32_t* idx, float* wts, const float* logits, int n, int experts, int top, void* stream)
{
    MIX_CHECK(idx && wts && logits && n >= 0 && experts > 0 && top > 0 && top <= experts, "mix_topk_softmax: bad arguments (top %d of %d)", top, experts);
    if (n == 0) return EXL3_MIX_OK;
    hipLaunchKernelGGL(topk_softmax_kernel, dim3((n + 63) / 64), dim3(64), 0, (hipStream_t) stream, idx, wts, logits, n, experts, top);
    return mix_check_launch("mix_topk_softmax");
}
