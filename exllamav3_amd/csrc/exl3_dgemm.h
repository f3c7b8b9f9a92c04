// Arguments and the output stage of exl3_dgemm (medium row counts), shared by the kernel units (one per bits-per-weight) and the launcher.
#pragma once
#include "exl3_common.cuh"
#include <atomic>
#include <type_traits>

#define DG_PITCH 136            // floats per row of the output tile in LDS: row groups 0 | 1 (and 2 | 3) of an accumulator touch different banks

template <int I, int N, typename F>
__device__ __forceinline__ void dg_static_for(F&& f)
{
    if constexpr (I < N) { f(std::integral_constant<int, I>{}); dg_static_for<I + 1, N>(f); }
}

#define DG_MAX_MATS 4
#define DG_OUT_F16 0
#define DG_OUT_F32 1
#define DG_OUT_ADD 2            // C (fp16) += result, one rounding
#define DG_OUT_F16_REF 3        // fp16 with the roundings of the small-m kernels (x suh, the rotated output and its product with svh each to fp16): the row counts that
                                // exl3_gemm takes from them keep their values -- a 4-bit cache turns a last bit of k or v into a whole level

struct DgemmMat
{
    const half_t* xh;           // [rows of whole tiles][k] activations rotated with this matrix's suh
    const uint32_t* B; const half_t* svh; const half_t* bias;
    void* C; int64_t ldc;       // row stride of C in elements
    int cb_first;               // first 128-column block of this matrix in the launch
};

// Up to 4 matrices of one k, K and codebook side by side (their column blocks are numbered through), or -- groups > 0 -- the same for every group (expert) e of rows
// [group_rows[e], group_rows[e + 1]) of the activations, matrix i of group e at index i * groups + e of the pointer tables (mat[i].B / svh / bias unused).
struct DgemmArgs
{
    DgemmMat mat[DG_MAX_MATS];
    const int32_t* group_rows; const uint64_t* group_B; const uint64_t* group_svh;
    float* slab;                // [S][m][128 nblk] partial sums when S > 1
    int num_mats, groups, m, k /* columns of one matrix: the tile stride of its packed words; 0 = from the next matrix's cb_first */, S, bps, mtiles, nblk, out, xh_bytes;
};

// the workgroup's tile: row tile x column block x k-slice
struct DgTile
{
    const half_t* xh; const uint32_t* B; const half_t* svh; const half_t* bias;
    void* C; int64_t ldc;
    int row0, row_end, cb /* in its matrix */, cb_all /* in the launch */, tiles_n, s, b0, b1;
};

// a table entry as a pointer into global memory (as a plain integer-to-pointer conversion it would be accessed with flat instructions, whose waits drain the LDS counter too)
template <typename T>
__device__ __forceinline__ const T* dg_global(uint64_t p) { return (const T*) (const __attribute__((address_space(1))) T*) p; }

// workgroup i runs on XCD i % 8; the row tiles of one (column block, slice) follow each other on one XCD and read its packed words from that XCD's L2.
// false: a workgroup of the rounded-up grid, or a row tile behind its group's last one
template <int BM>
__device__ __forceinline__ bool dg_locate(const DgemmArgs& a, DgTile& t)
{
    // the launch's scalars in one batch, the matrix's in a second one (left alone, the compiler loads each in front of its use: six round trips)
    const int mtiles = a.mtiles, S = a.S, nblk = a.nblk, bps = a.bps, num_mats = a.num_mats, nbk = a.k >> 7, groups = a.groups;
    const int f1 = a.mat[1].cb_first, f2 = a.mat[2].cb_first, f3 = a.mat[3].cb_first;
    asm volatile("" :: "s"(mtiles), "s"(S), "s"(nblk), "s"(bps), "s"(num_mats), "s"(nbk), "s"(groups), "s"(f1), "s"(f2), "s"(f3), "s"(a.m), "s"(a.xh_bytes));
    const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3, mq = seq / mtiles;
    const int unit = mq * 8 + xcd;
    int mt = seq - mq * mtiles;
    if (unit >= nblk * S) return false;
    t.s = unit / nblk; t.cb_all = unit - t.s * nblk;
    int mi = 0, lo = 0, hi = num_mats > 1 ? f1 : nblk;
    if (num_mats > 1 && t.cb_all >= f1) { mi = 1; lo = f1; hi = num_mats > 2 ? f2 : nblk; }
    if (num_mats > 2 && t.cb_all >= f2) { mi = 2; lo = f2; hi = num_mats > 3 ? f3 : nblk; }
    if (num_mats > 3 && t.cb_all >= f3) { mi = 3; lo = f3; hi = nblk; }
    t.tiles_n = 8 * (hi - lo);
    t.cb = t.cb_all - lo;
    t.xh = a.mat[mi].xh; t.C = a.mat[mi].C; t.ldc = a.mat[mi].ldc; t.B = a.mat[mi].B; t.svh = a.mat[mi].svh; t.bias = a.mat[mi].bias;
    asm volatile("" :: "s"(t.xh), "s"(t.C), "s"(t.ldc), "s"(t.B), "s"(t.svh), "s"(t.bias));
    t.row0 = mt * BM; t.row_end = a.m;
    if (groups > 0)
    {
        // the group whose row tiles hold tile mt: one group per lane, 64 at a time (one after the other, each boundary is a round trip to memory)
        const int lane = threadIdx.x & 63;
        int e = -1;
        for (int base = 0; base < groups && e < 0; base += 64)
        {
            const int g = base + lane;
            const int first = a.group_rows[min(g, groups)], end = a.group_rows[min(g + 1, groups)];
            int sum = (end - first + BM - 1) / BM;
            #pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const int p = __shfl_up(sum, o, 64); if (lane >= o) sum += p; }
            const unsigned long long hit = __ballot(sum > mt);
            if (hit)
            {
                const int w = __builtin_ctzll(hit);
                e = base + w;
                t.row_end = __builtin_amdgcn_readlane(end, w);
                t.row0 = __builtin_amdgcn_readlane(first, w) + (mt - (w ? __builtin_amdgcn_readlane(sum, w - 1) : 0)) * BM;
            }
            else mt -= __builtin_amdgcn_readlane(sum, 63);
        }
        if (e < 0) return false;
        const uint64_t pb = a.group_B[mi * groups + e], ps = a.group_svh[mi * groups + e];
        t.B = dg_global<uint32_t>(pb); t.svh = dg_global<half_t>(ps); t.bias = nullptr;
    }
    t.b0 = t.s * bps; t.b1 = min(t.b0 + bps, nbk);
    return true;
}

// four consecutive output columns of one row: f = (1 / sqrt(128)) svh, or svh itself for DG_OUT_F16_REF
__device__ __forceinline__ float4_t dg_scale(const DgemmArgs& a, const half4_t sc)
{
    const float r = a.out == DG_OUT_F16_REF ? 1.0f : HAD_R_SCALE_128;
    return float4_t{ r * (float) sc.x, r * (float) sc.y, r * (float) sc.z, r * (float) sc.w };
}

__device__ __forceinline__ void dg_put(const DgemmArgs& a, void* C, int64_t off, const float4_t h, const float4_t f, const half4_t bv)
{
    if (a.out == DG_OUT_F16_REF)
    {
        const half4_t sc = { (half_t) f.x, (half_t) f.y, (half_t) f.z, (half_t) f.w };
        half4_t o = half4_t{ f2h(h.x * HAD_R_SCALE_128), f2h(h.y * HAD_R_SCALE_128), f2h(h.z * HAD_R_SCALE_128), f2h(h.w * HAD_R_SCALE_128) } * sc;
        *((half4_t*) ((half_t*) C + off)) = o + bv;
        return;
    }
    float4_t o = { h.x * f.x + (float) bv.x, h.y * f.y + (float) bv.y, h.z * f.z + (float) bv.z, h.w * f.w + (float) bv.w };
    if (a.out == DG_OUT_F32) { *((float4_t*) ((float*) C + off)) = o; return; }
    half4_t* c = (half4_t*) ((half_t*) C + off);
    if (a.out == DG_OUT_ADD) { const half4_t r = *c; o.x += (float) r.x; o.y += (float) r.y; o.z += (float) r.z; o.w += (float) r.w; }
    *c = half4_t{ (half_t) o.x, (half_t) o.y, (half_t) o.z, (half_t) o.w };
}

// From accumulators to the output.  A wave holds the sums of its k half for all rows and its 64 columns: accumulator [i][u][set][r] of lane 16 kg + mj is row
// 16 i + 4 kg + r, column 64 ch + 32 u + 16 (mj >> 3) + 8 set + (mj & 7).  The two k halves swap halves of the rows through LDS, so that every wave ends with the
// finished sums of half the rows; with one slice the output Hadamard then runs over the column bits that lie in registers (set, u) and in the 16 lanes of a DPP row,
// and its last stage (the column half, another wave's) over the LDS tile on the way out.  Doing all of it row by row from LDS took twice as many vector
// instructions, and with one workgroup per CU nothing runs beside them.  part: [16 MT][DG_PITCH] floats over the operand buffers, which every wave has left behind.
template <int MT>
__device__ __forceinline__ void dg_epilogue(const DgemmArgs& a, const DgTile& t, float4_t (&acc)[MT][2][2], float* part, int wave, int lane)
{
    constexpr int H0 = MT / 2, BM = 16 * MT;
    const int ch = wave & 1, kh = wave >> 1, mj = lane & 15, kg = lane >> 4;
    float* base = part + 4 * kg * DG_PITCH + 64 * ch + 16 * (mj >> 3) + (mj & 7);
    auto at = [&] (int i, int u, int set, int r) -> float& { return base[(16 * i + r) * DG_PITCH + 32 * u + 8 * set]; };
    // (row tiles as compile-time indices, and the two halves' code kept apart by the empty statements -- merged, it would index the accumulators at run time: scratch)
    auto give = [&] (auto ic) __attribute__((always_inline))
    {
        constexpr int i = decltype(ic)::value;
        asm volatile("; %0" :: "n"(i));
        #pragma unroll
        for (int u = 0; u < 2; ++u)
            #pragma unroll
            for (int r = 0; r < 4; ++r) { at(i, u, 0, r) = acc[i][u][0][r]; at(i, u, 1, r) = acc[i][u][1][r]; }
        asm volatile("; %0" :: "n"(i));
        __builtin_amdgcn_sched_barrier(0);
    };
    float sg[4];
    #pragma unroll
    for (int b = 0; b < 4; ++b) sg[b] = (mj >> b) & 1 ? -1.0f : 1.0f;
    auto take = [&] (auto ic) __attribute__((always_inline))
    {
        constexpr int i = decltype(ic)::value;
        float v[2][2][4];
        asm volatile("; %0" :: "n"(i));
        #pragma unroll
        for (int u = 0; u < 2; ++u)
            #pragma unroll
            for (int r = 0; r < 4; ++r) { v[u][0][r] = acc[i][u][0][r] + at(i, u, 0, r); v[u][1][r] = acc[i][u][1][r] + at(i, u, 1, r); }
        if (a.S == 1)
        {
            #pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const float p0 = v[0][0][r] + v[0][1][r], m0_ = v[0][0][r] - v[0][1][r], p1 = v[1][0][r] + v[1][1][r], m1 = v[1][0][r] - v[1][1][r];
                v[0][0][r] = p0 + p1; v[1][0][r] = p0 - p1; v[0][1][r] = m0_ + m1; v[1][1][r] = m0_ - m1;
            }
            #pragma unroll
            for (int b = 0; b < 4; ++b)
                #pragma unroll
                for (int e = 0; e < 16; ++e) { float& x = v[e >> 3][(e >> 2) & 1][e & 3]; x = __builtin_fmaf(x, sg[b], xor_lane(x, 1 << b)); }
        }
        #pragma unroll
        for (int u = 0; u < 2; ++u)
            #pragma unroll
            for (int r = 0; r < 4; ++r) { at(i, u, 0, r) = v[u][0][r]; at(i, u, 1, r) = v[u][1][r]; }
        asm volatile("; %0" :: "n"(i));
        __builtin_amdgcn_sched_barrier(0);
    };
    if (kh) dg_static_for<0, H0>(give); else dg_static_for<H0, MT>(give);
    __syncthreads();
    if (kh) dg_static_for<H0, MT>(take); else dg_static_for<0, H0>(take);
    __syncthreads();

    const int l = lane & 31, hw = 2 * wave + (lane >> 5);
    if (a.S > 1)
    {
        const size_t ntot = (size_t) a.nblk * 128;
        float* slab = a.slab + (size_t) t.s * a.m * ntot + (size_t) t.cb_all * 128;
        #pragma unroll 4
        for (int i = 0; i < BM / 8; ++i)
        {
            const int row = 8 * i + hw;
            if (t.row0 + row < t.row_end) *((float4_t*) (slab + (size_t) (t.row0 + row) * ntot) + l) = *((const float4_t*) (part + row * DG_PITCH) + l);
        }
        return;
    }
    const half4_t sc = ((const half4_t*) (t.svh + t.cb * 128))[l];
    const half4_t bv = t.bias ? ((const half4_t*) (t.bias + t.cb * 128))[l] : half4_t{ 0, 0, 0, 0 };
    const float sgn = l < 16 ? 1.0f : -1.0f;
    const float4_t f = dg_scale(a, sc);
    #pragma unroll 4
    for (int i = 0; i < BM / 8; ++i)
    {
        const int row = 8 * i + hw;
        const float* p = part + row * DG_PITCH + 4 * (l & 15);
        const float4_t x = *((const float4_t*) p), y = *((const float4_t*) (p + 64));
        const float4_t h = { __builtin_fmaf(y.x, sgn, x.x), __builtin_fmaf(y.y, sgn, x.y), __builtin_fmaf(y.z, sgn, x.z), __builtin_fmaf(y.w, sgn, x.w) };
        if (t.row0 + row < t.row_end) dg_put(a, t.C, (int64_t) (t.row0 + row) * t.ldc + t.cb * 128 + 4 * l, h, f, bv);
    }
}

// Launch of one of the kernels.  More than 64 KB of LDS per workgroup (the narrow kernel's 128-row form, the wide one's all) is asked for once per kernel and device, in front of the first launch there.
template <void (*KERNEL)(const DgemmArgs)>
static void dg_start(dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a)
{
    static std::atomic<uint64_t> ready{ 0 };
    int dev = 0;
    if (lds > 65536 && hipGetDevice(&dev) == hipSuccess && !((ready.load(std::memory_order_relaxed) >> (dev & 63)) & 1))
    {
        (void) hipFuncSetAttribute((const void*) KERNEL, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds);
        ready.fetch_or(1ull << (dev & 63), std::memory_order_relaxed);
    }
    KERNEL<<<grid, dim3(256), lds, st>>>(a);
}
