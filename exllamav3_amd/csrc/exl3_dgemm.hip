// Launchers of exl3_dgemm (exl3_dgemm.kspec.hip, exl3_dgemm_wide.kspec.hip: quantized products for medium row counts on rotated activations), the rotation in front
// of them and the reduction behind a split one.
#include "exl3_api_internal.h"
#include "exl3_dgemm.h"
#include "exl3_dgemm_api.h"
#include <atomic>
#include <math.h>
#include <stdlib.h>
#include <string.h>

// ------------------------------------------------------------------------------------------------
// Rotation: xh_i[r] = fp16(H128 (x[map r] suh_i)) for up to 4 scale vectors from one read of the row.  16 lanes per 128-value block, 8 values (16 bytes) per lane:
// three butterfly stages in registers, four over a DPP row.  HBM-bound in theory; at a few hundred rows a launch of 3 - 5 us.
// ACT: the input is silu(g) u of two rows, rounded to fp16 like the activation kernel's output (the reference's intermediate).
// ------------------------------------------------------------------------------------------------
struct DgRotateArgs
{
    const half_t* x; const half_t* u; int64_t ldx; const int64_t* map;
    const half_t* suh[DG_MAX_MATS]; half_t* xh[DG_MAX_MATS];
    const int32_t* group_rows; const uint64_t* group_suh;                 // groups > 0: scale vector i of row r is table entry i * groups + (group of r)
    int count, groups, rows, k, ref;                                      // ref: x suh rounded to fp16 first (the small-m kernels' rounding)
};

template <bool ACT>
__global__ __launch_bounds__(256)
void exl3_dgemm_rotate_kernel(const DgRotateArgs a)
{
    const int l = threadIdx.x & 15, row = blockIdx.x, nbk = a.k >> 7, want = blockIdx.y * 16 + (threadIdx.x >> 4);
    const bool ok = want < nbk;                                           // (whole DPP rows of 16 lanes are in or out)
    const int blk = ok ? want : nbk - 1;
    const int64_t src = a.map ? a.map[row] : row;
    const int col = blk * 128 + 8 * l;
    half8_t xv = *((const half8_t*) (a.x + src * a.ldx + col));
    if constexpr (ACT)
    {
        const half8_t uv = *((const half8_t*) (a.u + src * a.ldx + col));
        #pragma unroll
        for (int i = 0; i < 8; ++i) { const float g = (float) xv[i]; xv[i] = f2h(g / (1.0f + expf(-g)) * (float) uv[i]); }
    }
    int e = 0;
    for (int base = 0; base < a.groups; base += 64)                       // the row's group: boundaries at or below it, one per lane
        e += __popcll(__ballot(base + (int) (threadIdx.x & 63) + 1 < a.groups && row >= a.group_rows[min(base + (int) (threadIdx.x & 63) + 1, a.groups)]));
    for (int i = 0; i < a.count; ++i)
    {
        const half_t* suh = a.groups > 0 ? dg_global<half_t>(a.group_suh[i * a.groups + e]) : a.suh[i];
        const half8_t sv = *((const half8_t*) (suh + col));
        float v[8];
        #pragma unroll
        for (int j = 0; j < 8; ++j) { v[j] = (float) xv[j] * (float) sv[j]; if (a.ref) v[j] = (float) f2h(v[j]); }
        #pragma unroll
        for (int b = 1; b < 8; b <<= 1)
            #pragma unroll
            for (int j = 0; j < 8; ++j) if (!(j & b)) { const float p = v[j], q = v[j | b]; v[j] = p + q; v[j | b] = p - q; }
        #pragma unroll
        for (int b = 1; b < 16; b <<= 1)
        {
            const float sg = (l & b) ? -1.0f : 1.0f;
            #pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = __builtin_fmaf(v[j], sg, xor_lane(v[j], b));
        }
        half8_t o;
        #pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = f2h(v[j] * HAD_R_SCALE_128);
        if (ok) *((half8_t*) (a.xh[i] + (size_t) row * a.k + col)) = o;
    }
}

static int dg_rotate(const DgRotateArgs& a, bool act, hipStream_t st)
{
    if (a.rows == 0) return EXL3_OK;
    const dim3 grid((unsigned) a.rows, (unsigned) (((a.k >> 7) + 15) / 16));
    if (act) exl3_dgemm_rotate_kernel<true><<<grid, dim3(256), 0, st>>>(a);
    else exl3_dgemm_rotate_kernel<false><<<grid, dim3(256), 0, st>>>(a);
    return exl3_check_launch("exl3_dgemm_rotate");
}

// ------------------------------------------------------------------------------------------------
// Sum of the slices' partial rows, output Hadamard, svh, bias.  One half-wave per (row, column block); the slices' loads are in flight eight at a time
// ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256)
void exl3_dgemm_reduce_kernel(const DgemmArgs a)
{
    const int l = threadIdx.x & 31, hw = threadIdx.x >> 5;
    const int64_t item = (int64_t) blockIdx.x * 8 + hw, items = (int64_t) a.m * a.nblk;
    const int64_t it = item < items ? item : items - 1;
    const int row = (int) (it / a.nblk), cb = (int) (it - (int64_t) row * a.nblk);
    int mi = 0;
    #pragma unroll
    for (int i = 1; i < DG_MAX_MATS; ++i) if (i < a.num_mats && cb >= a.mat[i].cb_first) mi = i;
    const size_t ntot = (size_t) a.nblk * 128, step = (size_t) a.m * ntot / 4;
    const float4_t* p = (const float4_t*) (a.slab + (size_t) row * ntot + (size_t) cb * 128) + l;
    float4_t v = { 0.f, 0.f, 0.f, 0.f };
    #pragma unroll 8
    for (int s = 0; s < a.S; ++s) v += p[(size_t) s * step];
    float h0 = v.x, h1 = v.y, h2 = v.z, h3 = v.w;
    had128_f32x4(h0, h1, h2, h3, l);
    if (item >= items) return;
    const int cbl = cb - a.mat[mi].cb_first;
    const half4_t sc = ((const half4_t*) (a.mat[mi].svh + cbl * 128))[l];
    const half4_t bv = a.mat[mi].bias ? ((const half4_t*) (a.mat[mi].bias + cbl * 128))[l] : half4_t{ 0, 0, 0, 0 };
    const float4_t f = dg_scale(a, sc);
    dg_put(a, a.mat[mi].C, (int64_t) row * a.mat[mi].ldc + cbl * 128 + 4 * l, float4_t{ h0, h1, h2, h3 }, f, bv);
}

#define DG_DECL(KK) void exl3_dgemm_launch_k##KK(int cb, int mt, dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a); \
                    void exl3_dgemm_wide_launch_k##KK(int cb, int mt, dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a);
DG_DECL(1) DG_DECL(2) DG_DECL(3) DG_DECL(4) DG_DECL(5) DG_DECL(6) DG_DECL(7) DG_DECL(8)
#undef DG_DECL

// 16-row tiles per workgroup: 4 .. 8 in the narrow kernel (two workgroups per CU), 10 .. 16 (even) in the wide one.  For m rows in mtiles equal parts:
static int dg_narrow_tiles(int m, int mtiles) { const int t = ((m + mtiles - 1) / mtiles + 15) / 16; return t <= 4 ? 4 : t; }
static int dg_wide_tiles(int m, int mtiles) { const int t = ((m + mtiles - 1) / mtiles + 15) / 16; return t <= 10 ? 10 : (t + 1) / 2 * 2; }

// groups of rows (their boundaries are on the device): the fewest row tiles
static int dg_row_tiles(int m)
{
    return m <= 128 ? dg_narrow_tiles(m, 1) : dg_wide_tiles(m, (m + 255) / 256);
}

struct DgPlan { int mt, mtiles, S; double us; };

// What a block of 128 k costs beside 1 .. 4 bits of the hashed-byte codebook (cb 2): wider words are two loads per lane from 5 bits and unaligned ones at 7, the codebooks that add two halves
// decode with more instructions.  wide: in the wide kernel, one / two: in the narrow one with one / two workgroups on a compute unit, deep: 7 and 8 bits in the narrow kernel's 112- and 128-row
// forms, whose second ring of words does not fit the registers.
struct DgKind { double wide, one, two, small, deep; };
static DgKind dg_kind(int K, int cb)
{
    const int w5 = K > 4, w7 = K > 6, c1 = cb == 1, c0 = cb == 0;
    return { 0.086 * w5 + 0.063 * w7 + 0.049 * c1 + 0.134 * c0, 0.103 * w5 + 0.054 * w7 + 0.172 * c1 + 0.223 * c0, 0.107 * w5 + 0.053 * w7 + 0.082 * c1 + 0.221 * c0,
             0.076 * w5 + 0.038 * w7 + 0.068 * c1 + 0.134 * c0, (double) w7 };
}

// Microseconds of one (m, k, n) product cut into `mtiles` row tiles and s k-slices of b blocks on `cus` compute units, without the rotation in front of it.
// Fitted to 38 800 launches: fourteen shapes from 2048 x 512 to 4096 x 14336, 40 .. 1000 rows, 2, 4, 6, 8 bits, three codebooks, every row tiling, up to five splits each.  The choices are 0.3 %
// slower than the best of the launches on average up to 128 rows (7 % at most) and 0.9 % above (13 %); without the terms of dg_kind they were 1.0 % (30 %) and 5.2 % (48 %) slower:
// 8192 x 8192, 8 bits, 420 rows 134 us, 84 now.
// Up to 128 rows (one row tile): a workgroup pays its prologue and epilogue once and `step` per 128 k.  Above: a wide workgroup has its CU alone, a last round that fills the chip in part runs
// faster than a full one; two narrow workgroups share a CU at about the cost of one after the other.  A split writes and reads its partial sums and launches their reduction:
// above 128 rows priced as in a stream, where that kernel follows without a gap (the launches were timed in graphs, whose next node costs 3 us more; and the sums of a wide kernel's eight slices
// take 9 us to add where four slices take 6).  Over 2 463 launches with cold weights, less that gap, the choices are 1.1 % slower than the best on average as before, 11 % at most (19); chunks of
// 180 .. 256 rows through four layers of 4096 / 14336: 4 % faster.
static double dg_cost(const DgKind& kind, int m, int k, int n, int mt, int mtiles, int s, int b, int cus)
{
    const double wgs = (double) mtiles * (n >> 7) * s;
    const double sums = s > 1 ? 1e-6 * s * (double) m * n : 0.0, deep = mt > 6 ? kind.deep : 0.0;
    if (m <= 128)
    {
        const double per_cu = ceil(wgs / cus), alone = 0.471 + 0.079 * mt + kind.small + 0.473 * deep, shared = 0.299 + 0.038 * mt + 0.83 * kind.small + 0.082 * deep;
        return per_cu * (per_cu == 1.0 ? b * alone + 6.7 : b * shared + 6.1) + (s > 1 ? 1.6 + 1.45 * sums + 0.08 * s : 0.0);
    }
    if (mt > 8)
    {
        const double rounds = ceil(wgs / cus), last = wgs / cus - (rounds - 1.0);
        return (rounds - 1.0 + 0.86 + 0.14 * last) * (b * (0.156 + kind.wide + 0.081 * mt) + 0.69 * mt) + (s > 1 ? 0.5 * sums + 0.10 * s : 0.0);
    }
    const double one = b * (0.215 + kind.one + 0.112 * mt + 0.487 * deep) + 0.03 * mt, two = b * (0.828 + kind.two + 0.122 * mt) + 0.73 * mt;
    const double rounds = ceil(wgs / (2.0 * cus)), left = wgs - (rounds - 1.0) * 2.0 * cus;
    return (rounds - 1.0) * two + (left > cus ? two * (0.50 + 0.50 * left / (2.0 * cus)) : one) + (s > 1 ? 1.0 + 0.36 * sums + 0.35 * s : 0.0);
}

// The cheapest kernel, row tiling and split whose partial sums fit max_floats
static DgPlan dg_plan(int m, int k, int n, int K, int cb, int cus, int64_t max_floats)
{
    const int nb = k >> 7;
    const DgKind kind = dg_kind(K, cb);
    DgPlan best = { 0, 0, 1, 0.0 };
    double cost = 1e30;
    auto tiling = [&] (int mt, int mtiles, bool alone)
    {
        for (int s = 1; s <= nb && s <= 16; ++s)
        {
            const int b = (nb + s - 1) / s;
            if ((nb + b - 1) / b != s) continue;
            if (s > 1 && (int64_t) s * m * n > max_floats) break;
            if (alone && (int64_t) mtiles * (n >> 7) * s > cus) break;
            const double c = dg_cost(kind, m, k, n, mt, mtiles, s, b, cus);
            if (c < cost) { cost = c; best = { mt, mtiles, s, c }; }
        }
    };
    if (m <= 128) tiling(dg_narrow_tiles(m, 1), 1, false);
    else
    {
        const int narrow = (m + 127) / 128;
        for (int t = narrow; t <= narrow + 2; ++t) tiling(dg_narrow_tiles(m, t), t, t > narrow);      // (shorter tiles than need be only where each has a CU of its own)
        for (int t = (m + 255) / 256; t <= narrow; ++t) tiling(dg_wide_tiles(m, t), t, false);
    }
    return best;
}

static int dg_device_cus(int* cus)
{
    static std::atomic<int> cached[64];                   // (a property of the device; several threads store the same value)
    int dev = 0;
    EXL3_CHECK_HIP(hipGetDevice(&dev), "exl3_dgemm");
    const bool known = dev >= 0 && dev < 64;
    if (known && (*cus = cached[dev].load(std::memory_order_relaxed)) != 0) return EXL3_OK;
    EXL3_CHECK_HIP(hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev), "exl3_dgemm");
    if (known) cached[dev].store(*cus, std::memory_order_relaxed);
    return EXL3_OK;
}

static int dg_launch(const DgemmArgs& a, int mt, int K, int cb, hipStream_t st)
{
    const dim3 grid((unsigned) ((a.nblk * a.S + 7) / 8 * 8 * a.mtiles));
    const size_t lds = (size_t) 16 * mt * DG_PITCH * 4;              // >= the two activation buffers of 16 mt x 256 bytes
    switch (K)
    {
        #define DG(KK) case KK: if (mt <= 8) exl3_dgemm_launch_k##KK(cb, mt, grid, lds, st, a); else exl3_dgemm_wide_launch_k##KK(cb, mt, grid, lds, st, a); break;
        DG(1) DG(2) DG(3) DG(4) DG(5) DG(6) DG(7) DG(8)
        #undef DG
    }
    int rc = exl3_check_launch("exl3_dgemm");
    if (rc != EXL3_OK || a.S == 1) return rc;
    exl3_dgemm_reduce_kernel<<<dim3((unsigned) (((int64_t) a.m * a.nblk + 7) / 8)), dim3(256), 0, st>>>(a);
    return exl3_check_launch("exl3_dgemm (reduce)");
}

// (the most rows any row tiling of m rows touches)
int exl3_dgemm_xh_rows(int m)
{
    if (m <= 128) return 16 * dg_narrow_tiles(m, 1);
    const int narrow = (m + 127) / 128;
    int rows = 0;
    for (int t = narrow; t <= narrow + 2; ++t) { const int r = 16 * dg_narrow_tiles(m, t) * t; rows = r > rows ? r : rows; }
    for (int t = (m + 255) / 256; t <= narrow; ++t) { const int r = 16 * dg_wide_tiles(m, t) * t; rows = r > rows ? r : rows; }
    return rows;
}

extern "C" int exl3_dgemm_plan_kind(int m, int k, int n, int K, int cb, int* xh_rows, int64_t* slab_floats)
{
    EXL3_CHECK_ARG(xh_rows && slab_floats && m >= 1 && k > 0 && n > 0 && k % 128 == 0 && n % 128 == 0, "exl3_dgemm_plan: m >= 1, k and n divisible by 128");
    EXL3_CHECK_ARG(K >= 1 && K <= 8 && cb >= 0 && cb <= 2, "exl3_dgemm_plan: K must be in [1, 8], codebook in [0, 2]");
    int cus = 0;
    const int rc = dg_device_cus(&cus);
    if (rc != EXL3_OK) return rc;
    const int S = dg_plan(m, k, n, K, cb, cus, INT64_MAX).S;
    *xh_rows = exl3_dgemm_xh_rows(m);
    *slab_floats = S > 1 ? (int64_t) S * m * n : 0;
    return EXL3_OK;
}

extern "C" int exl3_dgemm_plan(int m, int k, int n, int* xh_rows, int64_t* slab_floats) { return exl3_dgemm_plan_kind(m, k, n, 4, 2, xh_rows, slab_floats); }

// Whether the product is faster here than through a rebuilt fp16 matrix and a plain GEMM (128 < m < 1024; both called one after the other, launches included).  Here: the rotation and the launches,
// then the plan.  There: two launches; W^T written once, and for every 256 rows read again next to their products (its tiles), with a term for long contractions, whose few outputs leave compute
// units idle.  Fitted to 3 510 calls (thirteen shapes, 150 .. 1000 rows, 1 .. 8 bits, three codebooks; 4.1 % and 3.6 % rms); the margin leaves 27 of them more than 2 % slower than the other route, 8 %
// at most, and the mean 0.2 % above the better route's.  Row limits without a term for bits and codebook left 181 of them slower, 21 % at most (4096 x 6144, 8 bits, 560 rows: 69 us / 57).
extern "C" int exl3_dgemm_pays(int m, int k, int n, int K, int cb)
{
    EXL3_CHECK_ARG(m >= 1 && k > 0 && n > 0 && k % 128 == 0 && n % 128 == 0 && K >= 1 && K <= 8 && cb >= 0 && cb <= 2, "exl3_dgemm_pays: m >= 1, k and n divisible by 128, K in [1, 8], codebook in [0, 2]");
    int cus = 0;
    const int rc = dg_device_cus(&cus);
    if (rc != EXL3_OK) return rc;
    const double kn = 1e-6 * (double) k * n, tiles = (m + 255) / 256;
    const DgPlan plan = dg_plan(m, k, n, K, cb, cus, INT64_MAX);
    const double here = fmax(16.5, 9.5 + 1.243 * (plan.us + (plan.S > 1 ? 2.3 : 0.0)));      // (2.3: the gap in front of the reduction, which the tiling is not charged for)
    // (30.5: the host's time for that route's launches, which is what small calls one after the other take; behind a queue of other work they take their device time, 1024 x 1024 at 1000 rows 21 us here
    // and 16 there, 2048 x 2048 29 and 26.  Many rows are such a queue: beyond 768 of them the device's time decides, but for long contractions)
    const double there = fmax(m > 768 && k < 2 * n ? 0.0 : 30.5, 15.3 + 0.669 * kn + 0.126 * kn * tiles + 0.616e-3 * kn * m + 0.88e-3 * k + 1.365e-6 * (double) k * m);
    if (n >= 10240 && kn >= 55.0)
    {
        // Large matrices of many columns: the plain GEMM's tiles of 256 x 256 run in whole rounds over the chip, which the line above knows nothing of (4096 x 22016, 4 bits, 400 rows: 102 us here, 131
        // there, 126 by that line; 5120 x 27648, 600 rows 224 / 292 / 225).  Fitted to 420 calls of seven shapes, 6.4 % rms; the factor from 840 calls and 330 of gate and up together: the choice is
        // 0.3 % slower than the better route on average, 11 % at most (4096 x 28672, 8 bits, codebook 0, 512 rows), where the line above was 1.7 and 2.2 % and 35 % slower.
        const double rounds = ceil(tiles * ceil(n / 256.0) / cus);
        return here < 1.06 * (-11.5 + 0.805 * kn + 0.584e-3 * kn * m + 2.68e-3 * k * rounds + 0.191 * kn * tiles) ? 1 : 0;
    }
    return here < 0.97 * there ? 1 : 0;
}

extern "C" int exl3_dgemm(const void* x, int64_t ldx, const void* const* suhs, void* xh, int xh_rows, const void* const* Bs, const void* const* svhs,
                          const void* const* biases, void* const* Cs, const int64_t* ldcs, const int* ns, int count, int out, void* slab, int64_t slab_floats,
                          int m, int k, int K, int cb, int force_split, void* stream)
{
    EXL3_CHECK_ARG(x && suhs && xh && Bs && svhs && Cs && ldcs && ns, "exl3_dgemm: null pointer");
    EXL3_CHECK_ARG(count >= 1 && count <= DG_MAX_MATS, "exl3_dgemm: between 1 and 4 matrices");
    EXL3_CHECK_ARG(m >= 1 && k > 0 && k % 128 == 0 && ldx >= k && ldx % 8 == 0, "exl3_dgemm: m >= 1, k divisible by 128, rows 16-byte aligned");
    EXL3_CHECK_ARG(K >= 1 && K <= 8 && cb >= 0 && cb <= 2, "exl3_dgemm: K must be in [1, 8], codebook in [0, 2]");
    EXL3_CHECK_ARG(out >= DG_OUT_F16 && out <= DG_OUT_F16_REF + 1, "exl3_dgemm: bad output mode");
    EXL3_CHECK_ARG(((uintptr_t) x | (uintptr_t) xh | (uintptr_t) slab) % 16 == 0, "exl3_dgemm: 16-byte aligned buffers");
    int cus = 0;
    int rc = dg_device_cus(&cus);
    if (rc != EXL3_OK) return rc;
    DgemmArgs a; DgRotateArgs r;
    memset((void*) &a, 0, sizeof(a)); memset((void*) &r, 0, sizeof(r));
    const int rows = exl3_dgemm_xh_rows(m), nb = k >> 7;
    EXL3_CHECK_ARG(xh_rows >= rows && (int64_t) rows * k * 2 <= 0x7fffffffll, "exl3_dgemm: xh needs %d rows per scale vector, below 2 GiB", rows);
    r.x = (const half_t*) x; r.ldx = ldx; r.rows = m; r.k = k; r.ref = out >= DG_OUT_F16_REF;
    if (out > DG_OUT_F16_REF) out = DG_OUT_F32;           // (4: fp32 output behind the rounded input)
    for (int i = 0; i < count; ++i)
    {
        EXL3_CHECK_ARG(suhs[i] && Bs[i] && svhs[i] && Cs[i] && ns[i] > 0 && ns[i] % 128 == 0, "exl3_dgemm: null matrix / n not divisible by 128");
        EXL3_CHECK_ARG(ldcs[i] >= ns[i] && ldcs[i] % 4 == 0 && (uintptr_t) Cs[i] % (out == DG_OUT_F32 ? 16 : 8) == 0, "exl3_dgemm: bad output row stride / alignment");
        int same = -1;                                    // matrices that share their input scales share the rotated rows
        for (int j = 0; j < r.count; ++j) if (r.suh[j] == (const half_t*) suhs[i]) { same = j; break; }
        if (same < 0) { same = r.count++; r.suh[same] = (const half_t*) suhs[i]; r.xh[same] = (half_t*) xh + (size_t) same * xh_rows * k; }
        a.mat[i].xh = r.xh[same];
        a.mat[i].B = (const uint32_t*) Bs[i]; a.mat[i].svh = (const half_t*) svhs[i]; a.mat[i].bias = biases ? (const half_t*) biases[i] : nullptr;
        a.mat[i].C = Cs[i]; a.mat[i].ldc = ldcs[i]; a.mat[i].cb_first = a.nblk;
        a.nblk += ns[i] / 128;
    }
    a.num_mats = count; a.m = m; a.k = k; a.out = out; a.xh_bytes = rows * k * 2;
    DgPlan plan = dg_plan(m, k, 128 * a.nblk, K, cb, cus, slab ? slab_floats : 0);
    if (force_split < 0 && m > 128) { plan.mtiles = (m + 255) / 256; plan.mt = dg_wide_tiles(m, plan.mtiles); }
    const int mt = plan.mt;
    a.mtiles = plan.mtiles;
    int S = force_split != 0 ? abs(force_split) : plan.S;
    if (S > nb) S = nb;
    a.bps = (nb + S - 1) / S;
    a.S = (nb + a.bps - 1) / a.bps;
    EXL3_CHECK_ARG(a.S == 1 || (slab && slab_floats >= (int64_t) a.S * m * a.nblk * 128), "exl3_dgemm: slab too small for %d slices", a.S);
    a.slab = (float*) slab;
    rc = dg_rotate(r, false, (hipStream_t) stream);
    return rc != EXL3_OK ? rc : dg_launch(a, mt, K, cb, (hipStream_t) stream);
}

// ------------------------------------------------------------------------------------------------
// The same over groups of rows with matrices of their own (the experts of a sparse-MoE block): rows sorted by group, boundaries and pointers in device memory, so that
// nothing is read back on the host.  Row tiles: `tile_rows` is the caller's estimate of a group's rows (it only sizes the tiles).
// ------------------------------------------------------------------------------------------------
static int dg_group_tiles(int tile_rows)
{
    return dg_row_tiles(tile_rows < 1 ? 1 : tile_rows);
}

extern "C" int exl3_dgemm_grouped_xh_rows(int rows, int tile_rows) { return rows + 16 * dg_group_tiles(tile_rows); }

extern "C" int exl3_dgemm_grouped(const void* x, const void* act_u, int64_t ldx, const int64_t* row_map, const uint64_t* group_suh, void* xh, int xh_rows,
                                  const uint64_t* group_B, const uint64_t* group_svh, const int32_t* group_rows, int groups, void* const* Cs, int64_t ldc, int n, int count,
                                  int out, int rows, int tile_rows, int k, int K, int cb, void* stream)
{
    EXL3_CHECK_ARG(x && group_suh && xh && group_B && group_svh && group_rows && Cs, "exl3_dgemm_grouped: null pointer");
    EXL3_CHECK_ARG(count >= 1 && count <= 2 && groups >= 1 && groups <= 4096, "exl3_dgemm_grouped: one or two matrices per group");
    EXL3_CHECK_ARG(rows >= 0 && k > 0 && k % 128 == 0 && n > 0 && n % 128 == 0 && ldx >= k && ldx % 8 == 0 && ldc >= n && ldc % 4 == 0, "exl3_dgemm_grouped: k and n divisible by 128, aligned rows");
    EXL3_CHECK_ARG(K >= 1 && K <= 8 && cb >= 0 && cb <= 2 && (out == DG_OUT_F16 || out == DG_OUT_F32), "exl3_dgemm_grouped: K in [1, 8], codebook in [0, 2], fp16 or fp32 output");
    EXL3_CHECK_ARG(((uintptr_t) x | (uintptr_t) act_u | (uintptr_t) xh) % 16 == 0, "exl3_dgemm_grouped: 16-byte aligned buffers");
    const int mt = dg_group_tiles(tile_rows), need = rows + 16 * mt;
    EXL3_CHECK_ARG(xh_rows >= need && (int64_t) xh_rows * k * 2 <= 0x7fffffffll, "exl3_dgemm_grouped: xh needs %d rows per matrix, below 2 GiB", need);
    if (rows == 0) return EXL3_OK;
    DgemmArgs a; DgRotateArgs r;
    memset((void*) &a, 0, sizeof(a)); memset((void*) &r, 0, sizeof(r));
    r.x = (const half_t*) x; r.u = (const half_t*) act_u; r.ldx = ldx; r.map = row_map; r.group_rows = group_rows; r.group_suh = group_suh; r.groups = groups;
    r.count = count; r.rows = rows; r.k = k;
    for (int i = 0; i < count; ++i)
    {
        EXL3_CHECK_ARG(Cs[i] && (uintptr_t) Cs[i] % 16 == 0, "exl3_dgemm_grouped: 16-byte aligned outputs");
        r.xh[i] = (half_t*) xh + (size_t) i * xh_rows * k;
        a.mat[i].xh = r.xh[i]; a.mat[i].C = Cs[i]; a.mat[i].ldc = ldc; a.mat[i].cb_first = i * (n >> 7);
    }
    a.group_rows = group_rows; a.group_B = group_B; a.group_svh = group_svh; a.groups = groups; a.num_mats = count;
    a.m = rows; a.k = k; a.S = 1; a.bps = k >> 7; a.nblk = count * (n >> 7); a.out = out; a.xh_bytes = xh_rows * k * 2;
    const int most = (rows + 16 * mt - 1) / (16 * mt) + groups;           // every group ends in at most one partial tile
    a.mtiles = most < rows ? most : rows;
    const int rc = dg_rotate(r, act_u != nullptr, (hipStream_t) stream);
    return rc != EXL3_OK ? rc : dg_launch(a, mt, K, cb, (hipStream_t) stream);
}
