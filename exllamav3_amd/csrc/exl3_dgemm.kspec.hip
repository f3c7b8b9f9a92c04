// Quantized matrix product for medium row counts: 16-bit activations in the rotated basis times packed weights that are decoded in registers.
//
//   C = ((A suh) H) @ dequant(B) H svh (+ bias)      reference: modules/quant/exl3.py:161-218 (what the large-batch route computes), quant/exl3_gemm_kernel.cuh:8-80
//
// The input is already rotated (exl3_had_r_128); the output Hadamard and svh are applied at the end.  Between the small-m kernels (one pass over the packed
// weights per 64 rows) and the prefill route (decode every weight, rotate it on both sides, write 2 bytes per weight, read them again in a plain GEMM) lie the row
// counts where the first decodes too often and the second spends most of its time on weights: here a weight is decoded once per up to 128 rows and never leaves
// the registers of the wave that decoded it.
//
// Work split.  A workgroup of 4 waves owns 16 MT rows x one 128-column block x one k-slice.  Wave = (64-column half) x (64-deep half of every 128-deep
// Hadamard block): per block it decodes 4 tile rows x 4 tiles = 64 weights per lane into eight B operands of v_mfma_f32_16x16x32_f16 (the decoding lane's
// registers are the operand: lane 16 g + 8 t2 + c holds columns c, c + 8 of tile t2 for the 16 k of tile row g) and multiplies them with 2 MT A operands from
// LDS, so one 16-byte LDS read feeds four matrix instructions.  With 32 columns per wave the LDS port would be the bound (128 B per cycle and CU), with 128 the
// accumulators would not fit beside the operands.  Two workgroups share a CU: while one wave of a SIMD decodes (vector unit), the other multiplies (matrix unit).
//
// Activations: [16 MT][128] per block, 256-byte rows, the 16-byte chunk c of row r at position c ^ (r & 15): 16 lanes that read the same chunk of 16 rows touch
// all banks once.  Two buffers, filled by loads that write LDS directly, a whole block ahead.
#include "exl3_common.cuh"
#include "exl3_api_internal.h"
#include "exl3_lane_decode.cuh"
#include "exl3_dgemm.h"

template <int K, int CB, int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
void exl3_dgemm_kernel(const DgemmArgs a)
{
    constexpr int NW = 8 * K, BM = 16 * MT;
    extern __shared__ __attribute__((aligned(16))) char smem[];       // two activation buffers of BM x 256 B; later BM x DG_PITCH floats

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ch = wave & 1, kh = wave >> 1;

    DgTile t;
    if (!dg_locate<BM>(a, t)) return;
    const int b0 = t.b0, b1 = t.b1;

    // ---- packed words: tile rows 4 kh + g of a block, tiles 4 ch + 2 u + t2 of the column block
    const int g = lane >> 4, t2 = (lane >> 3) & 1, c = lane & 7;
    const size_t bstride = (size_t) 8 * t.tiles_n * NW;
    const uint32_t* __restrict__ strip = t.B + ((size_t) (4 * kh + g) * t.tiles_n + t.cb * 8 + 4 * ch + t2) * NW + (size_t) c * K;
    auto wptr = [&] (int b, int u) -> const uint32_t* { return strip + (size_t) min(b, b1 - 1) * bstride + (size_t) (2 * u) * NW; };

    // ---- activations, straight into LDS (16 bytes per lane, lane-linear): instruction j of wave w fills rows 16 j + 4 w .. + 3, lane l the position l & 15 of
    // row l >> 4 of them, so the permutation of a row's chunks is carried by the source address
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*) t.xh, (short) 0, a.xh_bytes, 0x00027000);
    const int srow = 4 * wave + (lane >> 4);
    const int voff = (t.row0 + srow) * a.k * 2 + (((lane & 15) ^ srow) << 4);
    auto fetch = [&] (int b, int buf, int j0, int j1)
    {
        const int so = min(b, b1 - 1) * 256;
        #pragma unroll
        for (int j = j0; j < j1; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*) (smem + buf * (BM * 256) + (16 * j + 4 * wave) * 256), 16, voff,
                                                     so + j * 32 * a.k, 0, 0);
    };
    auto barrier = [] ()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    float4_t acc[MT][2][2];
    #pragma unroll
    for (int i = 0; i < MT; ++i)
        #pragma unroll
        for (int u = 0; u < 2; ++u) { acc[i][u][0] = float4_t{ 0.f, 0.f, 0.f, 0.f }; acc[i][u][1] = acc[i][u][0]; }

    // packed words two blocks ahead of their use (one where two rings would not fit)
    constexpr int NR = K <= 6 || MT <= 6 ? 2 : 1;
    LaneWords<K> ring[NR][2];
    constexpr int WL = 2 * ((K + 3) / 4);                 // fewest load instructions of a block's words: what may still be in flight behind a fetch that has landed
    fetch(b0, 0, 0, MT);
    #pragma unroll
    for (int r = 0; r < NR; ++r) { load_lane_words<K>(ring[r][0], wptr(b0 + r, 0)); load_lane_words<K>(ring[r][1], wptr(b0 + r, 1)); }
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(NR * WL) : "memory");
    barrier();

    // A operand of (row 16 i + mj, k half h of tile row kg): chunk 8 kh + 2 kg + h
    const int mj = lane & 15, kg = lane >> 4;
    const int lds_r = mj * 256 + (((8 * kh + 2 * kg) ^ mj) << 4);

    // (the last block of a slice with an odd number of them requests nothing: what lands in LDS behind its barrier would land in the output tile)
    auto block = [&] (int b, int buf, LaneWords<K> (&slot)[2], auto last) __attribute__((always_inline))
    {
        constexpr bool MORE = !decltype(last)::value;
        // the next block's activations are requested between the decode groups (every wave read that buffer for the last time in front of the barrier behind us):
        // back to back the requests of four waves queue at the CU's one address unit and hold their waves there
        half8_t bf[2][2][2];                              // [u][column c / c + 8][k half]
        #pragma unroll
        for (int u = 0; u < 2; ++u)
        {
            uint32_t Wx[K + 1];
            #pragma unroll
            for (int i = 0; i < K; ++i) Wx[i + 1] = slot[u].w[i];
            const uint32_t wl = slot[u].w[K - 1];
            const uint32_t r1 = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) wl, 0x121, 0xf, 0xf, true);
            const uint32_t r9 = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) wl, 0x129, 0xf, 0xf, true);
            Wx[0] = (lane & 7) ? r1 : r9;
            union { uint32_t w[4]; half8_t h; } o[2][2];
            dg_static_for<0, 4>([&] (auto qc)
            {
                constexpr int q = decltype(qc)::value;
                half4_t x[2], y[2];
                decode_quad<K, CB, 0, 8 * q>(Wx, x);
                decode_quad<K, CB, 0, 8 * q + 4>(Wx, y);
                union { half4_t h; uint32_t w[2]; } ux, uy; ux.h = x[0]; uy.h = y[0];
                o[0][0].w[q] = ux.w[0]; o[0][1].w[q] = ux.w[1]; o[1][0].w[q] = uy.w[0]; o[1][1].w[q] = uy.w[1];
                __builtin_amdgcn_sched_barrier(0);      // eight weights in flight: the registers are the accumulators' and the operands'
                if (MORE && 4 * u + q < MT) fetch(b + 1, buf ^ 1, 4 * u + q, 4 * u + q + 1);
            });
            bf[u][0][0] = o[0][0].h; bf[u][0][1] = o[0][1].h; bf[u][1][0] = o[1][0].h; bf[u][1][1] = o[1][1].h;
        }
        if constexpr (MORE)
        {
            asm volatile("" ::: "memory");                // the words are requested behind the activations: the wait below counts them
            #pragma unroll
            for (int u = 0; u < 2; ++u) load_lane_words<K>(slot[u], wptr(b + NR, u));
        }
        const char* ab = smem + buf * (BM * 256);
        #pragma unroll
        for (int i = 0; i < MT; ++i)
            #pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                const half8_t af = *((const half8_t*) (ab + (lds_r ^ (h << 4)) + i * 4096));
                #pragma unroll
                for (int u = 0; u < 2; ++u)
                {
                    acc[i][u][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf[u][0][h], acc[i][u][0], 0, 0, 0);
                    acc[i][u][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, bf[u][1][h], acc[i][u][1], 0, 0, 0);
                }
            }
        if constexpr (MORE) asm volatile("s_waitcnt vmcnt(%0)" :: "n"(WL) : "memory");
        barrier();
    };
    int b = b0;
    for (; b + 2 <= b1; b += 2) { block(b, 0, ring[0], std::false_type{}); block(b + 1, 1, ring[NR - 1], std::false_type{}); }
    if (b < b1) block(b, 0, ring[0], std::true_type{});

    dg_epilogue<MT>(a, t, acc, (float*) smem, wave, lane);
}

#ifndef G2_K
#error "compile with -DG2_K=<bits per weight>"
#endif

template <int CB>
static void dg_launch_cb(int mt, dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a)
{
    switch (mt)
    {
        #define DG(M) case M: dg_start<exl3_dgemm_kernel<G2_K, CB, M>>(grid, lds, st, a); break;
        DG(4) DG(5) DG(6) DG(7) DG(8)
        #undef DG
    }
}

#define DG_CAT_(a, b) a##b
#define DG_CAT(a, b) DG_CAT_(a, b)
void DG_CAT(exl3_dgemm_launch_k, G2_K)(int cb, int mt, dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a)
{
    if (cb == 0) dg_launch_cb<0>(mt, grid, lds, st, a);
    else if (cb == 1) dg_launch_cb<1>(mt, grid, lds, st, a);
    else dg_launch_cb<2>(mt, grid, lds, st, a);
}
