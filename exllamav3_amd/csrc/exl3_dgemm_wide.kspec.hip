// exl3_dgemm for more than 128 rows: the same product as exl3_dgemm.kspec.hip with up to 256 rows per workgroup, one wave per SIMD.
//
// What bounds the narrow kernel is the vector unit: a matrix instruction and a vector instruction that issue from the two waves of a SIMD overlap only in part
// (64 v_mfma_f32_16x16x32_f16 and the 240 vector instructions that decode their weights take 1.16 us together, 0.54 and 0.5 alone), so the way to go faster
// is fewer decoded weights per matrix instruction.  With 256 rows a weight is decoded once per 16 row tiles: 256 accumulators and everything else in the 512
// registers of the only wave of a SIMD.  hipcc moves accumulators between the two halves of the register file when it allocates that by itself (560 moves per 256 matrix
// instructions), so the matrix instructions are written as asm statements whose accumulator operand is tied ("+a"): they are accumulation registers for good.
// The 256-row form keeps three registers in scratch memory, stored in front of the output stage and read in it, outside the loop; a form without them ran 0.2 % slower (1100 tokens through 8 experts).
//
// With one wave nothing else covers a latency, so everything is ahead of its use in program order: while block b is multiplied, block b + 1 is decoded (a piece of two to
// three vector instructions behind every matrix instruction), the activations of b + 1 are on their way into LDS, the packed words of b + 2 are in flight and an A operand
// is read three groups of four matrix instructions before it is needed.
#include "exl3_common.cuh"
#include "exl3_api_internal.h"
#include "exl3_lane_decode.cuh"
#include "exl3_dgemm.h"

__device__ __forceinline__ void dg_mfma(float4_t& acc, const half8_t& a, const half8_t& b)
{
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

union DgOperand { uint32_t w[4]; half8_t h; };

template <int K, int CB, int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void exl3_dgemm_wide_kernel(const DgemmArgs a)
{
    constexpr int NW = 8 * K, BM = 16 * MT, G = 2 * MT, NM = 8 * MT;      // groups of four matrix instructions, matrix instructions per block
    extern __shared__ __attribute__((aligned(16))) char smem[];       // two activation buffers of BM x 256 B; later BM x DG_PITCH floats

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ch = wave & 1, kh = wave >> 1;

    DgTile t;
    if (!dg_locate<BM>(a, t)) return;
    const int b0 = t.b0, b1 = t.b1;

    const int g = lane >> 4, t2 = (lane >> 3) & 1, c = lane & 7;
    const size_t bstride = (size_t) 8 * t.tiles_n * NW;
    const uint32_t* __restrict__ strip = t.B + ((size_t) (4 * kh + g) * t.tiles_n + t.cb * 8 + 4 * ch + t2) * NW + (size_t) c * K;
    auto wptr = [&] (int b, int u) -> const uint32_t* { return strip + (size_t) min(b, b1 - 1) * bstride + (size_t) (2 * u) * NW; };

    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*) t.xh, (short) 0, a.xh_bytes, 0x00027000);
    const int srow = 4 * wave + (lane >> 4);
    const int voff = (t.row0 + srow) * a.k * 2 + (((lane & 15) ^ srow) << 4);
    auto fetch = [&] (int b, int buf, int j)
    {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*) (smem + buf * (BM * 256) + (16 * j + 4 * wave) * 256), 16, voff,
                                                 min(b, b1 - 1) * 256 + j * 32 * a.k, 0, 0);
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

    LaneWords<K> ring[2][2];
    constexpr int WL = 2 * ((K + 3) / 4);                 // fewest load instructions of a block's words: what may still be in flight behind a fetch that has landed

    // ---- decode of one block in 128 pieces: 32 pairs of weights (one dword of an operand each) of four pieces
    uint32_t Wx[2][K + 1], px0, px1;
    auto words = [&] (const LaneWords<K> (&slot)[2])
    {
        #pragma unroll
        for (int u = 0; u < 2; ++u)
        {
            #pragma unroll
            for (int i = 0; i < K; ++i) Wx[u][i + 1] = slot[u].w[i];
            const uint32_t wl = slot[u].w[K - 1];
            const uint32_t r1 = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) wl, 0x121, 0xf, 0xf, true);
            const uint32_t r9 = (uint32_t) __builtin_amdgcn_update_dpp(0, (int) wl, 0x129, 0xf, 0xf, true);
            Wx[u][0] = (lane & 7) ? r1 : r9;
        }
    };
    auto piece = [&] (auto pc, DgOperand (&o)[2][2][2]) __attribute__((always_inline))
    {
        constexpr int P = decltype(pc)::value, pair = P >> 2, st = P & 3, u = pair >> 4, t = 2 * (pair & 15), q = t >> 3, set = (t >> 2) & 1, h = (t >> 1) & 1;
        if constexpr (st == 0) px0 = cb_product<CB>(lane_state<K, t>(Wx[u]));
        else if constexpr (st == 1) px1 = cb_product<CB>(lane_state<K, t + 1>(Wx[u]));
        else if constexpr (CB != EXL3_CB_MUL1)
        {
            if constexpr (st == 2) { px0 = cb_mask3inst(px0); px1 = cb_mask3inst(px1); }
            else o[u][set][h].w[q] = half2_as_u32(u32_as_half2(__builtin_amdgcn_perm(px1, px0, 0x05040100u)) + u32_as_half2(__builtin_amdgcn_perm(px1, px0, 0x07060302u)));
        }
        else
        {
            if constexpr (st == 2) px0 = __builtin_amdgcn_sad_hi_u8(px1, 0u, __builtin_amdgcn_sad_u8(px0, 0u, 0x64006400u));
            else
            {
                const half2_t kinv = { u16_as_half(0x1eeeu), u16_as_half(0x1eeeu) }, kbias = { u16_as_half(0xc931u), u16_as_half(0xc931u) };
                o[u][set][h].w[q] = half2_as_u32(__builtin_elementwise_fma(u32_as_half2(px0), kinv, kbias));
            }
        }
    };

    DgOperand bf[2][2][2][2];                             // [block parity][u][column c / c + 8][k half]
    #pragma unroll
    for (int j = 0; j < MT; ++j) fetch(b0, 0, j);
    #pragma unroll
    for (int u = 0; u < 2; ++u) load_lane_words<K>(ring[0][u], wptr(b0, u));
    words(ring[0]);
    #pragma unroll
    for (int r = 1; r < 3; ++r)
        #pragma unroll
        for (int u = 0; u < 2; ++u) load_lane_words<K>(ring[r & 1][u], wptr(b0 + r, u));
    dg_static_for<0, 128>([&] (auto pc) { piece(pc, bf[0]); });
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(2 * WL) : "memory");
    barrier();
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");      // (accumulators written by vector instructions, read by a matrix instruction that the compiler does not see)

    const int mj = lane & 15, kg = lane >> 4;
    const int lds_r = mj * 256 + (((8 * kh + 2 * kg) ^ mj) << 4);

    // (the last block of a slice with an odd number of them requests and decodes nothing: what lands in LDS behind its barrier would land in the output tile)
    auto block = [&] (int b, auto parity, LaneWords<K> (&slot)[2], auto last) __attribute__((always_inline))
    {
        constexpr int buf = decltype(parity)::value;
        constexpr bool MORE = !decltype(last)::value;
        const char* ab = smem + buf * (BM * 256);
        half8_t af[4];
        auto read = [&] (int gi) { af[gi & 3] = *((const half8_t*) (ab + (lds_r ^ ((gi & 1) << 4)) + (gi >> 1) * 4096)); };
        read(0); read(1); read(2);
        if constexpr (MORE) words(slot);
        __builtin_amdgcn_sched_barrier(0);
        dg_static_for<0, G>([&] (auto gc)
        {
            constexpr int gi = decltype(gc)::value, i = gi >> 1, h = gi & 1;
            if constexpr (gi + 3 < G) read(gi + 3);
            dg_static_for<0, 4>([&] (auto mc)
            {
                constexpr int m = decltype(mc)::value, n = 4 * gi + m, u = m >> 1, set = m & 1;
                dg_mfma(acc[i][u][set], af[gi & 3], bf[buf][u][set][h].h);
                if constexpr (MORE) dg_static_for<n * 128 / NM, (n + 1) * 128 / NM>([&] (auto pc) { piece(pc, bf[buf ^ 1]); });
                if constexpr (MORE && n % 3 == 1 && n / 3 < MT) fetch(b + 1, buf ^ 1, n / 3);
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        if constexpr (MORE)
        {
            #pragma unroll
            for (int u = 0; u < 2; ++u) load_lane_words<K>(slot[u], wptr(b + 3, u));
            asm volatile("s_waitcnt vmcnt(%0)" :: "n"(WL) : "memory");
        }
        barrier();
    };
    constexpr auto even = std::integral_constant<int, 0>{};
    constexpr auto odd = std::integral_constant<int, 1>{};
    int b = b0;
    for (; b + 2 <= b1; b += 2) { block(b, even, ring[1], std::false_type{}); block(b + 1, odd, ring[0], std::false_type{}); }
    if (b < b1) block(b, even, ring[1], std::true_type{});
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");    // the last matrix instructions have written their accumulators
    __builtin_amdgcn_sched_barrier(0);

    dg_epilogue<MT>(a, t, acc, (float*) smem, wave, lane);
}

#ifndef G2_K
#error "compile with -DG2_K=<bits per weight>"
#endif

template <int CB>
static void dgw_launch_cb(int mt, dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a)
{
    switch (mt)
    {
        #define DG(M) case M: dg_start<exl3_dgemm_wide_kernel<G2_K, CB, M>>(grid, lds, st, a); break;
        DG(10) DG(12) DG(14) DG(16)
        #undef DG
    }
}

#define DG_CAT_(a, b) a##b
#define DG_CAT(a, b) DG_CAT_(a, b)
void DG_CAT(exl3_dgemm_wide_launch_k, G2_K)(int cb, int mt, dim3 grid, size_t lds, hipStream_t st, const DgemmArgs& a)
{
    if (cb == 0) dgw_launch_cb<0>(mt, grid, lds, st, a);
    else if (cb == 1) dgw_launch_cb<1>(mt, grid, lds, st, a);
    else dgw_launch_cb<2>(mt, grid, lds, st, a);
}
