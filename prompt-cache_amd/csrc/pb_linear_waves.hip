// pb_linear over some tens or hundreds of rows: small tiles whose four waves split k instead of the tile.
//
// Workgroup = 32 rows x 32 result columns (gated: 16 of each half).  A wave takes every fourth chunk of 128 bytes of k for the whole tile, through a ring
// of LDS images of its own (global_load_lds, the layout of linear_dma_kernel): nothing that a wave does waits for another one until the four sums are
// added at the end, in the waves' order.
// What bounds it: with one workgroup a CU, a wave's own chain -- fp32 its MFMAs (1024 cycles a chunk), bf16 one trip to L2 per S - 1 chunks --, beyond
// that L2's 64 bytes a clock and CU (a chunk is 8 KB for 128 cycles of bf16 products).
#include <type_traits>

#include "pb_linear_parts.h"
#include "pb_linear_tiles.h"

namespace {
using namespace pcb;

__device__ const u32x4 zero_row = {0u, 0u, 0u, 0u};

template <typename E, int EPI, int S>
__global__ __launch_bounds__(256) void linear_waves_kernel(pcb_linear_args a) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int CE = 16 / sizeof(E), BK = 8 * CE, BM = 32, BN = TWO ? 16 : 32, ROWS = 64, NI = ROWS / 8, TN = TWO ? 1 : 2;
    __shared__ __attribute__((aligned(16))) E img[4][S][ROWS * BK];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), group = lane >> 4, l15 = lane & 15;
    const int K = a.K, M = a.M, N = a.N;
    const int mb = (M + BM - 1) / BM, total = mb * ((N + BN - 1) / BN), per = (total + 7) / 8;
    const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
    const int m_lo = t % mb * BM, n_lo = t / mb * BN, g = a.n_batch > 0 ? blockIdx.z : 0;
    const E* X = (const E*)a.x + g * a.x_batch_stride;
    const E* W = (const E*)a.w + g * a.w_group_stride;

    // a wave's instruction i fills rows 8 i .. + 7 of its image: A rows, W rows, W2 rows
    const E* src[NI];
    int kc[2];                                                       // the lane's k offset within the chunk (even and odd instructions)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = 8 * i + (lane >> 3);
        if (i < 2) kc[i] = ((lane & 7) ^ ((r >> 1) & 7)) * CE;
        if (8 * i < BM) {
            const int m = m_lo + r < M ? m_lo + r : M - 1;
            src[i] = X + (int64_t)(a.row_src ? a.row_src[m] : m) * a.ldx;
        } else {
            const bool second = TWO && 8 * i >= BM + BN;
            const int n0 = n_lo + r - BM - (second ? BN : 0), n = n0 < N ? n0 : N - 1;
            src[i] = (second ? (const E*)a.w2 : W) + (int64_t)n * a.ldw;
        }
    }
    const int chunks = (K + BK - 1) / BK, mine = (chunks - wave + 3) / 4;
    auto fetch = [&](int c, int buf) {
        const int k0 = (wave + 4 * c) * BK;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const void* p = src[i] + k0 + kc[i & 1];
            if (k0 + BK > K && k0 + kc[i & 1] >= K) p = &zero_row;
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                             (__attribute__((address_space(3))) void*)&img[wave][buf][i * 8 * BK], 16, 0, 0);
        }
    };
    auto frag = [&](int buf, int r, int ks) {
        Frag<E> f;
        const E* row = &img[wave][buf][r * BK];
        const int sw = (r >> 1) & 7;
        if constexpr (sizeof(E) == 2) {
            f.v = *reinterpret_cast<const u32x4*>(row + ((4 * ks + group) ^ sw) * CE);
        } else {
            const f4 lo = *reinterpret_cast<const f4*>(row + ((2 * group) ^ sw) * CE), hi = *reinterpret_cast<const f4*>(row + ((2 * group + 1) ^ sw) * CE);
#pragma unroll
            for (int e = 0; e < 4; ++e) f.v[e] = lo[e], f.v[4 + e] = hi[e];
        }
        return f;
    };
    Sum<E> sum[2][2];                                                // [row tile][column tile; gated: half]
#pragma unroll
    for (int p = 0; p < S - 1; ++p)
        if (p < mine) fetch(p, p);
    int buf = 0;
    for (int c = 0; c < mine; ++c) {
        // (loads land in order; the next chunk may be under way)
        static_assert(S <= 3, "at most one chunk beside the one at hand");
        if (S > 2 && c + 1 < mine)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NI) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        Frag<E> fa[BK / 32][2], fb[BK / 32][2];
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[ks][i] = frag(buf, 16 * i + l15, ks);
                fb[ks][i] = frag(buf, BM + 16 * i + l15, ks);
            }
        if (c + S - 1 < mine) fetch(c + S - 1, buf == 0 ? S - 1 : buf - 1);
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) sum[i][j].add(fb[ks][j], fa[ks][i]);
        buf = buf + 1 == S ? 0 : buf + 1;
    }
    // the waves' sums through LDS; wave w finishes tile w (row tile w / TN, column tile w % TN).  (The weights are the products' first operand: a lane has
    // four neighbouring columns of one row.)
    f4* const red = reinterpret_cast<f4*>(&img[0][0][0]);
    static_assert(sizeof(img) >= 4 * 4 * 64 * sizeof(f4), "room for the sums");
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) red[(wave * 4 + 2 * i + j) * 64 + lane] = sum[i][j].total();
    __syncthreads();
    if (wave >= 2 * TN) return;
    f4 acc = red[(TWO ? 2 * wave : wave) * 64 + lane], acc2 = red[(TWO ? 2 * wave + 1 : wave) * 64 + lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
        acc += red[(w * 4 + (TWO ? 2 * wave : wave)) * 64 + lane];
        if (TWO) acc2 += red[(w * 4 + 2 * wave + 1) * 64 + lane];
    }
    const int m = m_lo + 16 * (wave / TN) + l15, n = n_lo + 16 * (wave % TN) + 4 * group;
    if (m >= M) return;
    float bv[4], bv2[4], cs[4];
    Place to[4] = {};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const bool in = n + e < N;
        bv[e] = a.bias && in ? to_f32(((const E*)a.bias)[n + e]) : 0.0f;
        bv2[e] = TWO && a.bias2 && in ? to_f32(((const E*)a.bias2)[n + e]) : 0.0f;
        cs[e] = EPI == PCB_EPI_SCALE_ADD && in ? a.col_scale[n + e] : 0.0f;
        if (in) to[e] = place<E, EPI>(a, m, n + e);
    }
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (n + e < N) v[e] = finished<E, EPI>(a, to[e], n + e, acc[e], acc2[e], bv[e], bv2[e]);
    if (EPI != PCB_EPI_SCALE_ADD && n + 4 <= N) {
        const int size = to[0].wide ? 4 : (int)sizeof(E);
        if (to[3].p - to[0].p == 3 * size && to[1].p - to[0].p == size && to[3].wide == to[0].wide && (uintptr_t)to[0].p % (4 * size) == 0) {
            if (to[0].wide)
                store4((float*)to[0].p, v[0], v[1], v[2], v[3]);
            else
                store4((E*)to[0].p, v[0], v[1], v[2], v[3]);
            return;
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (n + e < N) put<E, EPI>(to[e], v[e], cs[e]);
}

template <typename E, int S>
int run(const pcb_linear_args& a, hipStream_t stream) {
    auto go = [&](auto epi) {
        hipLaunchKernelGGL((linear_waves_kernel<E, decltype(epi)::value, S>), dim3((uint32_t)(8 * ((pcb_linear_waves_tiles(a) + 7) / 8)), 1, a.n_batch > 0 ? a.n_batch : 1),
                           dim3(256), 0, stream, a);
        return pcb_check_launch("linear_waves_kernel");
    };
    switch (a.epilogue) {
        case PCB_EPI_STORE: return go(std::integral_constant<int, PCB_EPI_STORE>{});
        case PCB_EPI_SILU_MUL: return go(std::integral_constant<int, PCB_EPI_SILU_MUL>{});
        default: return go(std::integral_constant<int, PCB_EPI_SCALE_ADD>{});
    }
}

}  // namespace

int64_t pcb_linear_waves_tiles(const pcb_linear_args& a) {
    return (int64_t)pcb_ceil_div(a.M, 32) * pcb_ceil_div(a.N, a.epilogue == PCB_EPI_SILU_MUL ? 16 : 32);
}

// bf16: up to two workgroups a CU.  us, the tiles of linear_dma_kernel / here: 37 rows, 1024 columns, K = 1024 8.0 / 5.5, K = 4096 22.6 / 9.0; 200 x 1024,
// K = 2048 13.2 / 7.1; 64 x 5136, K = 2048 (322 workgroups) 13.4 / 9.4; 300 x 1024, K = 4096 (320) 23.5 / 12.4; 1000 x 512, K = 512 (512) 6.1 / 6.0;
// 130 x 4096, K = 1024 (640) 8.8 / 10.4.
// fp32: a round of the chip, and three over a deep k.  37 x 1024, K = 1024 17.5 / 9.5, K = 4096 60 / 25; 64 x 2048 gated, K = 1024 18.9 / 10.7;
// 300 x 2048, K = 2048 (640) 47.6 / 39.9, 75 x 4096 gated (768) 52 / 45; 130 x 5136 (805) 50.5 / 52.9.
// A wave has to have two chunks of k at least for its own ring to be worth the sums at the end, beyond 192 workgroups bf16 four: bf16 17 x 2048, K = 256
// 4.0 / 4.4, 17 x 11000 (344) K = 256 4.6 / 6.2, K = 512 5.7 / 6.9, 128 x 4096 (512) K = 512 6.2 / 6.7, gated 17 x 4096 (256) 6.1 / 6.5; fp32 64 x 512, K = 64 3.9 / 4.7.
bool pcb_linear_waves_fits(const pcb_linear_args& a) {
    if (a.n_groups > 0) return false;
    const int64_t wgs = pcb_linear_waves_tiles(a) * (a.n_batch > 0 ? a.n_batch : 1);
    if (a.dtype != PCB_BF16) return a.K >= 256 && (wgs <= 256 || (wgs <= 768 && a.K >= 2048));
    return a.K >= 1024 ? wgs <= 512 : a.K >= 512 && wgs <= 192;
}

// Three images to a wave's ring (96 KB: one workgroup a CU); two where bf16 has two workgroups a CU (300 x 1024, K = 1024: 6.7 us, 9.1 with three; 200 x
// 1024, 224 workgroups, K = 2048 7.6 and 7.1).
int pcb_linear_waves(const pcb_linear_args& a, hipStream_t stream) {
    if (a.dtype != PCB_BF16) return run<float, 3>(a, stream);
    return pcb_linear_waves_tiles(a) * (a.n_batch > 0 ? a.n_batch : 1) > 256 ? run<bf16_t, 2>(a, stream) : run<bf16_t, 3>(a, stream);
}
