// Weight-streaming projections of up to 32 rows in two planes, three to five tiles (pairs of tiles) a workgroup: pc_gemm_skinny.h's tiles, K split, reduction and
// epilogues with the next U k-steps' weights and activations under way while U are multiplied.  (One block of k-steps after the other leaves a wave without a load
// under way while it multiplies, and more bytes in flight do not make up for it: one or two k-steps of four tiles are what a CU's memory path holds.)
// us, one block after the other / so, weights from memory: 20 rows, 7b q|k|v 21.3 / 20.4, gate|up 36.5 / 33.1, o_proj in four slices 10.5 / 9.4, down_proj 22.0 / 21.6;
// 13b gate|up 52.4 / 51.1; 12 rows, 13b q|k|v 28.2 / 28.3, o_proj 16.6 / 12.1 and down_proj 33.0 / 23.7 with five tiles instead of eight.  Weights alone, 7b: 17.1, 28.7,
// 6.5, 16.2.  Not for 33 rows and more (down_proj 24.0 / 25.4: the activations are the larger part) nor one, two or eight tiles (18.5 / 21.5, 49.6 / 49.5).
#include <type_traits>

#include "pc_gemm_skinny.h"

using namespace pcg;

namespace {

// ODD: shares of an odd number of blocks, where the second of the last pair is not there (and not read; asked for unseen, as the other shares' all are, it cost as much as one
// that counts.  us, unseen / so: 800 tiles, 12 and 32 rows, K = 512 6.1 / 5.0 and 7.5 / 5.8, K = 1536 11.6 / 10.4 and 14.5 / 12.4, K = 2560 16.5 / 15.1 and 20.7 / 18.8; even ones the
// other way round, K = 1024, 12 rows 8.0 / 8.2, o_proj in four slices 9.0 / 9.3).
// TRACE (pc_dev_gemm_trace): a kernel of its own, since the places to stamp at cost 2 % of o_proj's
template <int MT, int T, int EPI, int U, bool ODD, bool TRACE>
__global__ __launch_bounds__(kThreads) void gemm_pipe_kernel(const GemmParams p) {
    constexpr int TT = EPI == EPI_SILU ? 2 * T : T, TPI = EPI == EPI_SILU ? 2 : 1;       // tiles, tiles of an output item
    constexpr int kRT = MT * TT < 8 ? MT * TT : 8, IPR = kRT / TPI;                      // tiles, items of a round of the reduction (64 KiB at most)
    constexpr int NOUT = MT * T, ROUNDS = (NOUT + IPR - 1) / IPR;
    __shared__ f4 red[kWaves][kRT][64];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int KS = p.KS, bx = blockIdx.x, by = blockIdx.y;
    if (TRACE) trace_stamp(p, bx, by, wave, 0);
    int ks0, ks1;
    wave_k_range<false>(p, by, wave, ks0, ks1);
    int tile[TT];
    wg_tiles<T, EPI>(p, bx, tile);
    const char* wt[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) wt[t] = (const char*)p.wf + (int64_t)tile[t] * KS * 1024;
    const int live = p.m_dev ? (*p.m_dev < p.M ? *p.m_dev : p.M) : p.M;
    bool ok[MT];
#pragma unroll
    for (int a = 0; a < MT; ++a) ok[a] = a * 16 + m < live;
    struct Block {
        h8 w[U][TT], h[U][MT], l[U][MT];
    } A, B;
    auto issue = [&](Block& b, int kb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int k = kb + u < ks1 ? kb + u : ks1 - 1;                         // (past the share the last k-step again, not multiplied)
            k = k < 0 ? 0 : k;
            const uint32_t at = (uint32_t)k * 1024u + (uint32_t)lane * 16u;
#pragma unroll
            for (int t = 0; t < TT; ++t) b.w[u][t] = __builtin_bit_cast(h8, __builtin_nontemporal_load((const u32x4*)(wt[t] + at)));
#pragma unroll
            for (int a = 0; a < MT; ++a) {
                const h8 zero = {0, 0, 0, 0, 0, 0, 0, 0};
                b.h[u][a] = b.l[u][a] = zero;
                if (ok[a]) {
                    b.h[u][a] = *(const h8*)((const char*)p.xf_hi + (int64_t)a * KS * 1024 + at);
                    b.l[u][a] = *(const h8*)((const char*)p.xf_lo + (int64_t)a * KS * 1024 + at);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    f4 acc[MT][TT];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[a][t] = f4{0.f, 0.f, 0.f, 0.f};
    auto consume = [&](const Block& b, int kb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (kb + u >= ks1) continue;                                     // (uniform over the wave)
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int a = 0; a < MT; ++a) {
                    acc[a][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b.w[u][t], b.h[u][a], acc[a][t], 0, 0, 0);
                    acc[a][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b.w[u][t], b.l[u][a], acc[a][t], 0, 0, 0);
                }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    issue(A, ks0);
    for (int kb = ks0; kb < ks1; kb += 2 * U) {
        if (!ODD || kb + U < ks1) issue(B, kb + U);
        consume(A, kb);
        if (kb + 2 * U < ks1) issue(A, kb + 2 * U);
        consume(B, kb + U);
    }
    if (TRACE) trace_stamp(p, bx, by, wave, 1);
    // the waves' shares in wave order, one output item a wave and round
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        if (r > 0) lds_barrier();
#pragma unroll
        for (int i = 0; i < IPR; ++i) {
            const int item = r * IPR + i;
            if (item < NOUT) {
                const int a = item / T, t = item - a * T;
                red[wave][i * TPI][lane] = acc[a][t];
                if (EPI == EPI_SILU) red[wave][i * TPI + TPI - 1][lane] = acc[a][TT - T + t];
            }
        }
        lds_barrier();
        if (TRACE && r == 0) trace_stamp(p, bx, by, wave, 2);
        const int item = r * IPR + wave;
        if (wave < IPR && item < NOUT) {
            const int a = item / T, t = item - a * T;
            f4 v = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                v += red[w][wave * TPI][lane];
                if (EPI == EPI_SILU) u += red[w][wave * TPI + TPI - 1][lane];
            }
            tile_epilogue_of<EPI, TRACE>(p, v, u, a * 16 + m, bx * T + t, g, by);
        }
    }
    if (TRACE) { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); trace_stamp(p, bx, by, wave, 3); }
}

template <int MT, int T, int EPI>
int go(const GemmParams& p, int units, hipStream_t s) {
    constexpr int U = EPI != EPI_SILU && (T == 4 || (MT == 1 && T == 3)) ? 2 : 1;
    const dim3 grid(pc_ceil_div(units, T), p.kslices);
    const bool odd = pc_ceil_div(pc_ceil_div(pc_ceil_div(p.KS, p.kslices), kWaves), U) & 1;
    if (p.trace)
        hipLaunchKernelGGL((gemm_pipe_kernel<MT, T, traced_epi(EPI), U, true, true>), grid, dim3(kThreads), 0, s, traced(p, EPI));
    else if (odd)
        hipLaunchKernelGGL((gemm_pipe_kernel<MT, T, EPI, U, true, false>), grid, dim3(kThreads), 0, s, p);
    else
        hipLaunchKernelGGL((gemm_pipe_kernel<MT, T, EPI, U, false, false>), grid, dim3(kThreads), 0, s, p);
    return pc_check_launch("gemm_pipe_kernel");
}

template <int MT, int T>
int by_epi(int epi, const GemmParams& p, int units, hipStream_t s) {
    switch (epi) {
        case EPI_STORE: return go<MT, T, EPI_STORE>(p, units, s);
        case EPI_ADD: return go<MT, T, EPI_ADD>(p, units, s);
        case EPI_SILU:
            if constexpr (T <= 4) return go<MT, T, EPI_SILU>(p, units, s);
            pc_set_error("pc_gemm (pipe): no gated unit with %d pairs a workgroup", T);
            return PC_ERR_ARG;
        case EPI_ROPE: return go<MT, T, EPI_ROPE>(p, units, s);
        default: return go<MT, T, EPI_GELU>(p, units, s);
    }
}

template <int MT>
int by_tiles(int epi, const GemmParams& p, int T, int units, hipStream_t s) {
    return T == 3 ? by_epi<MT, 3>(epi, p, units, s) : T == 4 ? by_epi<MT, 4>(epi, p, units, s) : by_epi<MT, 5>(epi, p, units, s);
}

}  // namespace

namespace pcg {
// Three and four tiles: plain results over up to 4096 of K a slice, beyond only over odd multiples of 512 (else tiles begin on the same channels, and the more steps a workgroup asks
// for at a time the better); gated ones of up to sixteen rows not where a block of four k-steps holds a wave's share, nor over multiples of 4096.  us, one block after the
// other / so: 560 and 800 tiles, 4 rows, K = 2048 9.2 / 8.9 and 13.0 / 12.7, 4096 14.8 / 14.9 and 23.4 / 23.6, 5120 17.7 / 18.6 and 23.4 / 23.8, 7168 23.5 / 24.5 and 31.1 / 32.0;
// 32 rows, K = 2048 11.5 / 11.6 and 14.8 / 14.3, 4096 19.0 / 19.7 and 26.1 / 26.8, 5120 23.5 / 25.3 and 30.4 / 31.2, 7168 31.6 / 34.1 and 40.9 / 42.5; 20 rows, K = 6656, 640 and 900
// tiles 28.9 / 28.0 and 35.2 / 34.7, 11008 46.8 / 48.8 and 61.2 / 62.8; gated, 688 pairs, 12 rows, K = 1024 11.4 / 12.0, 2048 17.3 / 16.3, 4096 29.7 / 30.8, 5120 40.0 / 38.8, 32
// rows, 640 pairs, K = 5120 43.2 / 42.0.  (Where a launch's weights lie moves such times by up to 3 %.)
// Three tiles over an odd multiple of 1024 (3072; of 1024 it makes no difference) not with more than 24 rows, whose operands have a second line in every group of lanes.  us, one block after
// the other / so, K = 3072, 520, 640 and 768 tiles: 32 rows 15.5 / 16.6, 16.5 / 17.4, 17.9 / 18.4, 24 rows 14.8 / 15.2, 15.9 / 16.0, 17.4 / 17.2; K = 2560 and 3584, 32 rows 0.95 to 1.01 of it.
bool pipe_takes(int epi, const GemmParams& p, int T) {
    if (epi == EPI_SILU) return p.M > 16 || (pc_ceil_div(p.KS, kWaves) != 4 && p.KS % 128 != 0);
    if (T == 3 && p.M > 24 && p.kslices == 1 && p.KS > 32 && p.KS % 64 == 32) return false;
    return p.KS <= 128 * p.kslices || p.KS % 32 == 16;
}

int launch_pipe(int epi, const GemmParams& p, int T, int units, hipStream_t s) {
    return p.M <= 16 ? by_tiles<1>(epi, p, T, units, s) : by_tiles<2>(epi, p, T, units, s);
}
}  // namespace pcg
