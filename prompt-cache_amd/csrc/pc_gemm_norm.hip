// Weight-streaming projections of up to sixteen rows behind an RMSNorm (q|k|v, gate|up, lm_head of a cached step or a decoded token): the norm's gain and the
// split into fp16 hi / lo happen in the launch, 1 / rms on the reduced tile (pc_gemm_skinny.h says how; tiles, K split and epilogues are that file's).
//
// What bounds them is the weight stream: 100 / 180 / 262 MB (q|k|v, gate|up, lm_head of a 7b model) read by themselves, in these tiles, take 17.1 / 28.7 /
// 42 us.  What came on top, a us each, were the rows' loads (two of every five instructions of q|k|v, four lanes of 64 in use for one row), gain and split (56
// instructions a k-step and wave, for sixteen rows whatever their number) and, a wave's blocks of k-steps being asked for one after the other, the waits between them:
//   normed_few_kernel   one and two rows: a wave turns its share of the rows into operand pieces once, all 64 lanes at work, and keeps them in LDS; its loop has
//                       weight loads and two LDS reads a k-step
//   normed_kernel       three rows and more: the next k-step's weights and rows are under way while this one is multiplied.  (Single k-steps: more bytes in flight
//                       cost more than the waits, q|k|v two k-steps at a time 20.0, four 21.6.)
// us, as blocks of four k-steps one after the other / so: 1 row, 7b q|k|v 20.3 / 18.6, gate|up 32.2 / 30.4, lm_head 49.9 / 41.9, 13b 29.4 / 25.9, 52.4 / 45.2,
// 57.6 / 49.8; 12 rows, 7b 20.7 / 19.8, 33.5 / 33.4, 13b 30.9 / 30.4, 51.0 / 49.3.
#include <type_traits>

#include "pc_gemm_skinny.h"

using namespace pcg;

namespace {

constexpr int kFewRows = 2;
constexpr int kFewLds = 48 * 1024;        // operand pieces of the rows: both planes, 4 bytes an element

__device__ __forceinline__ h8 weight(const char* tile, int ks, int lane) {
    return __builtin_bit_cast(h8, __builtin_nontemporal_load((const u32x4*)(tile + ((uint32_t)ks * 1024u + (uint32_t)lane * 16u))));
}

// the eight waves' sums of the workgroup's tiles in wave order, scaled by 1 / rms, to the epilogue: one tile (pair) a wave
template <int T, int EPI, bool TRACE>
__device__ __forceinline__ void reduce_normed(const GemmParams& p, const f4 (&acc)[EPI == EPI_SILU ? 2 * T : T], f4 (*red)[EPI == EPI_SILU ? 2 * T : T][64],
                                              const float (*ssl)[16], int wave, int lane, int m, int g) {
    constexpr int TT = EPI == EPI_SILU ? 2 * T : T;
#pragma unroll
    for (int t = 0; t < TT; ++t) red[wave][t][lane] = acc[t];
    if (TRACE) trace_stamp(p, blockIdx.x, 0, wave, 1);
    lds_barrier();
    if (TRACE) trace_stamp(p, blockIdx.x, 0, wave, 2);
    if (wave >= T) return;
    f4 v = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        v += red[w][wave][lane];
        if (EPI == EPI_SILU) u += red[w][T + wave][lane];
        tot += ssl[w][m];
    }
    const float rs = rsqrtf(tot / (float)(p.KS * 32) + p.eps);
    v *= rs;
    u *= rs;
    tile_epilogue_of<EPI, TRACE>(p, v, u, m, (int)blockIdx.x * T + wave, g, 0);
    if (TRACE) { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); trace_stamp(p, blockIdx.x, 0, wave, 3); }
}

template <int T, int EPI, int U, bool TRACE>
__global__ __launch_bounds__(kThreads) void normed_few_kernel(const GemmParams p) {
    constexpr int TT = EPI == EPI_SILU ? 2 * T : T;
    extern __shared__ __attribute__((aligned(16))) _Float16 pieces[];       // per wave: [row][hi, lo][ld]
    __shared__ f4 red[kWaves][TT][64];
    __shared__ float ssl[kWaves][16];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (TRACE) trace_stamp(p, blockIdx.x, 0, wave, 0);
    const int KS = p.KS, M = p.M;
    const int live = p.m_dev ? (*p.m_dev < M ? *p.m_dev : M) : M;           // (rows behind them are never read)
    int ks0, ks1;
    wave_k_range<false>(p, 0, wave, ks0, ks1);
    const int n = ks1 > ks0 ? (ks1 - ks0) * 32 : 0, ld = (KS + kWaves - 1) / kWaves * 32 + 32;   // (rows begin 64 bytes apart in the banks)
    _Float16* mine = pieces + wave * (M * 2 * ld);
    int tile[TT];
    wg_tiles<T, EPI>(p, blockIdx.x, tile);
    const char* wt[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) wt[t] = (const char*)p.wf + (int64_t)tile[t] * KS * 1024;
    h8 wA[U][TT], wB[U][TT];
    auto issue = [&](h8 (&w)[U][TT], int kb) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int t = 0; t < TT; ++t) w[u][t] = weight(wt[t], kb + u < ks1 ? kb + u : ks1 - 1, lane);
    };
    // ---- the rows: elements e .. e + 7 of the wave's share, a chunk of 512 at a time; the first chunk ahead of the weights
    f4 xa[kFewRows][2];
    h8 gm;
    auto ask = [&](int e) {
        const int at = e < n ? e : n > 0 ? n - 8 : -ks0 * 32;                // (clamped: nothing is kept of what lies behind the share)
#pragma unroll
        for (int r = 0; r < kFewRows; ++r) {
            const float* x = p.xn + (int64_t)(r < live ? r : 0) * (KS * 32) + ks0 * 32 + at;
            xa[r][0] = *(const f4*)x;
            xa[r][1] = *(const f4*)(x + 4);
        }
        gm = *(const h8*)(p.gamma + ks0 * 32 + at);
    };
    float ss[kFewRows];
#pragma unroll
    for (int r = 0; r < kFewRows; ++r) ss[r] = 0.f;
    auto keep = [&](int e) {
        if (e >= n) return;
#pragma unroll
        for (int r = 0; r < kFewRows; ++r)
            if (r < M) {                                                     // (uniform)
                h8 hi, lo;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float x = r < live ? (i < 4 ? xa[r][0][i] : xa[r][1][i - 4]) : 0.f;
                    ss[r] += x * x;
                    _Float16 a, b;
                    pc_split(x * (float)gm[i], a, b);
                    hi[i] = a;
                    lo[i] = b;
                }
                *(h8*)(mine + r * 2 * ld + e) = hi;
                *(h8*)(mine + (r * 2 + 1) * ld + e) = lo;
            }
    };
    ask(lane * 8);
    __builtin_amdgcn_sched_barrier(0);
    issue(wA, ks0);
    __builtin_amdgcn_sched_barrier(0);
    keep(lane * 8);
    for (int e = 512 + lane * 8; e - lane * 8 < n; e += 512) {
        ask(e);
        keep(e);
    }
#pragma unroll
    for (int r = 0; r < kFewRows; ++r) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss[r] += __shfl_xor(ss[r], o);
        if (lane == 0) ssl[wave][r] = ss[r];
    }
    // ---- the products (LDS of the wave's own: no barrier)
    f4 acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    const _Float16* hr = mine + (m < M ? m : 0) * 2 * ld + g * 8;
    auto consume = [&](const h8 (&w)[U][TT], int kb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (kb + u >= ks1) continue;                                     // (uniform over the wave)
            const h8 hi = *(const h8*)(hr + (kb + u - ks0) * 32), lo = *(const h8*)(hr + ld + (kb + u - ks0) * 32);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][t], hi, acc[t], 0, 0, 0);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[u][t], lo, acc[t], 0, 0, 0);
            }
        }
    };
    for (int kb = ks0; kb < ks1; kb += 2 * U) {
        issue(wB, kb + U);
        __builtin_amdgcn_sched_barrier(0);
        consume(wA, kb);
        __builtin_amdgcn_sched_barrier(0);
        if (kb + 2 * U < ks1) issue(wA, kb + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        consume(wB, kb + U);
        __builtin_amdgcn_sched_barrier(0);
    }
    reduce_normed<T, EPI, TRACE>(p, acc, red, ssl, wave, lane, m, g);
}

template <int T, int EPI, bool TRACE>
__global__ __launch_bounds__(kThreads) void normed_kernel(const GemmParams p) {
    constexpr int TT = EPI == EPI_SILU ? 2 * T : T;
    __shared__ f4 red[kWaves][TT][64];
    __shared__ float ssl[kWaves][16];
    __shared__ __attribute__((aligned(16))) _Float16 gain[kWaves * kGamHalfs];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (TRACE) trace_stamp(p, blockIdx.x, 0, wave, 0);
    const int KS = p.KS;
    const int live = p.m_dev ? (*p.m_dev < p.M ? *p.m_dev : p.M) : p.M;
    int ks0, ks1;
    wave_k_range<false>(p, 0, wave, ks0, ks1);
    int tile[TT];
    wg_tiles<T, EPI>(p, blockIdx.x, tile);
    const char* wt[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) wt[t] = (const char*)p.wf + (int64_t)tile[t] * KS * 1024;
    const bool ok = m < live;
    const float* xrow = p.xn + (int64_t)m * (KS * 32) + g * 8;
    h8 wA[TT], wB[TT];
    f4 xA[2], xB[2];
    auto issue = [&](h8 (&w)[TT], f4 (&x)[2], int k) {
        k = k < ks1 ? k : ks1 - 1;
#pragma unroll
        for (int t = 0; t < TT; ++t) w[t] = weight(wt[t], k, lane);
        x[0] = x[1] = f4{0.f, 0.f, 0.f, 0.f};
        if (ok) {
            x[0] = *(const f4*)(xrow + k * 32);
            x[1] = *(const f4*)(xrow + k * 32 + 4);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    issue(wA, xA, ks0);
    _Float16* gs = gain + wave * kGamHalfs;                                  // (the wave's own: no barrier)
    for (int j = lane * 8; j < (ks1 - ks0) * 32; j += 512) *(h8*)(gs + j) = *(const h8*)(p.gamma + ks0 * 32 + j);
    float ss = 0.f;
    f4 acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
    auto consume = [&](const h8 (&w)[TT], const f4 (&x)[2], int k) {
        const h8 gw = *(const h8*)(gs + (k - ks0) * 32 + g * 8);
        h8 hi, lo;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float xv = e < 4 ? x[0][e] : x[1][e - 4];
            ss += xv * xv;
            _Float16 a, b;
            pc_split(xv * (float)gw[e], a, b);
            hi[e] = a;
            lo[e] = b;
        }
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[t], hi, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[t], lo, acc[t], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int k = ks0; k < ks1; k += 2) {
        issue(wB, xB, k + 1);
        consume(wA, xA, k);
        if (k + 2 < ks1) issue(wA, xA, k + 2);
        if (k + 1 < ks1) consume(wB, xB, k + 1);
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (g == 0) ssl[wave][m] = ss;
    reduce_normed<T, EPI, TRACE>(p, acc, red, ssl, wave, lane, m, g);
}

// (pc_dev_gemm_trace: kernels of their own, since the places to stamp at cost 1 or 2 % of the shortest launches)
template <int T, int EPI, bool TRACE>
int go_few(const GemmParams& p, int units, size_t lds, hipStream_t s) {
    constexpr int U = EPI == EPI_SILU ? 1 : 4;
    static const hipError_t raised =
        hipFuncSetAttribute(reinterpret_cast<const void*>(normed_few_kernel<T, EPI, U, TRACE>), hipFuncAttributeMaxDynamicSharedMemorySize, kFewLds);
    (void)raised;
    hipLaunchKernelGGL((normed_few_kernel<T, EPI, U, TRACE>), dim3(pc_ceil_div(units, T)), dim3(kThreads), lds, s, p);
    return pc_check_launch("normed_few_kernel");
}

template <int T, int EPI>
int go(const GemmParams& p, int units, hipStream_t s) {
    if (p.trace)
        hipLaunchKernelGGL((normed_kernel<T, traced_epi(EPI), true>), dim3(pc_ceil_div(units, T)), dim3(kThreads), 0, s, traced(p, EPI));
    else
        hipLaunchKernelGGL((normed_kernel<T, EPI, false>), dim3(pc_ceil_div(units, T)), dim3(kThreads), 0, s, p);
    return pc_check_launch("normed_kernel");
}

size_t few_lds(const GemmParams& p) { return (size_t)p.M * 2 * (pc_ceil_div(p.KS, kWaves) * 32 + 32) * 2 * kWaves; }

}  // namespace

namespace pcg {

// Not plain results over a share of up to four k-steps a wave (us, 1 row, blocks of k-steps / so: K = 512, 300 and 800 tiles 4.4 / 4.8 and 5.9 / 7.7, K = 1024 5.4 / 5.3 and
// 8.0 / 9.1; K = 1152 0.90 and 0.96 of it, 1536 6.4 / 5.7 and 10.6 / 9.6, 2048 7.5 / 6.6 and 14.4 / 11.3; gated, K = 512, 300 and 860 pairs 5.9 / 5.5 and 8.7 / 7.9).
bool normed_few_takes(int epi, const GemmParams& p) {
    return p.xn && (epi == EPI_SILU || p.KS > 4 * kWaves) && !p.w8 && p.M <= kFewRows && p.kslices == 1 && p.kskew == 0 && (epi == EPI_STORE || epi == EPI_ROPE || epi == EPI_SILU) && few_lds(p) <= kFewLds;
}

// Tiles (pairs of tiles) a workgroup: the number that leaves the fewest of the chip's 256 CUs without one in the last round, of 3 (of 2, where tile images are not
// whole multiples of 64 KB: those of two and four tiles then lie on the same channels), 1 and the other.  us, 1 row, 1 / 2 / 3 / 4 tiles: K = 4096, 768 tiles
// 20.0 / 22.2 / 18.6 / 22.8, 688 pairs 29.6 / 35.9 / 30.4 / 33.0, 2000 tiles 41.9 / 46.4 / 43.0 / 49.6; K = 5120, 960 tiles 26.1 / 25.9 / 31.1 / 27.7, 864 pairs
// 46.0 / 45.2 / 57.7 / 46.3, 2000 tiles 50.6 / 49.8 / 51.2 / 51.6.
int launch_normed_few(int epi, const GemmParams& p, int units, hipStream_t s) {
    const bool even = p.KS % 64 != 0;
    const int cand[3] = {even ? 2 : 3, even ? 3 : 1, even ? 1 : 3};
    int T = 1;
    float best = 0.f;
    for (int c : cand) {
        const int wg = pc_ceil_div(units, c), rounds = pc_ceil_div(wg, 256);
        const float busy = (float)units / ((float)rounds * 256.f * (float)c);
        if (busy > best) T = c, best = busy;
    }
    const size_t lds = few_lds(p);
    auto sized = [&](auto t) {
        constexpr int TV = decltype(t)::value;
        auto go = [&](auto e) {
            constexpr int EPI = decltype(e)::value;
            return p.trace ? go_few<TV, traced_epi(EPI), true>(traced(p, EPI), units, lds, s) : go_few<TV, EPI, false>(p, units, lds, s);
        };
        return epi == EPI_STORE  ? go(std::integral_constant<int, EPI_STORE>{})
               : epi == EPI_ROPE ? go(std::integral_constant<int, EPI_ROPE>{})
                                 : go(std::integral_constant<int, EPI_SILU>{});
    };
    return T == 1 ? sized(std::integral_constant<int, 1>{}) : T == 2 ? sized(std::integral_constant<int, 2>{}) : sized(std::integral_constant<int, 3>{});
}

// Where single k-steps, the next under way, are the faster: not where a block of four holds a wave's whole share; over more than 4096 of K only over odd multiples of 512 (else tiles
// begin on the same channels, and the more steps a workgroup asks for at a time the better); two tiles a workgroup, few bytes under way, only with the loads of ten rows
// beside them.  us, blocks of four / so, at 3, 8 and 16 rows: plain, 300 tiles (two), K = 512 4.5 / 4.4, 4.8 / 4.8, 5.3 / 5.0, K = 1024 5.5 / 6.2, 5.9 / 6.5, 6.6 / 6.6, K = 2048
// 7.5 / 8.8, 8.1 / 8.9, 9.9 / 9.6, K = 4096 12.1 / 14.3, 13.2 / 14.4, 15.8 / 15.2, K = 5120 15.6 / 19.3, 16.4 / 18.0, 18.8 / 19.2, K = 8192 21.6 / 26.4, 24.0 / 26.9, 26.5 / 27.2; 640
// (three), K = 1024 1.07, 1.05, 1.00 of it, K = 1536 0.92, 0.88, 0.87, 4096 0.95, 1.00, 0.95, 5120 1.04, 1.08, 1.05, 8192 1.07, 1.10, 1.07, 11008 1.06, 1.06, 1.02; 960 (four) 4096 0.99,
// 1.01, 0.93, 5120 1.02, 1.03, 1.00, 8192 1.03, 1.05, 1.02, 13824 0.96, 0.96, 0.92; gated, 688 pairs (three), K = 4096 31.3 / 32.0, 31.7 / 31.8, 33.2 / 32.0, 640, K = 1024 1.02, 1.02, 0.99,
// K = 2048 0.93, 0.91, 0.90, 5120 1.01, 1.02, 1.01, 8192 1.09, 1.08, 1.06; 864 (four), K = 4096 44.5 / 45.4, 43.3 / 44.3, 43.5 / 43.8, 5120 53.1 / 52.1, 51.0 / 49.8, 52.7 / 50.7.  (Where a
// launch's weights lie moves such times by up to 3 %.)
bool normed_takes(int epi, const GemmParams& p, int T) {
    const int share = pc_ceil_div(p.KS, kWaves);
    const bool far = p.KS % 32 == 16;
    if (epi == EPI_SILU) return T == 4 ? p.KS % 128 != 0 : share <= 16 ? share != 4 && (p.KS % 128 != 0 || p.M > 9) : far;
    if (share <= 4) return share <= 2;
    return T > 2 ? share <= 16 || far : share <= 16 && p.M > 9;
}

// (two to four tiles, or pairs of tiles, a workgroup)
int launch_normed(int epi, const GemmParams& p, int T, int units, hipStream_t s) {
    auto sized = [&](auto t) {
        constexpr int TV = decltype(t)::value;
        return epi == EPI_STORE ? go<TV, EPI_STORE>(p, units, s) : epi == EPI_ROPE ? go<TV, EPI_ROPE>(p, units, s) : go<TV, EPI_SILU>(p, units, s);
    };
    return T == 2 ? sized(std::integral_constant<int, 2>{}) : T == 3 ? sized(std::integral_constant<int, 3>{}) : sized(std::integral_constant<int, 4>{});
}

}  // namespace pcg
