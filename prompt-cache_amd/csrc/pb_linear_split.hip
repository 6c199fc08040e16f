// pb_linear over many rows in fp32 on the bf16 matrix cores: every operand element as the sum of three bf16 (8 + 8 + 8 bits: hi + mid + lo is the element
// exactly, but for what an element below 2^-110 has below 2^-133, bf16's smallest; conversions and products keep subnormal numbers), a product as the six of the
// nine partial products that reach 2^-26 of it: hi hi in one sum, hi mid, mid hi, mid mid, hi lo, lo hi in another.  What is left out is at most 2^-26 of a term,
// and a sum of 32 terms is rounded once: against 64 bits 0.46 of the error of the fp32 matrix cores (K = 1024: 1.9e-7 / 4.1e-7), which do 256 multiply-adds a
// clock and CU where these do 4096 / 6.
//
// Workgroup = (32 TM) x (16 WN TN) results, 2 x WN waves of TM x TN blocks of 16 x 16.  Per k-step of 32 the rows go global -> registers (two steps ahead), are split
// there, each element once a workgroup, and lie in two LDS images of three planes; one barrier a k-step that waits for LDS only.
// What bounds it: issue.  An element's split is 5.5 VALU instructions (and its row's largest magnitude half of one, not counted here), a wave of eight in the 128 x 128
// tile has 88 of them and 48 MFMAs a step, two waves to a SIMD: 1200 clocks of the one, 1536 of the other, of which next to nothing overlaps (1.39 us a step; the two from different waves: 1.57 of what the slower
// takes).  Products first and then the splits, in every order that was tried, is as good as any finer mix of them (interleaved by hand 49, by the compiler
// 46, this 45 us where one is 1024 deep).
#include <type_traits>

#include "pb_linear_epi.h"
#include "pb_linear_tiles.h"

namespace {
using namespace pcb;

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f4 mma3(const u32x4& w, const u32x4& x, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, w), __builtin_bit_cast(b8, x), c, 0, 0, 0);
}

template <int EPI, int TM, int TN, int WN>
__global__ __launch_bounds__(128 * WN) void linear_split_kernel(pcb_linear_args a) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int BM = 32 * TM, BN = 16 * WN * TN, ROWS = BM + (TWO ? 2 : 1) * BN, RI = 16 * WN, NC = ROWS / RI, NB = TWO ? 2 * TN : TN;
    static_assert(ROWS % RI == 0 && BM % RI == 0, "whole chunks");
    __shared__ __attribute__((aligned(16))) char img[2][3][ROWS * 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN, g = lane >> 4, l15 = lane & 15;
    const int K = a.K, N = a.N;

    const int mb = (a.M + BM - 1) / BM, tiles = mb * ((N + BN - 1) / BN), per = (tiles + 7) / 8;
    const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);        // (tiles panel by panel, each XCD one run of them)
    if ((int)(blockIdx.x >> 3) >= per || t >= tiles) return;
    const int m_lo = t % mb * BM, m_hi = a.M, n_lo = t / mb * BN, z = a.n_batch > 0 ? blockIdx.z : 0;
    const float* W = (const float*)a.w + z * a.w_group_stride;
    const float* W2 = TWO ? (const float*)a.w2 + z * a.w_group_stride : nullptr;
    const float* X = (const float*)a.x + z * a.x_batch_stride;
    auto xrow = [&](int r) {                                         // image row r < BM (rows past the end repeat the last one: not stored)
        const int m = m_lo + r < m_hi ? m_lo + r : m_hi - 1;
        return X + (int64_t)(a.row_src ? a.row_src[m] : m) * a.ldx;
    };
    auto wrow = [&](int c) {                                         // weight row c of the image; gated: BN of W, BN of W2
        const bool second = TWO && c >= BN;
        const int n = n_lo + c - (second ? BN : 0);
        return (second ? W2 : W) + (int64_t)(n < N ? n : N - 1) * a.ldw;
    };
    // a thread's chunk i: four elements of image row RI i + tid / 8
    const int sr = tid >> 3, sk = 4 * (tid & 7);
    const float* src[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) src[i] = RI * i < BM ? xrow(RI * i + sr) : wrow(RI * i + sr - BM);
    // (always loaded, chunks past K from the row's last four: a load under a branch is waited for where the branches meet)
    f4 raw[2][NC];                                                   // k-steps of either parity
    auto load = [&](f4& to, int i, int step) {
        const int k = 32 * step + sk;
        to = *reinterpret_cast<const f4*>(src[i] + (k < K ? k : K - 4));
    };
    const int at = sr * 64 + (((tid & 7) >> 1) ^ ((sr >> 2) & 3)) * 16 + (tid & 1) * 8;
    // part q of a chunk, what it leaves stays (the 16-byte chunk c of row r lies at c ^ (r / 4 & 3): a fragment read touches every bank slot)
    float top[NC];                                                   // the largest magnitude of each chunk's elements so far
#pragma unroll
    for (int i = 0; i < NC; ++i) top[i] = 0.0f;
    auto peak = [&](const f4& r, int i, int h) {                     // half h of a chunk (a NaN is passed over: its sums are no numbers either)
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top[i]) : "v"(r[2 * h]), "v"(r[2 * h + 1]));
    };
    auto store = [&](f4& r, int i, int q, int buf) {
        const uint2 p = {bf16_pair(r[0], r[1]), bf16_pair(r[2], r[3])};
        if (q < 2) {
            r[0] -= __uint_as_float(p.x << 16);
            r[1] -= __uint_as_float(p.x & 0xffff0000u);
            r[2] -= __uint_as_float(p.y << 16);
            r[3] -= __uint_as_float(p.y & 0xffff0000u);
        }
        *reinterpret_cast<uint2*>(&img[buf][q][RI * i * 64 + at]) = p;
    };
    f4 big[TM][NB], small[TM][NB];                                   // hi hi; the five others
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) big[i][j] = small[i][j] = f4{0.f, 0.f, 0.f, 0.f};
    const int steps = (K + 31) / 32;
    const int fo = l15 * 64 + ((g ^ ((l15 >> 2) & 3)) << 4);
    u32x4 fa[TM][3], fb[NB][3];
    auto read = [&](int buf) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i][q] = *reinterpret_cast<const u32x4*>(&img[buf][q][(wm * TM + i) * 1024 + fo]);
#pragma unroll
            for (int j = 0; j < NB; ++j)
                fb[j][q] = *reinterpret_cast<const u32x4*>(&img[buf][q][(BM / 16 + (j >= TN ? WN * TN : 0) + wn * TN + j % TN) * 1024 + fo]);
        }
    };
    // product k of the six of every pair of blocks: the small ones of a kind one after the other, so that no two neighbours add to the same sum
    constexpr int MF = 6 * TM * NB, FROM = MF - 2 * NC;
    // Where a chunk's largest magnitude is taken: behind the last products, one instruction each, ahead of the chunk's split where there are few products.  us, behind /
    // ahead, K = 4096: 128 x 128 tiles 167 / 172 (without 167), 64 x 128 107.5 / 109 (102.5), 64 x 64 71.2 / 70.0 (68.3); ahead of the products, while their
    // operands come from LDS, 169.7, 107.5, 73.4.
    constexpr bool BEHIND = MF >= 24;
    auto product = [&](int k) {
        const int kind = k / (TM * NB), j = k / TM % NB, i = k % TM;
        const int w = kind == 0 ? 2 : kind == 3 || kind == 4 ? 1 : 0, x = kind == 1 ? 2 : kind == 3 || kind == 5 ? 1 : 0;
        f4& c = kind == 2 ? big[i][j] : small[i][j];
        c = mma3(fb[j][w], fa[i][x], c);
    };
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };   // (LDS only: the loads under way go on)
    // k-step s of parity P, behind its products the parts of step s + 1 and the loads of step s + 3
    auto stage = [&](auto parity, int s) {
        constexpr int P = decltype(parity)::value;
        meet();
        read(P);
        auto unit = [&](int u) {
            if (!BEHIND && u % 3 == 0) peak(raw[1 - P][u / 3], u / 3, 0), peak(raw[1 - P][u / 3], u / 3, 1);
            store(raw[1 - P][u / 3], u / 3, u % 3, 1 - P);
            if (u % 3 == 2) load(raw[1 - P][u / 3], u / 3, s + 3 < steps ? s + 3 : steps - 1);
        };
#pragma unroll
        for (int k = 0; k < MF; ++k) {
            product(k);
            if (BEHIND && k >= FROM) {
                __builtin_amdgcn_sched_barrier(0);
                peak(raw[1 - P][(k - FROM) / 2], (k - FROM) / 2, (k - FROM) & 1);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 3 * NC; ++u) unit(u);
    };
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        load(raw[0][i], i, 0);
        load(raw[1][i], i, steps > 1 ? 1 : 0);
    }
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        for (int h = 0; h < 2; ++h) peak(raw[0][i], i, h);
#pragma unroll
        for (int q = 0; q < 3; ++q) store(raw[0][i], i, q, 0);
        load(raw[0][i], i, steps > 2 ? 2 : steps - 1);
    }
    for (int s = 0; s + 1 < steps; s += 2) {
        stage(std::integral_constant<int, 0>{}, s);
        if (s + 2 >= steps) break;
        stage(std::integral_constant<int, 1>{}, s + 1);
    }
    meet();
    read((steps - 1) & 1);
    if (K % 32 != 0) {                                               // zeros for what lies past K (K is a multiple of four)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (8 * g + 2 * e >= K % 32) fa[i][q][e] = 0u;
    }
#pragma unroll
    for (int k = 0; k < MF; ++k) product(k);
    // What is no number here may have a sum: the parts of an infinity (or of a value that rounds to one) make NaN.  And what the parts of a sum's elements leave out,
    // 2^-134 of each at most, is K 2^-133 times the largest element of its row and column: results below 2^26 times that would show it (rows of zeros aside).  A wave
    // that has such a result works its blocks out on the fp32 matrix cores and takes it from there: a result depends on its own row and column alone.
    // What that costs, us: nothing but NaN 600 x 5136, K = 1024 134, 2048 x 2048 x 2048 257 (numbers: 54, 96; fp32 matrix cores from the start 78, 147).  Without and with
    // the maxima and this look: 2048 columns and K, 2048 rows 95.8 / 96.7, 600 x 2560, K = 1024 29.9 / 31.0, 600 x 5136 48.0 / 47.5, 400 x 2048 20.0 / 20.8.
    __shared__ __attribute__((aligned(16))) float tops[ROWS];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        float t = top[i];
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) t = fmaxf(t, __shfl_xor(t, o, 64));
        if ((tid & 7) == 0) tops[RI * i + sr] = t;
    }
    __syncthreads();
    // (first against the largest bound of a lane's results, a NaN through a sum of zeros)
    f4 v[TM][NB], tw[NB];
    float tx[TM], most = 0.0f, least = __builtin_inff(), none = 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i) most = fmaxf(most, tx[i] = tops[(wm * TM + i) * 16 + l15]);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        tw[j] = *reinterpret_cast<const f4*>(&tops[BM + (j >= TN ? BN : 0) + (wn * TN + j % TN) * 16 + 4 * g]);
        most = fmaxf(fmaxf(fmaxf(most, tw[j][0]), fmaxf(tw[j][1], tw[j][2])), tw[j][3]);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            v[i][j] = big[i][j] + small[i][j];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                least = fminf(least, fabsf(v[i][j][e]));
                none = __builtin_fmaf(v[i][j][e], 0.0f, none);
            }
        }
    const float share = (float)K * 0x1p-107f;
    auto lost = [&](int i, int j, int e) {
        const float r = fabsf(v[i][j][e]), x = tx[i], w = tw[j][e];
        return !(r <= 3.4028234663852886e38f) || (x > 0.0f && w > 0.0f && r < fmaxf(x, w) * share);
    };
    bool again = least < most * share || !(none == 0.0f);
    if (__any(again)) {
        again = false;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) again = again || lost(i, j, e);
    }
    if (__any(again)) {
        const float *xs[TM], *ws[NB];
#pragma unroll
        for (int i = 0; i < TM; ++i) xs[i] = xrow((wm * TM + i) * 16 + l15) + 4 * g;
#pragma unroll
        for (int j = 0; j < NB; ++j) ws[j] = wrow((j >= TN ? BN : 0) + (wn * TN + j % TN) * 16 + l15) + 4 * g;
        f4 nx[TM], nw[NB];
        auto ask = [&](int k) {                                      // (past K the first ones again, not counted)
            const int at = k + 4 * g < K ? k : -4 * g;
#pragma unroll
            for (int i = 0; i < TM; ++i) nx[i] = *reinterpret_cast<const f4*>(xs[i] + at);
#pragma unroll
            for (int j = 0; j < NB; ++j) nw[j] = *reinterpret_cast<const f4*>(ws[j] + at);
        };
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) big[i][j] = small[i][j] = f4{0.f, 0.f, 0.f, 0.f};
        ask(0);
#pragma unroll 1
        for (int k = 0; k < K; k += 16) {                            // (a lane's four elements are the k of four products; even and odd in sums of their own)
            const bool in = k + 4 * g < K;
            f4 x[TM], w[NB];
#pragma unroll
            for (int i = 0; i < TM; ++i) x[i] = in ? nx[i] : f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NB; ++j) w[j] = in ? nw[j] : f4{0.f, 0.f, 0.f, 0.f};
            if (k + 16 < K) ask(k + 16);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j) {
                        f4& c = e & 1 ? small[i][j] : big[i][j];
                        c = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j][e], x[i][e], c, 0, 0, 0);
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[i][j][e] = lost(i, j, e) ? big[i][j][e] + small[i][j][e] : v[i][j][e];
    }
    f4 acc[TM][TN], acc2[TWO ? TM : 1][TWO ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = v[i][j];
            if (TWO) acc2[TWO ? i : 0][TWO ? j : 0] = v[i][TN + j];
        }
    finish_tile<float, EPI, TM, TN, WN>(a, acc, acc2, m_lo, m_hi, n_lo, wm, wn, g, l15);
}

template <int EPI, int TM, int TN, int WN>
int launch(const pcb_linear_args& a, hipStream_t stream) {
    const int64_t tiles = (int64_t)pcb_ceil_div(a.N, 16 * WN * TN) * pcb_ceil_div(a.M, 32 * TM);
    hipLaunchKernelGGL((linear_split_kernel<EPI, TM, TN, WN>), dim3((uint32_t)(8 * ((tiles + 7) / 8)), 1, a.n_batch > 0 ? a.n_batch : 1), dim3(128 * WN), 0, stream, a);
    return pcb_check_launch("linear_split_kernel");
}

// workgroups of rows x cols (cols: weight rows) tiles
int64_t tiles_of(const pcb_linear_args& a, int rows, int cols) {
    const int W = a.epilogue == PCB_EPI_SILU_MUL ? 2 : 1;
    return (int64_t)pcb_ceil_div(a.M, rows) * pcb_ceil_div(W * a.N, cols) * (a.n_batch > 0 ? a.n_batch : 1);
}

// The tile whose workgroups on the fullest CU cost least, us a k-step of 32: one, two, .. eight of 64 x 64 0.56, 1.02, .. 4.06 (gated, four waves: 0.66, 1.03,
// .. 3.75), of 64 x 128 0.86, 1.83, .. 7.9, of 128 x 128 1.42, 3.0, 4.6, 6.4 -- the larger, the fewer splits a product.  At 570 sizes (100 .. 2048 rows, 512 ..
// 10272 columns, K = 256 .. 2048) on average 0.3 % from the fastest of them.
enum Shape { SMALL = 1, WIDE, LARGE };
Shape shape_of(const pcb_linear_args& a) {
    auto on_a_cu = [&](int rows, int cols) { return (float)((tiles_of(a, rows, cols) + 255) / 256); };
    const bool gated = a.epilogue == PCB_EPI_SILU_MUL;
    const float large = 1.45f * on_a_cu(128, 128), wide = 0.885f * on_a_cu(64, 128), small = gated ? 0.24f + 0.44f * on_a_cu(64, 64) : 0.52f * on_a_cu(64, 64);
    return large <= wide && large <= small ? LARGE : wide <= small ? WIDE : SMALL;
}

template <int EPI>
int dispatch(const pcb_linear_args& a, hipStream_t stream) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    switch (shape_of(a)) {
        case LARGE: return launch<EPI, 4, TWO ? 1 : 2, 4>(a, stream);
        case WIDE: return launch<EPI, 2, TWO ? 1 : 2, 4>(a, stream);
        default: return launch<EPI, 2, 1, TWO ? 2 : 4>(a, stream);
    }
}

}  // namespace

// From 145 tiles of 64 x 64 on (128 of them 0.70 .. 0.90 of the fp32 matrix cores' speed: tiles of 32 x 32 there, on all CUs), where the launch takes less by this
// estimate than by fp32_us() (pb_linear.hip): fitted to 2080 sizes of 17 .. 2048 rows, 145 .. 2048 such tiles, K = 256 .. 2048, plain and gated.  Slower than the fp32 matrix
// cores by more than 4 % at five of them (splitting whatever has 145 tiles: at 468, by up to half: 32 rows of 65920 columns, K = 1024 57.4 / 84.5, 600 x 1664 -- two
// rounds of the chip -- 26.7 / 32.3), on average 0.2 % behind the better of the two.  600 x 5136, K = 1024 78 -> 47.5 us, the gated pair of 2048 60 -> 46.3,
// 2048 x 2048 x 2048 147 -> 96.
bool pcb_linear_split_fits(const pcb_linear_args& a) { return a.n_groups == 0 && tiles_of(a, 64, 64) > 144; }

int pcb_linear_split_shape(const pcb_linear_args& a) { return shape_of(a); }

float pcb_linear_split_us(const pcb_linear_args& a) {
    const bool gated = a.epilogue == PCB_EPI_SILU_MUL;
    const float steps = (float)((a.K + 31) / 32);
    auto on_a_cu = [&](int rows, int cols) { return (float)((tiles_of(a, rows, cols) + 255) / 256); };
    switch (shape_of(a)) {
        case LARGE: return (1.29f * steps + 4.5f) * on_a_cu(128, 128) + 5.0f;
        case WIDE: return gated ? (0.765f * steps + 3.3f) * on_a_cu(64, 128) + 4.2f : (0.81f * steps + 2.4f) * on_a_cu(64, 128) + 4.7f;
        default:
            return gated ? (0.22f + 0.38f * on_a_cu(64, 64)) * steps + 6.2f + 0.75f * on_a_cu(64, 64) :
                           (0.045f + 0.425f * on_a_cu(64, 64)) * steps + 5.9f + 0.7f * on_a_cu(64, 64);
    }
}

int pcb_linear_split(const pcb_linear_args& a, hipStream_t stream) {
    switch (a.epilogue) {
        case PCB_EPI_STORE: return dispatch<PCB_EPI_STORE>(a, stream);
        case PCB_EPI_SILU_MUL: return dispatch<PCB_EPI_SILU_MUL>(a, stream);
        default: return dispatch<PCB_EPI_SCALE_ADD>(a, stream);
    }
}
