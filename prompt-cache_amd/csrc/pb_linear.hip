// pcb_linear: Y = A W^T for row-major activations and nn.Linear-layout weights in bf16 or fp32, with what decoder layers fuse
// around a projection: bias, gathered and scaled input rows, per-group weights (experts), a gated-unit epilogue, and the
// layer-scaled accumulation into an fp32 residual stream.
//
// Tiling: workgroup = 4 waves in a 2 x 2 grid, a wave owns TM x TN result tiles of 16 x 16, so the workgroup covers
// (32 TM) x (32 TN) of Y.  Per stage of two 32-element k-steps the A and B panels go global -> registers -> LDS (the next stage's
// loads are in flight while this stage's MFMAs run); waves read their operand fragments from LDS with one 16-byte read per fragment (bf16).
// Operands that can be read in 16-byte chunks take linear_dma_kernel below instead (large plain launches in bf16 pb_linear_tiles.hip, those of few tiles
// pb_linear_waves.hip); odd sizes
// and scaled rows this one.
#include <type_traits>

#include "pb_linear_parts.h"
#include "pb_linear_tiles.h"

namespace {
using namespace pcb;

template <typename E>
struct Tile {
    static constexpr int KS = sizeof(E) == 2 ? 2 : 1;   // 32-element k-steps per LDS stage (fp32 panels are twice as large)
    static constexpr int CE = 16 / sizeof(E);       // elements per 16-byte chunk
    static constexpr int CPR = 32 * KS / CE;         // chunks per staged row
    static constexpr int LD = 32 * KS + CE;          // LDS row stride in elements (16-byte aligned rows, skewed banks)
};

__device__ __forceinline__ u32x4 zero_chunk() { return u32x4{0u, 0u, 0u, 0u}; }

// one 16-byte chunk of row `p` (null: a row outside the matrix) starting at k element k, K elements in the row
template <typename E>
__device__ __forceinline__ u32x4 load_chunk(const E* p, int k, int K, bool vec, float scale, bool scaled) {
    constexpr int CE = Tile<E>::CE;
    u32x4 c = zero_chunk();
    if (p == nullptr || k >= K) return c;
    if (vec) {
        c = *reinterpret_cast<const u32x4*>(p + k);
    } else {
        __attribute__((aligned(16))) E tmp[CE];
#pragma unroll
        for (int e = 0; e < CE; ++e) tmp[e] = k + e < K ? p[k + e] : from_f32<E>(0.0f);
        c = *reinterpret_cast<u32x4*>(tmp);
    }
    if (scaled) {
        __attribute__((aligned(16))) E tmp[CE];
        *reinterpret_cast<u32x4*>(tmp) = c;
#pragma unroll
        for (int e = 0; e < CE; ++e) tmp[e] = from_f32<E>(scale * to_f32(tmp[e]));
        c = *reinterpret_cast<u32x4*>(tmp);
    }
    return c;
}

// the lane's elements of a whole k-step, p at element 0 of it in the lane's row (16-byte aligned): k elements 8 group .. + 7 in 16-byte reads.
// (Both operands use this map, so where an element sits in the k-step does not matter.  fp32 in the map of load_frag is eight 4-byte reads.)
__device__ __forceinline__ Frag<bf16_t> whole_frag(const bf16_t* p, int group) {
    Frag<bf16_t> f;
    f.v = *reinterpret_cast<const u32x4*>(p + 8 * group);
    return f;
}
__device__ __forceinline__ Frag<float> whole_frag(const float* p, int group) {
    Frag<float> f;
    const f4 lo = *reinterpret_cast<const f4*>(p + 8 * group), hi = *reinterpret_cast<const f4*>(p + 8 * group + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) f.v[e] = lo[e], f.v[4 + e] = hi[e];
    return f;
}

template <typename E, int EPI, int TM, int TN>
__global__ __launch_bounds__(256) void linear_kernel(pcb_linear_args a) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int BM = 32 * TM, BN = 32 * TN, BROWS = TWO ? 2 * BN : BN;
    constexpr int CE = Tile<E>::CE, CPR = Tile<E>::CPR, LD = Tile<E>::LD, KS = Tile<E>::KS;
    constexpr int A_CH = (BM * CPR + 255) / 256, B_CH = (BROWS * CPR + 255) / 256;
    __shared__ __attribute__((aligned(16))) E As[BM * LD];
    __shared__ __attribute__((aligned(16))) E Bs[BROWS * LD];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1, group = lane >> 4, l15 = lane & 15;
    const int K = a.K, N = a.N;

    // which rows: a plain launch tiles [0, M); a grouped launch walks the group offsets to find its group and tile
    int g = 0, m_lo, m_hi;
    if (a.n_groups > 0) {
        int t = blockIdx.y;
        m_lo = -1;
        for (g = 0; g < a.n_groups; ++g) {
            const int lo = a.group_off[g], hi = a.group_off[g + 1];
            const int nt = (hi - lo + BM - 1) / BM;
            if (t < nt) {
                m_lo = lo + t * BM;
                m_hi = hi;
                break;
            }
            t -= nt;
        }
        if (m_lo < 0) return;
    } else {
        m_lo = blockIdx.y * BM;
        m_hi = a.M;
        if (a.n_batch > 0) g = blockIdx.z;
        if (m_lo >= m_hi) return;
    }
    const int n_lo = blockIdx.x * BN;
    const E* W = (const E*)a.w + (int64_t)g * a.w_group_stride;
    const E* W2 = TWO ? (const E*)a.w2 + (int64_t)g * a.w_group_stride : nullptr;
    const E* X = (const E*)a.x + (a.n_batch > 0 ? (int64_t)blockIdx.z * a.x_batch_stride : 0);
    const bool vec = (K % CE == 0) && (a.ldx % CE == 0) && (a.ldw % CE == 0) && (((uintptr_t)X | (uintptr_t)W | (uintptr_t)W2) % 16 == 0);
    const bool scaled = a.row_scale != nullptr;

    // this thread's chunks of the two panels
    const E* a_row[A_CH];
    float a_scale[A_CH];
    int a_k[A_CH], a_at[A_CH];
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
        const int c = tid + 256 * i, r = c / CPR;
        a_k[i] = (c % CPR) * CE;
        a_at[i] = c < BM * CPR ? r * LD + a_k[i] : -1;
        const int m = m_lo + r;
        a_row[i] = nullptr;
        a_scale[i] = 1.0f;
        if (c < BM * CPR && m < m_hi) {
            a_row[i] = X + (int64_t)(a.row_src ? a.row_src[m] : m) * a.ldx;
            if (scaled) a_scale[i] = a.row_scale[m];
        }
    }
    const E* b_row[B_CH];
    int b_k[B_CH], b_at[B_CH];
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
        const int c = tid + 256 * i, r = c / CPR;
        b_k[i] = (c % CPR) * CE;
        b_at[i] = c < BROWS * CPR ? r * LD + b_k[i] : -1;
        const E* base = (TWO && r >= BN) ? W2 : W;
        const int n = n_lo + (TWO && r >= BN ? r - BN : r);
        b_row[i] = (c < BROWS * CPR && n < N) ? base + (int64_t)n * a.ldw : nullptr;
    }

    f4 acc[TM][TN], acc2[TWO ? TM : 1][TWO ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = f4{0.f, 0.f, 0.f, 0.f};
            if (TWO) acc2[i][j] = f4{0.f, 0.f, 0.f, 0.f};
        }

    u32x4 ra[A_CH], rb[B_CH];
#pragma unroll
    for (int i = 0; i < A_CH; ++i) ra[i] = load_chunk<E>(a_row[i], a_k[i], K, vec, a_scale[i], scaled);
#pragma unroll
    for (int i = 0; i < B_CH; ++i) rb[i] = load_chunk<E>(b_row[i], b_k[i], K, vec, 1.0f, false);

    for (int k0 = 0; k0 < K; k0 += 32 * KS) {
        __syncthreads();                           // the previous stage's fragment reads are done
#pragma unroll
        for (int i = 0; i < A_CH; ++i)
            if (a_at[i] >= 0) *reinterpret_cast<u32x4*>(&As[a_at[i]]) = ra[i];
#pragma unroll
        for (int i = 0; i < B_CH; ++i)
            if (b_at[i] >= 0) *reinterpret_cast<u32x4*>(&Bs[b_at[i]]) = rb[i];
        __syncthreads();
        if (k0 + 32 * KS < K) {
#pragma unroll
            for (int i = 0; i < A_CH; ++i) ra[i] = load_chunk<E>(a_row[i], k0 + 32 * KS + a_k[i], K, vec, a_scale[i], scaled);
#pragma unroll
            for (int i = 0; i < B_CH; ++i) rb[i] = load_chunk<E>(b_row[i], k0 + 32 * KS + b_k[i], K, vec, 1.0f, false);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            Frag<E> fa[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i] = load_frag(&As[((wm * TM + i) * 16 + l15) * LD + 32 * ks], group, 32, true);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const Frag<E> fb = load_frag(&Bs[((wn * TN + j) * 16 + l15) * LD + 32 * ks], group, 32, true);
#pragma unroll
                for (int i = 0; i < TM; ++i) acc[i][j] = mma(fa[i], fb, acc[i][j]);
                if (TWO) {
                    const Frag<E> fb2 = load_frag(&Bs[(BN + (wn * TN + j) * 16 + l15) * LD + 32 * ks], group, 32, true);
#pragma unroll
                    for (int i = 0; i < TM; ++i) acc2[i][j] = mma(fa[i], fb2, acc2[i][j]);
                }
            }
        }
    }

    const E* bias = (const E*)a.bias;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n_lo + (wn * TN + j) * 16 + l15;
        if (n >= N) continue;
        const float bv = bias ? to_f32(bias[n]) : 0.0f;
        const float bv2 = (TWO && a.bias2) ? to_f32(((const E*)a.bias2)[n]) : 0.0f;
        const float cs = (EPI == PCB_EPI_SCALE_ADD) ? a.col_scale[n] : 0.0f;
        Place to[TM][4];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m_lo + (wm * TM + i) * 16 + 4 * group + r;
                to[i][r] = place<E, EPI>(a, m < m_hi ? m : m_hi - 1, n);
            }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (m_lo + (wm * TM + i) * 16 + 4 * group + r < m_hi)
                    put<E, EPI>(to[i][r], finished<E, EPI>(a, to[i][r], n, acc[i][j][r], TWO ? acc2[i][j][r] : 0.0f, bv, bv2), cs);
    }
}

// ---- few rows: the weights stream once, straight from memory into the matrix cores --------------------------------------------
// Workgroup = 16 result columns x up to 16 rows; its SKW waves split the k range (k-step s goes to wave s % SKW) and add their
// partial tiles through LDS.  No LDS staging: a lane's B fragment is 16 contiguous bytes of its weight row (fp32: 32), its A fragment as many of
// its activation row (a handful of rows that stay in cache).  Bound by the launch and one trip to memory at 4 MB of weights, by the stream at
// 40 (10 272 x 2 048 bf16, 8 rows: 12.6 us, 3.3 TB/s).  fp32 in 16-byte reads instead of 4-byte ones, us: 1 row, 1024 x 1024 10.0 -> 5.6,
// 1024 x 4096 32.6 -> 13.4, 5136 x 1024 18.2 -> 9.5, 8 rows 27.6 -> 10.4.
template <typename E>
__device__ __forceinline__ void scale_frag(Frag<E>& f, float s);
template <>
__device__ __forceinline__ void scale_frag<bf16_t>(Frag<bf16_t>& f, float s) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t w = f.v[e];
        f.v[e] = bf16_pair(s * __uint_as_float(w << 16), s * __uint_as_float(w & 0xffff0000u));
    }
}
template <>
__device__ __forceinline__ void scale_frag<float>(Frag<float>& f, float s) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f.v[e] *= s;
}

// SKW: waves of a workgroup (eight, or sixteen where few workgroups walk a long k range).  LATE (bf16): where a result goes is worked out when it
// is there, row by row.  Ahead of the products it hides its loads, but holds back the loads of the wave that stores, by 0.2-0.5 us a workgroup:
// a gain as long as no workgroup waits for another one's place on the chip.
template <typename E, int EPI, int SKW, bool LATE>
__global__ __launch_bounds__(64 * SKW) void linear_skinny_kernel(pcb_linear_args a) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int CE = Tile<E>::CE;
    __shared__ f4 red[TWO ? 2 : 1][SKW][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, group = lane >> 4, l15 = lane & 15;
    const int K = a.K, N = a.N;
    int g = 0, m_lo, m_hi;
    if (a.n_groups > 0) {
        int t = blockIdx.y;
        m_lo = -1;
        for (g = 0; g < a.n_groups; ++g) {
            const int lo = a.group_off[g], hi = a.group_off[g + 1];
            const int nt = (hi - lo + 15) / 16;
            if (t < nt) {
                m_lo = lo + t * 16;
                m_hi = hi;
                break;
            }
            t -= nt;
        }
        if (m_lo < 0) return;
    } else {
        m_lo = blockIdx.y * 16;
        m_hi = a.M;
        if (a.n_batch > 0) g = blockIdx.z;
        if (m_lo >= m_hi) return;
    }
    const int n_lo = blockIdx.x * 16;
    const E* W = (const E*)a.w + (int64_t)g * a.w_group_stride;
    const E* W2 = TWO ? (const E*)a.w2 + (int64_t)g * a.w_group_stride : nullptr;
    const E* X = (const E*)a.x + (a.n_batch > 0 ? (int64_t)blockIdx.z * a.x_batch_stride : 0);
    const bool vec = (K % CE == 0) && (a.ldx % CE == 0) && (a.ldw % CE == 0) && (((uintptr_t)X | (uintptr_t)W | (uintptr_t)W2) % 16 == 0);
    const int n_b = n_lo + l15, m_a = m_lo + l15;
    const bool b_ok = n_b < N, a_ok = m_a < m_hi;
    const E* wrow = W + (int64_t)(b_ok ? n_b : 0) * a.ldw;
    const E* wrow2 = TWO ? W2 + (int64_t)(b_ok ? n_b : 0) * a.ldw : nullptr;
    const E* xrow = X + (int64_t)(a_ok ? (a.row_src ? a.row_src[m_a] : m_a) : 0) * a.ldx;
    // (the wave that stores asks for everything the epilogue needs before the products, or before it waits for the other waves)
    constexpr bool ADD = EPI == PCB_EPI_SCALE_ADD;
    const int n_c = n_lo + l15 < N ? n_lo + l15 : N - 1;
    float bv = 0.0f, bv2 = 0.0f, cs = 0.0f;
    Place to[4] = {};
    auto columns = [&] {
        if (a.bias) bv = to_f32(((const E*)a.bias)[n_c]);
        if (TWO && a.bias2) bv2 = to_f32(((const E*)a.bias2)[n_c]);
        if (ADD) cs = a.col_scale[n_c];
    };
    auto places = [&] {
        columns();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m_lo + 4 * group + r;
            if (TWO || m < m_hi) to[r] = place<E, EPI>(a, m < m_hi ? m : m_hi - 1, n_c);
        }
    };
    if (!LATE && wave == 0) places();
    const bool scaled = a.row_scale != nullptr;
    const float xs = (scaled && a_ok) ? a.row_scale[m_a] : 1.0f;
    Sum<E> sum, sum2;
    const int nsteps = (K + 31) / 32;
    // whole k-steps of rows that can be read in 16-byte pieces: nothing between the loads.  (Lanes past the last row or column read row 0
    // or column 0 instead: what they multiply is not stored.)
    int st = wave;
    if (vec && !scaled) {
        const int whole = K / 32;
#pragma unroll 8
        for (; st < whole; st += SKW) {
            const Frag<E> fa = whole_frag(xrow + 32 * st, group), fb = whole_frag(wrow + 32 * st, group);
            sum.add(fa, fb);
            if (TWO) sum2.add(fa, whole_frag(wrow2 + 32 * st, group));
        }
    }
#pragma unroll 2
    for (; st < nsteps; st += SKW) {
        const int k0 = 32 * st;
        Frag<E> fa = load_frag(xrow + k0, group, a_ok ? K - k0 : 0, vec);
        if (scaled) scale_frag<E>(fa, xs);
        const Frag<E> fb = load_frag(wrow + k0, group, b_ok ? K - k0 : 0, vec);
        sum.chain(fa, fb);
        if (TWO) sum2.chain(fa, load_frag(wrow2 + k0, group, b_ok ? K - k0 : 0, vec));
    }
    f4 acc = sum.total(), acc2 = sum2.total();
    if (LATE && ADD && wave == 0) places();
    red[0][wave][lane] = acc;
    if (TWO) red[1][wave][lane] = acc2;
    __syncthreads();
    if (wave != 0) return;
    acc = red[0][0][lane];
    if (TWO) acc2 = red[1][0][lane];
#pragma unroll
    for (int w = 1; w < SKW; ++w) {
        acc += red[0][w][lane];
        if (TWO) acc2 += red[1][w][lane];
    }
    const int n = n_lo + l15;
    if (n >= N) return;
    if (LATE && !ADD) columns();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = m_lo + 4 * group + r;
        if (m < m_hi) {
            if (LATE && !ADD) to[r] = place<E, EPI>(a, m, n);
            put<E, EPI>(to[r], finished<E, EPI>(a, to[r], n, acc[r], acc2[r], bv, bv2), cs);
        }
    }
}

// The few-row products of pb_linear_parts.h, a launch of their own.  LATE: as above.
// (few_rows() below says which launches take it, and what both cost)
template <typename E, int EPI, int PARTS, int U, bool LATE, int G, bool ONCE>
__global__ __launch_bounds__(512) void linear_parts_kernel(pcb_linear_args a) {
    __shared__ f4 red[EPI == PCB_EPI_SILU_MUL ? 2 * G : G][8][64];
    parts_block<E, EPI, PARTS, U, LATE, G, ONCE, sizeof(E) == 4 && EPI == PCB_EPI_SILU_MUL && PARTS == 1>(a, blockIdx.x, red);
}

// ---- many rows: both panels travel to LDS by themselves ------------------------------------------------------------------------------
// The same tiles (2 x 2 waves of TM x TN result tiles) for operands whose rows can be read in 16-byte chunks: global_load_lds carries a
// stage of 128 bytes of k (64 elements of bf16, 32 of fp32; 1 KiB per wave instruction: 8 rows) straight into a ring of two or three images, one
// barrier per stage, so no register and no branch stands between the loads.  Rows past the end repeat the last one (their results are not
// stored); chunks past K come from a block of zeros.  The 16-byte chunk c of row r sits at position c ^ ((r >> 1) & 7) of its 128-byte row,
// which spreads a fragment read over all banks; the loads write lane by lane, so the permutation is applied to each lane's source.
// A plain launch numbers its tiles panel by panel (all row blocks of a column panel in turn) and gives each XCD one run of them: a
// panel's weights are fetched into one L2.
// fp32 through here instead of linear_kernel (one stage in registers, fragments in eight 4-byte LDS reads), us: 600 rows, 2048 x 2048 257 -> 68,
// 1024 x 1024 120 -> 26, 1024 x 4096 470 -> 91, 5136 x 1024 141 -> 79; 2048 x 2048 x 2048 267 -> 149 (0.115 of 0.157 PFLOP/s).
__device__ const u32x4 zero_row = {0u, 0u, 0u, 0u};

__device__ __forceinline__ void dma16(const void* g, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g, (__attribute__((address_space(3))) void*)lds_wave_base, 16,
                                     0, 0);
}

template <typename E, int EPI, int TM, int TN, int STAGES>
__global__ __launch_bounds__(256) void linear_dma_kernel(pcb_linear_args a) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int BM = 32 * TM, BN = 32 * TN, ROWS = BM + (TWO ? 2 : 1) * BN, CE = Tile<E>::CE, BK = 8 * CE;
    constexpr int NI = ROWS / 32;                                    // wave instructions per wave and stage
    __shared__ __attribute__((aligned(16))) E img[STAGES][ROWS * BK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1, group = lane >> 4, l15 = lane & 15;
    const int K = a.K, N = a.N;

    int g = 0, m_lo = -1, m_hi = 0, n_lo;
    if (a.n_groups > 0) {
        int t = blockIdx.y;
        for (g = 0; g < a.n_groups; ++g) {
            const int lo = a.group_off[g], hi = a.group_off[g + 1];
            const int nt = (hi - lo + BM - 1) / BM;
            if (t < nt) {
                m_lo = lo + t * BM;
                m_hi = hi;
                break;
            }
            t -= nt;
        }
        if (m_lo < 0) return;
        n_lo = blockIdx.x * BN;
    } else {
        const int mb = (a.M + BM - 1) / BM, total = mb * ((N + BN - 1) / BN), per = (total + 7) / 8;
        const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
        m_lo = t % mb * BM;
        m_hi = a.M;
        n_lo = t / mb * BN;
        if (a.n_batch > 0) g = blockIdx.z;
    }
    const E* W = (const E*)a.w + (int64_t)g * a.w_group_stride;
    const E* W2 = TWO ? (const E*)a.w2 + (int64_t)g * a.w_group_stride : nullptr;
    const E* X = (const E*)a.x + (a.n_batch > 0 ? (int64_t)blockIdx.z * a.x_batch_stride : 0);

    // instruction i of this wave fills rows 8 (4 i + wave) .. + 7 of the image: A rows, then W rows, then W2 rows
    const E* src[NI];
    int kc[NI];                                                      // the lane's k offset within the stage
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = 8 * (4 * i + wave) + (lane >> 3);
        kc[i] = ((lane & 7) ^ ((r >> 1) & 7)) * CE;
        if (32 * i < BM) {
            int m = m_lo + r;
            m = m < m_hi ? m : m_hi - 1;
            src[i] = X + (int64_t)(a.row_src ? a.row_src[m] : m) * a.ldx;
        } else {
            const bool second = TWO && 32 * i >= BM + BN;
            int n = n_lo + r - BM - (second ? BN : 0);
            n = n < N ? n : N - 1;
            src[i] = (second ? W2 : W) + (int64_t)n * a.ldw;
        }
    }
    auto fetch = [&](int k0, int buf) {
        if (k0 + BK <= K) {
#pragma unroll
            for (int i = 0; i < NI; ++i) dma16(src[i] + k0 + kc[i], &img[buf][(4 * i + wave) * 8 * BK]);
        } else {
#pragma unroll
            for (int i = 0; i < NI; ++i)
                dma16(k0 + kc[i] < K ? (const void*)(src[i] + k0 + kc[i]) : (const void*)&zero_row, &img[buf][(4 * i + wave) * 8 * BK]);
        }
    };
    Sum<E> sum[TM][TN], sum2[TWO ? TM : 1][TWO ? TN : 1];
    // the lane's k elements 8 group .. + 7 of a 32-deep step: one chunk in bf16, two in fp32
    auto frag = [&](int buf, int r, int ks) {
        Frag<E> f;
        const E* row = &img[buf][r * BK];
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
    // STAGES - 1 stages are in flight: at the top of a step the wave waits for its own part of the stage at hand (loads land in order),
    // the barrier then says that everyone's has landed and that the buffer of the step before is read out
#pragma unroll
    for (int p = 0; p < STAGES - 1; ++p)
        if (p * BK < K) fetch(p * BK, p);
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += BK, buf = buf + 1 == STAGES ? 0 : buf + 1) {
        if (STAGES > 2 && k0 + BK < K)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * NI) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (k0 + (STAGES - 1) * BK < K) fetch(k0 + (STAGES - 1) * BK, buf == 0 ? STAGES - 1 : buf - 1);
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) {
            Frag<E> fa[TM];
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i] = frag(buf, (wm * TM + i) * 16 + l15, ks);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const Frag<E> fb = frag(buf, BM + (wn * TN + j) * 16 + l15, ks);
#pragma unroll
                for (int i = 0; i < TM; ++i) sum[i][j].add(fb, fa[i]);
                if (TWO) {
                    const Frag<E> fb2 = frag(buf, BM + BN + (wn * TN + j) * 16 + l15, ks);
#pragma unroll
                    for (int i = 0; i < TM; ++i) sum2[i][j].add(fb2, fa[i]);
                }
            }
        }
    }

    f4 acc[TM][TN], acc2[TWO ? TM : 1][TWO ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = sum[i][j].total();
            if (TWO) acc2[i][j] = sum2[i][j].total();
        }
    finish_tile<E, EPI, TM, TN>(a, acc, acc2, m_lo, m_hi, n_lo, wm, wn, group, l15);
}

template <typename E, int EPI, int TM, int TN, int STAGES>
int launch_dma(const pcb_linear_args& a, hipStream_t stream) {
    constexpr int BM = 32 * TM, BN = 32 * TN;
    const int nb = pcb_ceil_div(a.N, BN), mb = pcb_ceil_div(a.M, BM);
    const dim3 grid = a.n_groups > 0 ? dim3(nb, mb + a.n_groups) : dim3(8 * pcb_ceil_div(nb * mb, 8), 1, a.n_batch > 0 ? a.n_batch : 1);
    hipLaunchKernelGGL((linear_dma_kernel<E, EPI, TM, TN, STAGES>), grid, dim3(256), 0, stream, a);
    return pcb_check_launch("linear_dma_kernel");
}

// whether every operand row can be read in 16-byte chunks
bool dma_ok(const pcb_linear_args& a) {
    const int ce = a.dtype == PCB_BF16 ? 8 : 4;
    return !a.row_scale && a.K % ce == 0 && a.ldx % ce == 0 && a.ldw % ce == 0 && a.w_group_stride % ce == 0 && a.x_batch_stride % ce == 0 &&
           ((uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)a.w2) % 16 == 0 && (int64_t)pcb_ceil_div(a.N, 32) * pcb_ceil_div(a.M, 32) < (1 << 30);
}

// fp32 (1 / 16 of the bf16 rate): bound by the matrix cores, so what counts is that all CUs have the same share of tiles.  Whole rounds of
// the 256 CUs times a tile's work; a 128 x 128 tile costs 3.8 of 64 x 64 and a 32 x 64 tile 0.575 (us, 64-, 128- and 32-row tiles):
// 2048 x 2048 x 2048 158 / 149 / 166, 4096 x 4096, K = 1024 299 / 276 / 317, 1200 x 4096, K = 2048 188 / 267 / 203, 600 x 2564, K = 1024
// 44 / 76 / 47, 600 x 2048, K = 2048 79 / 146 / 68, 130 x 1024, K = 1024 25 / 75 / 17.
// (32 x 32 tiles, three to a CU, up to 768 of them: 600 x 1024, K = 1024 25.8 -> 21.5, 300 x 1024 18.1 -> 16.3, 200 x 2564 26.5 -> 22.1, 600 x 512,
// K = 512 10.3 -> 9.6; 600 x 2564 (1539) 42.9, 45.1 so.  What is below a round of the chip or deep is with pb_linear_waves.hip.)
struct Fp32Tile {
    int rows;                                                        // (0: 32 x 32)
    float rounds;
};
Fp32Tile fp32_tile(const pcb_linear_args& a, int rows) {
    const int64_t batch = a.n_batch > 0 ? a.n_batch : 1, extra = a.n_groups / 2;      // (groups: part tiles)
    auto rounds = [&](int bm, int bn) { return (float)((batch * (pcb_ceil_div(a.M, bm) + extra) * pcb_ceil_div(a.N, bn) + 255) / 256); };
    const bool gated = a.epilogue == PCB_EPI_SILU_MUL;
    const int tnw = gated ? 2 : 4;
    if (!gated && a.n_groups == 0 && batch * pcb_ceil_div(a.M, 32) * pcb_ceil_div(a.N, 32) <= 768) return {0, rounds(32, 32)};
    const float large = 3.8f * rounds(128, 32 * tnw), mid = rounds(64, 16 * tnw), small = 0.575f * rounds(32, 16 * tnw);
    if (rows > 64 && large <= mid && large <= small) return {128, rounds(128, 32 * tnw)};
    return rows > 32 && mid <= small ? Fp32Tile{64, mid} : Fp32Tile{32, rounds(32, 16 * tnw)};
}

// What a plain or batched launch takes on the fp32 matrix cores, us, by its kernel's rounds of the chip and k-steps of 32 (fitted to 2080 sizes, within 10 %)
float fp32_us(const pcb_linear_args& a) {
    const float steps = (float)pcb_ceil_div(a.K, 32);
    if (pcb_linear_waves_fits(a)) return 0.22f * steps * (float)((pcb_linear_waves_tiles(a) * (a.n_batch > 0 ? a.n_batch : 1) + 255) / 256);
    const Fp32Tile t = fp32_tile(a, a.M);
    switch (t.rows) {
        case 0: return 0.16f * t.rounds * steps + 6.4f;
        case 128: return (0.25f + 1.92f * t.rounds) * steps + 6.4f + 2.3f * t.rounds;
        case 64: return (0.1f + 0.545f * t.rounds) * steps + 5.2f + 0.5f * t.rounds;
        default: return (0.07f + 0.29f * t.rounds) * steps + 5.0f + 0.25f * t.rounds;
    }
}

template <typename E, int EPI>
int dispatch_dma(const pcb_linear_args& a, int rows, hipStream_t stream) {
    // the largest tile that still gives every CU a workgroup; grouped launches count the tiles their rows fill
    constexpr int TNW = EPI == PCB_EPI_SILU_MUL ? 2 : 4;
    const int64_t batch = a.n_batch > 0 ? a.n_batch : 1;
    auto tiles = [&](int bm, int bn) { return batch * pcb_ceil_div(a.M, bm) * pcb_ceil_div(a.N, bn); };
    if constexpr (sizeof(E) == 4) {
        const Fp32Tile t = fp32_tile(a, rows);
        if constexpr (EPI != PCB_EPI_SILU_MUL)
            if (t.rows == 0) return launch_dma<E, EPI, 1, 1, 3>(a, stream);
        if (t.rows == 128) return launch_dma<E, EPI, 4, TNW, 2>(a, stream);
        return t.rows == 64 ? launch_dma<E, EPI, 2, TNW / 2, 3>(a, stream) : launch_dma<E, EPI, 1, TNW / 2, 3>(a, stream);
    }
    // (two workgroups of a CU hide each other's loads behind their products; a lone one needs a stage more in flight)
    if (rows > 64 && tiles(128, 32 * TNW) > 256) return launch_dma<E, EPI, 4, TNW, 2>(a, stream);
    if (rows > 64 && tiles(128, 32 * TNW) == 256) return launch_dma<E, EPI, 4, TNW, 3>(a, stream);
    if (rows > 32 && tiles(64, 32 * TNW) >= 400) return launch_dma<E, EPI, 2, TNW, 3>(a, stream);
    if (rows > 32) return launch_dma<E, EPI, 2, TNW / 2, 3>(a, stream);
    return launch_dma<E, EPI, 1, TNW / 2, 3>(a, stream);
}

template <typename E, int EPI, int TM, int TN>
int launch(const pcb_linear_args& a, hipStream_t stream) {
    constexpr int BM = 32 * TM, BN = 32 * TN;
    const dim3 grid(pcb_ceil_div(a.N, BN), pcb_ceil_div(a.M, BM) + (a.n_groups > 0 ? a.n_groups : 0), a.n_batch > 0 ? a.n_batch : 1);
    hipLaunchKernelGGL((linear_kernel<E, EPI, TM, TN>), grid, dim3(256), 0, stream, a);
    return pcb_check_launch("linear_kernel");
}

// Which kernel takes a launch of up to sixteen rows: parts runs of k side by side in linear_parts_kernel (0: linear_skinny_kernel), late: where results
// go is worked out behind the products.  Measured with weights from memory at 4067 points, 64 .. 32000 columns, K = 64 .. 8192, 1 to 16 rows, every
// epilogue, both types: on average 1.3 % behind the fastest of them all, nowhere more than 8 % behind linear_skinny_kernel.  us below: linear_skinny_kernel /
// one run / two / four, the faster of late and not.  (g1, g2, g4: workgroups of 16, 8 and 4 columns.)
struct FewRows {
    int parts;
    bool late;
    int blocks = 1;                                                  // blocks of 16 / parts columns a workgroup has
};
FewRows few_rows(const pcb_linear_args& a) {
    const bool bf = a.dtype == PCB_BF16, gated = a.epilogue == PCB_EPI_SILU_MUL, add = a.epilogue == PCB_EPI_SCALE_ADD;
    if (!pcb_linear_pieces(a)) return {0, false};
    const int64_t batch = a.n_batch > 0 ? a.n_batch : 1, g1 = batch * pcb_ceil_div(a.N, 16), g2 = batch * pcb_ceil_div(a.N, 8),
                  g4 = batch * pcb_ceil_div(a.N, 4);
    // Late beyond three workgroups a CU (the gated unit in bf16 two), stores in bf16 also over K >= 512.  bf16, 32000 x 512, 4 rows added: not late 11.7,
    // late 10.0; fp32 gated 11000 x 64 6.4, 7.6.
    const FewRows skinny = {0, false},
                  one = {1, (g1 > (gated && bf ? 512 : 768) && (bf || !gated || a.K >= 512)) || (bf && a.epilogue == PCB_EPI_STORE && a.K >= 512)};
    // gated, many columns over next to no k: fp32 11000 x 64 5.4 / 6.4
    if (gated && a.K < 128) return g1 > 512 ? skinny : one;
    // more than eight rows in bf16: the kernel above over a deep k of few columns (its sixteen waves) or of more than a round of the chip.  16 rows, K = 4096:
    // 2048 columns 11.3 / 12.2, 4096 13.7 / 13.3, 5120 19.8 / 22.2, gated 4096 20.3 / 21.8, 5120 34.8 / 31.6
    if (a.M > 8) return bf && a.K >= 2048 && (g1 <= (gated && a.K >= 4096 ? 256 : 192) || (g1 > 256 && !gated)) ? skinny : one;
    // four runs up to three workgroups a CU.  1 row bf16: 2048 x 4096 8.5 / 8.4 / 5.9 / 5.7, 3072 x 2048 6.2 / 5.7 / 5.6 / 5.1; 4 rows, 3072 x 2048 6.5 / 6.3 / 6.3 /
    // 6.2, gated 10.3 / 10.5 / 9.5 / 8.6, 3072 x 1024 5.6 / 4.5 / 4.9 / 4.8, gated 6.8 / 6.5 / 6.6 / 6.5; 1 row fp32 1024 x 2048 9.0 / 7.5 / 5.3 / 4.5
    const bool late = a.epilogue == PCB_EPI_STORE ? bf || a.M <= 2 : gated && bf;
    // Stores in bf16 of more than a round of eight columns each: two runs and as many blocks of them a workgroup, up to four (deeper k three), as keeps the share of
    // the busiest CU smallest, the more the better.  Times of the rule before, 8 rows, K = 2048: 2568 columns (2) 0.93, 5136 (3) 0.78, 7424 (4) 0.80, 10272 (3)
    // 0.76, 32000 (4) 0.72; K = 4096 0.94, 0.77, 0.92 (2), 0.82, 0.74 (2); K = 1024 1.0, 0.89, 0.84, 0.91, 0.79; 4 rows, K = 2048 0.93, 0.89, 0.90, 0.88, 0.86.  One and
    // two rows only over K <= 1024 (10272 columns 0.85, 32000 0.79; K = 2048 1.02, 1.01).
    if (bf && a.epilogue == PCB_EPI_STORE && a.n_batch == 0 && a.K % 64 == 0 && a.K >= 1024 && g2 > 256 && (a.M > 2 || a.K <= 1024))
        return {2, true, pcb_parts_blocks(g2, a.K).blocks};
    if (a.M <= 4 && a.K % 128 == 0 && a.K >= (gated && bf ? 2048 : 1024) && g4 <= (a.M <= 2 || gated || a.K >= 2048 ? 768 : 512)) return {4, late};
    // (From here on, in bf16: sums into rows, the gated unit, batches, and plain stores of one and two rows over K > 1024 or of no more than a round.)
    // Two runs, of more than four rows not where 16 columns each are one round of the chip and eight are two (there the kernel above over a deep k; stores of 8 rows
    // over K = 4096, which a batch has as well: 2048 columns 9.6 / 10.3 / 7.1, 2560 9.8 / 10.6 / 10.6, 4096 13.6 / 11.6 / 11.3, 8192 18.3 / 20.1 / 20.4, 16384 35.8 / 36.0 / 36.4)
    if (a.K % 64 != 0 || a.K < (bf ? 1024 : 512)) return one;
    if (a.M > 4 && !gated) {
        const bool hole = g2 > 256 && g2 <= 400;
        if (bf && a.K >= 4096 && (hole || (g2 > 768 && g2 <= 1400))) return skinny;
        if (hole) return one;
    }
    // ... and while the chip has places for them: accumulations in bf16 8 rows, 4096 x 1024 5.6 / 4.9 / 5.1, 8192 x 1024 6.7 / 7.0 / 7.5, 8192 x 2048 10.8 / 11.7 /
    // 11.5; stores in bf16 at any size (32000 x 2048, 1 row 30.0 / 27.8 / 23.6), batches of them up to six rows (the same columns, 5 rows 32.1 / 31.1 / 29.8, 8 rows 34.3 / 34.6 /
    // 35.1), in fp32 two (2 rows 33.7 / 27.0 / 26.4); fp32, K = 2048, 4 rows, 8192 columns 20.1 / 17.3 / 17.5, 8 rows, 6144 20.4 / 16.9 / 15.8, 8192 21.8 / 18.1 / 19.9; 4 rows added, K = 512, 4096
    // columns 5.7 / 5.0 / 5.2, 8192 7.3 / 6.4 / 6.9
    const bool any = bf ? (add ? a.K >= 2048 && a.M <= 4 : gated || a.M <= 6) : a.epilogue == PCB_EPI_STORE && a.M <= 2;
    const int64_t most = any ? INT64_MAX : add ? (a.K < (bf ? 2048 : 1024) ? 640 : bf || a.M > 4 ? 768 : 1024) : bf || a.M <= 4 ? 1024 : 768;
    return g2 <= most ? FewRows{2, late} : one;
}

// Whether an fp32 launch of more than sixteen rows, read in 16-byte chunks, has its operands split (pb_linear_split.hip; at a tie, whose error is the smaller)
bool in_parts(const pcb_linear_args& a) { return pcb_linear_split_fits(a) && pcb_linear_split_us(a) < 1.01f * fp32_us(a); }

template <typename E>
int dispatch(const pcb_linear_args& a, hipStream_t stream) {
    // rows per group decide the row tile: many rows -> 128-row panels, few -> 32-row panels (the weights stream once)
    const int rows = a.n_groups > 0 ? pcb_ceil_div(a.M, a.n_groups) : a.M;
    // (a narrow result -- router logits, step sizes: N <= 64 -- takes the 32-row panels too: 128-row panels would leave M / 128
    // workgroups on the chip, each walking all of K)
    const bool big = rows > 64 && a.N > 64;
    if (rows <= 16) {
        const dim3 grid(pcb_ceil_div(a.N, 16), pcb_ceil_div(a.M, 16) + (a.n_groups > 0 ? a.n_groups : 0), a.n_batch > 0 ? a.n_batch : 1);
        const int64_t groups = (int64_t)grid.x * grid.y * grid.z;
        const bool deep = a.K >= 2048 && groups <= 192;
        // LATE beyond three workgroups a CU, of the gated unit over few k beyond four.  Of the launches that come this far (groups, odd rows, many columns
        // over a deep k), bf16, us, ahead of the products / late: stores 8 rows, 16384 x 1000 15.5 / 12.8, x 2024 28.8 / 22.1, x 4096 44.1 / 35.0, 32000 x 4096
        // 62.1 / 59.7; 8 groups of 2048 x 1024, one row each 13.4 / 10.2; accumulations 16384 x 1000 11.8 / 11.9, 32000 x 4096 64.4 / 59.5; gated, 1 row,
        // 16384 x 1000 23.4 / 22.2, 8 rows 26.2 / 25.7, 32000 x 2024 67.9 / 66.6, x 4096 111.6 / 117.9.
        const bool late = sizeof(E) == 2 && groups > (a.epilogue == PCB_EPI_SILU_MUL && a.K < 2048 ? 1024 : 768);
        const FewRows few = few_rows(a);
        if (few.parts > 0) {
            const bool once = pcb_weights_once((a.epilogue == PCB_EPI_SILU_MUL ? 2 : 1) * (int64_t)a.N, a.K, sizeof(E));
            auto launch = [&](auto epi, auto p, auto late, auto u, auto blocks) {
                constexpr int EPI = decltype(epi)::value, P = decltype(p)::value, G = decltype(blocks)::value;
                const dim3 grid(pcb_ceil_div(a.N, 16 / P * G), 1, a.n_batch > 0 ? a.n_batch : 1);
                if (P > 1 && once)
                    hipLaunchKernelGGL((linear_parts_kernel<E, EPI, P, decltype(u)::value, decltype(late)::value, G, (P > 1)>), grid, dim3(512), 0, stream, a);
                else
                    hipLaunchKernelGGL((linear_parts_kernel<E, EPI, P, decltype(u)::value, decltype(late)::value, G, false>), grid, dim3(512), 0, stream, a);
            };
            using One = std::integral_constant<int, 1>;
            using Two = std::integral_constant<int, 2>;
            using Three = std::integral_constant<int, 3>;
            using Four = std::integral_constant<int, 4>;
            // (fp32: more k-steps in flight cost workgroups)
            auto go = [&](auto epi, auto p, auto late) { launch(epi, p, late, std::integral_constant<int, sizeof(E) == 2 ? 4 : 2>{}, One{}); };
            if constexpr (sizeof(E) == 2)
                if (few.blocks > 1) {
                    using Store = std::integral_constant<int, PCB_EPI_STORE>;
                    auto sized = [&](auto u) {
                        few.blocks == 2   ? launch(Store{}, Two{}, std::true_type{}, u, Two{})
                        : few.blocks == 3 ? launch(Store{}, Two{}, std::true_type{}, u, Three{})
                                          : launch(Store{}, Two{}, std::true_type{}, u, Four{});
                    };
                    a.K <= 1024 ? sized(Two{}) : sized(Four{});
                    return pcb_check_launch("linear_parts_kernel");
                }
            auto kind = [&](auto epi) {
                // (what few_rows() does not ask for is not built: runs side by side are late in a plain store, in bf16 in the gated unit)
                constexpr bool LATE = decltype(epi)::value == PCB_EPI_STORE || (sizeof(E) == 2 && decltype(epi)::value == PCB_EPI_SILU_MUL);
                if (few.parts == 1)
                    return few.late ? go(epi, One{}, std::true_type{}) : go(epi, One{}, std::false_type{});
                if constexpr (LATE)
                    if (few.late) return few.parts == 4 ? go(epi, Four{}, std::true_type{}) : go(epi, Two{}, std::true_type{});
                if constexpr (!LATE || sizeof(E) == 4) few.parts == 4 ? go(epi, Four{}, std::false_type{}) : go(epi, Two{}, std::false_type{});
            };
            switch (a.epilogue) {
                case PCB_EPI_STORE: kind(std::integral_constant<int, PCB_EPI_STORE>{}); break;
                case PCB_EPI_SILU_MUL: kind(std::integral_constant<int, PCB_EPI_SILU_MUL>{}); break;
                default: kind(std::integral_constant<int, PCB_EPI_SCALE_ADD>{});
            }
            return pcb_check_launch("linear_parts_kernel");
        }
        auto go = [&](auto epi) {
            constexpr int EPI = decltype(epi)::value;
            if (deep)
                hipLaunchKernelGGL((linear_skinny_kernel<E, EPI, 16, false>), grid, dim3(64 * 16), 0, stream, a);
            else if (late)
                hipLaunchKernelGGL((linear_skinny_kernel<E, EPI, 8, sizeof(E) == 2>), grid, dim3(64 * 8), 0, stream, a);
            else
                hipLaunchKernelGGL((linear_skinny_kernel<E, EPI, 8, false>), grid, dim3(64 * 8), 0, stream, a);
        };
        switch (a.epilogue) {
            case PCB_EPI_STORE: go(std::integral_constant<int, PCB_EPI_STORE>{}); break;
            case PCB_EPI_SILU_MUL: go(std::integral_constant<int, PCB_EPI_SILU_MUL>{}); break;
            default: go(std::integral_constant<int, PCB_EPI_SCALE_ADD>{});
        }
        return pcb_check_launch("linear_skinny_kernel");
    }
    if (dma_ok(a)) {
        if (sizeof(E) == 4 && in_parts(a)) return pcb_linear_split(a, stream);
        if (pcb_linear_waves_fits(a)) return pcb_linear_waves(a, stream);
        // Plain launches whose 128 x 128 tiles reach more than half of the 256 CUs go to the whole-CU tiles of pb_linear_tiles.hip (row strides
        // such that a tile's rows lie within 32-bit offsets); below, the smaller tiles here give more CUs work: 300 x 2048, K = 2048 (48 tiles)
        // 13.1 us here, 14.9 there, 1024 x 1024 x 1024 (64) 8.3 / 9.6, 1024 x 2048, K = 2048 (128) 15.9 / 16.2, 300 x 8192 (192) 21.4 / 17.4.
        const int weight_rows = a.epilogue == PCB_EPI_SILU_MUL ? 2 * a.N : a.N;
        if (sizeof(E) == 2 && rows > 64 && a.n_groups == 0 && a.n_batch == 0 && !a.row_src && a.ldx < (1 << 22) && a.ldw < (1 << 22) &&
            (int64_t)pcb_ceil_div(a.M, 128) * pcb_ceil_div(weight_rows, 128) > 128)
            return pcb_linear_tiles(a, stream);
        switch (a.epilogue) {
            case PCB_EPI_STORE: return dispatch_dma<E, PCB_EPI_STORE>(a, rows, stream);
            case PCB_EPI_SILU_MUL: return dispatch_dma<E, PCB_EPI_SILU_MUL>(a, rows, stream);
            default: return dispatch_dma<E, PCB_EPI_SCALE_ADD>(a, rows, stream);
        }
    }
    auto go = [&](auto epi) {
        constexpr int EPI = decltype(epi)::value, W = EPI == PCB_EPI_SILU_MUL ? 2 : 1;
        return big ? launch<E, EPI, 4, 4 / W>(a, stream) : launch<E, EPI, 1, 2 / W>(a, stream);
    };
    switch (a.epilogue) {
        case PCB_EPI_STORE: return go(std::integral_constant<int, PCB_EPI_STORE>{});
        case PCB_EPI_SILU_MUL: return go(std::integral_constant<int, PCB_EPI_SILU_MUL>{});
        default: return go(std::integral_constant<int, PCB_EPI_SCALE_ADD>{});
    }
}

}  // namespace

int pcb_linear_check(const pcb_linear_args* a) {
    PCB_REQUIRE(a && a->struct_bytes == sizeof(pcb_linear_args), PCB_ERR_ARG, "pcb_linear: struct size mismatch");
    PCB_REQUIRE(a->dtype == PCB_BF16 || a->dtype == PCB_F32, PCB_ERR_ARG, "pcb_linear: unknown dtype");
    PCB_REQUIRE(a->M >= 0 && a->N > 0 && a->K > 0 && a->ldx >= a->K && a->ldw >= a->K, PCB_ERR_ARG, "pcb_linear: bad sizes");
    PCB_REQUIRE(a->epilogue >= PCB_EPI_STORE && a->epilogue <= PCB_EPI_SCALE_ADD, PCB_ERR_ARG, "pcb_linear: unknown epilogue");
    PCB_REQUIRE(a->act >= PCB_ACT_NONE && a->act <= PCB_ACT_SCALE && a->act2 >= PCB_ACT_NONE && a->act2 <= PCB_ACT_SCALE &&
                    a->act_split >= 0 &&
                    ((a->act | a->act2) == 0 || a->epilogue == PCB_EPI_STORE ||
                     (a->epilogue == PCB_EPI_SILU_MUL && a->act2 == 0 &&
                      (a->act == PCB_ACT_SILU || a->act == PCB_ACT_RELU || a->act == PCB_ACT_GELU_TANH))),
                PCB_ERR_ARG, "pcb_linear: an activation goes with the plain store epilogue (the gated one takes silu, relu or gelu_tanh)");
    PCB_REQUIRE((a->act != PCB_ACT_SOFTCAP && a->act2 != PCB_ACT_SOFTCAP) || a->act_param > 0.0f, PCB_ERR_ARG,
                "pcb_linear: the soft cap must be positive");
    if (a->M == 0) return PCB_OK;
    PCB_REQUIRE(a->x && a->w && a->y, PCB_ERR_ARG, "pcb_linear: null pointer");
    PCB_REQUIRE(a->n_groups >= 0 && (a->n_groups == 0 || a->group_off), PCB_ERR_ARG, "pcb_linear: groups need their offsets");
    PCB_REQUIRE(a->n_batch >= 0 && a->n_batch <= 65535 &&
                    (a->n_batch == 0 || (a->n_groups == 0 && a->epilogue == PCB_EPI_STORE && a->split_n == 0 && a->split_n3 == 0 && !a->bias &&
                                         !a->row_scale && a->x_batch_stride >= 0 && a->y_batch_stride >= 0 && a->w_group_stride >= 0)),
                PCB_ERR_ARG, "pcb_linear: a batch goes with plain stores (no groups, no split destinations, no bias)");
    PCB_REQUIRE(!a->row_gate || (a->epilogue == PCB_EPI_SILU_MUL && a->n_groups == 0 && a->ld_row_gate >= 1), PCB_ERR_ARG,
                "pcb_linear: a gate per row goes with the gated epilogue of a plain (ungrouped) launch");
    PCB_REQUIRE(a->epilogue != PCB_EPI_SILU_MUL || a->w2, PCB_ERR_ARG, "pcb_linear: the gated epilogue takes w2");
    PCB_REQUIRE(a->epilogue == PCB_EPI_SILU_MUL || !a->bias2, PCB_ERR_ARG, "pcb_linear: a second bias goes with the gated epilogue");
    PCB_REQUIRE(a->epilogue != PCB_EPI_SCALE_ADD || (a->col_scale && a->ldy >= a->N && !a->row_dst), PCB_ERR_ARG,
                "pcb_linear: scale-add needs col_scale and a plain fp32 destination");
    PCB_REQUIRE(a->split_n == 0 || (a->epilogue == PCB_EPI_STORE && a->split_n > 0 && a->split_n < a->N && a->y2 && a->row_off2 &&
                                    a->head_dim2 > 0 && a->ldy >= a->split_n) ||
                    (a->epilogue == PCB_EPI_STORE && a->split_n > 0 && a->split_n < a->N && a->y2 && a->y2_f32 && a->split_n3 == 0 &&
                     a->n_groups == 0 && a->head_stride2 >= a->N - a->split_n && a->ldy >= a->split_n),
                PCB_ERR_ARG, "pcb_linear: bad split destination");
    PCB_REQUIRE(a->split_n3 == 0 || (a->epilogue == PCB_EPI_STORE && a->split_n3 > a->split_n && a->split_n3 < a->N && a->y3 && a->row_off3 &&
                                     a->col_stride3 > 0 && (a->split_n > 0 || a->ldy >= a->split_n3)),
                PCB_ERR_ARG, "pcb_linear: bad column-wise destination");
    PCB_REQUIRE(a->split_n > 0 || a->split_n3 > 0 || a->epilogue == PCB_EPI_SCALE_ADD || a->ldy >= a->N, PCB_ERR_ARG, "pcb_linear: ldy < N");
    return PCB_OK;
}

PCB_EXPORT int pcb_linear_parts_form(const pcb_linear_args* a) {
    const int rc = pcb_linear_check(a);
    if (rc != PCB_OK) return rc;
    return a->dtype == PCB_F32 && a->M > 16 && dma_ok(*a) && in_parts(*a) ? pcb_linear_split_shape(*a) : 0;
}

PCB_EXPORT int pcb_linear(const pcb_linear_args* a, void* stream) {
    const int rc = pcb_linear_check(a);
    if (rc != PCB_OK || a->M == 0) return rc;
    return a->dtype == PCB_BF16 ? dispatch<pcb::bf16_t>(*a, (hipStream_t)stream) : dispatch<float>(*a, (hipStream_t)stream);
}
