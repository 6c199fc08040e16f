// pb_linear over many rows in bf16: four waves (2 x 2) in tiles of 128 or 256 rows x 128, 192 or 256 columns with a whole CU's
// LDS for their ring, main loop and staging order in mfma_tile_loop.h (16 x 16 MFMA blocks, 32 x 32 in the 128 x 128 tiles).
//
// What bounds it: power (at 128 x 128 LDS bandwidth nearly as much: a wave of 64 x 64 reads as many bytes as its MFMAs take cycles; eight waves in two
// halves of k, or four and five images, take 10 % fewer clocks a K-step and the same time).  Against linear_dma_kernel (pb_linear.hip: 16 x 16 MFMAs, two or three images, two
// workgroups to a CU), us, 2048 rows: 2048 x 2048 29.9 -> 19.9 (0.87 PFLOP/s), K = 8192 93.5 -> 72, 2560 columns 39.8 -> 31, 8192 columns
// 90.5 -> 65.6 (1.05 PFLOP/s; the gated pair 79.3 -> 60.7); 4096 x 4096 x 4096 161 -> 112 (1.23 PFLOP/s).  With a sigmoid on half of the columns: 5136
// columns 77.6 -> 63.0, 10272 132 -> 124 since it and silu do without expf's and the division's cases (over_one_plus_exp; and 192-column tiles).
#include "mfma_tile_loop.h"
#include "pb_linear_parts.h"
#include "pb_linear_tiles.h"

namespace {
using namespace pcb;

typedef __bf16 b8 __attribute__((ext_vector_type(8)));

struct Grid { int mb, nb; mfma_tile::Strips s; };

// The wave's sums in `patch` to where they go: quad pc of rows pr, pr + RPI .. (R of them, RPI = 64 / LPR), row pr = row m0 of the result,
// columns n .. n + 3 (n0: the wave's first).  First the patch is turned into results in place, then stored.  Short loops on purpose, and no
// load behind a store:
// - code that runs once comes in at about 2 bytes per ns (instruction misses): a 256 x 256 tile whose epilogue was unrolled took 20 us
//   longer than its products;
// - stores and loads count on one counter, so a wait for a load behind a store waits for the store's way to memory and back (2.4 us).
template <int EPI, int R>
__device__ __forceinline__ void store_columns(const pcb_linear_args& a, char* patch, int pr, int pc, int n0, int n, int m0) {
    typedef bf16_t E;
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int LPR = TWO ? 8 : 16, RPI = 64 / LPR;
    const int M = a.M, N = a.N, whole = act_end(a);                  // columns below `whole` go to y
    auto at = [&](int e, int c) { return (f4*)(patch + (RPI * e + pr) * 256 + ((c + pc) ^ ((RPI * e + pr) & 15)) * 16); };
    auto row = [&](int e) { const int m = m0 + RPI * e; return m < M ? m : M - 1; };
    auto four = [&](const E* p) {
        f4 b = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (p && n + k < N) b[k] = to_f32(p[n + k]);
        return b;
    };
    const int esz = (EPI == PCB_EPI_SCALE_ADD || a.out_f32) ? 4 : 2;
    const bool quad = a.ldy % 4 == 0 && (uintptr_t)a.y % (4 * esz) == 0 && n + 4 <= whole &&
                      (EPI != PCB_EPI_SCALE_ADD || !a.base || (a.ldbase % 4 == 0 && (uintptr_t)a.base % 16 == 0));
    auto largest = [](const f4(&v)[4]) {                             // (what is no number does not count: it stays none either way)
        float top = 0.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int k = 0; k < 4; ++k) top = fmaxf(top, fabsf(v[e][k]));
        return top;
    };
    if (EPI == PCB_EPI_STORE && (a.bias || (a.act | a.act2))) {
        const int mid = a.act_split > 0 && a.act_split < whole ? a.act_split : whole;
        f4 bv = four((const E*)a.bias);
        auto run = [&](auto code, int lo, int hi) {
#pragma unroll 1
            for (int e0 = 0; e0 < R; e0 += 4) {
                f4 v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = *at(e0 + e, 0) + bv;
                auto each = [&](auto f) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (n + k >= lo && n + k < hi) v[e][k] = f(v[e][k]);
                        *at(e0 + e, 0) = v[e];
                    }
                };
                constexpr int A = decltype(code)::value;
                if ((A == PCB_ACT_SIGMOID || A == PCB_ACT_SILU) && largest(v) <= PLAIN_EXP)
                    each([](float x) { return over_one_plus_exp(A == PCB_ACT_SILU ? x : 1.0f, x); });
                else
                    each([&](float x) { return apply_act(A, x, a.act_param); });
            }
            bv = f4{0.f, 0.f, 0.f, 0.f};
        };
        bool added = !a.bias;
#pragma unroll 1
        for (int part = 0; part < 2; ++part) {
            const int act = part ? a.act2 : a.act, lo = part ? mid : 0, hi = part ? whole : mid;
            if (n0 >= hi || n0 + 4 * LPR <= lo || act == PCB_ACT_NONE) continue;
            added = true;
            switch (act) {
                case PCB_ACT_SILU: run(std::integral_constant<int, PCB_ACT_SILU>{}, lo, hi); break;
                case PCB_ACT_SIGMOID: run(std::integral_constant<int, PCB_ACT_SIGMOID>{}, lo, hi); break;
                case PCB_ACT_RELU2: run(std::integral_constant<int, PCB_ACT_RELU2>{}, lo, hi); break;
                case PCB_ACT_SOFTPLUS: run(std::integral_constant<int, PCB_ACT_SOFTPLUS>{}, lo, hi); break;
                case PCB_ACT_SOFTCAP: run(std::integral_constant<int, PCB_ACT_SOFTCAP>{}, lo, hi); break;
                case PCB_ACT_RELU: run(std::integral_constant<int, PCB_ACT_RELU>{}, lo, hi); break;
                case PCB_ACT_GELU_TANH: run(std::integral_constant<int, PCB_ACT_GELU_TANH>{}, lo, hi); break;
                case PCB_ACT_LOGSIGMOID: run(std::integral_constant<int, PCB_ACT_LOGSIGMOID>{}, lo, hi); break;
                default: run(std::integral_constant<int, PCB_ACT_SCALE>{}, lo, hi);
            }
        }
        if (!added) run(std::integral_constant<int, PCB_ACT_NONE>{}, 0, 0);
    }
    if (EPI == PCB_EPI_SILU_MUL) {
        const f4 bv = four((const E*)a.bias), bv2 = four((const E*)a.bias2);
        auto gate = [&](auto code) {
#pragma unroll 1
            for (int e0 = 0; e0 < R; e0 += 4) {
                f4 v[4], u[4];
                float rg[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = *at(e0 + e, 0) + bv;
                    u[e] = *at(e0 + e, 8) + bv2;
                    rg[e] = a.row_gate ? to_f32(((const E*)a.row_gate)[row(e0 + e) * a.ld_row_gate]) : 1.0f;
                }
                auto each = [&](auto f) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) v[e][k] = f(v[e][k]) * u[e][k] * rg[e];
                        *at(e0 + e, 0) = v[e];
                    }
                };
                constexpr int A = decltype(code)::value;
                if (A == PCB_ACT_SILU && largest(v) <= PLAIN_EXP)
                    each([](float x) { return over_one_plus_exp(x, x); });
                else
                    each([](float x) { return gate_act(A, x); });
            }
        };
        if (a.act == PCB_ACT_RELU)
            gate(std::integral_constant<int, PCB_ACT_RELU>{});
        else if (a.act == PCB_ACT_GELU_TANH)
            gate(std::integral_constant<int, PCB_ACT_GELU_TANH>{});
        else
            gate(std::integral_constant<int, PCB_ACT_SILU>{});
    }
    if (EPI == PCB_EPI_SCALE_ADD) {
        const float* from = a.base ? a.base : (const float*)a.y;
        const int64_t ld = a.base ? a.ldbase : a.ldy;
        const f4 bv = four((const E*)a.bias);
        f4 cs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (n + k < N) cs[k] = a.col_scale[n + k];
        if (quad) {
#pragma unroll
            for (int e0 = 0; e0 < R; e0 += 16) {                     // (16 rows' residuals in one wait; R is 16 or 32)
                f4 b0[16];
#pragma unroll
                for (int e = 0; e < 16; ++e) b0[e] = *(const f4*)(from + row(e0 + e) * ld + n);
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (m0 + RPI * (e0 + e) < M)
                        *(f4*)((float*)a.y + (int64_t)(m0 + RPI * (e0 + e)) * a.ldy + n) = b0[e] + cs * (*at(e0 + e, 0) + bv);
            }
            return;
        }
#pragma unroll 1
        for (int k = 0; k < 4 && n + k < N; ++k)
#pragma unroll 1
            for (int e0 = 0; e0 < R; e0 += 8) {
                float b0[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) b0[e] = from[row(e0 + e) * ld + n + k];
                const float ck = a.col_scale[n + k], bk = a.bias ? to_f32(((const E*)a.bias)[n + k]) : 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float* p = (float*)at(e0 + e, 0) + k;
                    *p = b0[e] + ck * (*p + bk);
                }
            }
    }
    auto pack = [](const f4& r) { return uint2{bf16_pair(r[0], r[1]), bf16_pair(r[2], r[3])}; };
    if (quad && !a.row_dst) {
        char* y = (char*)a.y + ((int64_t)m0 * a.ldy + n) * esz;
        const int64_t step = (int64_t)RPI * a.ldy * esz;
#pragma unroll 1
        for (int e0 = 0; e0 < R; e0 += 4) {
            f4 v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = *at(e0 + e, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e, y += step) {
                if (m0 + RPI * (e0 + e) >= M) continue;
                if (esz == 4)
                    *(f4*)y = v[e];
                else
                    *(uint2*)y = pack(v[e]);
            }
        }
        return;
    }
    // whole quads in rows of their own: row_dst, the fp32 rows or the heads that split_n begins
    const bool split = EPI == PCB_EPI_STORE && a.split_n > 0 && n >= a.split_n && n + 4 <= (a.split_n3 > 0 ? a.split_n3 : N) && a.split_n % 4 == 0 &&
                       a.head_stride2 % 4 == 0 && (a.y2_f32 ? (uintptr_t)a.y2 % 16 == 0 : a.head_dim2 % 4 == 0 && (uintptr_t)a.y2 % 8 == 0);
    const int c = n - a.split_n;
    if (quad || split) {
        const bool wide = split ? a.y2_f32 : esz == 4;
        const int size = wide ? 4 : 2;
        char* y = split ? (char*)a.y2 + (a.y2_f32 ? c : (int64_t)(c / a.head_dim2) * a.head_stride2 + c % a.head_dim2) * size : (char*)a.y + (int64_t)n * size;
#pragma unroll 1
        for (int e0 = 0; e0 < R; e0 += 8) {
            int64_t off[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int m = row(e0 + e);
                off[e] = !split ? a.row_dst[m] * a.ldy : a.y2_f32 ? m * a.head_stride2 : a.row_off2[m];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (m0 + RPI * (e0 + e) >= M) continue;
                const f4 v = *at(e0 + e, 0);
                char* p = y + off[e] * size;
                if (wide) {
                    *(f4*)p = v;
                } else if (off[e] % 4 == 0) {
                    *(uint2*)p = pack(v);
                } else {
#pragma unroll
                    for (int k = 0; k < 4; ++k) ((E*)p)[k] = from_f32<E>(v[k]);
                }
            }
        }
        return;
    }
    // element by element: edges, unaligned rows, splits inside a quad, the column-wise destination
#pragma unroll 1
    for (int nk = n; nk < n + 4 && nk < N; ++nk) {
        const bool third = EPI == PCB_EPI_STORE && a.split_n3 > 0 && nk >= a.split_n3;
        const bool second = EPI == PCB_EPI_STORE && !third && a.split_n > 0 && nk >= a.split_n;
        const int d = nk - a.split_n;
        const int64_t col = third ? (int64_t)(nk - a.split_n3) * a.col_stride3
                            : !second ? nk
                            : a.y2_f32 ? d
                                       : (int64_t)(d / a.head_dim2) * a.head_stride2 + d % a.head_dim2;
        const bool wide = second ? a.y2_f32 : !third && esz == 4;
        char* y = (char*)(third ? a.y3 : second ? a.y2 : a.y);
#pragma unroll 1
        for (int e0 = 0; e0 < R; e0 += 8) {
            int64_t off[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int m = row(e0 + e);
                off[e] = col + (third    ? a.row_off3[m]
                                : second ? a.y2_f32 ? m * a.head_stride2 : a.row_off2[m]
                                         : (EPI != PCB_EPI_SCALE_ADD && a.row_dst ? a.row_dst[m] : m) * a.ldy);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if (m0 + RPI * (e0 + e) >= M) continue;
                const float r = ((const float*)at(e0 + e, 0))[nk - n];
                if (wide)
                    ((float*)y)[off[e]] = r;
                else
                    ((E*)y)[off[e]] = from_f32<E>(r);
            }
        }
    }
}

template <int MT, int NT, int S, int BLK>
constexpr int kTileLds = S * mfma_tile::Loop<MT, NT, S, 1, BLK>::kStage > 4 * 32 * MT * 256 ? S * mfma_tile::Loop<MT, NT, S, 1, BLK>::kStage : 4 * 32 * MT * 256;

// tile (mi, ni) of a product
template <int EPI, int MT, int NT, int S, int BLK>
__device__ __forceinline__ void tile_block(const pcb_linear_args& a, int mi, int ni, char* lds) {
    typedef bf16_t E;
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    using L = mfma_tile::Loop<MT, NT, S, 1, BLK>;
    constexpr int BM = L::BM, BN = TWO ? L::BN / 2 : L::BN, NI = L::NI;   // BN: result columns
    constexpr int P = 32 * MT * 256;                                 // bytes of a patch (see below)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int m_lo = mi * BM, n_lo = ni * BN, K = a.K, N = a.N, nk = (K + 63) / 64;

    // staging: a lane's 16-byte chunk of an instruction's row as a 32-bit offset from the operand's K-step (the address is otherwise uniform)
    const int srow = 8 * wave + (lane >> 3), cx = (lane & 7) ^ ((srow >> 1) & 7);
    const int last = (K - (nk - 1) * 64) / 8;                        // chunks of the last K-step (8: a whole one)
    const E* base[3] = {(const E*)a.x + (int64_t)m_lo * a.ldx, (const E*)a.w + (int64_t)n_lo * a.ldw,
                        TWO ? (const E*)a.w2 + (int64_t)n_lo * a.ldw : nullptr};
    uint32_t off[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = 32 * i + srow;
        if (32 * i < BM) {
            off[i] = (uint32_t)((m_lo + r < a.M ? r : a.M - 1 - m_lo) * (int)a.ldx + cx * 8) * 2u;
        } else {
            // (gated: the first half of a wave's columns is W's rows, the second the matching rows of W2)
            const int c = r - BM, n = TWO ? c / (32 * NT) * 16 * NT + c % (16 * NT) : c;
            off[i] = (uint32_t)((n_lo + n < N ? n : N - 1 - n_lo) * (int)a.ldw + cx * 8) * 2u;
        }
    }
    // (chunks past K: the row's first of the K-step again, whose products Loop leaves out)
    const uint32_t past = cx < last ? 0u : (uint32_t)(-16 * cx);
    auto stage = [&](int i, int t, char* buf) {
        const int which = 32 * i < BM ? 0 : TWO && (32 * i - BM) / (16 * NT) % 2 ? 2 : 1;
        const char* s = (const char*)(base[which] + (int64_t)t * 64);
        const uint32_t o = off[i] + (t == nk - 1 ? past : 0u);
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(s + o),
                                         (__attribute__((address_space(3))) void*)(buf + (4 * i + wave) * 1024), 16, 0, 0);
    };
    typename L::Acc acc[L::MB][L::NB];
    // (the weights are the products' first operand: a lane ends up with a row of a block and four neighbouring columns, BLK = 32: four times four)
    auto mma = [](typename L::Acc& c, const b8& x, const b8& w) {
        if constexpr (BLK == 16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x, c, 0, 0, 0);
        else
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, c, 0, 0, 0);
    };
    L::template run<b8>(acc, lds, nk, last, lane, wm, wn, mma, stage);

    // Results: 64 accumulator columns of a wave go into an LDS patch of its own (16-byte quad c of row r at c ^ (r & 15)), so that neighbouring
    // lanes store neighbouring columns.  Gated: 32 gate columns and the matching 32 of the other half side by side.
    __syncthreads();                                                 // (the images are read out)
    constexpr int PARTS = (NT + 1) / 2, ROOM = 4 * P * PARTS <= S * L::kStage ? PARTS : 1;   // patches that fit at a time
    char* patch = lds + wave * (P * ROOM);
    constexpr int LPR = TWO ? 8 : 16, RPI = 64 / LPR;                // lanes on a row, rows an access covers
    const int fr = lane % BLK, pr = lane / LPR, pc = lane % LPR;
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto put = [&](auto part, char* to) {
        constexpr int j = decltype(part)::value;
        constexpr int H = 32 / BLK;                                  // blocks of 32 columns
        constexpr bool ODD = NT % 2 != 0 && j == PARTS - 1;          // (the last half patch of an odd number of them)
#pragma unroll
        for (int i = 0; i < L::MB; ++i)
#pragma unroll
            for (int h = 0; h < (ODD ? H : 2 * H); ++h) {
                const typename L::Acc& c = acc[i][ODD ? L::NB - H + h : TWO ? H * j + h / H * (L::NB / 2) + h % H : 2 * H * j + h];
#pragma unroll
                for (int q = 0; q < BLK * BLK / 256; ++q)
                    *(f4*)(to + (BLK * i + fr) * 256 + ((BLK / 4 * h + mfma_tile::quad_of<BLK>(q, lane)) ^ (fr & 15)) * 16) =
                        f4{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
            }
    };
    auto store = [&](int j, char* from) {
        const int n0 = n_lo + (TWO ? wn * 16 * NT + 32 * j : wn * 32 * NT + 64 * j);
        if (NT % 2 != 0 && j == PARTS - 1 && pc >= 8) return;
        if (n0 < N) store_columns<EPI, 32 * MT / RPI>(a, from, pr, pc, n0, n0 + 4 * pc, m_lo + wm * 32 * MT + pr);
    };
    using First = std::integral_constant<int, 0>;
    using Second = std::integral_constant<int, PARTS - 1>;
    put(First{}, patch);
    if constexpr (ROOM == PARTS) {
        if constexpr (PARTS == 2) put(Second{}, patch + P);
        fence();
#pragma unroll 1
        for (int j = 0; j < PARTS; ++j) store(j, patch + j * P);
    } else {
        fence();
        store(0, patch);
        fence();
        put(Second{}, patch);
        fence();
        store(1, patch);
    }
}

template <int EPI, int MT, int NT, int S, int BLK>
__global__ __launch_bounds__(256, 1) void linear_tile_kernel(const pcb_linear_args a, const Grid g) {
    __shared__ __attribute__((aligned(16))) char lds[kTileLds<MT, NT, S, BLK>];
    int mi, ni;
    if (mfma_tile::tile_of(g.s, g.mb, g.nb, blockIdx.x, mi, ni)) tile_block<EPI, MT, NT, S, BLK>(a, mi, ni, lds);
}

// two products of the same rows in one grid: the first na column blocks are the first product's
template <int EPI, int MT, int NT, int S, int BLK>
__global__ __launch_bounds__(256, 1) void linear_tile_pair_kernel(const pcb_linear_args a, const pcb_linear_args b, const Grid g, int na) {
    __shared__ __attribute__((aligned(16))) char lds[kTileLds<MT, NT, S, BLK>];
    int mi, ni;
    if (!mfma_tile::tile_of(g.s, g.mb, g.nb, blockIdx.x, mi, ni)) return;
    if (ni < na)
        tile_block<PCB_EPI_STORE, MT, NT, S, BLK>(a, mi, ni, lds);
    else
        tile_block<EPI, MT, NT, S, BLK>(b, mi, ni - na, lds);
}

// (b: the second product of a pair, the first one is a plain store)
template <int EPI, int MT, int NT, int S, int BLK = (MT * NT > 4 ? 16 : 32)>
int launch(const pcb_linear_args& a, const pcb_linear_args* b, hipStream_t stream) {
    using L = mfma_tile::Loop<MT, NT, S, 1, BLK>;
    constexpr int BN = EPI == PCB_EPI_SILU_MUL ? L::BN / 2 : L::BN;
    const int mb = pcb_ceil_div(a.M, L::BM), na = b ? pcb_ceil_div(a.N, L::BN) : 0, nb = na + pcb_ceil_div(b ? b->N : a.N, BN);
    const mfma_tile::Strips s = mfma_tile::strips(mb, nb, L::BM, L::BN);
    const dim3 grid(8 * s.mh * s.nh);
    if constexpr (EPI != PCB_EPI_SCALE_ADD)
        if (b) {
            hipLaunchKernelGGL((linear_tile_pair_kernel<EPI, MT, NT, S, BLK>), grid, dim3(256), 0, stream, a, *b, (Grid{mb, nb, s}), na);
            return pcb_check_launch("linear_tile_pair_kernel");
        }
    hipLaunchKernelGGL((linear_tile_kernel<EPI, MT, NT, S, BLK>), grid, dim3(256), 0, stream, a, (Grid{mb, nb, s}));
    return pcb_check_launch("linear_tile_kernel");
}

// The tile whose whole rounds of the 256 CUs cost least.  A round, in us, one workgroup per CU, from K = 64 .. 8192 on a full chip:
// 128 x 128 4.5 + 0.53 per K-step, 128 x 192 5.6 + 0.645, 128 x 256 7 + 0.67, 256 x 192 8 + 0.95, 256 x 256 10 + 1.03 (K = 2048: 21, 26, 28, 38, 43).
// 2048 rows, K = 2048, 128 x 128 / 128 x 256 / 256 x 256 and what the rule took: N = 2048 20.0 / 28.0 / 42.7 -> 20.0, 8192 84 / 75 / 67 -> 66;
// 6000 rows, K = 512, N = 2048 21.2 / 24.9 / 22.3 -> 21.9.  Without and with the two of 192 columns: 2048 rows, N = 2560 31.7 / 29.9, 5136 55.3 / 49.7,
// 10272 106 / 102; 1500 x 3072 31.3 / 25.4; 4096 x 2560 52.0 / 45.4; 2400 x 2048, K = 8192 102 / 91.  (The gated unit's halves are whole pairs of
// 32-column blocks: not 192.)  With the present loop at 330 sizes on average 0.8 % from the fastest shape, 8 of them by more than 10 % (by grid_us() below 1.2 %, 11).
enum Shape { SQUARE, WIDE192, WIDE, TALL192, TALL };
int choose(const pcb_linear_args& a, const pcb_linear_args* b) {
    const bool gated = (b ? b : &a)->epilogue == PCB_EPI_SILU_MUL;
    auto cols = [](const pcb_linear_args& q) { return q.epilogue == PCB_EPI_SILU_MUL ? 2 * q.N : q.N; };      // weight rows
    auto rounds = [&](int bm, int bn) { return ((int64_t)pcb_ceil_div(a.M, bm) * (pcb_ceil_div(cols(a), bn) + (b ? pcb_ceil_div(cols(*b), bn) : 0)) + 255) / 256; };
    const float steps = (float)pcb_ceil_div(a.K, 64);
    const float square = rounds(128, 128) * (4.5f + 0.53f * steps), wide = rounds(128, 256) * (7.0f + 0.67f * steps),
                tall = rounds(256, 256) * (10.0f + 1.03f * steps);
    const float least = tall <= wide && tall <= square ? tall : wide <= square ? wide : square;
    if (!gated) {
        const float wide192 = rounds(128, 192) * (5.6f + 0.645f * steps), tall192 = rounds(256, 192) * (8.0f + 0.95f * steps);
        if (tall192 < least && tall192 <= wide192) return TALL192;
        if (wide192 < least) return WIDE192;
    }
    return tall == least ? TALL : wide == least ? WIDE : SQUARE;
}

template <int EPI>
int dispatch(const pcb_linear_args& a, hipStream_t stream) {
    const int shape = choose(a, nullptr);
    if constexpr (EPI != PCB_EPI_SILU_MUL) {
        if (shape == TALL192) return launch<EPI, 4, 3, 2>(a, nullptr, stream);
        if (shape == WIDE192) return launch<EPI, 2, 3, 3>(a, nullptr, stream);
    }
    if (shape == TALL) return launch<EPI, 4, 4, 2>(a, nullptr, stream);
    return shape == WIDE ? launch<EPI, 2, 4, 3>(a, nullptr, stream) : launch<EPI, 2, 2, 3>(a, nullptr, stream);
}

template <int EPI>
int dispatch_pair(const pcb_linear_args& a, const pcb_linear_args& b, int shape, hipStream_t stream) {
    if constexpr (EPI != PCB_EPI_SILU_MUL) {
        if (shape == TALL192) return launch<EPI, 4, 3, 2>(a, &b, stream);
        if (shape == WIDE192) return launch<EPI, 2, 3, 3>(a, &b, stream);
    }
    if (shape == TALL) return launch<EPI, 4, 4, 2>(a, &b, stream);
    return shape == WIDE ? launch<EPI, 2, 4, 3>(a, &b, stream) : launch<EPI, 2, 2, 3>(a, &b, stream);
}

}  // namespace

int pcb_linear_tiles(const pcb_linear_args& a, hipStream_t stream) {
    switch (a.epilogue) {
        case PCB_EPI_STORE: return dispatch<PCB_EPI_STORE>(a, stream);
        case PCB_EPI_SILU_MUL: return dispatch<PCB_EPI_SILU_MUL>(a, stream);
        default: return dispatch<PCB_EPI_SCALE_ADD>(a, stream);
    }
}

// What a grid of one or two products takes, us (choose() above ranks shapes by whole rounds of a full chip; this is for comparing grids that fill it differently, and
// the kernels of smaller tiles): whole rounds, half a round's products for a part of one and the rest of it in proportion (a full chip runs at a lower clock), and
// the activations behind the last products, 0.056 a number and thread.
static float grid_us(const pcb_linear_args& a, const pcb_linear_args* b, int shape) {
    static constexpr struct { int bm, bn; float base, step; } T[] = {
        {128, 128, 4.8f, 0.57f}, {128, 192, 7.0f, 0.77f}, {128, 256, 11.0f, 0.88f}, {256, 192, 10.0f, 1.3f}, {256, 256, 12.7f, 1.5f}};
    const auto& t = T[shape];
    auto blocks = [&](const pcb_linear_args& q) { return (int64_t)pcb_ceil_div(q.epilogue == PCB_EPI_SILU_MUL ? 2 * q.N : q.N, t.bn); };
    auto acts = [&](const pcb_linear_args& q) { return q.epilogue == PCB_EPI_SILU_MUL ? 0.5f : (q.act | q.act2) ? 1.0f : 0.0f; };
    const int64_t tiles = pcb_ceil_div(a.M, t.bm) * (blocks(a) + (b ? blocks(*b) : 0)), rest = tiles % 256;
    const float steps = t.step * (float)pcb_ceil_div(a.K, 64), act = b && acts(*b) > acts(a) ? acts(*b) : acts(a);
    const float whole = (float)(tiles / 256), part = rest ? 0.5f + (float)rest / 512.0f : 0.0f;
    return steps * (whole + part) + t.base * (whole > 0.0f ? whole + part : 1.0f) + 0.056f * act * (float)(t.bm * t.bn / 256);
}

// ... and a product by itself, through the kernel that pb_linear has for it: waves, these tiles, or tiles of 64 x 64
static float alone_us(const pcb_linear_args& q) {
    const float steps = (float)pcb_ceil_div(q.K, 64);
    const int cols = q.epilogue == PCB_EPI_SILU_MUL ? 2 * q.N : q.N;
    if (pcb_linear_waves_fits(q)) {
        const int64_t wgs = pcb_linear_waves_tiles(q);
        return wgs <= 256 ? 3.5f + (float)wgs / 230.0f + 0.087f * steps : 4.6f + 0.19f * steps;
    }
    if ((int64_t)pcb_ceil_div(q.M, 128) * pcb_ceil_div(cols, 128) > 128) return grid_us(q, nullptr, choose(q, nullptr));
    return (int64_t)pcb_ceil_div(q.M, 64) * pcb_ceil_div(cols, 64) <= 256 ? 4.2f + 0.33f * steps : 4.8f + 0.42f * steps;
}

// Two products in one grid fill the rounds that each leaves part empty: one grid where that takes 5 % less by these estimates than the two by themselves (gated units
// beyond 128 rows only; their code is longer, 1.5).  Of 600 sizes that go out in one so -- 65 .. 4800 rows, 64 .. 12000 columns, K = 64 .. 8192 -- two are slower for it,
// by 8 and 23 %, on average they take 0.79 of the time.  (Judged by this grid's times alone, without the kernels of smaller tiles, 153 of 1160 lost more than 2 %, up
// to 1.6: 76 rows, K = 8192, 240 and 152 columns 27.3 / 43.9.)
// Apart / in one, us, 2560 and 8192 fp32 columns, K = 2048: 255 rows 38.1 / 25.1, 377 40.1 / 25.4, 679 52.4 / 35.0, 1484 77.8 / 57.7, 2195 120 / 103; 2048
// with a sigmoid and a gated 4096: 142 rows 32.3 / 24.7, 558 50.9 / 40.1, 2195 124 / 106 (1805 83 / 102: apart); 640 and 2048, K = 512: 310 rows 12.0 / 9.0.
int pcb_linear_tiles_pair_shape(const pcb_linear_args& a, const pcb_linear_args& b) {
    auto fits = [](const pcb_linear_args& q) {
        return q.dtype == PCB_BF16 && q.M > 64 && q.n_groups == 0 && q.n_batch == 0 && !q.row_src && q.ldx < (1 << 22) && q.ldw < (1 << 22) && pcb_linear_pieces(q);
    };
    const bool gated = b.epilogue == PCB_EPI_SILU_MUL;
    if (!fits(a) || !fits(b) || a.M != b.M || a.K != b.K || a.epilogue != PCB_EPI_STORE || b.epilogue == PCB_EPI_SCALE_ADD || (gated && a.M <= 128)) return -1;
    const int shape = choose(a, &b);
    return grid_us(a, &b, shape) + (gated ? 1.5f : 0.0f) < 0.95f * (alone_us(a) + alone_us(b)) ? shape : -1;
}

int pcb_linear_tiles_pair(const pcb_linear_args& a, const pcb_linear_args& b, int shape, hipStream_t stream) {
    return b.epilogue == PCB_EPI_SILU_MUL ? dispatch_pair<PCB_EPI_SILU_MUL>(a, b, shape, stream) : dispatch_pair<PCB_EPI_STORE>(a, b, shape, stream);
}
