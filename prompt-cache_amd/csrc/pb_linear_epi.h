// What pb_linear's kernels do with finished sums (pb_linear.hip, pb_linear_tiles.hip): bias, activation, gated unit, where each element goes.
#pragma once
#include <type_traits>

#include "pb_common.h"

namespace pcb {

__device__ __forceinline__ float apply_act(int act, float v, float param) {
    switch (act) {
        case PCB_ACT_SILU: return v / (1.0f + expf(-v));
        case PCB_ACT_SIGMOID: return 1.0f / (1.0f + expf(-v));
        case PCB_ACT_RELU2: return v > 0.0f ? v * v : 0.0f;
        case PCB_ACT_SOFTPLUS: return v > 20.0f ? v : log1pf(expf(v));
        case PCB_ACT_SOFTCAP: return param * tanhf(v / param);
        case PCB_ACT_RELU: return v > 0.0f ? v : 0.0f;
        case PCB_ACT_GELU_TANH: return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
        case PCB_ACT_LOGSIGMOID: return param * (fminf(v, 0.0f) - log1pf(expf(-fabsf(v))));
        case PCB_ACT_SCALE: return param * v;
        default: return v;
    }
}

// the gated epilogue's function: silu (the default), relu or the tanh-form gelu, which is z sigmoid(2 u) for tanh's argument u.  Kept short:
// an epilogue too long to unroll would index the accumulators, which throws them out of the registers.
__device__ __forceinline__ float gate_act(int act, float v) {
    const float t = act == PCB_ACT_GELU_TANH ? 1.5957691216057308f * (v + 0.044715f * v * v * v) : v;
    const float s = v / (1.0f + expf(-t));
    return act == PCB_ACT_RELU ? fmaxf(v, 0.0f) : s;
}

// num / (1 + e^-v) for |v| <= 87 (num = 1: sigmoid, v: silu), where nothing over- or underflows and neither the exponential nor the quotient needs its
// cases: e^x = 2^n 2^f with x log2 e = n + f (log2 e in two parts, the product's rounding put back), a quotient corrected once.  17 instructions where
// expf and a division are some forty; the same bits as theirs but for four of 1.7e7 values spread over +-87.
constexpr float PLAIN_EXP = 87.0f;
__device__ __forceinline__ float over_one_plus_exp(float num, float v) {
#pragma clang fp contract(off)
    const float x = -v, p = x * 1.44269502e+00f, n = __builtin_rintf(p);
    const float rest = __builtin_fmaf(x, 1.92596303e-08f, __builtin_fmaf(x, 1.44269502e+00f, -p));
    const float d = 1.0f + __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((p - n) + rest), (int)n);
    const float r = __builtin_amdgcn_rcpf(d), q = num * r;
    return __builtin_fmaf(__builtin_fmaf(-d, q, num), r, q);
}

// columns that pass through act / act2 of a plain store: the split-off parts are stored as they are
__device__ __forceinline__ int act_end(const pcb_linear_args& a) {
    return a.split_n > 0 ? a.split_n : (a.split_n3 > 0 ? a.split_n3 : a.N);
}

// Where one finished element goes (see pcb_linear_args) and, for the scaled accumulation, what it is added to.  A kernel asks for all its
// elements' places before its first store: loads and stores count on one counter, so a load behind a store waits for the store's way to memory.
struct Place {
    char* p;
    bool wide;                                                       // fp32 (else E)
    float base;                                                      // scaled accumulation: what it is added to; gated epilogue: the row's gate
};
template <typename E, int EPI>
__device__ __forceinline__ Place place(const pcb_linear_args& a, int m, int n) {
    if (EPI == PCB_EPI_SCALE_ADD) {
        float* y = (float*)a.y + (int64_t)m * a.ldy + n;
        return Place{(char*)y, true, a.base ? a.base[(int64_t)m * a.ldbase + n] : *y};
    }
    if (a.split_n3 > 0 && n >= a.split_n3) return Place{(char*)((E*)a.y3 + a.row_off3[m] + (int64_t)(n - a.split_n3) * a.col_stride3), false, 0.0f};
    if (a.split_n > 0 && n >= a.split_n) {
        const int c = n - a.split_n;
        if (a.y2_f32) return Place{(char*)((float*)a.y2 + m * a.head_stride2 + c), true, 0.0f};
        return Place{(char*)((E*)a.y2 + a.row_off2[m] + (int64_t)(c / a.head_dim2) * a.head_stride2 + c % a.head_dim2), false, 0.0f};
    }
    const int64_t at = (int64_t)(a.row_dst ? a.row_dst[m] : m) * a.ldy + n + (a.n_batch > 0 ? (int64_t)blockIdx.z * a.y_batch_stride : 0);
    const float gate = EPI == PCB_EPI_SILU_MUL && a.row_gate ? to_f32(((const E*)a.row_gate)[m * a.ld_row_gate]) : 1.0f;
    return a.out_f32 ? Place{(char*)((float*)a.y + at), true, gate} : Place{(char*)((E*)a.y + at), false, gate};
}
template <typename E, int EPI>
__device__ __forceinline__ void put(const Place& t, float v, float cs) {
    if (EPI == PCB_EPI_SCALE_ADD)
        *(float*)t.p = t.base + cs * v;
    else if (t.wide)
        *(float*)t.p = v;
    else
        *(E*)t.p = from_f32<E>(v);
}

// one result element through bias, activation and gate
template <typename E, int EPI>
__device__ __forceinline__ float finished(const pcb_linear_args& a, const Place& t, int n, float acc, float acc2, float bv, float bv2) {
    float v = acc + bv;
    if (EPI == PCB_EPI_STORE && (a.act | a.act2) && n < act_end(a))
        v = apply_act((a.act_split > 0 && n >= a.act_split) ? a.act2 : a.act, v, a.act_param);
    if (EPI == PCB_EPI_SILU_MUL) {
        v = gate_act(a.act, v) * (acc2 + bv2);
        if (a.row_gate) v *= t.base;
    }
    return v;
}

// The results of a wave's TM x TN tiles of 16 x 16 (rows (wm TM + i) 16 + l15 of m_lo .. m_hi - 1, columns (wn TN + j) 16 + 4 group .. + 3 behind n_lo) to where
// they go; acc2: the gated unit's other half
template <typename E, int EPI, int TM, int TN, int WN = 2>
__device__ __forceinline__ void finish_tile(const pcb_linear_args& a, f4 (&acc)[TM][TN], f4 (&acc2)[EPI == PCB_EPI_SILU_MUL ? TM : 1][EPI == PCB_EPI_SILU_MUL ? TN : 1],
                                            int m_lo, int m_hi, int n_lo, int wm, int wn, int group, int l15) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int BN = 16 * WN * TN;                                 // (WN waves side by side)
    const int N = a.N;
    // Bias, gate and activation first, in the accumulators -- an activation is chosen once, around the loop over them --, then the stores
    const E* bias = (const E*)a.bias;
    const E* bias2 = TWO ? (const E*)a.bias2 : nullptr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n_lo + (wn * TN + j) * 16 + 4 * group;
        if (bias || TWO) {
            float bv[4], bv2[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool in = n + e < N;
                bv[e] = bias && in ? to_f32(bias[n + e]) : 0.0f;
                bv2[e] = TWO && bias2 && in ? to_f32(bias2[n + e]) : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                float rg = 1.0f;
                if (TWO && a.row_gate) {
                    const int m = m_lo + (wm * TM + i) * 16 + l15;
                    rg = to_f32(((const E*)a.row_gate)[(m < m_hi ? m : m_hi - 1) * a.ld_row_gate]);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[i][j][e] += bv[e];
                    if (TWO) acc[i][j][e] = gate_act(a.act, acc[i][j][e]) * (acc2[TWO ? i : 0][TWO ? j : 0][e] + bv2[e]) * rg;
                }
            }
        }
    }
    if (EPI == PCB_EPI_STORE && (a.act | a.act2)) {
        const int end = act_end(a), mid = a.act_split > 0 && a.act_split < end ? a.act_split : end;
        auto run = [&](auto code, int lo, int hi) {
            constexpr int A = decltype(code)::value;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n_lo + (wn * TN + j) * 16 + 4 * group;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e >= lo && n + e < hi) {
#pragma unroll
                        for (int i = 0; i < TM; ++i) acc[i][j][e] = apply_act(A, acc[i][j][e], a.act_param);
                    }
            }
        };
        auto pass = [&](int act, int lo, int hi) {
            if (n_lo >= hi || n_lo + BN <= lo) return;
            switch (act) {
                case PCB_ACT_SILU: run(std::integral_constant<int, PCB_ACT_SILU>{}, lo, hi); break;
                case PCB_ACT_SIGMOID: run(std::integral_constant<int, PCB_ACT_SIGMOID>{}, lo, hi); break;
                case PCB_ACT_RELU2: run(std::integral_constant<int, PCB_ACT_RELU2>{}, lo, hi); break;
                case PCB_ACT_SOFTPLUS: run(std::integral_constant<int, PCB_ACT_SOFTPLUS>{}, lo, hi); break;
                case PCB_ACT_SOFTCAP: run(std::integral_constant<int, PCB_ACT_SOFTCAP>{}, lo, hi); break;
                case PCB_ACT_RELU: run(std::integral_constant<int, PCB_ACT_RELU>{}, lo, hi); break;
                case PCB_ACT_GELU_TANH: run(std::integral_constant<int, PCB_ACT_GELU_TANH>{}, lo, hi); break;
                case PCB_ACT_LOGSIGMOID: run(std::integral_constant<int, PCB_ACT_LOGSIGMOID>{}, lo, hi); break;
                case PCB_ACT_SCALE: run(std::integral_constant<int, PCB_ACT_SCALE>{}, lo, hi); break;
                default: break;
            }
        };
#pragma unroll 1
        for (int part = 0; part < 2; ++part) pass(part ? a.act2 : a.act, part ? mid : 0, part ? end : mid);
    }
    const int whole = act_end(a);                                    // columns that go to y
    const int esz = (EPI == PCB_EPI_SCALE_ADD || a.out_f32 || sizeof(E) == 4) ? 4 : 2;
    const bool quads = a.ldy % 4 == 0 && (uintptr_t)a.y % (4 * esz) == 0 && a.y_batch_stride % 4 == 0 &&
                       (EPI != PCB_EPI_SCALE_ADD || !a.base || (a.ldbase % 4 == 0 && (uintptr_t)a.base % 16 == 0));
    const int64_t y0 = a.n_batch > 0 ? (int64_t)blockIdx.z * a.y_batch_stride : 0;
    // (what the stores need is loaded before the first of them)
    int64_t dst[TM];
    f4 base[EPI == PCB_EPI_SCALE_ADD ? TM : 1][EPI == PCB_EPI_SCALE_ADD ? TN : 1], cs[EPI == PCB_EPI_SCALE_ADD ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int mm = m_lo + (wm * TM + i) * 16 + l15, m = mm < m_hi ? mm : m_hi - 1;
        dst[i] = (int64_t)(EPI != PCB_EPI_SCALE_ADD && a.row_dst ? a.row_dst[m] : m) * a.ldy + y0;
        if constexpr (EPI == PCB_EPI_SCALE_ADD) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n_lo + (wn * TN + j) * 16 + 4 * group;
                if (i == 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) cs[j][e] = n + e < N ? a.col_scale[n + e] : 0.0f;
                }
                if (quads && n + 4 <= N) base[i][j] = *reinterpret_cast<const f4*>(a.base ? a.base + (int64_t)m * a.ldbase + n : (const float*)a.y + dst[i] + n);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n_lo + (wn * TN + j) * 16 + 4 * group;
        const bool quad = quads && n + 4 <= whole;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = m_lo + (wm * TM + i) * 16 + l15;
            if (m >= m_hi) continue;
            const f4 v = acc[i][j];
            if (quad) {
                if constexpr (EPI == PCB_EPI_SCALE_ADD)
                    *reinterpret_cast<f4*>((float*)a.y + dst[i] + n) = base[i][j] + cs[j] * v;
                else if (esz == 4)
                    *reinterpret_cast<f4*>((float*)a.y + dst[i] + n) = v;
                else
                    *reinterpret_cast<uint2*>((E*)a.y + dst[i] + n) = uint2{bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3])};
            } else {
                Place to[4] = {};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) to[e] = place<E, EPI>(a, m, n + e);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) put<E, EPI>(to[e], v[e], EPI == PCB_EPI_SCALE_ADD ? cs[EPI == PCB_EPI_SCALE_ADD ? j : 0][e] : 0.0f);
            }
        }
    }
}

}  // namespace pcb
