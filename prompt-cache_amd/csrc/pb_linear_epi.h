// What pb_linear's kernels do with finished sums (pb_linear.hip, pb_linear_tiles.hip): bias, activation, gated unit, where each element goes.
#pragma once
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

}  // namespace pcb
