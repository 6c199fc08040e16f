// Pieces the attention kernels of libpromptcache_blocks.so share: softmax weights as an operand of the second product.
#pragma once
#include "pb_common.h"

// bf16 prompts of the usual head counts in one pass without a band (pb_attn_talk_prompt.hip): which calls it takes, and the launch
bool pcb_talk_prompt_fits(const pcb_attn_talk_args& a);
int pcb_talk_prompt(const pcb_attn_talk_args& a, hipStream_t stream);

#ifdef __HIPCC__
namespace pcb {

// e^x of a score less its row's maximum (x <= 0, -infinity for a key the row does not see): 2^(x log2 e) on the hardware's exp2, the product's
// rounding put back (log2 e in two parts), so that the error does not grow with |x|.  Seven instructions; below e^-87 it is 0.  NaN stays NaN
// (v_maximum3_f32; fmaxf would return the bound for it).
__device__ __forceinline__ float exp_le0(float x) {
    x = __builtin_elementwise_maximum(x, -200.0f);
    const float p = x * 1.44269502e+00f, lo = __builtin_fmaf(x, 1.92596303e-08f, __builtin_fmaf(x, 1.44269502e+00f, -p));
    const float e = __builtin_amdgcn_exp2f(p);
    return __builtin_fmaf(e, lo * 6.93147182e-01f, e);
}

// the largest over the four lane groups (16 lanes apart)
__device__ __forceinline__ float max4(float v) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// eight softmax weights of a lane.  bf16: a hi + lo pair of bf16 values (two MFMAs), so that they are not rounded to 8 bits; fp32: as
// they are
template <typename E>
struct PFrag;
template <>
struct PFrag<bf16_t> {
    Frag<bf16_t> hi, lo;
};
template <>
struct PFrag<float> {
    Frag<float> hi;
};

__device__ __forceinline__ void make_p(PFrag<bf16_t>& f, const float (&p)[8]) {
    // hi = p, lo = what that leaves, both rounded to nearest: hi + lo carries 17 bits of p's mantissa.  Six instructions a pair of weights; cutting the upper
    // 16 bits off instead took twelve.
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t w = bf16_pair(p[2 * e], p[2 * e + 1]);
        f.hi.v[e] = w;
        f.lo.v[e] = bf16_pair(p[2 * e] - __uint_as_float(w << 16), p[2 * e + 1] - __uint_as_float(w & 0xffff0000u));
    }
}
__device__ __forceinline__ void make_p(PFrag<float>& f, const float (&p)[8]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) f.hi.v[e] = p[e];
}

__device__ __forceinline__ f4 mma_p(const Frag<bf16_t>& v, const PFrag<bf16_t>& p, f4 c) {
    c = mma(v, p.hi, c);
    return mma(v, p.lo, c);
}
__device__ __forceinline__ f4 mma_p(const Frag<float>& v, const PFrag<float>& p, f4 c) { return mma(v, p.hi, c); }

// ---- value operands out of an LDS tile kept key by key ([key][column], ld elements per key) ------------------------------------------
// The second product is O^T = V^T P^T: its A operand wants, per lane (value column l & 15, group l >> 4), eight keys of that column.  Key
// k index (group g, e) stands for key 4 g + e (e < 4) and 16 + 4 g + e - 4 (e >= 4) of the 32-key step -- what the lanes hold of the
// weights after S^T = K Q^T.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// `t` points at (key 0 of the step, column 0 of the 16-column block); transposed 8-byte reads: the 16 lanes of a group give the addresses
// of a 4-key x 16-column block (lane i: key i / 4, columns 4 (i % 4) ..) and receive its columns
__device__ __forceinline__ Frag<bf16_t> load_v_lds(const bf16_t* t, int ld, int g, int i) {
    const bf16_t* p = t + (4 * g + (i >> 2)) * ld + 4 * (i & 3);
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 16 * ld));
    Frag<bf16_t> f;
    const uint2 ua = __builtin_bit_cast(uint2, a), ub = __builtin_bit_cast(uint2, b);
    f.v = u32x4{ua.x, ua.y, ub.x, ub.y};
    return f;
}
__device__ __forceinline__ Frag<float> load_v_lds(const float* t, int ld, int g, int i) {
    Frag<float> f;
#pragma unroll
    for (int e = 0; e < 8; ++e) f.v[e] = t[(e < 4 ? 4 * g + e : 16 + 4 * g + e - 4) * ld + i];
    return f;
}

// elements per LDS row for `cols` columns (a multiple of 16): rows 8 (mod 16) dwords apart, so that four neighbouring keys of a transposed
// read fall on different banks
template <typename E>
__host__ __device__ constexpr int v_ld(int cols) {
    return sizeof(E) == 2 ? cols + (cols / 2 % 16 == 8 ? 0 : 16) : cols + 8;
}

}  // namespace pcb
#endif
