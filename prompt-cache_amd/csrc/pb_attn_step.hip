// pcb_attn_step: a decoding step of an attention layer behind its projection: norm, rotation and cache store of the step's row (what pcb_head_prep does) in
// the launch that attends over the slot's cached rows (pcb_attn_rows, pcb_attn_latent); the merge of their runs is a launch of its own, as there.
//
// One workgroup = one query row x up to 16 query heads of one key head x one run of the keys, four waves.  They prepare the row's queries into LDS -- and the new key
// and value into LDS and the cache where the run has them -- while the run's first rows are on their way, one wave making the turns.  Keys go straight from
// memory into the matrix cores' operands (a lane's 16 bytes of a row), values through LDS, whose transposed reads the second product wants.  Scores S^T = K Q^T: wave w takes
// the 16 keys 16 w .. of a block and leaves them in LDS; then every wave takes all of them and a quarter of the value columns, O^T = V^T P^T.  The new row
// is taken from LDS, so nothing waits for its way to memory.
// What bounds it: the chain of a workgroup -- launch, the tile, projected row and first keys (the turns' float64 sincos beside them), norm, one block of keys --
// 7.2 us, where head_prep's was 5.4 and the single rows' attention's 5.6; beyond one block a workgroup ~1.3 a block.  us, a decoding step of Fivesun in a graph, three
// launches a layer / two: 8 requests of 300 keys, width 2048 bf16 299 / 290, 64 of 300 443 / 428, 48 of 1000 446 / 425, one of 100 239 / 231; 2 of 300, width 1024
// fp32 224 / 203, 64 of 500 442 / 411.  (A workgroup that walks all keys of a row by itself, so that nothing is merged: one of 100 keys 230, 8 of 300 294, 2 of 300 in fp32
// 241, one of 1000 287 for 245: a CU's own path to memory, ~45 GB/s.)
#include "pb_attn_common.h"

namespace {
using namespace pcb;

constexpr int LW = 4;                                                // waves of a workgroup
constexpr int MAX_PAIRS = 64;

__device__ __forceinline__ void put8(bf16_t* p, const float (&v)[8]) {
    store4(p, v[0], v[1], v[2], v[3]);
    store4(p + 4, v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void put8(float* p, const float (&v)[8]) {
    store4(p, v[0], v[1], v[2], v[3]);
    store4(p + 4, v[4], v[5], v[6], v[7]);
}

// KSQ: 32-element k-steps of a key; VBW: 16-column value blocks per wave; LATENT: the values are the keys' leading columns
template <typename E, int KSQ, int VBW, bool LATENT>
__global__ __launch_bounds__(64 * LW) void attn_step_kernel(pcb_attn_step_args a) {
    constexpr int CE = 16 / sizeof(E), BK = sizeof(E) == 2 ? 64 : 32, NKT = BK / 16, NK2 = BK / 32;
    constexpr int KC = KSQ * 32, VC = VBW * 16 * LW, QC = LATENT ? 64 : KC, QLD = QC + CE, VLD = v_ld<E>(VC), LPR = 64 * LW / BK, VCH = VC / CE / LPR;
    static_assert(VC / CE % LPR == 0, "whole chunks per thread");
    __shared__ __attribute__((aligned(16))) E Qs[16 * QLD], Kn[KC], Vn[LATENT ? 8 : VC], Vs[BK * VLD];   // (LATENT: the queries' turned parts)
    __shared__ f4 Ss[NKT][64];
    __shared__ float cs[MAX_PAIRS], sn[MAX_PAIRS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, c = lane & 15;
    const int32_t* tile = a.tiles + 4 * blockIdx.x;
    const int slot = tile[0], pos = tile[1];
    const int64_t row = tile[3];
    const int per = a.H / a.Hkv, hb = (per + 15) / 16;
    const int hk = blockIdx.y / hb, j0 = blockIdx.y % hb * 16, h0 = hk * per + j0;
    const int n_h = per - j0 < 16 ? per - j0 : 16;
    const int dim = a.dim, vdim = a.vdim, np = a.rot_dims / 2;
    const E* P = (const E*)a.p + row * a.ldp;
    E* K = (E*)a.k + (int64_t)slot * a.k_slot_stride + (int64_t)hk * a.k_head_stride;
    E* V = (E*)a.v + (int64_t)slot * a.v_slot_stride + (int64_t)hk * a.v_head_stride;

    int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;      // the oldest key the row sees
    if (a.block > 0) lo = max(lo, pos / a.block * a.block);
    int kb_lo = lo / BK, kb_hi = pos / BK;
    if (a.n_splits > 1) {                                            // this workgroup's run of the blocks (it may be empty)
        const int run = (kb_hi - kb_lo + a.n_splits) / a.n_splits;
        kb_lo += (int)blockIdx.z * run;
        kb_hi = kb_lo + run - 1 < kb_hi ? kb_lo + run - 1 : kb_hi;
    }
    const bool last = kb_lo <= kb_hi && kb_hi == pos / BK, first = last && j0 == 0;      // the run has the new row; it stores it

    // ---- what this wave prepares of the row, eight columns a lane, requested first: query heads, 16 lanes each (LATENT: their turned parts, 8 lanes each, waves
    // 0 and 1); wave 2 also key and value (LATENT: the latent, 32 lanes), wave 3 the turns (LATENT: and the key's turned part)
    constexpr int LPH = LATENT ? 8 : 16;
    const int qd = LATENT ? dim - vdim : dim, qh = wave * (64 / LPH) + lane / LPH, qc = 8 * (lane % LPH);
    const bool q_on = qh < n_h && qc < qd;
    Frag<E> xq, xk;
    zero8(xq);
    zero8(xk);
    const bool whole = (((uintptr_t)a.p | (uintptr_t)((a.ldp | a.q_at | a.q_head_stride | a.k_at | a.k_cols | a.v_at) * (int64_t)sizeof(E))) & 15) == 0;
    auto eight = [&](const E* p) {                                   // (rows that begin anywhere: element by element)
        if (whole) return load8(p);
        __attribute__((aligned(16))) E t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = p[e];
        return load8(t);
    };
    if (q_on) xq = eight(P + a.q_at + (int64_t)(h0 + qh) * a.q_head_stride + qc);
    const bool value = !LATENT && lane >= 16;
    const int kc = 8 * (LATENT ? lane : lane % 16);
    const bool k_on = last && (LATENT ? (wave == 2 ? kc < vdim : wave == 3 && kc < qd) : wave == 2 && lane < 32 && kc < (value ? vdim : dim));
    if (k_on) xk = eight(P + (LATENT ? a.k_at + (wave == 3 ? vdim : 0) : value ? a.v_at + (int64_t)hk * vdim : a.k_at + (int64_t)hk * a.k_cols) + kc);

    // ---- the run's first rows
    Frag<E> kf[KSQ];
    u32x4 rv[VCH];
    const int lr = tid / LPR, lc = tid % LPR * CE;                   // this thread's value row of a block and its first column
    auto fetch = [&](int kb) {
        if (wave < NKT) {
            const int j = kb * BK + wave * 16 + c;
            const E* p = K + (int64_t)(j < pos ? j : lo) * a.k_row_stride + 8 * g; // (from the new row on: any row; not used)
#pragma unroll
            for (int ks = 0; ks < KSQ; ++ks) {
                zero8(kf[ks]);
                if (32 * ks + 8 * g < dim) kf[ks] = load8(p + 32 * ks);
            }
        }
        const int j = kb * BK + lr;
        const E* p = V + (int64_t)(j < pos ? j : lo) * a.v_row_stride;
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int k = lc + i * LPR * CE;
            rv[i] = u32x4{0u, 0u, 0u, 0u};
            if (k < vdim) rv[i] = *reinterpret_cast<const u32x4*>(p + k);
        }
    };
    if (kb_lo <= kb_hi) fetch(kb_lo);
    Frag<E> qf[KSQ];
    const int qr = c < n_h ? c : n_h - 1;                            // (lanes past the last head repeat it; nothing of theirs is stored)
    if (LATENT) {                                                    // the folded queries, as they are
        const E* q = (const E*)a.q + row * a.ldq + (int64_t)(h0 + qr) * dim + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSQ; ++ks)
            if (32 * ks < vdim) qf[ks] = load8(q + 32 * ks);
    }
    if (wave == 3 && lane < np) {
        double s, t;
        sincos((double)pos * a.freqs[lane], &s, &t);
        cs[lane] = (float)t * a.rot_mag;
        sn[lane] = (float)s * a.rot_mag;
    }
    __syncthreads();                                                 // (the turns)
    auto norm = [&](float (&v)[8], int D, const float* gain, int col, bool on) {
        float ss = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
        ss += __shfl_xor(ss, 1, 64);
        ss += __shfl_xor(ss, 2, 64);
        ss += __shfl_xor(ss, 4, 64);
        ss += __shfl_xor(ss, 8, 64);
        if (LATENT) ss += __shfl_xor(ss, 16, 64);
        const float inv = 1.0f / sqrtf(ss / (float)D + a.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= inv;
        if (on && gain) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= gain[col + e];
        }
    };
    auto turn = [&](float (&v)[8], int col) {
        if (col >= a.rot_dims) return;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float u = v[2 * e], w = v[2 * e + 1], ct = cs[col / 2 + e], st = sn[col / 2 + e];
            v[2 * e] = u * ct - w * st;
            v[2 * e + 1] = w * ct + u * st;
        }
    };
    float v[8];
    if (wave * (64 / LPH) < n_h) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = at8(xq, e);
        if (!LATENT) norm(v, dim, a.q_gain, qc, q_on);
        if (q_on) {
            turn(v, qc);
            put8(&Qs[qh * QLD + qc], v);
        }
    }
    if (last && wave >= 2) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = at8(xk, e);
        if (wave == 2) norm(v, LATENT || value ? vdim : dim, value ? nullptr : a.k_gain, kc, k_on);
        if (k_on) {
            if (value && a.blend) {
                const float lam = a.blend[0];
                const float* o = a.other + row * a.ld_other + (int64_t)hk * vdim + kc;
                float t[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) t[e] = (1.0f - lam) * v[e] + lam * o[e];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = t[e];
            }
            if (value && a.keep && first) {
                float* k = a.keep + row * a.ld_keep + (int64_t)hk * vdim + kc;
#pragma unroll
                for (int e = 0; e < 8; ++e) k[e] = v[e];
            }
            if (LATENT ? wave == 3 : !value) turn(v, kc);
            const int at = LATENT && wave == 3 ? vdim + kc : kc;
            put8(value ? &Vn[at] : &Kn[at], v);
            if (first) put8((value ? V + (int64_t)pos * a.v_row_stride : K + (int64_t)pos * a.k_row_stride) + at, v);
        }
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < KSQ; ++ks) {
        if (LATENT && 32 * ks < vdim) continue;
        zero8(qf[ks]);
        if (32 * ks + 8 * g < dim) qf[ks] = load8(&Qs[qr * QLD + 32 * ks + 8 * g - (LATENT ? vdim : 0)]);
    }
    const E* const new_v = LATENT ? Kn : Vn;
    const float sc = a.scale * 1.44269504088896f, NEG = -__builtin_inff();         // (scores in units of ln 2)
    float m = NEG, l = 0.0f;
    f4 o[VBW];
#pragma unroll
    for (int vb = 0; vb < VBW; ++vb) o[vb] = f4{0.f, 0.f, 0.f, 0.f};
    for (int kb = kb_lo; kb <= kb_hi; ++kb) {
        const bool fresh = kb * BK + lr >= pos;                      // (rows past the new one repeat it: finite, and masked)
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int k = lc + i * LPR * CE;
            if (fresh && k < vdim) rv[i] = *reinterpret_cast<const u32x4*>(&new_v[k]);
            *reinterpret_cast<u32x4*>(&Vs[lr * VLD + k]) = rv[i];
        }
        if (wave < NKT) {
            if (kb * BK + wave * 16 + c >= pos) {
#pragma unroll
                for (int ks = 0; ks < KSQ; ++ks)
                    if (32 * ks + 8 * g < dim) kf[ks] = load8(&Kn[32 * ks + 8 * g]);
            }
            f4 acc = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KSQ; ++ks) acc = mma(kf[ks], qf[ks], acc);
            Ss[wave][lane] = acc;
        }
        __syncthreads();
        if (kb < kb_hi) fetch(kb + 1);
        float s[NKT][4], bm = NEG;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt) {
            const f4 acc = Ss[kt][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int key = kb * BK + kt * 16 + 4 * g + e;
                s[kt][e] = key <= pos && key >= lo ? acc[e] * sc : NEG;
                bm = fmaxf(bm, s[kt][e]);
            }
        }
        bm = max4(bm);
        const float m_new = fmaxf(m, bm);
        const float m_use = m_new == NEG ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use);       // (m = -inf: 0)
        float psum = 0.0f;
        PFrag<E> pf[NK2];
#pragma unroll
        for (int k2 = 0; k2 < NK2; ++k2) {
            float p[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                p[e] = __builtin_amdgcn_exp2f(s[2 * k2 + (e >> 2)][e & 3] - m_use);
                psum += p[e];
            }
            make_p(pf[k2], p);
        }
        l = l * alpha + psum;
        m = m_new;
#pragma unroll
        for (int vb = 0; vb < VBW; ++vb) {
            const int vc = (wave * VBW + vb) * 16;
            if (vc >= vdim) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[vb][e] *= alpha;
#pragma unroll
            for (int k2 = 0; k2 < NK2; ++k2) o[vb] = mma_p(load_v_lds(&Vs[k2 * 32 * VLD + vc], VLD, g, c), pf[k2], o[vb]);
        }
        if (kb < kb_hi) __syncthreads();                             // (this block's reads are done)
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (c >= n_h) return;
    const int h = h0 + c;
    if (a.n_splits > 1 || (LATENT && a.up)) {                        // as the merging launches of pcb_attn_rows and pcb_attn_latent read it
        const int64_t run = ((int64_t)blockIdx.x * a.H + h) * a.n_splits + blockIdx.z;
        if (wave == 0 && g == 0) *reinterpret_cast<float2*>(a.part + (int64_t)a.n_rows * a.H * a.n_splits * vdim + 2 * run) = float2{m, l};
#pragma unroll
        for (int vb = 0; vb < VBW; ++vb) {
            const int vc = (wave * VBW + vb) * 16 + 4 * g;
            if (vc < vdim) *reinterpret_cast<f4*>(a.part + run * vdim + vc) = o[vb];
        }
        return;
    }
    float keep = 1.0f;
    if (a.sink) {
        const float sk = a.sink[h] * 1.44269504088896f;
        const float top = fmaxf(m, sk);
        keep = __builtin_amdgcn_exp2f(m - top);
        l = l * keep + __builtin_amdgcn_exp2f(sk - top);
    }
    float by = keep / l;
    if (a.gate) by *= to_f32(((const E*)a.gate)[row * a.ldg + h]);
    E* out = (E*)a.out + row * a.ldo + (int64_t)h * vdim;
#pragma unroll
    for (int vb = 0; vb < VBW; ++vb) {
        const int vc = (wave * VBW + vb) * 16 + 4 * g;
        if (vc < vdim) store4(out + vc, o[vb][0] * by, o[vb][1] * by, o[vb][2] * by, o[vb][3] * by);
    }
}

// one workgroup per (row, head): the runs' factors once, then their partial results rescaled to the common maximum and summed.  (What a thread adds up of the
// first runs is requested ahead of the factors.)
template <typename E>
__global__ __launch_bounds__(128) void attn_step_merge_kernel(pcb_attn_step_args a) {
    constexpr int AHEAD = 8;
    __shared__ float fac[64];
    const int h = blockIdx.y, vdim = a.vdim, Z = a.n_splits, lane = threadIdx.x & 63;
    const int64_t run = ((int64_t)blockIdx.x * a.H + h) * Z;
    const float* pp = a.part + run * vdim;
    const float* ml = a.part + (int64_t)a.n_rows * a.H * Z * vdim + 2 * run;
    const int64_t row = a.tiles[4 * blockIdx.x + 3];
    float first[AHEAD];
    const int c0 = threadIdx.x < vdim ? threadIdx.x : 0;
#pragma unroll
    for (int z = 0; z < AHEAD; ++z) first[z] = z < Z ? pp[(int64_t)z * vdim + c0] : 0.0f;
    if (threadIdx.x < 64) {
        const float NEG = -__builtin_inff();
        const float sk = a.sink ? a.sink[h] * 1.44269504088896f : NEG;
        const float gate = a.gate ? to_f32(((const E*)a.gate)[row * a.ldg + h]) : 1.0f;
        const float2 mz = lane < Z ? *reinterpret_cast<const float2*>(ml + 2 * lane) : float2{NEG, 0.0f};
        const float top = fmaxf(wave_max(mz.x), sk);                 // (the row sees itself: a number)
        const float w = __builtin_amdgcn_exp2f(mz.x - top);
        const float den = wave_sum(w * mz.y) + (a.sink ? __builtin_amdgcn_exp2f(sk - top) : 0.0f);
        fac[lane] = w / den * gate;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < vdim; c += 128) {
        float o = 0.0f;
        if (c == c0) {
#pragma unroll
            for (int z = 0; z < AHEAD; ++z)
                if (z < Z) o += fac[z] * first[z];
        }
#pragma unroll 8
        for (int z = c == c0 ? AHEAD : 0; z < Z; ++z) o += fac[z] * pp[(int64_t)z * vdim + c];     // (an empty run left zeros)
        ((E*)a.out)[row * a.ldo + (int64_t)h * vdim + c] = from_f32<E>(o);
    }
}

// The same for a latent's runs with the heads' own up-projections and gates behind it: one workgroup per (row, head), the head's rows of `up` on their way while the
// runs are merged, four lanes an output.  What bounds it: the way of the runs and of up's 49 KB to a CU.  A merge, a launch of H small products and one of gates were
// 14 us of a step (8 rows, 16 heads of 128 over a latent of 192, 5 runs), this is 8.
template <typename E>
__global__ __launch_bounds__(256) void attn_step_up_kernel(pcb_attn_step_args a) {
    constexpr int AHEAD = 8, PASS = 2, CH = 6;                       // 64 outputs a pass, chunks of 32 columns
    __shared__ float fac[64];
    __shared__ __attribute__((aligned(16))) float merged[32 * CH];
    const int tid = threadIdx.x, lane = tid & 63, h = blockIdx.y, vdim = a.vdim, up = a.up_dim, Z = a.n_splits > 1 ? a.n_splits : 1;
    const int64_t run = ((int64_t)blockIdx.x * a.H + h) * Z;
    const float* pp = a.part + run * vdim;
    const float* ml = a.part + (int64_t)a.n_rows * a.H * Z * vdim + 2 * run;
    const int64_t row = a.tiles[4 * blockIdx.x + 3];
    const int c0 = tid < vdim ? tid : 0;
    const float2 mz = *reinterpret_cast<const float2*>(ml + 2 * (lane < Z ? lane : 0));
    float first[AHEAD];
#pragma unroll
    for (int z = 0; z < AHEAD; ++z) first[z] = pp[(int64_t)(z < Z ? z : 0) * vdim + c0];
    E gate[PASS];
    Frag<E> w[PASS][CH];
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
        const int j = 64 * p + tid / 4 < up ? 64 * p + tid / 4 : up - 1;
        gate[p] = ((const E*)a.up_gate)[row * a.ld_up_gate + (int64_t)h * up + j];
        const E* wr = (const E*)a.up + ((int64_t)h * up + j) * vdim;
#pragma unroll
        for (int i = 0; i < CH; ++i) w[p][i] = load8(wr + (32 * i < vdim ? 32 * i : 0) + 8 * (tid & 3));
    }
    __builtin_amdgcn_sched_barrier(0);
    auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };      // (what is under way stays so)
    if (tid < 64) {
        const float m = lane < Z ? mz.x : -__builtin_inff(), l = lane < Z ? mz.y : 0.0f;
        const float f = __builtin_amdgcn_exp2f(m - wave_max(m));     // (the row sees itself: the largest is a number)
        fac[lane] = f / wave_sum(f * l);
    }
    barrier();
    if (tid < vdim) {
        float o = 0.0f;
#pragma unroll
        for (int z = 0; z < AHEAD; ++z)
            if (z < Z) o += fac[z] * first[z];
#pragma unroll 8
        for (int z = AHEAD; z < Z; ++z) o += fac[z] * pp[(int64_t)z * vdim + tid];      // (an empty run left zeros)
        merged[tid] = o;
    }
    barrier();
#pragma unroll
    for (int p = 0; p < PASS; ++p) {
        const int j = 64 * p + tid / 4;
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (32 * i < vdim)
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[e & 3] += at8(w[p][i], e) * merged[32 * i + 8 * (tid & 3) + e];
        float o = (acc[0] + acc[1]) + (acc[2] + acc[3]);
        o += __shfl_xor(o, 1, 64);
        o += __shfl_xor(o, 2, 64);
        if ((tid & 3) == 0 && j < up) ((E*)a.out)[row * a.ldo + (int64_t)h * up + j] = from_f32<E>(o * to_f32(gate[p]));
    }
}

template <typename E>
int dispatch(const pcb_attn_step_args& a, hipStream_t stream) {
    const int per = a.H / a.Hkv;
    const dim3 grid(a.n_rows, a.Hkv * ((per + 15) / 16), a.n_splits > 1 ? a.n_splits : 1), block(64 * LW);
    if (a.latent)
        hipLaunchKernelGGL((attn_step_kernel<E, 8, 3, true>), grid, block, 0, stream, a);
    else if (a.dim <= 64 && a.vdim <= 64)
        hipLaunchKernelGGL((attn_step_kernel<E, 2, 1, false>), grid, block, 0, stream, a);
    else
        hipLaunchKernelGGL((attn_step_kernel<E, 4, 2, false>), grid, block, 0, stream, a);
    if (a.up)
        hipLaunchKernelGGL(attn_step_up_kernel<E>, dim3(a.n_rows, a.H), dim3(256), 0, stream, a);
    else if (a.n_splits > 1)
        hipLaunchKernelGGL(attn_step_merge_kernel<E>, dim3(a.n_rows, a.H), dim3(128), 0, stream, a);
    return pcb_check_launch("attn_step_kernel");
}

}  // namespace

PCB_EXPORT int pcb_attn_step_fits(int32_t dtype, int32_t H, int32_t Hkv, int32_t dim, int32_t vdim, int32_t rot_dims, int32_t latent) {
    if ((dtype != PCB_BF16 && dtype != PCB_F32) || H <= 0 || Hkv <= 0 || H % Hkv != 0 || dim % 8 != 0 || vdim % 8 != 0 || dim <= 0 || vdim <= 0) return 0;
    if (rot_dims % 8 != 0 || rot_dims < 0 || rot_dims > 2 * MAX_PAIRS) return 0;
    if (latent) return Hkv == 1 && vdim % 32 == 0 && vdim <= 192 && dim - vdim <= 64 && dim >= vdim && dim <= 256 && rot_dims == dim - vdim;
    return dim <= 128 && vdim <= 128 && rot_dims <= dim;
}

PCB_EXPORT int pcb_attn_step(const pcb_attn_step_args* a, void* stream) {
    PCB_REQUIRE(a && a->struct_bytes == sizeof(pcb_attn_step_args), PCB_ERR_ARG, "pcb_attn_step: struct size mismatch");
    PCB_REQUIRE(pcb_attn_step_fits(a->dtype, a->H, a->Hkv, a->dim, a->vdim, a->rot_dims, a->latent), PCB_ERR_ARG,
                "pcb_attn_step: heads it does not take (columns in eights: keys and values of up to 128, a latent of up to 192 in"
                " thirty-twos with up to 64 rotated)");
    PCB_REQUIRE(a->n_rows >= 0 && a->n_rows <= 65535 && a->Hkv * ((a->H / a->Hkv + 15) / 16) <= 65535, PCB_ERR_ARG, "pcb_attn_step: bad sizes");
    if (a->n_rows == 0) return PCB_OK;
    PCB_REQUIRE(a->p && a->tiles && a->k && a->v && a->out && (a->rot_dims == 0 || a->freqs) && (!a->latent || a->q), PCB_ERR_ARG, "pcb_attn_step: null pointer");
    PCB_REQUIRE((!a->blend || (a->other && a->ld_other >= (int64_t)a->Hkv * a->vdim)) && (!a->keep || a->ld_keep >= (int64_t)a->Hkv * a->vdim) &&
                    (!a->gate || a->ldg >= a->H) && a->ldo >= (int64_t)a->H * (a->up ? a->up_dim : a->vdim) && (!a->latent || a->ldq >= (int64_t)a->H * a->dim) &&
                    a->k_cols >= (a->latent ? 0 : a->dim) && a->k_row_stride >= a->dim && a->v_row_stride >= a->vdim && a->k_slot_stride >= 0 && a->k_head_stride >= 0 &&
                    a->v_slot_stride >= 0 && a->v_head_stride >= 0 && a->q_head_stride >= 0 && a->q_at >= 0 && a->k_at >= 0 && a->v_at >= 0,
                PCB_ERR_ARG, "pcb_attn_step: bad strides");
    PCB_REQUIRE(!a->up || (a->latent && !a->sink && !a->gate && a->up_gate && a->up_dim > 0 && a->up_dim <= 128 && a->up_dim % 8 == 0 && a->part &&
                           (uintptr_t)a->up % 16 == 0 && a->ld_up_gate >= (int64_t)a->H * a->up_dim),
                PCB_ERR_ARG, "pcb_attn_step: up-projections of a latent's heads, up to 128 columns in eights, with their gates and scratch");
    PCB_REQUIRE((a->n_splits <= 1 && !a->up) || (a->part && (uintptr_t)a->part % 16 == 0 && a->n_splits <= 64), PCB_ERR_ARG,
                "pcb_attn_step: up to 64 runs, with their scratch in whole 16 bytes");
    const int es = a->dtype == PCB_BF16 ? 2 : 4;
    const int64_t whole = a->k_slot_stride | a->k_head_stride | a->k_row_stride | a->v_slot_stride | a->v_head_stride | a->v_row_stride | a->ldo | (a->latent ? a->ldq : 0);
    PCB_REQUIRE(whole * es % 16 == 0 && ((uintptr_t)a->k | (uintptr_t)a->v | (uintptr_t)a->out | (uintptr_t)a->q) % 16 == 0, PCB_ERR_ARG,
                "pcb_attn_step: cached rows and results begin at whole 16 bytes");
    pcb_attn_step_args q = *a;
    if (q.n_splits < 1) q.n_splits = 1;                              // (both launches lay the runs out by it)
    return q.dtype == PCB_BF16 ? dispatch<pcb::bf16_t>(q, (hipStream_t)stream) : dispatch<float>(q, (hipStream_t)stream);
}
