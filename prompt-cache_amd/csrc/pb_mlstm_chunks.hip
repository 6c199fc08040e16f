// The matrix memory of an mLSTM layer on the matrix cores, for whole segments of tokens (pcb_mlstm_prompt), and as one-token steps
// (pcb_mlstm_step).  Both go on to the head's output norm and gate.  (pb_mlstm.hip: the same memory token by token, for sizes these do not take.)
//
// Within a segment let F_t be the running sum of the log forget gates, b_j = li_j - F_j, and (S, n, m) the state before it.  Then
//   M_t = max(m, max_{j <= t} b_j),   m_t = F_t + M_t                     (the recurrence's running maximum, unrolled)
//   P_tj = (q_t k_j) exp(b_j - M_t)  (j <= t),   e_t = exp(m - M_t)
//   num_t = e_t S^T q_t + sum_j P_tj v_j,   q_t n_t = e_t (n q_t) + sum_j P_tj,   h_t = num_t / (max(|q_t n_t|, exp(-m_t)) + 1e-6)
// and the segment's own contribution to the state is S' = sum_j exp(b_j - B) k_j v_j^T, n' = sum_j exp(b_j - B) k_j, m' = F_end + B with
// B = max_j b_j.  F and b are differences of long sums: they are summed in 64 bits and kept as a float and its remainder.
//
//   1. mlstm_local_kernel   per (segment, head): S', n', m', F_end
//   2. mlstm_starts_kernel  the segments of a request in a row: every segment's start state; S and n behind the last one go to the slot
//   3. mlstm_rows_kernel    per (segment, head): h_t, its norm and gate; the slot's m
//
// All products with states or weights are fp32 (v_mfma_f32_16x16x4_f32); q k^T is the type's own product, exact in bf16.  Nothing passes through
// LDS but the gates: column tile n of a product stands for the columns 8 i + n (i = lane & 15), so that one 16-byte read of eight neighbouring
// elements of a row (32 in fp32) feeds eight tiles, and the scores are taken as K Q^T, whose result is the next product's operand as it lies.
//
// What bounds it (2048 tokens, 16 heads of 128, us): two passes token by token and the chain 318 + 60, then the norm 10; the three
// launches 22 + 18 + 31.  1 and 3: the fp32 products (7 and 14 at the rate of the matrix cores) and a workgroup's own chain of loads; 2: memory (67 MB).
#include <type_traits>

#include "pb_common.h"

namespace {
using namespace pcb;

__device__ __forceinline__ float soft_cap(float z, float cap) { return cap > 0.0f ? cap * tanhf(z / cap) : z; }
__device__ __forceinline__ float log_sigmoid(float z) { return fminf(z, 0.0f) - log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ f4 mma4(float a, float b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

__device__ __forceinline__ void load2(const bf16_t* p, float (&o)[2]) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(p);
    o[0] = __uint_as_float(w << 16), o[1] = __uint_as_float(w & 0xffff0000u);
}
__device__ __forceinline__ void load2(const float* p, float (&o)[2]) { o[0] = p[0], o[1] = p[1]; }
struct __attribute__((packed, aligned(4))) Floats8 {
    float v[8];
};
struct __attribute__((packed, aligned(4))) Floats4 {
    float v[4];
};

__device__ __forceinline__ double up(double v, int o) { return __shfl_up(v, o, 64); }

// one wave: the gates of the segment's n tokens, lane l the NT tokens from l NT on.  b[u] = li - F, F[u] = the running sum, 64 bits; tokens past n
// have b = -infinity, as those with a closed input gate (li = -infinity): nothing of them is taken, a segment of such tokens alone leaves S' = n' = 0 and
// m' = -infinity.  (A log forget gate below -1e8 counts as -1e8: what it forgets is gone either way, and sums and differences stay finite.)
template <typename E, int NT>
__device__ __forceinline__ void segment_gates(const pcb_mlstm_args& a, int64_t row0, int n, int h, int lane, double (&b)[NT], double (&F)[NT]) {
    const E* gi = (const E*)a.gi + row0 * a.ldgi + h;
    const E* gf = (const E*)a.gf + row0 * a.ldgf + h;
    float li[NT], lf[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int t = lane * NT + u, tc = t < n ? t : n - 1;
        li[u] = to_f32(gi[tc * a.ldgi]);
        lf[u] = to_f32(gf[tc * a.ldgf]);
    }
    double run = 0.0;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const float l = log_sigmoid(soft_cap(lf[u], a.gate_cap));
        run += lane * NT + u < n ? (l < -1e8f ? -1e8f : l) : 0.0f;
        F[u] = run;
    }
    double before = run;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double x = up(before, o);
        if (lane >= o) before += x;
    }
    before -= run;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        F[u] += before;
        b[u] = lane * NT + u < n ? (double)soft_cap(li[u], a.gate_cap) - F[u] : -__builtin_inf();
    }
}

// ---- 1. the segments' own contributions ---------------------------------------------------------------------------------------------------
// Wave w owns the key rows 8 i + 2 w, + 1 (two row tiles), all value columns: 16 result tiles, fed by one read of k (two elements) and one of v.
template <typename E, int NT>
__global__ __launch_bounds__(256) void mlstm_local_kernel(pcb_mlstm_args a, float* __restrict__ local, float* __restrict__ f_sum) {
    __shared__ float ws[64 * NT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, group = lane >> 4, l15 = lane & 15;
    const int32_t* rq = a.reqs + 4 * blockIdx.x;
    const int h = blockIdx.y, n = rq[2], dim = a.dim, vdim = a.vdim;
    const int64_t row0 = rq[3], rec = (int64_t)dim * vdim + dim + 1;
    float* st = local + ((int64_t)blockIdx.x * a.H + h) * rec;
    if (wave == 0) {
        double b[NT], F[NT];
        segment_gates<E, NT>(a, row0, n, h, lane, b, F);
        double top = b[0];
#pragma unroll
        for (int u = 1; u < NT; ++u) top = b[u] > top ? b[u] : top;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double x = __shfl_xor(top, o, 64);
            top = x > top ? x : top;
        }
#pragma unroll
        for (int u = 0; u < NT; ++u) ws[lane * NT + u] = b[u] == -__builtin_inf() ? 0.0f : expf((float)(b[u] - top));      // (top may be -infinity too)
        if (lane == 63) {                                                  // (its running sum is the whole segment's)
            f_sum[(int64_t)blockIdx.x * a.H + h] = (float)F[NT - 1];
            st[rec - 1] = (float)(F[NT - 1] + top);
        }
    }
    const bool d_ok = 8 * l15 < dim, c_ok = 8 * l15 < vdim;
    const E* k = (const E*)a.k + row0 * a.ldk + (int64_t)h * dim + (d_ok ? 8 * l15 + 2 * wave : 0);
    const E* v = (const E*)a.v + row0 * a.ldv + (int64_t)h * vdim + (c_ok ? 8 * l15 : 0);
    f4 acc[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[i][c] = f4{0.f, 0.f, 0.f, 0.f};
    float sn[2] = {0.0f, 0.0f};
    float kk[4][2];
    Frag<E> fv[4];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = j0 + 4 * u + group, jc = j < n ? j : n - 1;
            load2(k + jc * a.ldk, kk[u]);
            fv[u] = load8(v + jc * a.ldv);
        }
    };
    fetch(0);
    __syncthreads();
    for (int j0 = 0; j0 < n; j0 += 16) {                                   // (weights of tokens past the end are zero)
        float x[4][2];
        Frag<E> fn[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float w = ws[j0 + 4 * u + group];
            x[u][0] = w * kk[u][0], x[u][1] = w * kk[u][1];
            sn[0] += x[u][0], sn[1] += x[u][1];
            fn[u] = fv[u];
        }
        fetch(j0 + 16);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                acc[0][c] = mma4(x[u][0], at8(fn[u], c), acc[0][c]);
                acc[1][c] = mma4(x[u][1], at8(fn[u], c), acc[1][c]);
            }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        sn[i] += __shfl_xor(sn[i], 16, 64);
        sn[i] += __shfl_xor(sn[i], 32, 64);
        if (group == 0 && d_ok) st[(int64_t)dim * vdim + 8 * l15 + 2 * wave + i] = sn[i];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int d = 8 * (4 * group + r) + 2 * wave + i;
            if (d >= dim || !c_ok) continue;
            Floats8 o;
#pragma unroll
            for (int c = 0; c < 8; ++c) o.v[c] = acc[i][c][r];
            *reinterpret_cast<Floats8*>(st + (int64_t)d * vdim + 8 * l15) = o;
        }
    }
}

// ---- 2. every segment's start -----------------------------------------------------------------------------------------------------------------
// One workgroup per (chain, head, 1024 state elements).  The contributions of eight segments are requested at a time: one by one, each waits for
// a trip to memory (32 segments of 16 heads of 128 x 128: 60 us so, 18 eight at
// a time).  S and n behind the last segment go to the slot (every thread owns its
// elements); m is left to the third launch, since the other workgroups of this one still read it.
constexpr int AHEAD = 8;
__global__ __launch_bounds__(256) void mlstm_starts_kernel(const float* __restrict__ local, const float* __restrict__ f_sum, float* __restrict__ start,
                                                           float* state, int64_t slot_stride, const int32_t* __restrict__ chains, int H, int64_t rec) {
    const int32_t* ch = chains + 4 * blockIdx.x;
    const int slot = ch[0], pos0 = ch[1], seg0 = ch[2], n_seg = ch[3], h = blockIdx.y;
    const int64_t elems = rec - 1;
    float* st = state + (int64_t)slot * slot_stride + (int64_t)h * rec;
    float mm = pos0 > 0 ? st[elems] : 0.0f;
    const int64_t e0 = (int64_t)blockIdx.z * 1024 + threadIdx.x;
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = (pos0 > 0 && e0 + 256 * u < elems) ? st[e0 + 256 * u] : 0.0f;
    for (int g0 = 0; g0 < n_seg; g0 += AHEAD) {
        float lc[AHEAD][4], F[AHEAD], ml[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int64_t g = seg0 + (g0 + i < n_seg ? g0 + i : n_seg - 1);
            const float* p = local + (g * H + h) * rec;
            F[i] = f_sum[g * H + h];
            ml[i] = p[elems];
#pragma unroll
            for (int u = 0; u < 4; ++u) lc[i][u] = p[e0 + 256 * u < elems ? e0 + 256 * u : 0];
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            if (g0 + i >= n_seg) break;
            float* sg = start + ((int64_t)(seg0 + g0 + i) * H + h) * rec;
            if (blockIdx.z == 0 && threadIdx.x == 0) sg[elems] = mm;
            const float m_new = fmaxf(F[i] + mm, ml[i]);
            const float keep = expf(F[i] + mm - m_new), take = expf(ml[i] - m_new);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (e0 + 256 * u < elems) sg[e0 + 256 * u] = v[u];
                v[u] = keep * v[u] + take * lc[i][u];
            }
            mm = m_new;
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (e0 + 256 * u < elems) st[e0 + 256 * u] = v[u];
}

// A row's last tile holds tokens behind it: of weight 0, but 0 times infinity (or times what is no number) is none.  Such values are taken out of the tile,
// and what they belong to -- their column, from their token's own row on -- is set to NaN.  v: the lane's tokens `first` .. + 3 of the tile, eight columns.
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < __builtin_inff(); }
__device__ __forceinline__ void clear(Frag<bf16_t>& f, int e) { f.v[e >> 1] &= e & 1 ? 0xffffu : 0xffff0000u; }
__device__ __forceinline__ void clear(Frag<float>& f, int e) { f.v[e] = 0.0f; }
template <typename E>
__device__ __forceinline__ bool all_finite(const Frag<E> (&v)[4]) {
    float z = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 8; ++c) z = __builtin_fmaf(at8(v[r], c), 0.0f, z);
    return z == 0.0f;
}
template <typename E>
__device__ __forceinline__ void keep_behind(Frag<E> (&v)[4], f4 (&acc)[8], int first) {
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        int j = 16;
#pragma unroll
        for (int r = 3; r >= 0; --r)
            if (!finite(at8(v[r], c))) {
                j = first + r;
                clear(v[r], c);
            }
        j = min(j, __shfl_xor(j, 16, 64));
        j = min(j, __shfl_xor(j, 32, 64));
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (first + e >= j) acc[c][e] = __builtin_nanf("");
    }
}

// ---- 3. the rows ----------------------------------------------------------------------------------------------------------------------------------
// A wave owns 16 rows.  The norm's and the gate's part is that of pcb_gated_norm with a norm per head.
template <typename E, int NT>
__global__ __launch_bounds__(256 * NT, NT > 1 ? 1 : sizeof(E) == 2 ? 3 : 2) void mlstm_rows_kernel(pcb_mlstm_args a, pcb_mlstm_norm_args o, const float* __restrict__ local,
                                                              const float* __restrict__ f_sum, const float* __restrict__ start) {
    __shared__ float bh[64 * NT], bl[64 * NT], Mh[64 * NT], Ml[64 * NT], em[64 * NT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, group = lane >> 4, l15 = lane & 15;
    const int32_t* rq = a.reqs + 4 * blockIdx.x;
    const int h = blockIdx.y, n = rq[2], dim = a.dim, vdim = a.vdim;
    const int64_t row0 = rq[3], rec = (int64_t)dim * vdim + dim + 1, at = ((int64_t)blockIdx.x * a.H + h) * rec;
    const float* S = start + at;
    const float* sn = S + (int64_t)dim * vdim;
    const float m0 = S[rec - 1];
    const int t0 = 16 * wave, t = t0 + l15;
    const int64_t tc = row0 + (t < n ? t : n - 1);
    const E* q = (const E*)a.q + tc * a.ldq + (int64_t)h * dim;
    const int ns = (dim + 31) / 32;
    Frag<E> fq[4];
    float qn = 0.0f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int d = 32 * s + 8 * group;
        zero8(fq[s]);
        if (d < dim) fq[s] = load8(q + d);
    }
    const bool c_ok = 8 * l15 < vdim;
    const int c0 = c_ok ? 8 * l15 : 0;
    f4 acc[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] = f4{0.f, 0.f, 0.f, 0.f};
    // SR rows of S ahead of the products: the next ones are under way meanwhile, the first ones while wave 0 adds up the gates
    constexpr int SR = NT == 4 ? 2 : 4, PER = 8 / SR;
    Floats8 xs[SR];
    float xn[SR];
    auto state_rows = [&](int p) {
#pragma unroll
        for (int e = 0; e < SR; ++e) {
            const int d = 32 * (p / PER) + 8 * group + SR * (p % PER) + e, dc = d < dim ? d : 0;
            xs[e] = *reinterpret_cast<const Floats8*>(S + (int64_t)dc * vdim + c0);
            xn[e] = sn[dc];
        }
    };
    state_rows(0);
    if (wave == 0) {
        double b[NT], F[NT];
        segment_gates<E, NT>(a, row0, n, h, lane, b, F);
        double run = b[0];
#pragma unroll
        for (int u = 1; u < NT; ++u) run = b[u] > run ? b[u] : run;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {                                 // the largest b of this lane's tokens and all before them
            const double x = up(run, s);
            if (lane >= s && x > run) run = x;
        }
        double M = up(run, 1);
        if (lane == 0 || (double)m0 > M) M = (double)m0;
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int t = lane * NT + u;
            M = b[u] > M ? b[u] : M;
            const float hi = (float)b[u], Hi = (float)M;
            bh[t] = hi;
            bl[t] = b[u] == -__builtin_inf() ? 0.0f : (float)(b[u] - (double)hi);
            Mh[t] = Hi;
            Ml[t] = (float)(M - (double)Hi);
            em[t] = expf(-(float)(F[u] + M));
        }
        if (lane == 0 && a.end_slots && a.end_slots[blockIdx.x] >= 0) {
            const float m1 = f_sum[(int64_t)blockIdx.x * a.H + h] + m0, m2 = local[at + rec - 1];
            a.end_state[(int64_t)a.end_slots[blockIdx.x] * a.end_slot_stride + (int64_t)h * rec + rec - 1] = fmaxf(m1, m2);
        }
    }
    if (t0 < n) {
#pragma unroll
        for (int p = 0; p < 4 * PER; ++p) {
            if (p >= ns * PER) continue;
            Floats8 x[SR];
#pragma unroll
            for (int e = 0; e < SR; ++e) {
                x[e] = xs[e];
                qn += at8(fq[p / PER], SR * (p % PER) + e) * xn[e];
            }
            if (p + 1 < ns * PER) state_rows(p + 1);
#pragma unroll
            for (int e = 0; e < SR; ++e)
#pragma unroll
                for (int c = 0; c < 8; ++c) acc[c] = mma4(at8(fq[p / PER], SR * (p % PER) + e), x[e].v[c], acc[c]);
        }
    }
    const E* K = (const E*)a.k + row0 * a.ldk + (int64_t)h * dim;
    const E* V = (const E*)a.v + row0 * a.ldv + (int64_t)h * vdim + c0;
    Frag<E> fk[4], fv[4];
    auto keys = [&](int j0) {
        const int jk = j0 + l15 < n ? j0 + l15 : n - 1;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int d = 32 * u + 8 * group;
            zero8(fk[u]);
            if (d < dim) fk[u] = load8(K + jk * a.ldk + d);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = j0 + 4 * group + r;
            fv[r] = load8(V + (j < n ? j : n - 1) * a.ldv);
        }
    };
    keys(0);
    __syncthreads();
    if (t0 >= n) return;                                                   // (uniform over the wave; no barrier follows)
    qn += __shfl_xor(qn, 16, 64);
    qn += __shfl_xor(qn, 32, 64);
    const float th = Mh[t], tl = Ml[t];
    const float et = expf((m0 - th) - tl) * a.q_scale;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float x = __shfl(et, 4 * group + r, 64);
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[c][r] *= x;
    }
    float ps = 0.0f;
    for (int j0 = 0; j0 <= t0; j0 += 16) {
        if (j0 == t0 && __any(!all_finite(fv))) keep_behind(fv, acc, 4 * group);
        f4 s = f4{0.f, 0.f, 0.f, 0.f};
        Frag<E> v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (u < ns) s = mma(fk[u], fq[u], s);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = fv[r];
        if (j0 < t0) keys(j0 + 16);
        // the lane's results: row t, keys j0 + 4 group + r
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int j = j0 + 4 * group + r;
            const float p = j <= t ? s[r] * (expf((bh[j] - th) + (bl[j] - tl)) * a.q_scale) : 0.0f;
            ps += p;
#pragma unroll
            for (int c = 0; c < 8; ++c) acc[c] = mma4(p, at8(v[r], c), acc[c]);
        }
    }
    ps += __shfl_xor(ps, 16, 64);
    ps += __shfl_xor(ps, 32, 64);
    const float den = fmaxf(fabsf(et * qn + ps), em[t]) + 1e-6f;
    const float* gain = o.gain ? o.gain + (int64_t)h * vdim + c0 : nullptr;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int tr = t0 + 4 * group + r;
        const float dr = __shfl(den, 4 * group + r, 64);
        float y[8], ss = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            y[c] = acc[c][r] / dr;
            if (c_ok) ss += y[c] * y[c];
        }
#pragma unroll
        for (int x = 1; x < 16; x <<= 1) ss += __shfl_xor(ss, x, 64);
        if (tr >= n || !c_ok) continue;
        const float inv = 1.0f / sqrtf(ss / (float)vdim + o.eps);
        float g[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) g[c] = 1.0f;
        if (o.gate) {
            const E* gp = (const E*)o.gate + (row0 + tr) * o.ldg + (int64_t)h * vdim + c0;
            float g0[4], g1[4];
            load4(gp, true, 4, g0);
            load4(gp + 4, true, 4, g1);
#pragma unroll
            for (int c = 0; c < 4; ++c) g[c] = g0[c], g[4 + c] = g1[c];
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) y[c] *= inv * (gain ? gain[c] : 1.0f) * g[c];
        E* out = (E*)o.out + (row0 + tr) * o.ldo + (int64_t)h * vdim + c0;
        store4(out, y[0], y[1], y[2], y[3]);
        store4(out + 4, y[4], y[5], y[6], y[7]);
    }
}

// ---- one token per request --------------------------------------------------------------------------------------------------------------------
// One workgroup of 1024 threads per (request, head); a row of S is shared by LR lanes of four columns each, so a thread has NI rows, all of them
// requested at once with everything else.  A step is one trip to memory and two sums.
// us, 8 requests x 16 heads of 128: block by block as a prompt 22, the norm 4.5; so 7.9 (17 MB); 2 x 8 heads in fp32 17.7 + 4.5, 5.9.
template <typename E, int LR, int NI>
__global__ __launch_bounds__(1024) void mlstm_step_kernel(pcb_mlstm_args a, pcb_mlstm_norm_args o) {
    constexpr int RP = 1024 / LR, LDP = 4 * LR + 4;
    __shared__ __attribute__((aligned(16))) float part[16][LDP];
    __shared__ float part_n[16], red[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t* rq = a.reqs + 4 * blockIdx.x;
    const int slot = rq[0], pos0 = rq[1], h = blockIdx.y, dim = a.dim, vdim = a.vdim;
    const int64_t row = rq[3], rec = (int64_t)dim * vdim + dim + 1;
    float* st = a.state + (int64_t)slot * a.slot_stride + (int64_t)h * rec;
    float* st_n = st + (int64_t)dim * vdim;
    const int c = 4 * (tid % LR), d0 = tid / LR;
    const bool c_ok = c < vdim;
    const int cc = c_ok ? c : 0;
    const E* q = (const E*)a.q + row * a.ldq + (int64_t)h * dim;
    const E* k = (const E*)a.k + row * a.ldk + (int64_t)h * dim;
    Floats4 S[NI];
    float n[NI], kd[NI], qd[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int d = d0 + RP * i, dc = d < dim ? d : 0;
        S[i] = *reinterpret_cast<const Floats4*>(st + (int64_t)dc * vdim + cc);
        n[i] = st_n[dc];
        kd[i] = to_f32(k[dc]);
        qd[i] = to_f32(q[dc]) * a.q_scale;
    }
    float m = st_n[dim];
    float v[4];
    load4((const E*)a.v + row * a.ldv + (int64_t)h * vdim + cc, true, 4, v);
    const float zi = to_f32(((const E*)a.gi)[row * a.ldgi + h]), zf = to_f32(((const E*)a.gf)[row * a.ldgf + h]);
    // (what the last part needs)
    const int64_t oc = (int64_t)h * vdim + tid;
    const bool mine = tid < vdim;
    const float gate = mine && o.gate ? to_f32(((const E*)o.gate)[row * o.ldg + oc]) : 1.0f;
    const float gain = mine && o.gain ? o.gain[oc] : 1.0f;

    const float li = soft_cap(zi, a.gate_cap), lf = log_sigmoid(soft_cap(zf, a.gate_cap));
    if (pos0 <= 0) m = 0.0f;
    const float m_new = fmaxf(lf + m, li);
    const float keep = expf(lf + m - m_new), take = expf(li - m_new);
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f}, accn = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int d = d0 + RP * i;
        if (d >= dim) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            S[i].v[e] = keep * (pos0 > 0 ? S[i].v[e] : 0.0f) + kd[i] * (take * v[e]);
            acc[e] += S[i].v[e] * qd[i];
        }
        n[i] = keep * (pos0 > 0 ? n[i] : 0.0f) + take * kd[i];
        accn += n[i] * qd[i];
        if (c_ok) *reinterpret_cast<Floats4*>(st + (int64_t)d * vdim + c) = S[i];
    }
    // (the rows of a wave meet by shuffles, the waves in LDS)
#pragma unroll
    for (int x = LR; x < 64; x <<= 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += __shfl_xor(acc[e], x, 64);
        accn += __shfl_xor(accn, x, 64);
    }
    if (lane < LR) *reinterpret_cast<f4*>(&part[wave][c]) = f4{acc[0], acc[1], acc[2], acc[3]};
    if (lane == 0) part_n[wave] = accn;
    __syncthreads();
    // (n and m are written behind the barrier: every thread has read m)
    if (c == 0) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (d0 + RP * i < dim) st_n[d0 + RP * i] = n[i];
    }
    if (tid == 0) st_n[dim] = m_new;
    float y = 0.0f;
    if (wave < 4 && mine) {
        float num = 0.0f, nq = 0.0f;
#pragma unroll
        for (int w = 0; w < 16; ++w) num += part[w][tid], nq += part_n[w];
        y = num / (fmaxf(fabsf(nq), expf(-m_new)) + 1e-6f);
    }
    if (wave < 4) {
        const float ss = wave_sum(y * y);
        if (lane == 0) red[wave] = ss;
    }
    __syncthreads();
    if (!mine) return;
    const float inv = 1.0f / sqrtf(((red[0] + red[1]) + (red[2] + red[3])) / (float)vdim + o.eps);
    ((E*)o.out)[row * o.ldo + oc] = from_f32<E>(y * (inv * gain * gate));
}

// eight neighbouring columns of a row in 16-byte pieces, gate and output in pieces of four
bool aligned(const pcb_mlstm_args& a, const pcb_mlstm_norm_args& o) {
    const int es = a.dtype == PCB_BF16 ? 2 : 4;
    auto whole = [&](const void* p, int64_t ld, int bytes) { return (uintptr_t)p % bytes == 0 && ld * es % bytes == 0; };
    return a.dim % 8 == 0 && a.vdim % 8 == 0 && whole(a.q, a.ldq, 16) && whole(a.k, a.ldk, 16) && whole(a.v, a.ldv, 16) &&
           (!o.gate || whole(o.gate, o.ldg, 4 * es)) && whole(o.out, o.ldo, 4 * es);
}
int check(const pcb_mlstm_args* a, const pcb_mlstm_norm_args* o, const char* what) {
    PCB_REQUIRE(a && o && a->struct_bytes == sizeof(pcb_mlstm_args) && o->struct_bytes == sizeof(pcb_mlstm_norm_args), PCB_ERR_ARG,
                "%s: struct size mismatch", what);
    PCB_REQUIRE(a->dtype == PCB_BF16 || a->dtype == PCB_F32, PCB_ERR_ARG, "%s: unknown dtype", what);
    PCB_REQUIRE(a->n_reqs >= 0 && a->H > 0 && a->dim > 0 && a->vdim > 0 && a->ldq >= (int64_t)a->H * a->dim && a->ldk >= (int64_t)a->H * a->dim &&
                    a->ldv >= (int64_t)a->H * a->vdim && a->ldgi >= a->H && a->ldgf >= a->H && o->ldo >= (int64_t)a->H * a->vdim &&
                    (!o->gate || o->ldg >= (int64_t)a->H * a->vdim) &&
                    a->slot_stride >= (int64_t)a->H * ((int64_t)a->dim * a->vdim + a->dim + 1),
                PCB_ERR_ARG, "%s: bad sizes", what);
    PCB_REQUIRE(a->n_reqs == 0 || (a->q && a->k && a->v && a->gi && a->gf && a->reqs && a->state && o->out), PCB_ERR_ARG, "%s: null pointer", what);
    return PCB_OK;
}

template <typename E>
int step(const pcb_mlstm_args& a, const pcb_mlstm_norm_args& o, hipStream_t stream) {
    const dim3 grid(a.n_reqs, a.H), block(1024);
    auto go = [&](auto lr, auto ni) {
        hipLaunchKernelGGL((mlstm_step_kernel<E, decltype(lr)::value, decltype(ni)::value>), grid, block, 0, stream, a, o);
    };
    if (a.vdim <= 64)
        a.dim <= 128 ? go(std::integral_constant<int, 16>{}, std::integral_constant<int, 2>{})
                     : go(std::integral_constant<int, 16>{}, std::integral_constant<int, 4>{});
    else if (a.vdim <= 128)
        a.dim <= 128 ? go(std::integral_constant<int, 32>{}, std::integral_constant<int, 4>{})
                     : go(std::integral_constant<int, 32>{}, std::integral_constant<int, 8>{});
    else
        go(std::integral_constant<int, 64>{}, std::integral_constant<int, 8>{});
    return pcb_check_launch("mlstm_step_kernel");
}

template <typename E, int NT>
int prompt(const pcb_mlstm_args& a, const pcb_mlstm_norm_args& o, const int32_t* chains, int n_chains, float* local, float* f_sum, float* start,
           hipStream_t stream) {
    const int64_t rec = (int64_t)a.dim * a.vdim + a.dim + 1;
    const dim3 grid(a.n_reqs, a.H);
    hipLaunchKernelGGL((mlstm_local_kernel<E, NT>), grid, dim3(256), 0, stream, a, local, f_sum);
    hipLaunchKernelGGL(mlstm_starts_kernel, dim3(n_chains, a.H, (unsigned)((rec - 1 + 1023) / 1024)), dim3(256), 0, stream, local, f_sum, start, a.state,
                       a.slot_stride, chains, a.H, rec);
    hipLaunchKernelGGL((mlstm_rows_kernel<E, NT>), grid, dim3(256 * NT), 0, stream, a, o, local, f_sum, start);
    return pcb_check_launch("mlstm_rows_kernel");
}

}  // namespace

PCB_EXPORT int pcb_mlstm_step(const pcb_mlstm_args* a, const pcb_mlstm_norm_args* o, void* stream) {
    int rc = check(a, o, "pcb_mlstm_step");
    if (rc != PCB_OK || a->n_reqs == 0) return rc;
    PCB_REQUIRE(a->dim <= 256 && a->vdim <= 256 && (a->dim <= 128 || a->vdim <= 128) && a->vdim % 4 == 0 && a->ldv % 4 == 0 &&
                    (uintptr_t)a->v % (a->dtype == PCB_BF16 ? 8 : 16) == 0,
                PCB_ERR_ARG, "pcb_mlstm_step: up to 256 x 128 or 128 x 256 columns per head, values in whole chunks of four");
    return a->dtype == PCB_BF16 ? step<pcb::bf16_t>(*a, *o, (hipStream_t)stream) : step<float>(*a, *o, (hipStream_t)stream);
}

PCB_EXPORT int pcb_mlstm_prompt(const pcb_mlstm_args* a, const pcb_mlstm_norm_args* o, const int32_t* chains, int32_t n_chains, int32_t max_tokens,
                                float* local, float* f_sum, float* start, void* stream) {
    int rc = check(a, o, "pcb_mlstm_prompt");
    if (rc != PCB_OK || a->n_reqs == 0) return rc;
    PCB_REQUIRE(chains && n_chains > 0 && local && f_sum && start && a->end_slots && a->end_state == a->state && a->end_slot_stride == a->slot_stride,
                PCB_ERR_ARG, "pcb_mlstm_prompt: chains, scratch and end slots within the states are needed");
    PCB_REQUIRE(a->dim <= 128 && a->vdim <= 128 && max_tokens > 0 && max_tokens <= 256 && aligned(*a, *o), PCB_ERR_ARG,
                "pcb_mlstm_prompt: up to 128 columns per head in whole chunks of eight, segments of up to 256 tokens");
    hipStream_t s = (hipStream_t)stream;
    if (a->dtype == PCB_BF16)
        return max_tokens <= 64    ? prompt<pcb::bf16_t, 1>(*a, *o, chains, n_chains, local, f_sum, start, s)
               : max_tokens <= 128 ? prompt<pcb::bf16_t, 2>(*a, *o, chains, n_chains, local, f_sum, start, s)
                                   : prompt<pcb::bf16_t, 4>(*a, *o, chains, n_chains, local, f_sum, start, s);
    return max_tokens <= 64    ? prompt<float, 1>(*a, *o, chains, n_chains, local, f_sum, start, s)
           : max_tokens <= 128 ? prompt<float, 2>(*a, *o, chains, n_chains, local, f_sum, start, s)
                               : prompt<float, 4>(*a, *o, chains, n_chains, local, f_sum, start, s);
}
