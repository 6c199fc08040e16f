// pcb_attn_talk for bf16 prompts with heads of 128 columns and four query heads to a key head (4, 8 or 16 heads): scores, mixing, softmax and values in
// one pass over the keys, without a band of scores in memory.
//
// A unit is 16 / H x 4 queries of all heads: "lane heads" 0 .. 15 = (query quarter, head).  It walks its keys 64 at a time with four waves, each of which
// first has 16 of the keys and all lane heads, then the 16 rows (heads x queries) of one key head and quarter and all 64 keys:
//   scores   Q K^T with the four heads of a key head x four queries as rows: a result lane then holds head = its lane group, query = its register,
//            which is what the mixing's product (weights in fp32, v_mfma_f32_16x16x4_f32) wants as an operand: nothing is moved in between
//   softmax  the mixed scores come out as lane = lane head, registers = neighbouring keys; the four waves agree on the maxima through LDS
//   values   weights as a hi + lo pair of bf16 through LDS, values by transposed reads of the key tile
// The next keys are requested into registers before a tile is worked on and pass into the second of two tiles in LDS beside the exchange of the maxima, so
// that a tile's values and the next one's scores have no barrier between them.
//
// What bounds it: a tile's chain (scores, maxima, weights, values, three barriers) at two waves per SIMD: matrix cores busy 27 %, vector unit 33 %, LDS 25 %
// of the time; LDS bank conflicts, 23 % before the spreads below, are 1 %.  us (scores into a band of memory and values behind it, then here), window 1024:
// 2048 rows of 16 heads 110.6 and 68.5, 8 heads 72.7 and 41.6, 4 heads 60.7 and 31.6; 6 x 300 rows of 16 heads 50.8 and 28.7, 100 rows 30.4 and 17.4, 9 rows
// 29.5 and 14.3; 200 rows of 16 heads behind 1000 keys 70.7 and 32.  One tile in LDS and four barriers: 16 heads 72.4, 8 heads 41.8, 4 heads 32.4.
#include <type_traits>

#include "pb_attn_common.h"

namespace {
using namespace pcb;

constexpr int D = 128, KT = 64;

// Where things lie in LDS, so that the lanes of one access fall on different banks.
// A key row is 16 chunks of eight columns; chunk c of key j lies at c ^ key_spread(j): reads of chunks c, c + 1 of 16 keys (operand of the scores) and
// transposed reads of 2 x 16 columns of 8 neighbouring keys.
__device__ __forceinline__ int key_spread(int j) { return (((j & 7) ^ (j >> 1 & 4)) << 1) | (j >> 3 & 1); }
// A row of weights (64 keys, block b of 16 rows, row r) is 8 chunks of eight; chunk c lies at c ^ row_spread(b, r), its halves change places in the
// blocks 2 and 3.
__device__ __forceinline__ int row_spread(int b, int r) { return (r >> 1) ^ (b & 1); }

// HKV key heads (H = 4 HKV).  `parts` workgroups share the keys of the same rows: each leaves [part][row][head]{D sums} and, behind all of these,
// {maximum, denominator} in the scratch, to be merged by talk_merge_kernel.
template <int HKV, int NU>
__global__ __launch_bounds__(256 * NU, 2) void talk_prompt_kernel(pcb_attn_talk_args a, const int32_t* __restrict__ tiles, int parts, int n_rows) {
    constexpr int H = 4 * HKV, UQ = 16 / HKV, WQ = NU * UQ;      // queries of a unit, of a workgroup
    constexpr int RP = 16 * NU, NCH = KT * HKV / RP;              // key rows staged at a time; 16-byte chunks of a key tile per thread
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    bf16_t* Ks = reinterpret_cast<bf16_t*>(lds);                 // [HKV][KT][D], two of them
    bf16_t* Kn = Ks + HKV * KT * D;                              // the next tile's
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), sub = wave & 3, unit = wave >> 2, g = lane >> 4, l15 = lane & 15;
    bf16_t* const Ps = Kn + HKV * KT * D + unit * 2 * 64 * KT;   // the unit's weights: [hi, lo][4][16 rows][KT]
    const int32_t* const t = tiles + 4 * (gridDim.x - 1 - blockIdx.x);        // (later rows see more keys: they start first)
    const int w_rows = t[2] - WQ * (int)blockIdx.y, w_first = t[1] + WQ * (int)blockIdx.y;
    if (w_rows <= 0) return;                                     // (uniform over the workgroup)
    const int last = w_first + (w_rows < WQ ? w_rows : WQ) - 1;
    const int window = a.window > 0 ? a.window : 0x3fffffff;
    const int j_min = w_first - window + 1 > 0 ? w_first - window + 1 : 0;
    const int nq = w_rows - UQ * unit, q0 = w_first + UQ * unit, row0 = t[3] + WQ * blockIdx.y + UQ * unit;       // the unit's rows
    const int n_kt = (last - j_min + KT) / KT;                   // key tiles, this workgroup's among them
    const int j_lo = j_min + KT * (int)((int64_t)n_kt * blockIdx.z / parts), j_hi = j_min + KT * (int)((int64_t)n_kt * (blockIdx.z + 1) / parts);
    const bf16_t* const C = (const bf16_t*)a.cache + (int64_t)t[0] * a.slot_stride;

    u32x4 next[NCH];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int u = 0; u < NCH; ++u) {
            const int j = j0 + (tid >> 4) + RP * (u % (KT / RP));
            // (keys past the last repeat it: masked)
            next[u] = *reinterpret_cast<const u32x4*>(C + (int64_t)(u / (KT / RP)) * a.head_stride + (int64_t)(j <= last ? j : last) * D + 8 * (tid & 15));
        }
    };
    fetch(j_lo);

    // for scores, mixing and softmax a wave has all heads and queries x 16 keys of the tile
    Frag<bf16_t> fq[4][4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int rq = (l15 & 3) + 4 * (c / HKV);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
            zero8(fq[c][st]);
            if (rq < nq) fq[c][st] = load8((const bf16_t*)a.q + (int64_t)(row0 + rq) * a.ldq + (4 * (c % HKV) + (l15 >> 2)) * D + 32 * st + 8 * g);
        }
    }
    // Scores are kept in units of ln 2, so that a weight is one v_exp_f32: scale and log2 e go into the mixing's weights (rounded once, from 64 bits), and the
    // distance bias, which is linear, is mixed once.  That leaves out the roundings of every head's scaled and biased score: the weights' error against
    // 64 bits is 0.2 to 1.0 of that of scores mixed from those (2048 keys of 16 heads 3.2e-6, 1.5e-5 that way; no bias 2.7e-7, 2.8e-7).
    const double log2e = 1.4426950408889634;
    const int my = l15 % H;                                      // this lane's head
    const int i0 = q0 + 4 * (l15 / H);                           // position of its query 0
    float mix[HKV], slope;
    {
        double s = 0.0;
        for (int h = 0; h < H; ++h) s += (double)a.talk[my * H + h] * (a.slopes ? (double)a.slopes[h] : 0.0);
        slope = (float)(s * log2e);
#pragma unroll
        for (int c = 0; c < HKV; ++c) mix[c] = (float)((double)a.talk[my * H + 4 * c + g] * (double)a.scale * log2e);
    }
    float rm[4], rl[4];                                          // running maximum and this lane's part of the denominator, per query
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        rm[r] = a.sink ? 0.0f : -INFINITY;                       // (the sink is a score of 0)
        rl[r] = a.sink && sub == 0 && g == 0 && blockIdx.z == 0 ? 1.0f : 0.0f;
    }
    // for the values it has the 16 rows (heads of a key head x queries) of block `sub`: rows 4 head + query
    f4 acc[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) acc[n] = f4{0.f, 0.f, 0.f, 0.f};

    auto stage = [&](bf16_t* K) {
#pragma unroll
        for (int u = 0; u < NCH; ++u) {
            const int j = (tid >> 4) + RP * (u % (KT / RP));
            *reinterpret_cast<u32x4*>(K + ((u / (KT / RP)) * KT + j) * D + 8 * ((tid & 15) ^ key_spread(j & 15))) = next[u];
        }
    };
    stage(Ks);
    __syncthreads();
    for (int j0 = j_lo; j0 < j_hi; j0 += KT) {
        if (j0 + KT < j_hi) fetch(j0 + KT);

        const int js = j0 + 16 * sub;                            // this wave's keys
        f4 s[4];
#pragma unroll
        for (int k = 0; k < HKV; ++k) {
            Frag<bf16_t> fk[4];
#pragma unroll
            for (int st = 0; st < 4; ++st) fk[st] = load8(Ks + (k * KT + 16 * sub + l15) * D + 8 * ((4 * st + g) ^ key_spread(l15)));
#pragma unroll
            for (int c = k; c < 4; c += HKV) {
                s[c] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < 4; ++st) s[c] = mma(fq[c][st], fk[st], s[c]);
            }
        }
        // mixed scores p[query][key 4 g + e]
        f4 p[4];
        const float dj = (float)(js + 4 * g - i0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // (heads of another quarter are products of their own: what a lane does not keep must not reach what it keeps)
#pragma unroll
            for (int v = 0; v < 4 / HKV; ++v) {
                f4 m = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < HKV; ++c) m = __builtin_amdgcn_mfma_f32_16x16x4f32(s[HKV * v + c][r], mix[c], m, 0, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) p[r][e] = v == 0 || l15 / H == v ? m[e] : p[r][e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) p[r][e] = __builtin_fmaf(slope, dj + (float)(e - r), p[r][e]);
        }
        if (js + 15 > q0 || q0 + UQ - 1 - js >= window) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if ((uint32_t)(i0 + r - (js + 4 * g + e)) >= (uint32_t)window) p[r][e] = -INFINITY;
        }
        // The four waves' maxima pass through the weights' memory: wave w reads them where none but itself will write weights (keys 4 (w & 1) + 8 {0, 1}
        // of 32 (w >> 1), queries 0, 1 | 2, 3), group g writes the copy for wave g.
        float top[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) top[r] = max4(fmaxf(fmaxf(p[r][0], p[r][1]), fmaxf(p[r][2], p[r][3])));
        auto place = [&](int b, int r, int c, int w) {           // chunk c (of the wave's 32 keys) of row r in block b, the half that wave w writes
            return Ps + (b * 16 + r) * KT + 8 * ((4 * (w >> 1) + c) ^ row_spread(b, r)) + 4 * ((w & 1) ^ (b >> 1));
        };
        __syncthreads();                                         // (the tile before is read out: its weights and its keys)
#pragma unroll
        for (int x = 0; x < 2; ++x) *reinterpret_cast<float2*>(place(sub, l15, x, g)) = make_float2(top[2 * x], top[2 * x + 1]);
        if (j0 + KT < j_hi) stage(Kn);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const float2 o = *reinterpret_cast<const float2*>(place(k, l15, x, sub));
                top[2 * x] = fmaxf(top[2 * x], o.x), top[2 * x + 1] = fmaxf(top[2 * x + 1], o.y);
            }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // (the lanes' reads come before any lane's weights)
        float al[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float m_new = fmaxf(rm[r], top[r]), m = m_new == -INFINITY ? 0.0f : m_new;      // (no key seen yet: every weight 0)
            al[r] = __builtin_amdgcn_exp2f(rm[r] - m);
            rm[r] = m_new;
            float sum = 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                p[r][e] = __builtin_amdgcn_exp2f(p[r][e] - m);
                sum += p[r][e];
            }
            rl[r] = rl[r] * al[r] + sum;
            uint2 hi, lo;
            hi.x = bf16_pair(p[r][0], p[r][1]), hi.y = bf16_pair(p[r][2], p[r][3]);
            lo.x = bf16_pair(p[r][0] - __uint_as_float(hi.x << 16), p[r][1] - __uint_as_float(hi.x & 0xffff0000u));
            lo.y = bf16_pair(p[r][2] - __uint_as_float(hi.y << 16), p[r][3] - __uint_as_float(hi.y & 0xffff0000u));
            // of every 32 keys, k elements 8 g .. + 3 = keys 4 g .. + 3, 8 g + 4 .. = keys 16 + 4 g ..
            bf16_t* const w = place(l15 >> 2, 4 * (l15 & 3) + r, g, sub);
            *reinterpret_cast<uint2*>(w) = hi;
            *reinterpret_cast<uint2*>(w + 64 * KT) = lo;
        }
        __syncthreads();

        if (__any(!(al[0] == 1.0f && al[1] == 1.0f && al[2] == 1.0f && al[3] == 1.0f))) {        // (a maximum rarely moves after the first tiles)
            f4 f;
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = __shfl(al[e], 4 * sub + g, 64);
#pragma unroll
            for (int n = 0; n < 8; ++n) acc[n] *= f;
        }
#pragma unroll
        for (int ks = 0; ks < KT / 32; ++ks) {
            const bf16_t* const w = Ps + (sub * 16 + l15) * KT + 8 * ((4 * ks + g) ^ row_spread(sub, l15));
            const Frag<bf16_t> ph = load8(w), pl = load8(w + 64 * KT);
            const int j = 32 * ks + 4 * g + (l15 >> 2), far = sub >> 1 ? -16 * D : 16 * D;
#pragma unroll
            for (int n = 0; n < 8; ++n) {
                const int c = 2 * n + ((l15 & 3) >> 1);
                const bf16_t* const v = Ks + ((sub % HKV) * KT + j + 16 * (sub >> 1)) * D + 8 * (c ^ key_spread(j & 15)) + 4 * (l15 & 1);
                const uint2 va = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)v));
                const uint2 vb = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(v + far)));
                Frag<bf16_t> fv;
                fv.v = u32x4{va.x, va.y, vb.x, vb.y};
                acc[n] = mma(ph, fv, acc[n]);
                acc[n] = mma(pl, fv, acc[n]);
            }
        }
        bf16_t* const k = Ks;
        Ks = Kn, Kn = k;
    }
    __syncthreads();

    // denominators: over the lane groups and the four waves
    float* const sums = reinterpret_cast<float*>(Ps);
    f4 mine;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        rl[r] += __shfl_xor(rl[r], 16, 64);
        mine[r] = rl[r] + __shfl_xor(rl[r], 32, 64);
    }
    if (g == 0) *reinterpret_cast<f4*>(sums + sub * 64 + 4 * l15) = mine;
    __syncthreads();
    f4 den = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 4; ++k) den += *reinterpret_cast<const f4*>(sums + k * 64 + 4 * (4 * sub + g));
    const int h = 4 * (sub % HKV) + g;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float top = __shfl(rm[e], 4 * sub + g, 64);
        const int rq = 4 * (sub / HKV) + e;
        if (rq >= nq) continue;
        if (parts > 1) {
            const int64_t at = ((int64_t)blockIdx.z * n_rows + row0 + rq) * H + h;
#pragma unroll
            for (int n = 0; n < 8; ++n) a.scratch[at * D + 16 * n + l15] = acc[n][e];
            if (l15 == 0) *reinterpret_cast<float2*>(a.scratch + (int64_t)parts * n_rows * H * D + 2 * at) = make_float2(top, den[e]);
        } else {
            bf16_t* const o = (bf16_t*)a.out + (int64_t)(row0 + rq) * a.ldo + h * D + l15;
            const float inv = 1.0f / den[e];
#pragma unroll
            for (int n = 0; n < 8; ++n) o[16 * n] = from_f32<bf16_t>(acc[n][e] * inv);
        }
    }
}

// The parts' results of a row, in order: a wave per head of a row, two columns a lane, everything requested at once.
constexpr int MAX_PARTS = 16;
__global__ __launch_bounds__(256) void talk_merge_kernel(pcb_attn_talk_args a, const int32_t* __restrict__ tiles, int parts, int n_rows) {
    const int lane = threadIdx.x & 63, H = a.H, e = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int32_t* const t = tiles + 4 * blockIdx.x;
    if (e >= t[2] * H) return;
    const int64_t n = (int64_t)n_rows * H, at = (int64_t)t[3] * H + e;
    const float2 s = *reinterpret_cast<const float2*>(a.scratch + parts * n * D + 2 * ((lane < parts ? lane : 0) * n + at));
    const float m = wave_max(s.x), w = lane < parts && s.x != -INFINITY ? __builtin_amdgcn_exp2f(s.x - m) : 0.0f;
    const float l = wave_sum(s.y * w);
    float2 o = make_float2(0.0f, 0.0f);
    for (int p0 = 0; p0 < parts; p0 += 4) {
        float2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const float2*>(a.scratch + ((p0 + u < parts ? p0 + u : parts - 1) * n + at) * D + 2 * lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const float f = __shfl(w, p0 + u, 64);               // (0 beyond the last)
            o.x += v[u].x * f, o.y += v[u].y * f;
        }
    }
    const float inv = 1.0f / l;
    *reinterpret_cast<uint32_t*>((bf16_t*)a.out + ((int64_t)t[3] + e / H) * a.ldo + (e % H) * D + 2 * lane) = bf16_pair(o.x * inv, o.y * inv);
}

}  // namespace

bool pcb_talk_prompt_fits(const pcb_attn_talk_args& a) {
    return a.dtype == PCB_BF16 && a.head_dim == D && a.talk && a.H == 4 * a.Hkv && (a.H == 4 || a.H == 8 || a.H == 16) && a.ldq % 8 == 0 &&
           a.slot_stride % 8 == 0 && a.head_stride % 8 == 0 && ((uintptr_t)a.q | (uintptr_t)a.cache) % 16 == 0;
}

int pcb_talk_prompt(const pcb_attn_talk_args& a, hipStream_t stream) {
    const int32_t* const tiles = a.tiles64 ? a.tiles64 : a.tiles;
    const int n_tiles = a.tiles64 ? a.n_tiles64 : a.n_tiles, tile_rows = a.tiles64 ? 64 : 16;
    const int n_rows = 16 * a.n_tiles;                           // (what the scratch is laid out for)
    auto go = [&](auto hkv, auto nu) {
        constexpr int HKV = decltype(hkv)::value, NU = decltype(nu)::value, LDS = 2 * (2 * HKV * KT * D + NU * 2 * 64 * KT), WQ = NU * 16 / HKV;
        static const hipError_t raised =
            hipFuncSetAttribute(reinterpret_cast<const void*>(talk_prompt_kernel<HKV, NU>), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
        (void)raised;
        // Workgroups share a row's keys while that gives no more of them than CUs and each keeps three tiles: below that the merge costs what it
        // saves.  us, one workgroup a row / the rule / twice as many: 16 heads, 1000 rows 62 / 49 / 61; 20 rows behind 1000 keys 63 / 26 / 22; 500
        // behind 8000 without a window 423 / 130 / 141; 2048 rows 72 / 72 / 95.  4 heads, 6 x 300 rows 17 / 17 / 20.
        const int keys = a.window > 0 && a.window < a.max_kv_len - WQ ? a.window + WQ : a.max_kv_len;
        int parts = 256 / pcb_ceil_div(n_rows, WQ);
        if (parts > pcb_ceil_div(keys, KT) / 3) parts = pcb_ceil_div(keys, KT) / 3;
        if (parts > MAX_PARTS) parts = MAX_PARTS;
        const int64_t room = a.scratch_floats / ((int64_t)n_rows * a.H * (D + 2));
        if (parts > room) parts = (int)room;
        if (parts < 1) parts = 1;
        hipLaunchKernelGGL((talk_prompt_kernel<HKV, NU>), dim3(n_tiles, pcb_ceil_div(tile_rows, WQ), parts), dim3(256 * NU), LDS, stream, a, tiles, parts,
                           n_rows);
        if (parts > 1) hipLaunchKernelGGL(talk_merge_kernel, dim3(n_tiles, tile_rows * a.H / 4), dim3(256), 0, stream, a, tiles, parts, n_rows);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    // (two units beside one another share a key tile: with 16 heads, whose tile fills the LDS, 72 us for 2048 rows, 95 alone; with 8 heads 58 and 42)
    if (a.H == 16)
        go(std::integral_constant<int, 4>{}, Two{});
    else if (a.H == 8)
        go(Two{}, One{});
    else
        go(One{}, One{});
    return pcb_check_launch("talk_prompt_kernel");
}
