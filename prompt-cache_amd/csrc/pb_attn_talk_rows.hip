// pcb_attn_talk_rows: the attention of pcb_attn_talk for single rows (one new token per request), in one launch.
//
// Workgroup = one row x KPW of the keys it sees (a multiple of 64, such that a row has at most max_parts workgroups; by the row's own position, since a
// captured step launches for the cache's capacity), all heads, 64 keys at a time:
//   scores   a wave takes 16 keys against every head: K Q^T on the matrix cores, the heads of one key head as columns; with scale and distance
//            bias into LDS
//   mixing   a lane per key, a wave for every fourth head: the heads' sums are lane-local, maximum and denominator of a head are sums over the wave
//   values   a thread owns eight columns of one key head and every n-th key, for all query heads of that key head: fp32 multiply-adds, the weights
//            from LDS as they are.  Its key rows are requested beside those of the scores.
// A row of one workgroup is finished there; of several, each leaves (sum, maximum, denominator) per head and the last one to arrive merges them in
// order, whoever is last.
//
// What bounds it: latency -- one trip to memory, three barriers, one more trip where rows are merged.  us, one row, 8 heads of 128 over 2, 45 keys:
// scores through the band and the values behind them 13.5 + 12.4 (two launches, 2 and 8 workgroups), 7.8 here.
// 16 heads over 4, window 1024: 8 rows of 1500 keys 46.6 and 21.0, 64 rows 85.7 and 41.5; no window, one row of 8000 keys 219.8 and 50.2; one row of 1000
// keys in a cache of 16384, 45.6 and 20.4 (110.8 with a workgroup's keys by the capacity).
#include <type_traits>

#include "pb_common.h"

namespace {
using namespace pcb;

constexpr int KB = 64;                 // keys at a time
// Workgroups that a row of `blocks` blocks of 64 keys may have, of n_rows rows: eight where the rows alone fill the chip, else sixteen, up to four rows
// over more than 48 blocks 32 (where each query head has its own keys a block of 16 heads in fp32 takes 20 us).  us, eight / sixteen, 64 rows of 1000 keys:
// 32 heads of 64 columns 61 / 90, 16 of 128 40 / 44; sixteen / 32, one row of 8000 keys: 16 heads over 4 67 / 50, 16 heads of 64 with keys of their own
// in fp32 173 / 100 (111 through the band); 2000 keys 27 / 30.
__host__ __device__ __forceinline__ int max_parts(int n_rows, int blocks) { return n_rows <= 4 ? (blocks > 48 ? 32 : 16) : n_rows <= 48 ? 16 : 8; }

constexpr int ANY = 1 << 20;            // (as many blocks as there may be)

// Hand-over between workgroups of one launch: stores that go through to memory, s_waitcnt vmcnt(0) (stores count there on gfx9), barrier, one relaxed
// arrival; loads that bypass this CU's caches.
typedef __attribute__((address_space(1))) unsigned long long gu64;
typedef __attribute__((address_space(1))) uint32_t gu32;
__device__ __forceinline__ void put2(float* p, float a, float b) {
    const unsigned long long x = ((unsigned long long)__float_as_uint(b) << 32) | __float_as_uint(a);
    __hip_atomic_store((gu64*)p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 get2(const float* p) {
    const unsigned long long x = __hip_atomic_load((gu64*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((uint32_t)x), __uint_as_float((uint32_t)(x >> 32)));
}

__device__ __forceinline__ void put8(bf16_t* p, const Frag<bf16_t>& f) { *reinterpret_cast<u32x4*>(p) = f.v; }
__device__ __forceinline__ void put8(float* p, const Frag<float>& f) {
    *reinterpret_cast<f4*>(p) = f4{f.v[0], f.v[1], f.v[2], f.v[3]};
    *reinterpret_cast<f4*>(p + 4) = f4{f.v[4], f.v[5], f.v[6], f.v[7]};
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

template <typename E, int HMAX, int REP>
__global__ __launch_bounds__(256, 2) void talk_rows_kernel(pcb_attn_talk_args a, float* __restrict__ part, uint32_t* __restrict__ counters) {
    constexpr int PG = 2;                                         // key heads whose fragments are requested together
    constexpr int VB = sizeof(E) == 2 ? 8 : 4;           // key rows of a thread in flight
    constexpr int HP = HMAX / 4;                         // heads a wave mixes
    constexpr int QLD = 128 + 16 / sizeof(E);
    extern __shared__ __attribute__((aligned(16))) float red[];          // [slices][H * D]: at the end
    __shared__ float sc[KB][HMAX + 1], P[HMAX][KB], keep_s[HMAX], m_s[HMAX], l_s[HMAX];
    __shared__ __attribute__((aligned(16))) float talk_s[HMAX * HMAX];
    __shared__ __attribute__((aligned(16))) E Qs[HMAX][QLD];             // columns past head_dim: zeros
    __shared__ int last_s;
    const int H = a.H, Hkv = H / REP, D = a.head_dim, HD = H * D;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = lane >> 4, l15 = lane & 15;
    // (weights of the mixing: on their way while the tile's record is, in LDS by the first barrier)
    constexpr int TW = (HMAX * HMAX + 255) / 256;
    float tw[TW];
#pragma unroll
    for (int u = 0; u < TW; ++u) {
        const int e = tid + 256 * u, h = e / HMAX, g = e % HMAX;
        tw[u] = a.talk && h < H && g < H ? a.talk[h * H + g] : 0.0f;
    }
    const int32_t* t = a.tiles + 4 * blockIdx.x;
    const int slot = t[0], i = t[1], row = t[3];
    const int j_min = a.window > 0 && i - a.window + 1 > 0 ? i - a.window + 1 : 0;
    const int blocks = (i - j_min + KB) / KB, most = max_parts(gridDim.x, blocks), kpw = KB * ((blocks + most - 1) / most);
    const int parts = (i - j_min + kpw) / kpw;           // workgroups of this row
    if ((int)blockIdx.y >= parts) return;                // (uniform over the workgroup)
    const int j_lo = j_min + kpw * blockIdx.y, j_hi = j_lo + kpw <= i ? j_lo + kpw - 1 : i;      // its keys, j_hi included
    const E* Q = (const E*)a.q + (int64_t)row * a.ldq;
    const E* C = (const E*)a.cache + (int64_t)slot * a.slot_stride;
    constexpr int QC = HMAX * 16 / 256 > 0 ? HMAX * 16 / 256 : 1;        // eight columns of a head per thread and pass
    Frag<E> fq[QC];
#pragma unroll
    for (int u = 0; u < QC; ++u) {
        const int h = (tid + 256 * u) >> 4, d = 8 * (tid & 15);
        zero8(fq[u]);
        if (h < H && d < D) fq[u] = load8(Q + (int64_t)h * D + d);
    }
    // values: this thread's columns and keys
    const int cols = D / 8, combos = cols * Hkv, slices = 256 / combos;
    const int slice = tid / combos, combo = tid % combos, vc = combo / cols, vd = combo % cols * 8;
    const bool active = slice < slices;
    const E* V = C + (int64_t)vc * a.head_stride + vd;
    float acc[REP][8];
#pragma unroll
    for (int r = 0; r < REP; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r][e] = 0.0f;
    float rm[HP], rl[HP];                                // running maximum (the sink is a score of 0) and denominator of the wave's heads
#pragma unroll
    for (int u = 0; u < HP; ++u) rm[u] = a.sink ? 0.0f : -INFINITY, rl[u] = 0.0f;

    for (int j0 = j_lo; j0 <= j_hi; j0 += KB) {
        Frag<E> fv[VB];
        auto values = [&](int kk) {
#pragma unroll
            for (int u = 0; u < VB; ++u) {
                const int j = j0 + kk + slices * u;
                fv[u] = load8(V + (int64_t)(j <= j_hi ? j : j_hi) * D);
            }
        };
        const int jk = j0 + 16 * wave + l15;
        const E* krow = C + (int64_t)(jk <= j_hi ? jk : j_hi) * D;
        for (int c0 = 0; c0 < Hkv; c0 += PG) {
            Frag<E> fk[PG][4];
            float slope[PG];
#pragma unroll
            for (int u = 0; u < PG; ++u) {
                const int c = c0 + u < Hkv ? c0 + u : Hkv - 1;
                slope[u] = a.slopes ? a.slopes[c * REP + (l15 < REP ? l15 : 0)] : 0.0f;
#pragma unroll
                for (int st = 0; st < 4; ++st) {         // (columns past head_dim meet zeros)
                    const int d = 32 * st + 8 * group;
                    fk[u][st] = load8(krow + (int64_t)c * a.head_stride + (d < D ? d : 0));
                }
            }
            if (c0 == 0 && active) values(slice);
            if (c0 == 0 && j0 == j_lo) {
#pragma unroll
                for (int u = 0; u < QC; ++u)
                    if ((tid + 256 * u) >> 4 < HMAX) put8(&Qs[(tid + 256 * u) >> 4][8 * (tid & 15)], fq[u]);
#pragma unroll
                for (int u = 0; u < TW; ++u)
                    if (tid + 256 * u < HMAX * HMAX) talk_s[tid + 256 * u] = tw[u];
                __syncthreads();
            }
#pragma unroll
            for (int u = 0; u < PG; ++u) {
                const int h0 = (c0 + u < Hkv ? c0 + u : Hkv - 1) * REP;
                f4 s = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int st = 0; st < 4; ++st)
                    s = mma(fk[u][st], load8(&Qs[h0 + (l15 < REP ? l15 : 0)][32 * st + 8 * group]), s);
                // lane: head h0 + l15, keys j0 + 16 wave + 4 group + r
                if (l15 < REP && c0 + u < Hkv) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int kk = 16 * wave + 4 * group + r;
                        sc[kk][h0 + l15] = s[r] * a.scale - slope[u] * (float)(i - (j0 + kk));
                    }
                }
            }
        }
        __syncthreads();
        // ---- mixing: lane = key, this wave's heads = wave, wave + 4, ..
        {
            float s[HMAX], x[HP];
#pragma unroll
            for (int g = 0; g < HMAX; ++g) s[g] = g < H ? sc[lane][g] : 0.0f;
            const bool seen = j0 + lane <= j_hi;
#pragma unroll
            for (int u = 0; u < HP; ++u) {
                float v = 0.0f;
                if (a.talk) {
#pragma unroll
                    for (int g = 0; g < HMAX; g += 4) {
                        const f4 w = *reinterpret_cast<const f4*>(&talk_s[(wave + 4 * u) * HMAX + g]);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v += w[e] * s[g + e];
                    }
                } else {
                    v = sc[lane][wave + 4 * u];          // (of a head past the last one: whatever stands there, unused)
                }
                x[u] = seen ? v : -INFINITY;
            }
            float top[HP], sum[HP];
#pragma unroll
            for (int u = 0; u < HP; ++u) top[u] = x[u];
            auto over_wave = [&](float(&v)[HP], auto f) {
#pragma unroll
                for (int u = 0; u < HP; ++u) {
                    v[u] = f(v[u], dpp<0xb1>(v[u]));               // quad_perm [1,0,3,2]
                    v[u] = f(v[u], dpp<0x4e>(v[u]));               // quad_perm [2,3,0,1]
                    v[u] = f(v[u], dpp<0x141>(v[u]));              // row_half_mirror
                    v[u] = f(v[u], dpp<0x140>(v[u]));              // row_mirror
                }
#pragma unroll
                for (int o = 16; o < 64; o <<= 1)
#pragma unroll
                    for (int u = 0; u < HP; ++u) v[u] = f(v[u], __shfl_xor(v[u], o, 64));
            };
            over_wave(top, [](float p, float q) { return fmaxf(p, q); });
#pragma unroll
            for (int u = 0; u < HP; ++u) {
                const float m = fmaxf(rm[u], top[u]);
                const float keep = rm[u] == -INFINITY ? 0.0f : expf(rm[u] - m);
                x[u] = expf(x[u] - m);
                sum[u] = x[u];
                rl[u] *= keep;
                rm[u] = m;
                if (wave + 4 * u < H) {
                    P[wave + 4 * u][lane] = x[u];
                    if (lane == 0) keep_s[wave + 4 * u] = keep;
                }
            }
            over_wave(sum, [](float p, float q) { return p + q; });
#pragma unroll
            for (int u = 0; u < HP; ++u) rl[u] += sum[u];
        }
        __syncthreads();
        if (active) {
            if (j0 != j_lo) {
#pragma unroll
                for (int r = 0; r < REP; ++r) {
                    const float keep = keep_s[vc * REP + r];
#pragma unroll
                    for (int e = 0; e < 8; ++e) acc[r][e] *= keep;
                }
            }
            const int n = j_hi - j0 + 1 < KB ? j_hi - j0 + 1 : KB;
            for (int kk = slice; kk < n; kk += slices * VB) {
                Frag<E> v[VB];
#pragma unroll
                for (int u = 0; u < VB; ++u) v[u] = fv[u];
                if (kk + slices * VB < n) values(kk + slices * VB);
#pragma unroll
                for (int u = 0; u < VB; ++u) {
                    const int k1 = kk + slices * u;
#pragma unroll
                    for (int r = 0; r < REP; ++r) {
                        const float p = k1 < n ? P[vc * REP + r][k1] : 0.0f;
#pragma unroll
                        for (int e = 0; e < 8; ++e) acc[r][e] += p * at8(v[u], e);
                    }
                }
            }
        }
        __syncthreads();
    }
    // ---- the slices meet
    if (active) {
        float* to = red + slice * HD + vc * REP * D + vd;
#pragma unroll
        for (int r = 0; r < REP; ++r) {
            *reinterpret_cast<f4*>(to + r * D) = f4{acc[r][0], acc[r][1], acc[r][2], acc[r][3]};
            *reinterpret_cast<f4*>(to + r * D + 4) = f4{acc[r][4], acc[r][5], acc[r][6], acc[r][7]};
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int u = 0; u < HP; ++u)
            if (wave + 4 * u < H) m_s[wave + 4 * u] = rm[u], l_s[wave + 4 * u] = rl[u];
    }
    __syncthreads();
    E* out = (E*)a.out + (int64_t)row * a.ldo;
    const int rec = HD + 2 * H, stride = max_parts(gridDim.x, ANY);
    float* mine = part + ((int64_t)blockIdx.x * stride + blockIdx.y) * rec;
#pragma unroll 1
    for (int e = 2 * tid; e < HD; e += 512) {
        float v0 = 0.0f, v1 = 0.0f;
#pragma unroll 4
        for (int s = 0; s < slices; ++s) {
            const float2 v = *reinterpret_cast<const float2*>(red + s * HD + e);
            v0 += v.x, v1 += v.y;
        }
        if (parts == 1) {
            const int h = e / D;                         // (D is even: both columns are the head's)
            const float inv = 1.0f / (l_s[h] + (a.sink ? expf(-m_s[h]) : 0.0f));
            out[e] = from_f32<E>(v0 * inv);
            out[e + 1] = from_f32<E>(v1 * inv);
        } else {
            put2(mine + e, v0, v1);
        }
    }
    if (parts == 1) return;
    if (tid < H) put2(mine + HD + 2 * tid, m_s[tid], l_s[tid]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        gu32* c = (gu32*)(counters + blockIdx.x);
        const uint32_t old = __hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_s = old + 1u == (uint32_t)parts;
        if (last_s) __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);       // (as the next launch wants it)
    }
    __syncthreads();
    if (!last_s) return;
    const float* all = part + (int64_t)blockIdx.x * stride * rec;
    float* w_s = red;                                    // [parts][H]: a part's weight over the row's denominator
    if (tid < H) {
        float m = a.sink ? 0.0f : -INFINITY, l = 0.0f;
        auto ask = [&](int b0, float2(&ml)[16]) {
#pragma unroll
            for (int b = 0; b < 16; ++b) ml[b] = get2(all + (int64_t)(b0 + b < parts ? b0 + b : 0) * rec + HD + 2 * tid);
#pragma unroll
            for (int b = 0; b < 16; ++b) m = b0 + b < parts ? fmaxf(m, ml[b].x) : m;
        };
        auto weigh = [&](int b0, float2(&ml)[16]) {
#pragma unroll
            for (int b = 0; b < 16; ++b) {
                ml[b].x = b0 + b < parts ? expf(ml[b].x - m) : 0.0f;
                if (b0 + b < parts) l += ml[b].x * ml[b].y;
            }
        };
        float2 lo[16], hi[16];
        ask(0, lo);
        if (parts > 16) ask(16, hi);
        weigh(0, lo);
        if (parts > 16) weigh(16, hi);
        if (a.sink) l += expf(-m);
        const float inv = 1.0f / l;
#pragma unroll
        for (int b = 0; b < 16; ++b) {
            w_s[b * H + tid] = lo[b].x * inv;
            if (parts > 16) w_s[(16 + b) * H + tid] = hi[b].x * inv;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int e = 2 * tid; e < HD; e += 512) {
        const int h = e / D;
        float v0 = 0.0f, v1 = 0.0f;
#pragma unroll 1
        for (int b0 = 0; b0 < parts; b0 += 8) {
            float2 v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = get2(all + (int64_t)(b0 + u < parts ? b0 + u : 0) * rec + e);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (b0 + u < parts) {
                    const float w = w_s[(b0 + u) * H + h];
                    v0 += w * v[u].x, v1 += w * v[u].y;
                }
        }
        out[e] = from_f32<E>(v0);
        out[e + 1] = from_f32<E>(v1);
    }
}

template <typename E>
int run(const pcb_attn_talk_args& a, float* part, uint32_t* counters, hipStream_t stream) {
    const int rep = a.H / a.Hkv, most = a.window > 0 && a.window < a.max_kv_len ? a.window : a.max_kv_len;
    const int blocks = pcb_ceil_div(most, KB), parts = max_parts(a.n_tiles, blocks);
    const dim3 grid(a.n_tiles, blocks < parts ? blocks : parts);
    const int slices = 256 / (a.head_dim / 8 * a.Hkv);
    size_t lds = (size_t)slices * a.H * a.head_dim * sizeof(float);            // (8 KiB times the query heads of a key head, at most)
    if (lds < 32 * (size_t)a.H * sizeof(float)) lds = 32 * (size_t)a.H * sizeof(float);
    auto go = [&](auto hmax, auto r) {
        auto kern = talk_rows_kernel<E, decltype(hmax)::value, decltype(r)::value>;
        static const hipError_t raised =
            hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 64 * 1024);
        (void)raised;
        hipLaunchKernelGGL(kern, grid, dim3(256), lds, stream, a, part, counters);
    };
    auto heads = [&](auto r) {
        if (a.H <= 8)
            go(std::integral_constant<int, 8>{}, r);
        else if (a.H <= 16)
            go(std::integral_constant<int, 16>{}, r);
        else
            go(std::integral_constant<int, 32>{}, r);
    };
    switch (rep) {
        case 1: heads(std::integral_constant<int, 1>{}); break;
        case 2: heads(std::integral_constant<int, 2>{}); break;
        case 4: heads(std::integral_constant<int, 4>{}); break;
        default: heads(std::integral_constant<int, 8>{});
    }
    return pcb_check_launch("talk_rows_kernel");
}

bool fits(int dtype, int H, int Hkv, int D) {
    const int rep = Hkv > 0 ? H / Hkv : 0;
    return (dtype == PCB_BF16 || dtype == PCB_F32) && H > 0 && H <= 32 && Hkv > 0 && H % Hkv == 0 && (rep == 1 || rep == 2 || rep == 4 || rep == 8) &&
           D > 0 && D <= 128 && D % 8 == 0 && D / 8 * Hkv <= 256;
}

}  // namespace

PCB_EXPORT int32_t pcb_attn_talk_rows_fits(int32_t dtype, int32_t H, int32_t Hkv, int32_t head_dim) { return fits(dtype, H, Hkv, head_dim); }
PCB_EXPORT int64_t pcb_attn_talk_rows_part(int32_t n_rows, int32_t H, int32_t head_dim) {
    return (int64_t)n_rows * max_parts(n_rows, ANY) * ((int64_t)H * head_dim + 2 * H);
}

PCB_EXPORT int pcb_attn_talk_rows(const pcb_attn_talk_args* a, float* part, int64_t part_floats, int32_t* counters, void* stream) {
    PCB_REQUIRE(a && a->struct_bytes == sizeof(pcb_attn_talk_args), PCB_ERR_ARG, "pcb_attn_talk_rows: struct size mismatch");
    PCB_REQUIRE(fits(a->dtype, a->H, a->Hkv, a->head_dim), PCB_ERR_ARG,
                "pcb_attn_talk_rows: up to 32 heads, 1, 2, 4 or 8 to a key head, of up to 128 columns in whole chunks of eight");
    PCB_REQUIRE(a->n_tiles >= 0 && a->max_kv_len > 0, PCB_ERR_ARG, "pcb_attn_talk_rows: bad sizes");
    if (a->n_tiles == 0) return PCB_OK;
    PCB_REQUIRE(a->q && a->tiles && a->cache && a->out && part && counters, PCB_ERR_ARG, "pcb_attn_talk_rows: null pointer");
    PCB_REQUIRE(a->ldq >= (int64_t)a->H * a->head_dim && a->ldo >= (int64_t)a->H * a->head_dim, PCB_ERR_ARG,
                "pcb_attn_talk_rows: row strides shorter than heads * head_dim");
    const int64_t per = a->dtype == PCB_BF16 ? 8 : 4;
    PCB_REQUIRE(a->ldq % per == 0 && a->slot_stride % per == 0 && a->head_stride % per == 0 && ((uintptr_t)a->q | (uintptr_t)a->cache) % 16 == 0 &&
                    (uintptr_t)part % 8 == 0,
                PCB_ERR_ARG, "pcb_attn_talk_rows: rows of queries and keys are read in 16-byte pieces");
    PCB_REQUIRE(part_floats >= pcb_attn_talk_rows_part(a->n_tiles, a->H, a->head_dim), PCB_ERR_ARG, "pcb_attn_talk_rows: scratch too small");
    return a->dtype == PCB_BF16 ? run<pcb::bf16_t>(*a, part, (uint32_t*)counters, (hipStream_t)stream)
                                : run<float>(*a, part, (uint32_t*)counters, (hipStream_t)stream);
}
