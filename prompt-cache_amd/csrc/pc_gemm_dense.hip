// Many-row projections (schema encode, no-cache prefill, long questions): the MFMA-bound regime of the path.
//
// Replaces  q_proj/k_proj/v_proj   promptcache/model/llama2.py:345-347   (one fused [q|k|v] GEMM)
//           o_proj + residual       promptcache/model/llama2.py:405, :638
//           gate/up + SiLU*up       promptcache/model/llama2.py:242
//           down_proj + residual    promptcache/model/llama2.py:242, :644
//           lm_head                 promptcache/model/llama2.py:1050
//           (Falcon / MPT: query_key_value, dense, dense_h_to_4h + GELU, dense_4h_to_h; falcon.py:393-405, :726-731)
// inside SchemaCache._process (cache_engine.py:243-248): the module-KV precompute.
//
// Y[m][n] = sum_k (Xhi[m][k] + Xlo[m][k]) * W[n][k]       X: split-precision fp16 planes [M][K] (hi = fp16(x),
//                                                          lo = fp16(x - hi); lo optional), W: nn.Linear [N][K] fp16
// Why two planes: an fp16 activation costs 2^-12 per projection input, and through 32 layers that alone moves
// 7b-shape logits by 2-3e-2 against the reference's fp32 CPU path.  Both planes meet the SAME weight
// fragment inside one tile pass: a weight fragment is read from LDS once and feeds the hi and the lo MFMA, the two
// partial products meet in the fp32 accumulator, and the epilogue (residual add, SiLU*up, GELU, fp32 store) runs on the
// accumulator tile -- no [2T][N] fp32 intermediate ever exists.
//
// Tile: workgroup = 4 waves (2 x 2), block tile 64 MT (M) x 64 NT (N) x 64 (K), wave tile 32 MT x 32 NT: 128 x 256 with both planes or
// one, 256 x 256 with one plane over many rows, 128 x 128 for launches whose 256-wide grid would leave CUs idle (launch_dense_tile).
// What bounds it: power (the matrix cores run these launches at 1.4-1.7 GHz; the same launches on zeros are 1.2-1.3 x faster), LDS bandwidth
// next.  Per 16-deep k-slab and both planes a wave of 64 x 128 reads 8 KiB of LDS for 16 MFMAs, two waves of 64 x 64 read 12 KiB for as
// many: the same block tile on eight waves kept the LDS pipe as busy as the matrix pipe.  Eight waves with an epilogue that read residuals
// between its stores -> this kernel, us, random data: both planes, 1 737 rows, q|k|v 329 -> 307, o_proj 113 -> 103, down 288 -> 265
// (1.18 PFLOP/s executed), 32 000 columns 816 -> 758, 3 584 rows down 598 -> 532; one plane, gate|up, 1 737 / 2 940 / 3 584 rows 370 -> 324,
// 600 -> 528, 729 -> 561 (256 x 256 tiles, 1.15 PFLOP/s).
// mfma_f32_16x16x32_f16 (32x32x16 in the 128 x 128 tiles of one plane; which and why: mfma_tile_loop.h).  Per 32 x 32 results and 16 of k: MT (2 MT with both
// planes) activation fragments and NT weight fragments
// (16 B per lane each, ds_read_b128) for MT NT (2 MT NT) MFMAs.
// Staging, LDS image and main loop: mfma_tile_loop.h.
// Which global weight row lands in which LDS row is free as well (per-lane source address): the SiLU launch puts 32
// gate rows and the 32 matching up rows side by side in one 64-column group, so gate_j and up_j meet in the same lane.
// Epilogue: the accumulator tile goes through the (now idle) LDS, 64 columns of a wave at a time, so that every global store is 16 B per
// lane on full rows.
// Grid: 1-D, XCD-aware: block id b runs on XCD b % 8; the tiles are cut into 8 rectangles (px row strips by 8 / px column strips),
// one per XCD, walked M-block by M-block: the 32 tiles that run on an XCD at a time share few activation rows AND few weight panels
// (with one column strip each an XCD walks all M-blocks: 2 048 x 8 192 x 2 048 in 256 x 256 tiles 93 us, in 4 x 2 strips 71).  Where no
// such cut reaches the rounds of an even share, the column-by-column order is dealt to the XCDs in 8 runs (mfma_tile_loop.h).
// Roofline: MFMA.  flops per launch = 2 * (TWO ? 2 : 1) * M * N * K against the 2.5 PFLOP/s dense fp16 peak.
#include <hip/hip_fp16.h>
#include <string.h>

#include <type_traits>

#include "mfma_tile_loop.h"
#include "pc_common.h"
#ifdef PC_DEV_SWEEPS
#include "pc_dev.h"
#endif

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int BK = 64;
enum { EPI_STORE = 0, EPI_ADD = 1, EPI_SILU = 2, EPI_ROPE = 3, EPI_GELU = 4 };

struct DenseParams {
    const _Float16* xh; const _Float16* xl; int64_t ldx;   // [M][K] planes (xl may be null), row stride in halfs
    const _Float16* w; int64_t ldw;                        // [N][K]
    const float* wscale;                                   // optional per-output-row scale (int8 codes held in fp16)
    // LLM.int8 (pc_int8.hip): xh holds activation CODES, xscale[m] = SCA[m] / 127; corr[m][n] (global weight-row index n) is
    // added before the epilogue's nonlinearity when *corr_has != 0
    const float* xscale; const float* corr; int64_t ldc; const int32_t* corr_has;
    // LO8: the lo activation plane as INT8 codes [M][K] with one scale per row (lo ~ code * xl8_scale[m]) against an int8
    // image of the weights [N][K] with one scale per row (W ~ code * w8_scale[n]): the residual product runs on
    // v_mfma_i32_32x32x32_i8 -- twice the fp16 MFMA rate, exact integer sums -- and joins the fp32 accumulator in the epilogue
    const signed char* xl8; const float* xl8_scale; int64_t ldx8;
    const signed char* w8; const float* w8_scale; int64_t ldw8;
    float* y; int64_t ldy;                                 // EPI_STORE / EPI_ADD
    _Float16* oh; _Float16* ol; int64_t ldo;               // EPI_SILU / EPI_GELU output planes
    int32_t M, N, K, mb, nb, nfeat;                        // nfeat: SiLU features (= N / 2)
    mfma_tile::Strips strips;                              // which tiles (M-block, weight panel) an XCD owns
    // split-K (EPI_STORE instantiation only): grid.y slices of `kper` K-steps, slice z stores its partial sums to
    // y + z * slab_stride; dense_reduce_kernel then adds the slabs in fixed order (launch_dense_splitk)
    int32_t kper; int64_t slab_stride;
    // EPI_ROPE (the fused q|k|v projection at head_dim 128, llama2.py:345-364): rotation table [M][64] (cos, sin), rotated q as
    // hi / lo planes [M][q_ts], rotated k and plain v into the arena planes (+ their residual planes) behind each batch row's past
    const float2* cs; _Float16* q_hi; _Float16* q_lo; int64_t q_ts;
    _Float16* k_arena; _Float16* v_arena; int64_t a_bs, a_hs;
    _Float16* k_lo; _Float16* v_lo; int64_t lo_bs, lo_hs; int32_t lo_row0;
    int32_t H, Hkv, q_len, past_len; const int32_t* past_lens;
};

__device__ __forceinline__ void glds16(const _Float16* g, char* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                     (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}

// the block tile of a launch: W x W waves of 32 MT x 32 NT, S LDS images in the ring (as many as the 160 KiB of a CU hold)
template <int W, bool TWO, bool NARROW, bool TALL>
struct Tile {
    static constexpr int MT = TALL ? 4 : 2, NT = NARROW ? 2 : 4, S = TWO || TALL ? 2 : 3, BLK = TWO || !NARROW ? 16 : 32;
    static constexpr int BM = 32 * W * MT, BN = 32 * W * NT;
};

// The 64 columns of group `grp` (of the launch's weight rows; EPI_SILU: 32 gate and the matching 32 up features, EPI_ROPE: 32 features of a
// head's first half and their rotary partners), rows mrow0 .. + 32 MT - 1, from a wave's patch to where they go.
// Loads come before stores and loops are short: a wait for a load behind a store waits for the store's way to memory and back (they count
// on one counter), and unrolled code that runs once is paid in instruction misses.
template <int EPI, int MT>
__device__ __forceinline__ void store_group(const DenseParams& p, char* patch, int lane, int grp, int mrow0) {
    constexpr bool PAIRS = EPI == EPI_SILU || EPI == EPI_ROPE;
    constexpr int LPR = PAIRS ? 8 : 16, RPI = 64 / LPR, R = 32 * MT / RPI;       // lanes on a row, rows an access covers, accesses
    const int pr = lane / LPR, pc = lane % LPR;
    auto at = [&](int e, int c) { return (f4*)(patch + (RPI * e + pr) * 256 + ((c + pc) ^ ((RPI * e + pr) & 15)) * 16); };
    auto mrow = [&](int e) { return mrow0 + RPI * e + pr; };
    auto row = [&](int e) { return mrow(e) < p.M ? mrow(e) : p.M - 1; };
    const int n = EPI == EPI_SILU ? grp * 32 + pc * 4 : grp * 64 + pc * 4;
    if (EPI != EPI_ROPE && n >= (EPI == EPI_SILU ? p.nfeat : p.N)) return;
    if (EPI != EPI_ROPE && p.wscale) {
#pragma unroll
        for (int h = 0; h < (EPI == EPI_SILU ? 2 : 1); ++h) {
            const int col = n + h * p.nfeat;
            const f4 sv = *(const f4*)(p.wscale + col);
            const bool corr = p.xscale && *p.corr_has;
#pragma unroll 1
            for (int e0 = 0; e0 < R; e0 += 4) {
                f4 cv[4];
                float xs[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    xs[e] = p.xscale ? p.xscale[row(e0 + e)] : 1.0f;
                    cv[e] = corr ? *(const f4*)(p.corr + (int64_t)row(e0 + e) * p.ldc + col) : f4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f4 v = *at(e0 + e, 8 * h) * sv;
                    if (p.xscale) v *= xs[e];
                    if (corr) v += cv[e];
                    *at(e0 + e, 8 * h) = v;
                }
            }
        }
    }
    if constexpr (EPI == EPI_SILU || EPI == EPI_GELU) {
#pragma unroll 1
        for (int e0 = 0; e0 < R; e0 += 2)
#pragma unroll
            for (int e = e0; e < e0 + 2; ++e) {
                const f4 v = *at(e, 0), u = EPI == EPI_SILU ? *at(e, 8) : v;
                h4 hi, lo;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const float s = EPI == EPI_SILU ? (v[k] / (1.0f + __expf(-v[k]))) * u[k]                       // act_fn(gate) * up, llama2.py:242
                                                    : 0.5f * v[k] * (1.0f + erff(v[k] * 0.70710678118654752f));   // nn.GELU(), falcon.py:726
                    _Float16 sh, sl;
                    pc_split(s, sh, sl);
                    hi[k] = sh; lo[k] = sl;
                }
                if (mrow(e) < p.M) {
                    *(h4*)(p.oh + (int64_t)mrow(e) * p.ldo + n) = hi;
                    if (p.ol) *(h4*)(p.ol + (int64_t)mrow(e) * p.ldo + n) = lo;
                }
            }
    } else if constexpr (EPI == EPI_ROPE) {
        // RoPE at the supplied positions (llama2.py:200-213, :357-359) and the KV append (:361-364):
        // 8 lanes per row, a lane holds features d0 .. d0+3 and d0+64 .. d0+67 of head `hd`
        const int hd = grp >> 1, d0 = (grp & 1) * 32 + pc * 4;
        if (hd >= p.H + 2 * p.Hkv) return;
        const bool rot = hd < p.H + p.Hkv, is_q = hd < p.H;
        const int kh = rot ? hd - p.H : hd - p.H - p.Hkv;
#pragma unroll 1
        for (int e0 = 0; e0 < R; e0 += 8) {
            f4 w01[8], w23[8];
            int64_t off[8], off_lo[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int m = row(e0 + e);
                if (rot) {
                    w01[e] = *(const f4*)(p.cs + (int64_t)m * 64 + d0);          // (cos, sin) of pairs d0, d0+1
                    w23[e] = *(const f4*)(p.cs + (int64_t)m * 64 + d0 + 2);      // ... d0+2, d0+3
                }
                if (is_q) {
                    off[e] = off_lo[e] = (int64_t)m * p.q_ts + hd * 128 + d0;
                } else {
                    const int b = m / p.q_len, t = m - b * p.q_len;
                    const int past = p.past_lens ? p.past_lens[b] : p.past_len;
                    off[e] = b * p.a_bs + kh * p.a_hs + (int64_t)(past + t) * 128 + d0;
                    off_lo[e] = b * p.lo_bs + kh * p.lo_hs + (int64_t)(past + t - p.lo_row0) * 128 + d0;
                }
            }
            _Float16* dh = is_q ? p.q_hi : rot ? p.k_arena : p.v_arena;
            _Float16* dl = is_q ? p.q_lo : rot ? p.k_lo : p.v_lo;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const f4 x0 = *at(e0 + e, 0), x1 = *at(e0 + e, 8);
                f4 a = x0, c = x1;
                if (rot) {
                    const float cs_[4] = {w01[e][0], w01[e][2], w23[e][0], w23[e][2]}, sn_[4] = {w01[e][1], w01[e][3], w23[e][1], w23[e][3]};
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        // q*cos + rotate_half(q)*sin (llama2.py:208): the low half pairs with -high, the high half with +low.  Which product
                        // stays unrounded is written out: left to the compiler, it changed with the code around it, and with it the last
                        // bits of every cached key (which the layers behind it turn into 3e-4 of the logits).
                        a[k] = fmaf(x0[k], cs_[k], -(x1[k] * sn_[k]));
                        c[k] = fmaf(x1[k], cs_[k], x0[k] * sn_[k]);
                    }
                }
                h4 ah, al, ch, cl;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    _Float16 t0, t1, t2, t3;
                    pc_split(a[k], t0, t1);
                    pc_split(c[k], t2, t3);
                    ah[k] = t0; al[k] = t1; ch[k] = t2; cl[k] = t3;
                }
                if (mrow(e0 + e) >= p.M) continue;
                *(h4*)(dh + off[e]) = ah;
                *(h4*)(dh + off[e] + 64) = ch;
                if (dl) { *(h4*)(dl + off_lo[e]) = al; *(h4*)(dl + off_lo[e] + 64) = cl; }
            }
        }
    } else {
        float* y = p.y + (int64_t)blockIdx.y * p.slab_stride + n;
#pragma unroll 1
        for (int e0 = 0; e0 < R; e0 += 16) {
            f4 old[16];
            if (EPI == EPI_ADD)
#pragma unroll
                for (int e = 0; e < 16; ++e) old[e] = *(const f4*)(y + (int64_t)row(e0 + e) * p.ldy);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                f4 v = *at(e0 + e, 0);
                if (EPI == EPI_ADD) v += old[e];
                if (mrow(e0 + e) < p.M) *(f4*)(y + (int64_t)mrow(e0 + e) * p.ldy) = v;
            }
        }
    }
}

// W: waves across and down a workgroup; TWO: both activation planes; NARROW: 128 columns instead of 256; TALL: 256 rows instead of 128
template <int W, int EPI, bool TWO, bool NARROW, bool TALL>
__global__ __launch_bounds__(256, 1) void gemm_dense_kernel(const DenseParams p) {
    static_assert(W == 2 && !(TWO && TALL), "four waves; two planes of 256 rows and their weights do not fit the LDS twice");
    using T = Tile<W, TWO, NARROW, TALL>;
    constexpr int MT = T::MT, NT = T::NT, S = T::S;
    using L = mfma_tile::Loop<MT, NT, S, TWO ? 2 : 1, T::BLK>;
    constexpr int PL = TWO ? 2 : 1, BM = L::BM, BN = L::BN;
    constexpr int NI = L::NI, NX = PL * BM / 32;                 // staging instructions per wave, of them for activations
    __shared__ __attribute__((aligned(16))) char lds[S * L::kStage];   // images: Xhi | Xlo | W

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    // block -> (M-block, weight panel), XCD-aware
    int mi, ni;
    if (!mfma_tile::tile_of(p.strips, p.mb, p.nb, blockIdx.x, mi, ni)) return;
    const int m0 = mi * BM;
    const int K = p.K, nkt = (K + BK - 1) / BK;          // K-steps of the whole product
    const int t0 = blockIdx.y * p.kper;                  // this slice's first K-step (kper = nkt without split-K)
    const int nk = (p.kper < nkt - t0) ? p.kper : nkt - t0;

    // global weight row of LDS weight-tile row r; -1 = past the end (clamped source, never stored)
    auto wrow = [&](int r) -> int {
        if (EPI == EPI_SILU) {
            const int f = (ni * NT + (r >> 6)) * 32 + (r & 31);
            return f < p.nfeat ? ((r >> 5) & 1) * p.nfeat + f : -1;
        }
        if (EPI == EPI_ROPE) {
            // a 64-column group = 32 features d of one head's first half next to their rotary partners d + 64, so
            // x[d] and x[d + 64] meet in the same row of a patch, 32 columns apart
            const int wt = r >> 6, c = r & 63;
            const int hd = ni * (BN / 128) + (wt >> 1);
            const int d = (c < 32) ? (wt & 1) * 32 + c : 64 + (wt & 1) * 32 + (c - 32);
            const int n = hd * 128 + d;
            return n < p.N ? n : -1;
        }
        const int n = ni * BN + r;
        return n < p.N ? n : -1;
    };

    // ---- staging sources: per lane one 16-byte chunk of one row per instruction; instruction i fills image rows 8 (4 i + wave) .. + 7 ----
    const int srow = 8 * wave + (lane >> 3);
    const int cx = (lane & 7) ^ ((srow >> 1) & 7);       // source chunk of the lane (the same in every instruction: 32 rows apart)
    const _Float16* src[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int r = 32 * i + srow;
        if (i < NX) {
            const bool lo = TWO && i >= NX / PL;
            const int m = m0 + r - (lo ? BM : 0);
            src[i] = (lo ? p.xl : p.xh) + (int64_t)(m < p.M ? m : p.M - 1) * p.ldx + cx * 8;
        } else {
            const int gr = wrow(r - PL * BM);
            src[i] = p.w + (int64_t)(gr < 0 ? 0 : gr) * p.ldw + cx * 8;
        }
    }
    // (chunks past K: the row's first chunk of the K-step, whose products the main loop leaves out)
    const int last = (K - (nkt - 1) * BK) / 8;           // valid chunks of the product's last K-step (8: a whole one)
    const int64_t past = cx < last ? 0 : -8 * cx;
    auto stage = [&](int i, int tl, char* buf) {
        const int t = t0 + tl;
        glds16(src[i] + ((int64_t)t * BK + (t == nkt - 1 ? past : 0)), buf + (4 * i + wave) * 1024);
    };
    const int keep = t0 + nk == nkt ? last : 8;          // chunks of this slice's last K-step

    typename L::Acc acc[L::MB][L::NB];
    auto mma = [](typename L::Acc& c, const h8& a, const h8& w) {
        if constexpr (T::BLK == 16)
            c = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, a, c, 0, 0, 0);
        else
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(w, a, c, 0, 0, 0);
    };
    L::template run<h8>(acc, lds, nk, keep, lane, wm, wn, mma, stage);

    // ---- epilogue: 64 accumulator columns of a wave at a time through an LDS patch of its own -> full-row global stores ----
    // (the weights are the products' first operand: a lane holds a row of a block and four neighbouring columns, in 32 x 32 blocks four times four;
    // patch: [32 MT][64] fp32, 16-byte quad c of row r at c ^ (r & 15))
    __syncthreads();                                       // every wave is done with the staging buffers
    constexpr int P = 32 * MT * 256, PARTS = NT / 2, ROOM = 4 * P * PARTS <= S * L::kStage ? PARTS : 1;   // patches that fit at a time
    char* patch = lds + wave * (P * ROOM);
    const int fr = lane % T::BLK;
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto put = [&](auto part, char* to) {
        constexpr int j = decltype(part)::value;
        constexpr int H = 64 / T::BLK;                     // blocks of 64 columns
#pragma unroll
        for (int i = 0; i < L::MB; ++i)
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int q = 0; q < T::BLK * T::BLK / 256; ++q) {
                    const typename L::Acc& c = acc[i][H * j + h];
                    *(f4*)(to + (T::BLK * i + fr) * 256 + ((T::BLK / 4 * h + mfma_tile::quad_of<T::BLK>(q, lane)) ^ (fr & 15)) * 16) =
                        f4{c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]};
                }
    };
    using First = std::integral_constant<int, 0>;
    using Second = std::integral_constant<int, PARTS - 1>;
    const int grp = ni * (BN / 64) + wn * PARTS;           // the wave's first 64-column group
    put(First{}, patch);
    if constexpr (ROOM == PARTS) {
        if constexpr (PARTS == 2) put(Second{}, patch + P);
        fence();
#pragma unroll 1
        for (int j = 0; j < PARTS; ++j) store_group<EPI, MT>(p, patch + j * P, lane, grp + j, m0 + wm * 32 * MT);
    } else {
        fence();
        store_group<EPI, MT>(p, patch, lane, grp, m0 + wm * 32 * MT);
        fence();
        put(Second{}, patch);
        fence();
        store_group<EPI, MT>(p, patch, lane, grp + 1, m0 + wm * 32 * MT);
    }
}

// Split-K tail: y[m][n] (+)= sum_z slab[z][m][n], slabs added in slice order (deterministic), 16 B per lane.
template <bool ADD>
__global__ __launch_bounds__(256) void dense_reduce_kernel(const float* __restrict__ slab, int64_t slab_stride, int ks,
                                                           float* __restrict__ y, int64_t ldy, int M, int N) {
    const int n4 = N >> 2;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)M * n4) return;
    const int m = (int)(i / n4), n = (int)(i - (int64_t)m * n4) * 4;
    const float* sp = slab + (int64_t)m * N + n;
    f4 v = *(const f4*)sp;
    for (int z = 1; z < ks; ++z) {
        const f4 x = *(const f4*)(sp + z * slab_stride);
        v[0] += x[0]; v[1] += x[1]; v[2] += x[2]; v[3] += x[3];
    }
    float* yp = y + (int64_t)m * ldy + n;
    if (ADD) {
        const f4 old = *(const f4*)yp;
        v[0] += old[0]; v[1] += old[1]; v[2] += old[2]; v[3] += old[3];
    }
    *(f4*)yp = v;
}

template <int EPI, bool TWO, bool NARROW, bool TALL>
int launch_dense_as(DenseParams& p, hipStream_t s, int kslices) {
    constexpr int BM = Tile<2, TWO, NARROW, TALL>::BM, BN = Tile<2, TWO, NARROW, TALL>::BN;
    p.mb = pc_ceil_div(p.M, BM);
    p.nb = (EPI == EPI_SILU) ? pc_ceil_div(p.nfeat, BN / 2) : pc_ceil_div(p.N, BN);
    const int nkt = pc_ceil_div(p.K, BK);
    p.kper = pc_ceil_div(nkt, kslices);
    p.strips = mfma_tile::strips(p.mb, p.nb, (TWO ? 2 : 1) * BM, BN);
    hipLaunchKernelGGL((gemm_dense_kernel<2, EPI, TWO, NARROW, TALL>), dim3(8 * p.strips.mh * p.strips.nh, pc_ceil_div(nkt, p.kper)), dim3(256), 0, s, p);
    return pc_check_launch("gemm_dense_kernel");
}

#ifdef PC_DEV_SWEEPS
#include "pc_gemm_dense_dev.h"
#endif

// the 128-row tiles, BN = 256 or 128 columns
template <int BN, int EPI>
int launch_dense(DenseParams& p, hipStream_t s, int kslices = 1) {
    if (p.xl8) {
#ifdef PC_DEV_SWEEPS
        return lockstep::launch<BN == 256 ? 2 : 4, EPI>(p, s, kslices);
#else
        pc_set_error("pc_gemm_dense: the int8 residual plane (x_lo8) needs a -DPC_DEV_SWEEPS build (csrc/pc_dev.h)");
        return PC_ERR_ARG;
#endif
    }
    if (p.xl) return launch_dense_as<EPI, true, BN == 128, false>(p, s, kslices);
    return launch_dense_as<EPI, false, BN == 128, false>(p, s, kslices);
}

// Few-row launches of the N = hidden projections (o_proj, down_proj at a few hundred rows: 64-128 tiles of 128 x 256 for
// 256 CUs): the K range is cut into slices that run as separate workgroups and meet in a fixed-order reduction.
// Returns 0 when split-K does not apply (the caller then launches the plain form).
template <int EPI>
int launch_dense_splitk(DenseParams& p, hipStream_t s, float* ws, int64_t ws_bytes, int* launched) {
    static const int forced_ks = [] { const char* e = getenv("PC_DENSE_KS"); return e ? atoi(e) : 0; }();
    static const int forced_bn = [] { const char* e = getenv("PC_DENSE_BN"); return e ? atoi(e) : 0; }();
    *launched = 0;
    if (!ws || p.xscale || (EPI != EPI_ADD && EPI != EPI_STORE)) return 0;
    const int nkt = pc_ceil_div(p.K, BK), mb = pc_ceil_div(p.M, 128);
    // widest panel whose slices still fill the chip: 256-wide tiles do twice the MFMAs per LDS byte of 128-wide ones
    const int b256 = mb * pc_ceil_div(p.N, 256), b128 = mb * pc_ceil_div(p.N, 128);
    bool narrow = forced_bn ? forced_bn == 128 : false;
    int ks = forced_ks ? forced_ks : 256 / b256;
    if (!forced_ks && !forced_bn && ks < 2 && 256 / b128 >= 2) { narrow = true; ks = 256 / b128; }
    if (ks > 8) ks = 8;
    while (ks > 1 && nkt / ks < 8) --ks;                     // keep >= 8 K-steps per slice
    if (ks < 2 || (int64_t)ks * p.M * p.N * 4 > ws_bytes) return 0;
    float* y = p.y; const int64_t ldy = p.ldy;
    p.y = ws; p.ldy = p.N; p.slab_stride = (int64_t)p.M * p.N;
    const int rc = narrow ? launch_dense<128, EPI_STORE>(p, s, ks) : launch_dense<256, EPI_STORE>(p, s, ks);
    if (rc) return rc;
    const int nslab = pc_ceil_div(pc_ceil_div(p.K, BK), p.kper);
    const int64_t items = (int64_t)p.M * (p.N >> 2);
    const dim3 grid((unsigned)((items + 255) / 256)), block(256);
    if (EPI == EPI_ADD) hipLaunchKernelGGL((dense_reduce_kernel<true>), grid, block, 0, s, ws, p.slab_stride, nslab, y, ldy, p.M, p.N);
    else hipLaunchKernelGGL((dense_reduce_kernel<false>), grid, block, 0, s, ws, p.slab_stride, nslab, y, ldy, p.M, p.N);
    *launched = 1;
    return pc_check_launch("dense_reduce_kernel");
}

template <int EPI>
int launch_dense_tile(DenseParams& p, hipStream_t s) {
    static const int forced = [] { const char* e = getenv("PC_DENSE_BN"); return e ? atoi(e) : 0; }();
    // 256-wide weight panels (twice the MFMAs per LDS byte) unless the 128-wide grid needs fewer tile-rounds of the 256
    // CUs: a 128-wide tile pass takes 0.62 of a 256-wide one (measured at K = 4096 and 11008,
    // profiles/r02_dense_splitk.txt), e.g. 1000 x 4096: 128 wide tiles = one round of half the chip, 256 narrow tiles =
    // one round of all of it
    const int cols = (EPI == EPI_SILU) ? p.nfeat * 2 : p.N;
    const int mb = pc_ceil_div(p.M, 128);
    const int b256 = mb * pc_ceil_div(cols, 256), b128 = mb * pc_ceil_div(cols, 128);
    const bool narrow = forced ? forced == 128 : (b256 <= 512 && 0.62f * pc_ceil_div(b128, 256) < 1.0f * pc_ceil_div(b256, 256));
    // One plane: 256 x 256 tiles where their whole rounds of the 256 CUs cost less than the 128 x 256 tiles' total.  Per round at K = 4096
    // (one plane, N = 12288 / 22016 / 32000, 1 737 / 2 940 / 3 584 rows): 95-111 us against 61-70 us, the latter hardly quantised.
    // (Both planes: 256-row tiles need 32-deep K-steps and gain 4 % at best, 3 584 x 12 288; 128-row tiles throughout.)
    const int b2 = pc_ceil_div(p.M, 256) * pc_ceil_div(cols, 256);
    if (!p.xl && !p.xl8 && !forced && !narrow && 1.52f * 256.f * pc_ceil_div(b2, 256) < (float)b256) return launch_dense_as<EPI, false, false, true>(p, s, 1);
    return narrow ? launch_dense<128, EPI>(p, s) : launch_dense<256, EPI>(p, s);
}

}  // namespace

namespace {
struct Lo8Operands { const void* x_lo8; const float* x_lo8_scale; int64_t ldx8; const void* w8; const float* w8_scale; int64_t ldw8; };
int gemm_dense_impl(const void* x_hi, const void* x_lo, int64_t ldx, const void* w, int64_t ldw, const float* w_scale,
                    const float* x_scale, const float* corr, int64_t ldc, const int32_t* corr_has, int32_t M, int32_t N,
                    int32_t K, int32_t epilogue, float* y, int64_t ldy, void* out_hi, void* out_lo, int64_t ldo, void* stream,
                    void* workspace = nullptr, int64_t ws_bytes = 0, const Lo8Operands* lo8 = nullptr) {
    PC_REQUIRE(M > 0 && N > 0 && K > 0 && K % 8 == 0 && N % 4 == 0, PC_ERR_ARG, "pc_gemm_dense: need M, N, K > 0, K%%8==0, N%%4==0");
    PC_REQUIRE(x_hi && w, PC_ERR_ARG, "pc_gemm_dense: null pointer");
    PC_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x_hi & 15) == 0 && ((uintptr_t)w & 15) == 0 &&
               ((uintptr_t)x_lo & 15) == 0, PC_ERR_ARG, "pc_gemm_dense: operands must be 16-byte aligned with row strides %% 8 == 0");
    PC_REQUIRE(!w_scale || ((uintptr_t)w_scale & 15) == 0, PC_ERR_ARG, "pc_gemm_dense: w_scale must be 16-byte aligned");
    DenseParams p;
    memset(&p, 0, sizeof(p));
    p.xh = (const _Float16*)x_hi; p.xl = (const _Float16*)x_lo; p.ldx = ldx;
    p.w = (const _Float16*)w; p.ldw = ldw; p.wscale = w_scale;
    PC_REQUIRE(!x_scale || (w_scale && !x_lo && corr && corr_has && ldc >= N && ldc % 4 == 0 && ((uintptr_t)corr & 15) == 0), PC_ERR_ARG,
               "pc_gemm_dense_a8: int8 activations need w_scale, no lo plane, corr (16-byte aligned, ldc >= N) and corr_has");
    p.xscale = x_scale; p.corr = corr; p.ldc = ldc; p.corr_has = corr_has;
    p.M = M; p.N = N; p.K = K;
    if (lo8) {
        PC_REQUIRE(lo8->x_lo8 && lo8->x_lo8_scale && lo8->w8 && lo8->w8_scale && !x_lo && !x_scale && !w_scale, PC_ERR_ARG,
                   "pc_gemm_dense_lo8: needs the int8 residual plane, its row scales, the int8 weight image and its row scales (and no "
                   "fp16 lo plane / LLM.int8 operands)");
        PC_REQUIRE(K % 64 == 0 && lo8->ldx8 >= K && lo8->ldw8 >= K && lo8->ldx8 % 16 == 0 && lo8->ldw8 % 16 == 0 &&
                   (((uintptr_t)lo8->x_lo8 | (uintptr_t)lo8->w8) & 15) == 0, PC_ERR_ARG,
                   "pc_gemm_dense_lo8: K %% 64 == 0, int8 planes 16-byte aligned with row strides %% 16 == 0");
        p.xl8 = (const signed char*)lo8->x_lo8; p.xl8_scale = lo8->x_lo8_scale; p.ldx8 = lo8->ldx8;
        p.w8 = (const signed char*)lo8->w8; p.w8_scale = lo8->w8_scale; p.ldw8 = lo8->ldw8;
    }
    hipStream_t s = (hipStream_t)stream;
    if (epilogue == EPI_SILU || epilogue == EPI_GELU) {
        PC_REQUIRE(out_hi && ldo % 4 == 0 && ((uintptr_t)out_hi & 7) == 0 && ((uintptr_t)out_lo & 7) == 0, PC_ERR_ARG,
                   "pc_gemm_dense: activation epilogues need an 8-byte aligned out_hi plane (out_lo optional)");
        p.oh = (_Float16*)out_hi; p.ol = (_Float16*)out_lo; p.ldo = ldo;
        if (epilogue == EPI_SILU) {
            PC_REQUIRE(N % 8 == 0 && ldo >= N / 2, PC_ERR_ARG, "pc_gemm_dense: SiLU epilogue needs N = 2*inter, inter %% 4 == 0, ldo >= inter");
            p.nfeat = N / 2;
            return launch_dense_tile<EPI_SILU>(p, s);
        }
        PC_REQUIRE(ldo >= N, PC_ERR_ARG, "pc_gemm_dense: GELU epilogue needs ldo >= N");
        return launch_dense_tile<EPI_GELU>(p, s);
    }
    PC_REQUIRE(y && ldy >= N && ldy % 4 == 0 && ((uintptr_t)y & 15) == 0, PC_ERR_ARG, "pc_gemm_dense: bad fp32 output");
    p.y = y; p.ldy = ldy;
    PC_REQUIRE(epilogue == EPI_ADD || epilogue == EPI_STORE, PC_ERR_ARG, "pc_gemm_dense: unknown epilogue %d", epilogue);
    PC_REQUIRE(!workspace || ((uintptr_t)workspace & 15) == 0, PC_ERR_ARG, "pc_gemm_dense_ws: workspace must be 16-byte aligned");
    int launched = 0;
    const int rc = epilogue == EPI_ADD ? launch_dense_splitk<EPI_ADD>(p, s, (float*)workspace, ws_bytes, &launched)
                                       : launch_dense_splitk<EPI_STORE>(p, s, (float*)workspace, ws_bytes, &launched);
    if (rc || launched) return rc;
    p.y = y; p.ldy = ldy; p.slab_stride = 0;
    if (epilogue == EPI_ADD) return launch_dense_tile<EPI_ADD>(p, s);
    return launch_dense_tile<EPI_STORE>(p, s);
}
}  // namespace

PC_EXPORT int pc_gemm_dense(const void* x_hi, const void* x_lo, int64_t ldx, const void* w, int64_t ldw,
                            const float* w_scale, int32_t M, int32_t N, int32_t K, int32_t epilogue, float* y, int64_t ldy,
                            void* out_hi, void* out_lo, int64_t ldo, void* stream) {
    return gemm_dense_impl(x_hi, x_lo, ldx, w, ldw, w_scale, nullptr, nullptr, 0, nullptr, M, N, K, epilogue, y, ldy, out_hi,
                           out_lo, ldo, stream);
}

// pc_gemm_dense with a caller-owned scratch buffer: plain-store / residual-add launches whose tile grid would leave most
// of the 256 CUs idle (a few hundred rows against N = hidden) cut K into slices -- partial slabs [slices][M][N] fp32 in
// `workspace`, added in slice order by a second launch.  Without room for the slabs the call is pc_gemm_dense.
PC_EXPORT int pc_gemm_dense_ws(const void* x_hi, const void* x_lo, int64_t ldx, const void* w, int64_t ldw,
                               const float* w_scale, int32_t M, int32_t N, int32_t K, int32_t epilogue, float* y, int64_t ldy,
                               void* out_hi, void* out_lo, int64_t ldo, void* workspace, int64_t ws_bytes, void* stream) {
    return gemm_dense_impl(x_hi, x_lo, ldx, w, ldw, w_scale, nullptr, nullptr, 0, nullptr, M, N, K, epilogue, y, ldy, out_hi,
                           out_lo, ldo, stream, workspace, ws_bytes);
}

#ifdef PC_DEV_SWEEPS      // (dev builds only: see pc_dev.h)
// pc_gemm_dense with the residual activation plane as int8 codes (pc_quant_rows_i8) against an int8 image of the weights: the
// second plane's product runs on v_mfma_i32_32x32x32_i8 at twice the fp16 MFMA rate (include/promptcache_hip.h).
PC_EXPORT int pc_gemm_dense_lo8(const void* x_hi, int64_t ldx, const void* x_lo8, const float* x_lo8_scale, int64_t ldx8, const void* w,
                                int64_t ldw, const void* w8, const float* w8_scale, int64_t ldw8, int32_t M, int32_t N, int32_t K,
                                int32_t epilogue, float* y, int64_t ldy, void* out_hi, void* out_lo, int64_t ldo, void* workspace,
                                int64_t ws_bytes, void* stream) {
    const Lo8Operands lo8{x_lo8, x_lo8_scale, ldx8, w8, w8_scale, ldw8};
    return gemm_dense_impl(x_hi, nullptr, ldx, w, ldw, nullptr, nullptr, nullptr, 0, nullptr, M, N, K, epilogue, y, ldy, out_hi, out_lo,
                           ldo, stream, workspace, ws_bytes, &lo8);
}
#endif  // PC_DEV_SWEEPS

// The fused q|k|v projection of a many-row pass at head_dim 128 (include/promptcache_hip.h: pc_dense_qkv_args): projection,
// RoPE at the supplied positions, rotated q as hi / lo planes, rotated k and v appended to the arena (+ residual planes) -- the
// [M][(H + 2 Hkv) D] fp32 intermediate and a separate pc_rope_append launch are not needed.
PC_EXPORT int pc_gemm_dense_qkv_rope(const pc_dense_qkv_args* a, void* stream) {
    PC_REQUIRE(a && a->struct_bytes == (uint32_t)sizeof(pc_dense_qkv_args), PC_ERR_ARG,
               "pc_gemm_dense_qkv_rope: args is NULL or struct_bytes != sizeof(pc_dense_qkv_args) (ABI mismatch)");
    PC_REQUIRE(a->D == 128 && a->B > 0 && a->H > 0 && a->Hkv > 0 && a->q_len > 0 && a->K > 0 && a->K % 8 == 0, PC_ERR_ARG,
               "pc_gemm_dense_qkv_rope: head_dim must be 128 (got %d); B, H, Hkv, q_len, K > 0; K %% 8 == 0", a->D);
    PC_REQUIRE(a->x_hi && a->w && a->cs && a->q_hi && a->k_arena && a->v_arena, PC_ERR_ARG, "pc_gemm_dense_qkv_rope: null pointer");
    PC_REQUIRE(a->ldx >= a->K && a->ldw >= a->K && a->ldx % 8 == 0 && a->ldw % 8 == 0 && ((uintptr_t)a->x_hi & 15) == 0 &&
               ((uintptr_t)a->w & 15) == 0 && ((uintptr_t)a->x_lo & 15) == 0 && ((uintptr_t)a->cs & 15) == 0, PC_ERR_ARG,
               "pc_gemm_dense_qkv_rope: operands and the rotation table must be 16-byte aligned with row strides %% 8 == 0");
    PC_REQUIRE(a->q_token_stride % 4 == 0 && a->arena_head_stride % 4 == 0 && a->arena_batch_stride % 4 == 0 &&
               ((uintptr_t)a->q_hi & 7) == 0 && ((uintptr_t)a->q_lo & 7) == 0 && ((uintptr_t)a->k_arena & 7) == 0 &&
               ((uintptr_t)a->v_arena & 7) == 0, PC_ERR_ARG, "pc_gemm_dense_qkv_rope: outputs must keep 8-byte alignment");
    PC_REQUIRE((a->k_lo == nullptr) == (a->v_lo == nullptr), PC_ERR_ARG, "pc_gemm_dense_qkv_rope: k_lo and v_lo go together");
    PC_REQUIRE(!a->k_lo || (a->lo_head_stride % 4 == 0 && a->lo_batch_stride % 4 == 0 && a->lo_row0 >= 0 &&
                            (a->past_lens ? a->lo_row0 == 0 : a->lo_row0 <= a->past_len)), PC_ERR_ARG,
               "pc_gemm_dense_qkv_rope: residual planes: 8-byte aligned strides, lo_row0 in [0, past_len] (0 with past_lens)");
    PC_REQUIRE((int64_t)a->past_len + a->q_len <= a->cap, PC_ERR_BOUNDS,
               "pc_gemm_dense_qkv_rope: past_len %d + q_len %d exceeds arena rows %d", a->past_len, a->q_len, a->cap);
    DenseParams p;
    memset(&p, 0, sizeof(p));
    p.xh = (const _Float16*)a->x_hi; p.xl = (const _Float16*)a->x_lo; p.ldx = a->ldx;
    p.w = (const _Float16*)a->w; p.ldw = a->ldw;
    p.M = a->B * a->q_len; p.N = (a->H + 2 * a->Hkv) * 128; p.K = a->K;
    if (a->x_lo8) {
        PC_REQUIRE(!a->x_lo && a->x_lo8_scale && a->w8 && a->w8_scale && a->K % 64 == 0 && a->ldx8 >= a->K && a->ldw8 >= a->K &&
                   a->ldx8 % 16 == 0 && a->ldw8 % 16 == 0 && (((uintptr_t)a->x_lo8 | (uintptr_t)a->w8) & 15) == 0, PC_ERR_ARG,
                   "pc_gemm_dense_qkv_rope: the int8 residual plane replaces x_lo; K %% 64 == 0; int8 planes 16-byte aligned, row strides %% 16 == 0");
        p.xl8 = (const signed char*)a->x_lo8; p.xl8_scale = a->x_lo8_scale; p.ldx8 = a->ldx8;
        p.w8 = (const signed char*)a->w8; p.w8_scale = a->w8_scale; p.ldw8 = a->ldw8;
    }
    p.cs = (const float2*)a->cs; p.q_hi = (_Float16*)a->q_hi; p.q_lo = (_Float16*)a->q_lo; p.q_ts = a->q_token_stride;
    p.k_arena = (_Float16*)a->k_arena; p.v_arena = (_Float16*)a->v_arena; p.a_bs = a->arena_batch_stride; p.a_hs = a->arena_head_stride;
    p.k_lo = (_Float16*)a->k_lo; p.v_lo = (_Float16*)a->v_lo; p.lo_bs = a->lo_batch_stride; p.lo_hs = a->lo_head_stride;
    p.lo_row0 = a->lo_row0;
    p.H = a->H; p.Hkv = a->Hkv; p.q_len = a->q_len; p.past_len = a->past_len; p.past_lens = a->past_lens;
    return launch_dense_tile<EPI_ROPE>(p, (hipStream_t)stream);
}

// LLM.int8 form of pc_gemm_dense (pc_int8.hip): xq = activation CODES of pc_quant_act_i8 held in fp16 (row-major [M][K]), w =
// weight codes held in fp16, y = (sum_k w[n][k] * xq[m][k]) * w_scale[n] * x_scale[m] (+ corr[m][n] when *corr_has), then
// the epilogue.  The integer dot product is accumulated in fp32 by the fp16 MFMAs: exact below 2^24 per accumulator.
PC_EXPORT int pc_gemm_dense_a8(const void* xq, int64_t ldx, const void* w_codes, int64_t ldw, const float* w_scale,
                               const float* x_scale, const float* corr, int64_t ldc, const int32_t* corr_has, int32_t M,
                               int32_t N, int32_t K, int32_t epilogue, float* y, int64_t ldy, void* out_hi, void* out_lo,
                               int64_t ldo, void* stream) {
    PC_REQUIRE(w_scale && x_scale, PC_ERR_ARG, "pc_gemm_dense_a8: null pointer");
    return gemm_dense_impl(xq, nullptr, ldx, w_codes, ldw, w_scale, x_scale, corr, ldc, corr_has, M, N, K, epilogue, y, ldy,
                           out_hi, out_lo, ldo, stream);
}
