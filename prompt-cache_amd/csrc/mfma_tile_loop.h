// The main loop of the LDS-tiled products (pc_gemm_dense.hip, pb_linear_tiles.hip): four waves (2 x 2) of 32 MT x 32 NT results, both operands
// as 128-byte rows (64 k of 2 bytes) in a ring of S LDS images, PL row operands ("planes") against one column operand.
//
// Image of a K-step: PL x 64 MT rows, then 64 NT columns, as rows of 128 bytes; the 16-byte chunk c of row r sits at position
// c ^ ((r >> 1) & 7), so that a fragment read touches every bank slot.  A wave's staging instruction i (global_load_lds, 1 KiB) fills rows
// 32 i + 8 wave .. + 7.  One barrier per K-step, fragments read one part of the products ahead, in two register sets; the last
// part of K-step t is multiplied behind the barrier, next to the first reads of K-step t + 1 and the first half of the staging of K-step t
// + S (its image was just freed); the second half goes out in the next part.
//
// BLK: results in blocks of 16 x 16 (32-deep slabs, two a K-step) or 32 x 32 (16-deep, four).  What bounds these loops on a full chip is power: a workgroup of
// 128 x 128, 128 x 256 or 256 x 256 takes 745, 1230 or 2200 clocks a K-step (of 512, 1024, 2048 of its MFMAs) whether it is alone, at 2.4 GHz, or one of 256, at 1.3
// to 1.6 GHz; with zeros as operands 256 of them run at 2.2.  MFMAs alone on random operands in registers, 256 CUs: 1.61 PFLOP/s in 32 x 32 x 16, 1.69 in
// 16 x 16 x 32, and so it is here, 32 x 32 / 16 x 16, us: two planes, 1737 x 12288, K = 4096 306 / 297, 3584 x 4096, K = 11008 530 / 517, 3584 x 12288 599 / 575; one
// plane, 2048 rows, K = 2048, 128 x 192 tiles 27.1 / 25.9, 128 x 256 34.4 / 33.1, 256 x 256 over 4096 x 4096 x 4096 103.9 / 101.7.  128 x 128 tiles of one plane are not
// as close to that limit and take 22.4 us for 21.4, 38.4 for 36.2 (2048 x 2048, K = 2048, 4096): 32 x 32.  Nor is anything else where few CUs have a tile: two planes,
// 70 x 640, K = 5120 (5 tiles) 46.1 / 51.5, 102 x 2560, K = 1024 (20) 14.0 / 15.1, from 64 tiles on equal, 256 and more 0.96 .. 0.99; one plane, 256 x 256 tiles on 192 CUs
// (1500 x 8192, K = 2048) 47.5 / 48.8, on all 0.95 .. 0.98 (2048 x 8192, K = 8192 194 / 187); over K <= 256 1 .. 3 % more.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace mfma_tile {

template <int N>
using I = std::integral_constant<int, N>;

template <int MT, int NT, int S, int PL, int BLK>
struct Loop {
    static constexpr int BM = 64 * MT, BN = 64 * NT, ROWS = PL * BM + BN;
    static constexpr int kStage = ROWS * 128, NI = ROWS / 32;        // bytes of an image, staging instructions of a wave
    static constexpr int MB = 32 * MT / BLK, NB = 32 * NT / BLK;     // a wave's blocks of results
    typedef float Acc __attribute__((ext_vector_type(BLK * BLK / 64)));

    // acc[i][j] = rows x columns.  V: a lane's eight elements of a fragment; mma(acc, row fragment, column fragment);
    // stage(i, t, image): this wave's staging instruction i of K-step t.  nk >= 1 K-steps, of the last one only the first `last` 16-byte
    // chunks count (1 .. 8; what is staged for the others is multiplied as zeros).  Returns with no load in flight.
    template <typename V, typename Mma, typename Stage>
    static __device__ __forceinline__ void run(Acc (&acc)[MB][NB], char* lds, int nk, int last, int lane, int wm, int wn, Mma mma, Stage stage) {
        constexpr int G = 64 / BLK, SLABS = 8 / G;
        constexpr bool SOON = S == 2 && PL * SLABS == 2;             // (the part after next waits for what is staged)
        constexpr int D0 = SOON ? NI : NI / 2;
        // lane = (row fr of the block, 16-byte chunk fg of the slab)
        const int fr = lane % BLK, fg = lane / BLK;
        int foff[SLABS];
#pragma unroll
        for (int ks = 0; ks < SLABS; ++ks) foff[ks] = fr * 128 + (((G * ks + fg) ^ ((fr >> 1) & 7)) << 4);
        const int a_base = (wm * 32 * MT) * 128, b_base = (PL * BM + wn * 32 * NT) * 128;
        // The products of a K-step go in U parts, plane pl of slab ks being part PL ks + pl: fa[part % 2] x fb[ks % 2]
        constexpr int U = PL * SLABS, MF = MB * NB;
        static_assert((SOON ? 2 * NI : NI - D0) <= MF, "at most one staging instruction behind a product");
        V fa[2][MB], fb[2][NB];
        auto read_one = [&](const char* buf, int u, int q) {         // operand q of part u: its plane's rows, behind the columns if it begins a slab
            const int pl = u % PL, ks = u / PL, c = pl == 0 ? NB : 0;
            if (q < c)
                fb[ks % 2][q] = *(const V*)(buf + b_base + q * BLK * 128 + foff[ks]);
            else
                fa[u % 2][q - c] = *(const V*)(buf + a_base + (pl * BM + (q - c) * BLK) * 128 + foff[ks]);
        };
        // part u's products, between them the reads of the next part (none behind the last one of all) and the staging instructions [d0, d1) of K-step t.
        // (Left alone, hipcc sinks the reads next to their first use and waits for them there.)
        auto part = [&](auto fresh, auto u_, auto next, const char* buf, int t, char* to, auto d0_, auto d1_) {
            constexpr int u = decltype(u_)::value, d0 = decltype(d0_)::value, d1 = decltype(d1_)::value;
            constexpr int un = (u + 1) % U, R = decltype(next)::value ? MB + (un % PL == 0 ? NB : 0) : 0;
            constexpr int gap = MF >= (BLK == 32 ? 2 : 4) * R ? 2 : 1, per = gap == 1 && BLK == 32 ? 2 : 1;
#pragma unroll
            for (int k = 0; k < MF; ++k) {
                const int i = k / NB, j = k % NB;
                if (decltype(fresh)::value) acc[i][j] = Acc{};
                mma(acc[i][j], fa[u % 2][i], fb[u / PL % 2][j]);
                __builtin_amdgcn_sched_barrier(0);
                if (k % gap == 0)
#pragma unroll
                    for (int e = 0; e < per; ++e)
                        if (per * (k / gap) + e < R) read_one(buf, un, per * (k / gap) + e);
                // (no loop here: with one, the unrolled whole passes what the compiler unrolls)
                constexpr int len = SOON ? 2 * (d1 - d0) : MF, over = len > 0 ? len : 1;
                const int n = d0 + k * (d1 - d0) / over;
                if (k < len && n < d0 + (k + 1) * (d1 - d0) / over) stage(n, t, to);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto clamp = [&](int t) { return t < nk ? t : nk - 1; };     // (past the end the last K-step goes into the idle image again)
        auto keep = [&](int u, int t) {                              // zeros for the chunks past K
            if (last == 8 || t + 1 < nk) return;
            const bool in = G * (u / PL) + fg < last;
#pragma unroll
            for (int q = 0; q < MB; ++q) fa[u % 2][q] = in ? fa[u % 2][q] : V{};
            if (u % PL == 0)
#pragma unroll
                for (int q = 0; q < NB; ++q) fb[u / PL % 2][q] = in ? fb[u / PL % 2][q] : V{};
        };
#pragma unroll
        for (int st = 0; st < S - 1; ++st)
#pragma unroll
            for (int i = 0; i < NI; ++i) stage(i, clamp(st), lds + st * kStage);
#pragma unroll
        for (int i = 0; i < D0; ++i) stage(i, clamp(S - 1), lds + (S - 1) * kStage);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * NI + D0) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int q = 0; q < MB + NB; ++q) read_one(lds, 0, q);
        // the first part is multiplied onto a constant zero, before the loop: clearing the accumulators first is an instruction a register
        // that runs once, and code that runs once comes in at the pace of instruction misses
        int cur = 0, prev = (S - 1) * kStage;                        // images of K-steps t and t + S - 1
        keep(0, 0);
        part(std::true_type{}, I<0>{}, std::true_type{}, lds, clamp(S - 1), lds + prev, I<D0>{}, I<NI>{});
        auto middle = [&](int t, auto end) {                         // parts 1 .. U - 2
            auto one = [&](auto u) {
                if (decltype(end)::value) keep(decltype(u)::value, t);
                part(std::false_type{}, u, std::true_type{}, lds + cur, 0, nullptr, I<0>{}, I<0>{});
            };
            if constexpr (U > 2) one(I<1>{}), one(I<2>{});
            static_assert(U == 2 || U == 4, "two or four parts");
        };
        int t = 0;
        for (; t + 1 < nk; ++t) {
            middle(t, std::false_type{});
            // K-step t + 1 has landed (S - 2 younger ones may be in flight), for everyone behind the barrier; all reads of K-step t are complete
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * NI) : "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            prev = cur;
            cur = cur + kStage == S * kStage ? 0 : cur + kStage;
            part(std::false_type{}, I<U - 1>{}, std::true_type{}, lds + cur, clamp(t + S), lds + prev, I<0>{}, I<D0>{});
            keep(0, t + 1);
            part(std::false_type{}, I<0>{}, std::true_type{}, lds + cur, clamp(t + S), lds + prev, I<D0>{}, I<NI>{});
        }
        middle(t, std::true_type{});
        keep(U - 1, t);
        part(std::false_type{}, I<U - 1>{}, std::false_type{}, nullptr, 0, nullptr, I<0>{}, I<0>{});
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // (clamped re-loads of the last K-step)
    }
};

// what a lane holds of an accumulator of BLK x BLK results whose first operand are the columns: quad q of row lane % BLK, columns quad_of(q, lane) * 4 .. + 3
template <int BLK>
static __device__ __forceinline__ int quad_of(int q, int lane) { return BLK == 16 ? lane >> 4 : 2 * q + (lane >> 5); }

// How a grid of mb x nb tiles is dealt to the XCDs: cut into 8 rectangles (px row strips by 8 / px column strips of mh x nh tiles), fewest
// rounds of an XCD's 32 CUs first, then fewest operand rows per K-step (row_cost for a tile's rows, col_cost for its columns) among 32 tiles
// that run at a time.  Where no cut reaches the rounds of an even share, the tiles go out in 8 runs of mh, column by column (px = 0, nh = 1):
// 3 x 81 tiles of 128 x 128 are 33 in a rectangle and 31 in a run (257 x 10272, K = 2048: 28.7 us in two rounds, 16.8 in one).  Launch 8 mh nh workgroups.
struct Strips { int px, mh, nh; };
static inline Strips strips(int mb, int nb, int row_cost, int col_cost) {
    Strips s{1, mb, (nb + 7) / 8};
    int64_t best = -1;
    for (int px = 1; px <= 8; px *= 2) {
        const int mh = (mb + px - 1) / px, nh = (nb + 8 / px - 1) / (8 / px), reach = mh < 32 ? mh : 32;
        const int64_t cost = (((int64_t)mh * nh + 31) / 32 << 32) + (int64_t)reach * row_cost + (int64_t)((32 + reach - 1) / reach) * col_cost;
        if (best < 0 || cost < best) { best = cost; s = Strips{px, mh, nh}; }
    }
    const int64_t run = ((int64_t)mb * nb + 7) / 8;
    if ((run + 31) / 32 < best >> 32) s = Strips{0, (int)run, 1};
    return s;
}
// the tile of workgroup `block` of such a launch; false: none
static __device__ __forceinline__ bool tile_of(const Strips& s, int mb, int nb, int block, int& mi, int& ni) {
    const int xcd = block & 7, slot = block >> 3;
    if (s.px == 0) {
        const int t = xcd * s.mh + slot;
        mi = t % mb;
        ni = t / mb;
    } else {
        mi = xcd % s.px * s.mh + slot % s.mh;
        ni = xcd / s.px * s.nh + slot / s.mh;
    }
    return mi < mb && ni < nb;
}

}  // namespace mfma_tile
