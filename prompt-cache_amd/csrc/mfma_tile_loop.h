// The main loop of the LDS-tiled products (pc_gemm_dense.hip, pb_linear_tiles.hip): four waves (2 x 2) of 32 MT x 32 NT result blocks, both operands
// as 128-byte rows (64 k of 2 bytes) in a ring of S LDS images, PL row operands ("planes") against one column operand.
//
// Image of a K-step: PL x 64 MT rows, then 64 NT columns, as rows of 128 bytes; the 16-byte chunk c of row r sits at position
// c ^ ((r >> 1) & 7), so that a fragment read touches every bank slot.  A wave's staging instruction i (global_load_lds, 1 KiB) fills rows
// 32 i + 8 wave .. + 7.  One barrier per K-step, fragments read one 16-deep slab ahead of their products, in two register sets; the last
// slab of K-step t is multiplied behind the barrier, next to the first reads of K-step t + 1 and the first half of the staging of K-step t
// + S (its image was just freed); the second half goes out in the next slab.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace mfma_tile {

template <int MT, int NT, int S, int PL>
struct Loop {
    static constexpr int BM = 64 * MT, BN = 64 * NT, ROWS = PL * BM + BN;
    static constexpr int kStage = ROWS * 128, NI = ROWS / 32;        // bytes of an image, staging instructions of a wave

    // acc[i][j] = rows x columns.  V: a lane's eight elements of a fragment; mma(acc, row fragment, column fragment);
    // stage(i, t, image): this wave's staging instruction i of K-step t.  nk >= 1 K-steps, of the last one only the first `last` 16-byte
    // chunks count (1 .. 8; what is staged for the others is multiplied as zeros).  Returns with no load in flight.
    template <typename V, typename Acc, typename Mma, typename Stage>
    static __device__ __forceinline__ void run(Acc (&acc)[MT][NT], char* lds, int nk, int last, int lane, int wm, int wn, Mma mma, Stage stage) {
        constexpr int R = PL * MT + NT, MF = PL * MT * NT, D0 = NI / 2;
        // lane = (row fr of the 32-row block, k-half fh)
        const int fr = lane & 31, fh = lane >> 5;
        int foff[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) foff[ks] = fr * 128 + (((2 * ks + fh) ^ ((fr >> 1) & 7)) << 4);
        const int a_base = (wm * 32 * MT) * 128, b_base = (PL * BM + wn * 32 * NT) * 128;
        struct Frags { V a[PL * MT], b[NT]; };
        auto read_one = [&](Frags& f, const char* buf, int ks, int q) {
            if (q < NT) {
                f.b[q] = *(const V*)(buf + b_base + q * 32 * 128 + foff[ks]);
            } else {
                const int pl = (q - NT) / MT, i = (q - NT) % MT;
                f.a[q - NT] = *(const V*)(buf + a_base + (pl * BM + i * 32) * 128 + foff[ks]);
            }
        };
        auto mfma_one = [&](const Frags& f, int q) {
            const int pl = q / (MT * NT), i = q / NT % MT, j = q % NT;
            mma(acc[i][j], f.a[pl * MT + i], f.b[j]);
        };
        // (left alone, hipcc sinks the reads next to their first use and waits for them there)
        auto slab = [&](const Frags& f, Frags& nx, const char* buf, int ks) {
#pragma unroll
            for (int q = 0; q < R; ++q) read_one(nx, buf, ks, q);
#pragma unroll
            for (int q = 0; q < MF; ++q) mfma_one(f, q);
#pragma unroll
            for (int k = 0; k < MF; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          // one MFMA
                if (MF >= 2 * R) {
                    if (k < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           // one DS read
                } else {
                    if (2 * k + 1 < R) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                    else if (2 * k < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
            }
        };
        // a slab that also carries the staging instructions [d0, d1) of K-step t; one read behind every second MFMA where that
        // places them all, else two behind each
        auto slab_staging = [&](auto fresh, const Frags& f, Frags& nx, const char* buf, int ks, int t, char* to, int d0, int d1) {
#pragma unroll
            for (int k = 0; k < MF; ++k) {
                if (decltype(fresh)::value && k < MT * NT) acc[k / NT][k % NT] = Acc{};
                mfma_one(f, k);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (MF >= 2 * R) {
                    if (k % 2 == 0 && k / 2 < R) read_one(nx, buf, ks, k / 2);
                } else {
                    if (2 * k < R) read_one(nx, buf, ks, 2 * k);
                    if (2 * k + 1 < R) read_one(nx, buf, ks, 2 * k + 1);
                }
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    if (i >= d0 + k * (d1 - d0) / MF && i < d0 + (k + 1) * (d1 - d0) / MF) stage(i, t, to);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto clamp = [&](int t) { return t < nk ? t : nk - 1; };     // (past the end the last K-step goes into the idle image again)
        Frags fa, fb;
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
        for (int q = 0; q < R; ++q) read_one(fa, lds, 0, q);
        // the first slab is multiplied onto a constant zero, before the loop: clearing the accumulators first is 16 instructions a block
        // that run once, and code that runs once comes in at the pace of instruction misses
        int cur = 0, prev = (S - 1) * kStage;                        // images of K-steps t and t + S - 1
        auto keep = [&](Frags& f, int ks, int t) {                   // zeros for the chunks past K
            if (last == 8 || t + 1 < nk) return;
            const bool in = 2 * ks + fh < last;
#pragma unroll
            for (int q = 0; q < PL * MT; ++q) f.a[q] = in ? f.a[q] : V{};
#pragma unroll
            for (int q = 0; q < NT; ++q) f.b[q] = in ? f.b[q] : V{};
        };
        keep(fa, 0, 0);
        slab_staging(std::true_type{}, fa, fb, lds, 1, clamp(S - 1), lds + prev, D0, NI);
        int t = 0;
        for (; t + 1 < nk; ++t) {
            slab(fb, fa, lds + cur, 2);
            slab(fa, fb, lds + cur, 3);
            // K-step t + 1 has landed (S - 2 younger ones may be in flight), for everyone behind the barrier; all reads of K-step t are complete
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((S - 2) * NI) : "memory");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            prev = cur;
            cur = cur + kStage == S * kStage ? 0 : cur + kStage;
            slab_staging(std::false_type{}, fb, fa, lds + cur, 0, clamp(t + S), lds + prev, 0, D0);
            keep(fa, 0, t + 1);
            slab_staging(std::false_type{}, fa, fb, lds + cur, 1, clamp(t + S), lds + prev, D0, NI);
        }
        keep(fb, 1, t);
        slab(fb, fa, lds + cur, 2);
        keep(fa, 2, t);
        slab(fa, fb, lds + cur, 3);
        keep(fb, 3, t);
#pragma unroll
        for (int q = 0; q < MF; ++q) mfma_one(fb, q);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // (clamped re-loads of the last K-step)
    }
};

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
