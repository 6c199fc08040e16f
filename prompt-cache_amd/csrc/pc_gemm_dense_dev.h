// Dev builds only (-DPC_DEV_SWEEPS; included by pc_gemm_dense.hip): the eight-wave form of the many-row projections with its two measured
// negative results -- the ping-pong main loop (PC_DENSE_PP=1, tools/dense_pp_ab.py) and the residual activation plane on the int8 MFMA
// (pc_gemm_dense_lo8, tools/dense_lo8_ab.py).
#pragma once

namespace lockstep {
constexpr int BM = 128;
constexpr int kXT = BM * BK * 2;                 // bytes of one activation plane tile (16 KiB)

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));

template <int WM, int EPI, bool TWO, bool PP, bool LO8 = false>
__global__ __launch_bounds__(512) void lockstep_kernel(const DenseParams p) {
    static_assert(!(LO8 && (TWO || PP)), "LO8 replaces the fp16 lo plane; lockstep main loop only");
    constexpr int WN = 8 / WM, MT = BM / (32 * WM), NT = 2, BN = 64 * WN;
    constexpr int kWT = BN * BK * 2;             // bytes of the weight tile
    // stage image: Xhi | Xlo | W   (LO8: Xhi | Xlo8 (64-byte rows) | W | W8 (64-byte rows))
    constexpr int oW = LO8 ? kXT + kXT / 2 : 2 * kXT;
    constexpr int oW8 = oW + kWT;
    constexpr int kStage = LO8 ? oW8 + kWT / 2 : 2 * kXT + kWT;
    constexpr int NXI = 2, NWI = BN / 64;        // staging instructions per wave: 2 per activation plane, BN/64 for W
    constexpr int NW8 = BN / 128;                // ... and for the int8 weight tile (16 rows x 64 B per instruction); Xlo8: one
    __shared__ __attribute__((aligned(16))) char lds[2 * kStage];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave - wm * WN;
    // block -> (M-block, weight panel), XCD-aware
    const int b = blockIdx.x, xcd = b & 7, slot = b >> 3;
    const int nloc = slot / p.mb, mi = slot - nloc * p.mb, ni = nloc * 8 + xcd;
    if (ni >= p.nb) return;
    const int m0 = mi * BM;
    const int K = p.K, nkt = (K + BK - 1) / BK;          // K-steps of the whole product
    const int t0 = blockIdx.y * p.kper;                  // this slice's first K-step (kper = nkt without split-K)
    const int nk = (p.kper < nkt - t0) ? p.kper : nkt - t0;

    // global weight row of LDS weight-tile row r; -1 = past the end (clamped source, never stored)
    auto wrow = [&](int r) -> int {
        if (EPI == EPI_SILU) {
            const int f = (ni * WN + (r >> 6)) * 32 + (r & 31);
            return f < p.nfeat ? ((r >> 5) & 1) * p.nfeat + f : -1;
        }
        if (EPI == EPI_ROPE) {
            // a wave tile (64 columns) = 32 features d of one head's first half next to their rotary partners d + 64, so
            // x[d] and x[d + 64] meet in the same lane and accumulator index of the two 32-wide MFMA blocks
            const int wt = r >> 6, c = r & 63;
            const int hd = ni * (BN / 128) + (wt >> 1);
            const int d = (c < 32) ? (wt & 1) * 32 + c : 64 + (wt & 1) * 32 + (c - 32);
            const int n = hd * 128 + d;
            return n < p.N ? n : -1;
        }
        const int n = ni * BN + r;
        return n < p.N ? n : -1;
    };

    // ---- staging sources: per lane one 16-byte chunk of one row per instruction ----
    const int srow = lane >> 3, scp = lane & 7;          // row inside the 8-row group, chunk POSITION in the LDS row
    const _Float16* gx[NXI];
    const _Float16* gw[NWI];
    int cx[NXI], cw[NWI];                                // source chunk index (for the K tail)
    const int64_t lo_delta = TWO ? (p.xl - p.xh) : 0;
#pragma unroll
    for (int j = 0; j < NXI; ++j) {
        const int r = wave * 16 + j * 8 + srow;
        const int gm = (m0 + r < p.M) ? m0 + r : p.M - 1;
        cx[j] = scp ^ ((r >> 1) & 7);
        gx[j] = p.xh + (int64_t)gm * p.ldx + cx[j] * 8;
    }
#pragma unroll
    for (int j = 0; j < NWI; ++j) {
        const int r = wave * (BN / 8) + j * 8 + srow;
        int gr = wrow(r);
        gr = gr < 0 ? 0 : gr;
        cw[j] = scp ^ ((r >> 1) & 7);
        gw[j] = p.w + (int64_t)gr * p.ldw + cw[j] * 8;
    }
    // LO8: one instruction of 16 rows x 64 B per wave for the activation codes, NW8 for the weight codes; lane -> (row, chunk
    // POSITION); position c of row r holds source chunk c ^ ((r >> 2) & 3): the 16 lanes of every ds_read_b128 group then fall
    // into 16 distinct 16-byte bank slots (64-byte rows: slot = 4 (r & 3) + position)
    [[maybe_unused]] const signed char* gx8 = nullptr;
    [[maybe_unused]] const signed char* gw8[NW8 > 0 ? NW8 : 1];
    if constexpr (LO8) {
        const int r = wave * 16 + (lane >> 2);
        const int gm = (m0 + r < p.M) ? m0 + r : p.M - 1;
        gx8 = p.xl8 + (int64_t)gm * p.ldx8 + (((lane & 3) ^ ((r >> 2) & 3)) << 4);
#pragma unroll
        for (int j = 0; j < NW8; ++j) {
            const int rw = wave * (BN / 8) + j * 16 + (lane >> 2);
            int gr = wrow(rw);
            gr = gr < 0 ? 0 : gr;
            gw8[j] = p.w8 + (int64_t)gr * p.ldw8 + (((lane & 3) ^ ((rw >> 2) & 3)) << 4);
        }
    }
    const bool ktail = (K % BK) != 0;
    auto stage = [&](int tl, char* buf) {
        const int t = t0 + tl;
        const bool tail = ktail && t == nkt - 1;
        const int64_t ko = (int64_t)t * BK;
        const int kchunks = tail ? (K - t * BK) / 8 : 8;          // valid 16-byte chunks in this K-step
#pragma unroll
        for (int j = 0; j < NXI; ++j) {
            const bool ok = !tail || cx[j] < kchunks;
            const _Float16* sh = ok ? gx[j] + ko : p.zeros;
            glds16(sh, buf + (wave * 16 + j * 8) * 128);
            if (TWO) glds16(ok ? gx[j] + lo_delta + ko : p.zeros, buf + kXT + (wave * 16 + j * 8) * 128);
        }
#pragma unroll
        for (int j = 0; j < NWI; ++j) {
            // chunks past K pair with zero activations: any finite weight bytes do (the row's first chunk)
            const _Float16* sw = (!tail || cw[j] < kchunks) ? gw[j] + ko : gw[j] - cw[j] * 8;
            glds16(sw, buf + oW + (wave * (BN / 8) + j * 8) * 128);
        }
        if constexpr (LO8) {                           // (K % 64 == 0 with LO8: no tail)
            glds16((const _Float16*)(gx8 + ko), buf + kXT + wave * 1024);
#pragma unroll
            for (int j = 0; j < NW8; ++j) glds16((const _Float16*)(gw8[j] + ko), buf + oW8 + (wave * (BN / 8) + j * 16) * 64);
        }
    };

    // ---- fragment addressing: lane = (row fr of the 32-row subtile, k-half fh) ----
    const int fr = lane & 31, fh = lane >> 5;
    int foff[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) foff[ks] = fr * 128 + (((2 * ks + fh) ^ ((fr >> 1) & 7)) << 4);
    const int a_base = (wm * 32 * MT) * 128;              // + 32*i rows, + kXT for the lo plane
    const int b_base = oW + (wn * 64) * 128;              // + 32*j rows
    // LO8: a lane's 16 codes of a 32-deep block kb are chunk 2 kb + fh of its row (A and B pair slot by slot, so which sixteen k
    // of the block a lane holds is free as long as both sides agree)
    [[maybe_unused]] int foff8[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) foff8[kb] = fr * 64 + (((2 * kb + fh) ^ ((fr >> 2) & 3)) << 4);
    [[maybe_unused]] const int a8_base = kXT + (wm * 32 * MT) * 64, b8_base = oW8 + (wn * 64) * 64;
    [[maybe_unused]] i16v iacc[LO8 ? MT : 1][LO8 ? NT : 1];
    if constexpr (LO8) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) iacc[i][j][r] = 0;
    }

    f16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // ---- main loop: one barrier per K-step, fragment reads one 16-deep slab ahead of the MFMAs ----
    // Two fragment register sets alternate over the 4 slabs of a K-step.  The reads of slab s+1 are issued in front of
    // the MFMAs of slab s, so their LDS latency passes under 4*MT MFMAs of 32 cycles each; the last slab of K-step t is
    // multiplied AFTER the barrier, next to the first reads of K-step t+1 and the LDS-DMA issue of K-step t+2, so the
    // matrix pipe has work while the workgroup re-synchronises.
    struct Frags { h8 ah[MT], al[TWO ? MT : 1], bw[NT]; };
    auto load_frags = [&](Frags& f, const char* buf, int ks) {
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            f.ah[i] = *(const h8*)(buf + a_base + i * 32 * 128 + foff[ks]);
            if (TWO) f.al[i] = *(const h8*)(buf + kXT + a_base + i * 32 * 128 + foff[ks]);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) f.bw[j] = *(const h8*)(buf + b_base + j * 32 * 128 + foff[ks]);
    };
    auto mfmas = [&](const Frags& f) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bw[j], acc[i][j], 0, 0, 0);
        if (TWO) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.bw[j], acc[i][j], 0, 0, 0);
        }
    };
    // Pin the issue order of one (reads of the next slab, MFMAs of this slab) pair: a read in front of every MFMA until
    // the reads run out.  Left alone, hipcc sinks the ds_reads next to their first use and waits lgkmcnt(0) right
    // behind them (seen in the ISA: four exposed LDS round trips per K-step).
    auto interleave = [&]() {
        // one MFMA, then two reads, until the reads run out: every read of the next slab is in flight at least three
        // MFMAs (~100 cycles) before the wait in front of that slab's first MFMA
        constexpr int R = MT * (TWO ? 2 : 1) + NT, MF = MT * NT * (TWO ? 2 : 1);
#pragma unroll
        for (int k = 0; k < MF; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                          // one MFMA
            if (2 * k + 1 < R) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);       // two DS reads
            else if (2 * k < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // (an odd one left)
        }
    };
    // The slab multiplied right behind the K-step barrier also carries the LDS-DMA issue of K-step t + 2 (its buffer was just
    // freed).  Rounds 2-4 issued the 8 (LO8: 11) DMA instructions in one burst in front of that slab's MFMAs: both waves of a SIMD
    // spend ~60-100 issue cycles per instruction there while the matrix pipe, drained by the barrier, has nothing to do (seen in
    // the ISA: barrier, 8 x global_load_lds, then the first MFMA).  Round 5 spreads them BETWEEN that slab's MFMAs: one MFMA, two
    // fragment reads (until they run out), the slab's share of the DMA instructions, next MFMA -- for launches with two fp16 planes
    // (-0.6 ... -2.6 % per layer at 800 ... 6000 rows); one-plane and int8-residual launches measured 1-5 % SLOWER that way and keep
    // the burst (profiles/r05_variants.txt).  -DPC_DENSE_SPREAD_DMA=0: the burst everywhere.
#ifndef PC_DENSE_SPREAD_DMA
#define PC_DENSE_SPREAD_DMA 1
#endif
    // one MFMA / one fragment read / a range of the DMA instructions of a K-step, by index (compile-time after unrolling)
    auto mfma_one = [&](const Frags& f, int idx) {
        const int pl = idx / (MT * NT), i = (idx / NT) % MT, j = idx % NT;
        if (TWO && pl == 1) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.bw[j], acc[i][j], 0, 0, 0);
        else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bw[j], acc[i][j], 0, 0, 0);
    };
    auto read_one = [&](Frags& f, const char* buf, int ks, int idx) {
        constexpr int NA = MT * (TWO ? 2 : 1);
        if (idx < NA) {
            const int i = TWO ? idx >> 1 : idx;
            if (TWO && (idx & 1)) f.al[i] = *(const h8*)(buf + kXT + a_base + i * 32 * 128 + foff[ks]);
            else f.ah[i] = *(const h8*)(buf + a_base + i * 32 * 128 + foff[ks]);
        } else {
            const int j = idx - NA;
            f.bw[j] = *(const h8*)(buf + b_base + j * 32 * 128 + foff[ks]);
        }
    };
    auto stage_range = [&](int tl, char* buf, int q0, int q1) {
        const int t = t0 + tl;
        const bool tail = ktail && t == nkt - 1;
        const int64_t ko = (int64_t)t * BK;
        const int kchunks = tail ? (K - t * BK) / 8 : 8;
        int q = 0;
#pragma unroll
        for (int j = 0; j < NXI; ++j) {
            const bool ok = !tail || cx[j] < kchunks;
            if (q >= q0 && q < q1) glds16(ok ? gx[j] + ko : p.zeros, buf + (wave * 16 + j * 8) * 128);
            ++q;
            if (TWO) {
                if (q >= q0 && q < q1) glds16(ok ? gx[j] + lo_delta + ko : p.zeros, buf + kXT + (wave * 16 + j * 8) * 128);
                ++q;
            }
        }
#pragma unroll
        for (int j = 0; j < NWI; ++j) {
            if (q >= q0 && q < q1)
                glds16((!tail || cw[j] < kchunks) ? gw[j] + ko : gw[j] - cw[j] * 8, buf + oW + (wave * (BN / 8) + j * 8) * 128);
            ++q;
        }
        if constexpr (LO8) {
            if (q >= q0 && q < q1) glds16((const _Float16*)(gx8 + ko), buf + kXT + wave * 1024);
            ++q;
#pragma unroll
            for (int j = 0; j < NW8; ++j) {
                if (q >= q0 && q < q1) glds16((const _Float16*)(gw8[j] + ko), buf + oW8 + (wave * (BN / 8) + j * 16) * 64);
                ++q;
            }
        }
    };
    if constexpr (PP) {
        // ---- ping-pong main loop (round 5; the guide's two-waves-per-SIMD regime).  MEASURED SLOWER than the lockstep loop below
        // on this kernel (0.87-0.90 x with both planes, profiles/r05_dense_pp_ab.txt) in all three forms tried -- fragment reads
        // waited for inside their load segment; read one phase ahead with hipcc's waits (lgkmcnt(0) every other phase: its
        // scoreboard merges conservatively at the group branches); read ahead as raw ds_read_b128 with explicit counted waits
        // (this form) -- kept for A/B behind -DPC_DEV_SWEEPS.  Eight barriers per K-step and one wave per SIMD feeding the
        // matrix pipe at a time lose to two waves per SIMD interleaving their MFMAs with one barrier per K-step; what is left
        // between the lockstep loop (1.09-1.15 PFLOP/s executed on random data) and the ~1.3 the guide's 8-phase template
        // reaches at 4096^3 is not in the wave pairing. ----
        // The loop above keeps the two waves of a SIMD in lockstep: both issue MFMAs at once (54 % of wave time were issue stalls
        // behind the shared pipe, profiles/r02_pmc_gemm_dense.txt) and both sit out the barrier and the first fragment reads of
        // the next K-step together (MFMA pipes busy 63 % of the kernel's cycles).  Here the workgroup's eight waves are two GROUPS
        // of four (one wave of each group per SIMD) that run the same program ONE BARRIER APART: a K-step is four phases (one
        // 16-deep slab each), a phase is a LOAD segment (the slab's 6 fragment reads, waited for) and a COMPUTE segment (its 8
        // MFMAs = 256 matrix-pipe cycles), every segment ends in a raw s_barrier -- so while group 0 is in its compute segment
        // group 1 is in its load segment and vice versa: the SIMD's matrix pipe always has exactly one wave feeding it, and the
        // LDS reads, the waits and the barrier latency of one wave pass under the MFMAs of the other.  One fragment register
        // set instead of two.
        //   barrier n separates interval n from n + 1.  Group 0: load (t, s) in interval 8t + 2s, compute in 8t + 2s + 1; group 1
        //   one interval later.  A load segment only ISSUES the fragment reads of the NEXT slab (two register sets); they are
        //   consumed one phase later, so the segment is a few dozen issue cycles and the LDS latency never sits in front of a
        //   barrier (first version: reads waited for inside their load segment -- the load segment then took longer than the
        //   partner's 256-cycle compute segment and the loop ran at ITS pace: 0.81-0.93 x the lockstep loop).
        //   Slab 0 of K-step t + 1 is read in load (t, 3): group 0 in interval 8t + 6, so K-step t + 1 must have landed, for all
        //   waves, by barrier 8t + 6: the LDS-DMA goes out in two pieces between MFMAs -- group 0 in compute (t, 0), (t, 1), waited
        //   for at the end of compute (t, 2); group 1 in load (t, 0) and compute (t, 0), waited for at the end of load (t, 2) -- at
        //   least two intervals of flight for the last piece.  The buffer it lands in held K-step t - 1, whose last reads (group
        //   1, issued in its load (t - 1, 2)) are complete at the start of interval 8t: every issue point above lies behind
        //   barrier 8t + 1.
        // Same MFMA order per accumulator as the loop above: bit-identical results.
        constexpr int NI = NXI * (TWO ? 2 : 1) + NWI;          // LDS-DMA instructions per wave and K-step
        auto stage_piece = [&](int tl, char* buf, int piece) {
            const int t = t0 + tl;
            const bool tail = ktail && t == nkt - 1;
            const int64_t ko = (int64_t)t * BK;
            const int kchunks = tail ? (K - t * BK) / 8 : 8;
            const int q0 = piece * NI / 2, q1 = (piece + 1) * NI / 2;
            int q = 0;
#pragma unroll
            for (int j = 0; j < NXI; ++j) {
                const bool ok = !tail || cx[j] < kchunks;
                if (q >= q0 && q < q1) glds16(ok ? gx[j] + ko : p.zeros, buf + (wave * 16 + j * 8) * 128);
                ++q;
                if (TWO) {
                    if (q >= q0 && q < q1) glds16(ok ? gx[j] + lo_delta + ko : p.zeros, buf + kXT + (wave * 16 + j * 8) * 128);
                    ++q;
                }
            }
#pragma unroll
            for (int j = 0; j < NWI; ++j) {
                if (q >= q0 && q < q1)
                    glds16((!tail || cw[j] < kchunks) ? gw[j] + ko : gw[j] - cw[j] * 8, buf + 2 * kXT + (wave * (BN / 8) + j * 8) * 128);
                ++q;
            }
        };
        const int grp = __builtin_amdgcn_readfirstlane(wave >> 2);
        Frags fr2[2];                                           // slab s lives in set s & 1: read one phase ahead of its MFMAs
        // The fragment reads of the ping-pong loop are raw ds_read_b128 statements hipcc does not count: a read issued in load
        // segment s is consumed in compute segment s + 1 behind an explicit `s_waitcnt lgkmcnt(R)` (R = reads per slab: only
        // the NEWER slab's reads may still be in flight).  Left to hipcc, the uniform `if (group)` branches between a read and
        // its use make the waitcnt pass merge its scoreboards conservatively: lgkmcnt(0) in every other phase, i.e. the LDS
        // latency of the just-issued reads in front of the MFMAs -- what the read-ahead is there to hide.  The loop holds no
        // other LDS or scalar-memory instruction (checked in the ISA: lgkmcnt counts in order only without SMEM in flight).
        constexpr int NR = MT * (TWO ? 2 : 1) + NT;
        const uint32_t lds32 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
        auto load_frags_raw = [&](Frags& f, uint32_t buf_off, int ks) {
            const uint32_t aa = lds32 + buf_off + a_base + foff[ks], ab = lds32 + buf_off + b_base + foff[ks];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.ah[i]) : "v"(aa), "i"(i * 32 * 128));
                if (TWO) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.al[i]) : "v"(aa), "i"(kXT + i * 32 * 128));
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.bw[j]) : "v"(ab), "i"(j * 32 * 128));
        };
        stage(0, lds);
        stage(nk > 1 ? 1 : 0, lds + kStage);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // both K-steps (the prologue is not where the time goes)
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        load_frags_raw(fr2[0], 0, 0);
        if (grp) {                                              // group 1 runs one interval behind
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        auto half_a = [&](const Frags& f) {                     // first half of a slab's MFMAs (hi plane; without a lo plane: the first row block)
#pragma unroll
            for (int i = 0; i < (TWO ? MT : (MT + 1) / 2); ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bw[j], acc[i][j], 0, 0, 0);
        };
        auto half_b = [&](const Frags& f) {
            if (TWO) {
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.al[i], f.bw[j], acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int i = (MT + 1) / 2; i < MT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bw[j], acc[i][j], 0, 0, 0);
            }
        };
        for (int t = 0; t < nk; ++t) {
            char* cur = lds + (t & 1) * kStage;
            char* nxt = lds + ((t + 1) & 1) * kStage;
            const int u1 = t + 1 < nk ? t + 1 : nk - 1;         // (clamped: past the end the last K-step goes into the idle buffer again)
#pragma unroll
            for (int sl = 0; sl < 4; ++sl) {
                // ---- load segment: only ISSUES the next slab's fragment reads (slab 0 of K-step t + 1 behind slab 3: its DMA was
                // waited for two barriers ago); they complete under the partner group's MFMAs and this group's own ----
                if (sl < 3) load_frags_raw(fr2[(sl + 1) & 1], (t & 1) * kStage, sl + 1);
                else load_frags_raw(fr2[0], ((t + 1) & 1) * kStage, 0);     // (past the last K-step: the clamped re-load of it, never multiplied)
                if (grp) {
                    if (sl == 0) stage_piece(u1, nxt, 0);
                    if (sl == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                // ---- compute segment: the slab read one phase ago; the newer slab's NR reads stay in flight ----
                static_assert(NR == 6 || NR == 4 || NR == 3, "reads per slab");
                if constexpr (NR == 6) asm volatile("s_waitcnt lgkmcnt(6)" ::: "memory");
                else if constexpr (NR == 4) asm volatile("s_waitcnt lgkmcnt(4)" ::: "memory");
                else asm volatile("s_waitcnt lgkmcnt(3)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_setprio(1);
                half_a(fr2[sl & 1]);
                __builtin_amdgcn_sched_barrier(0);
                if (!grp) {
                    if (sl < 2) stage_piece(u1, nxt, sl);
                } else {
                    if (sl == 0) stage_piece(u1, nxt, 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                half_b(fr2[sl & 1]);
                __builtin_amdgcn_s_setprio(0);
                if (sl == 2 && !grp) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the read-ahead behind the last slab: landed before its registers die)
        if (!grp) {                                             // group 0 waits for group 1's last compute segment
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if constexpr (LO8) {
        // ---- lockstep main loop with the lo plane on the int8 MFMA (round 5) ----
        // Per K-step: 16 fp16 MFMAs for the hi plane (as without a lo plane) + 8 v_mfma_i32_32x32x32_i8 for the residual plane
        // (two 32-deep blocks x MT x NT) instead of 16 more fp16 ones: 24 matrix-pipe slots instead of 32.  One int8 fragment set:
        // block kb is read one slab ahead of its MFMAs like the fp16 fragments (kb 0 next to slab 0, kb 1 next to slab 2).
        struct F8 { i4v a[MT], b[NT]; };
        F8 f8;
        auto load8 = [&](const char* buf, int kb) {
#pragma unroll
            for (int i = 0; i < MT; ++i) f8.a[i] = *(const i4v*)(buf + a8_base + i * 32 * 64 + foff8[kb]);
#pragma unroll
            for (int j = 0; j < NT; ++j) f8.b[j] = *(const i4v*)(buf + b8_base + j * 32 * 64 + foff8[kb]);
        };
        auto imfmas = [&]() {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) iacc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f8.a[i], f8.b[j], iacc[i][j], 0, 0, 0);
        };
        // (reads of the next slab, MFMAs of this one): one MFMA, then two reads, until the reads run out
        auto pin = [&](auto r_, auto mf_) {
            constexpr int R = decltype(r_)::value, MF = decltype(mf_)::value;
#pragma unroll
            for (int k = 0; k < MF; ++k) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if (2 * k + 1 < R) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                else if (2 * k < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        };
        using RH = std::integral_constant<int, MT + NT>;             // reads of one fp16 slab
        using RB = std::integral_constant<int, 2 * (MT + NT)>;       // ... plus one int8 block
        using MH = std::integral_constant<int, MT * NT>;             // MFMAs of one fp16 slab
        using MB = std::integral_constant<int, 2 * MT * NT>;         // ... plus one int8 block
        Frags fa, fb;
        stage(0, lds);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (nk > 1) stage(1, lds + kStage);
        load_frags(fa, lds, 0);
        load8(lds, 0);
        for (int t = 0; t + 1 < nk; ++t) {
            const char* cur = lds + (t & 1) * kStage;
            load_frags(fb, cur, 1);
            mfmas(fa);
            imfmas();
            pin(RH{}, MB{});
            load_frags(fa, cur, 2);
            load8(cur, 1);
            mfmas(fb);
            pin(RB{}, MH{});
            load_frags(fb, cur, 3);
            mfmas(fa);
            imfmas();
            pin(RH{}, MB{});
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            const int tn = t + 2 < nk ? t + 2 : nk - 1;
            // (the DMA issue spread between this slab's MFMAs -- see the fp16 loop below -- measured SLOWER here: 4177 vs 4136 us per
            // layer at 6000 rows, profiles/r05_variants.txt)
            stage(tn, lds + (t & 1) * kStage);
            load_frags(fa, lds + ((t + 1) & 1) * kStage, 0);
            load8(lds + ((t + 1) & 1) * kStage, 0);
            mfmas(fb);
            pin(RB{}, MH{});
        }
        {
            const char* cur = lds + ((nk - 1) & 1) * kStage;
            load_frags(fb, cur, 1);
            mfmas(fa);
            imfmas();
            pin(RH{}, MB{});
            load_frags(fa, cur, 2);
            load8(cur, 1);
            mfmas(fb);
            pin(RB{}, MH{});
            load_frags(fb, cur, 3);
            mfmas(fa);
            imfmas();
            pin(RH{}, MB{});
            mfmas(fb);
        }
        // the residual product joins the fp32 accumulator: y += int_sum * xl8_scale[row] * w8_scale[col]
        {
            float wsc[NT];
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                int gr = wrow(wn * 64 + 32 * j + fr);
                wsc[j] = p.w8_scale[gr < 0 ? 0 : gr];
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 32 * MT + 32 * i + 8 * (r >> 2) + 4 * fh + (r & 3);
                    const float xs = p.xl8_scale[m < p.M ? m : p.M - 1];
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j][r] = __builtin_fmaf((float)iacc[i][j][r], xs * wsc[j], acc[i][j][r]);
                }
        }
    } else {
    Frags fa, fb;
    stage(0, lds);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (nk > 1) stage(1, lds + kStage);
    load_frags(fa, lds, 0);
    for (int t = 0; t + 1 < nk; ++t) {
        const char* cur = lds + (t & 1) * kStage;
        load_frags(fb, cur, 1);
        mfmas(fa);
        interleave();
        load_frags(fa, cur, 2);
        mfmas(fb);
        interleave();
        load_frags(fb, cur, 3);
        mfmas(fa);
        interleave();
        // K-step t+1 has landed (this wave's LDS-DMA drained, then everyone's via the barrier), and every wave's reads
        // of K-step t are complete (__syncthreads waits lgkmcnt(0)): its buffer may be overwritten.  The stage index
        // is clamped instead of branched on (past the end it re-loads the last K-step into the idle buffer): a branch
        // here splits the block and hipcc then waits for the fresh reads below before the MFMAs that do not need them.
        __builtin_amdgcn_sched_barrier(0);      // slab 2's MFMAs stay in front of the barrier: they cover slab 3's reads
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const int tn = t + 2 < nk ? t + 2 : nk - 1;
        if constexpr (PC_DENSE_SPREAD_DMA && TWO) {
            constexpr int MF = MT * NT * (TWO ? 2 : 1), R = MT * (TWO ? 2 : 1) + NT, V = NXI * (TWO ? 2 : 1) + NWI;
            const char* nb = lds + ((t + 1) & 1) * kStage;
#pragma unroll
            for (int k = 0; k < MF; ++k) {
                mfma_one(fb, k);
                __builtin_amdgcn_sched_barrier(0);
                if (2 * k < R) read_one(fa, nb, 0, 2 * k);
                if (2 * k + 1 < R) read_one(fa, nb, 0, 2 * k + 1);
                stage_range(tn, lds + (t & 1) * kStage, k * V / MF, (k + 1) * V / MF);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            stage(tn, lds + (t & 1) * kStage);
            load_frags(fa, lds + ((t + 1) & 1) * kStage, 0);
            mfmas(fb);
            interleave();
        }
    }
    {
        const char* cur = lds + ((nk - 1) & 1) * kStage;
        load_frags(fb, cur, 1);
        mfmas(fa);
        interleave();
        load_frags(fa, cur, 2);
        mfmas(fb);
        interleave();
        load_frags(fb, cur, 3);
        mfmas(fa);
        interleave();
        mfmas(fb);
    }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // (the clamped re-load of the last K-step)

    // ---- epilogue: accumulators -> wave-private LDS tile [32*MT][64] fp32 -> full-row global stores ----
    __syncthreads();                                       // every wave is done with the staging buffers
    float* st = (float*)(lds + wave * (32 * MT * 64 * 4));
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                st[(32 * i + 8 * (r >> 2) + 4 * fh + (r & 3)) * 64 + 32 * j + fr] = acc[i][j][r];
    const int mrow0 = m0 + wm * 32 * MT;
    if (EPI == EPI_SILU) {
        // the wave's 64 columns are [32 gate features | the same 32 up features]: 8 lanes per row, 4 features per lane
        const int fbase = (ni * WN + wn) * 32 + (lane & 7) * 4;
#pragma unroll
        for (int it = 0; it < 4 * MT; ++it) {
            const int row = it * 8 + (lane >> 3), m = mrow0 + row;
            f4 g = *(const f4*)(st + row * 64 + (lane & 7) * 4);
            f4 u = *(const f4*)(st + row * 64 + 32 + (lane & 7) * 4);
            if (m < p.M && fbase < p.nfeat) {
                if (p.wscale) {
                    const f4 sg = *(const f4*)(p.wscale + fbase), su = *(const f4*)(p.wscale + p.nfeat + fbase);
                    g[0] *= sg[0]; g[1] *= sg[1]; g[2] *= sg[2]; g[3] *= sg[3];
                    u[0] *= su[0]; u[1] *= su[1]; u[2] *= su[2]; u[3] *= su[3];
                }
                if (p.xscale) {
                    const float xs = p.xscale[m];
                    g[0] *= xs; g[1] *= xs; g[2] *= xs; g[3] *= xs;
                    u[0] *= xs; u[1] *= xs; u[2] *= xs; u[3] *= xs;
                    if (*p.corr_has) {
                        const f4 cg = *(const f4*)(p.corr + (int64_t)m * p.ldc + fbase);
                        const f4 cu = *(const f4*)(p.corr + (int64_t)m * p.ldc + p.nfeat + fbase);
                        g[0] += cg[0]; g[1] += cg[1]; g[2] += cg[2]; g[3] += cg[3];
                        u[0] += cu[0]; u[1] += cu[1]; u[2] += cu[2]; u[3] += cu[3];
                    }
                }
                h4 hi, lo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float s = (g[e] / (1.0f + __expf(-g[e]))) * u[e];      // act_fn(gate) * up, llama2.py:242
                    _Float16 sh, sl;
                    pc_split(s, sh, sl);
                    hi[e] = sh; lo[e] = sl;
                }
                *(h4*)(p.oh + (int64_t)m * p.ldo + fbase) = hi;
                if (p.ol) *(h4*)(p.ol + (int64_t)m * p.ldo + fbase) = lo;
            }
        }
        return;
    }
    if (EPI == EPI_ROPE) {
        // RoPE at the supplied positions (llama2.py:200-213, :357-359) and the KV append (:361-364) on the accumulator tile:
        // 8 lanes per row, a lane holds features d0 .. d0+3 and d0+64 .. d0+67 of head `hd`
        const int hd = ni * (BN / 128) + (wn >> 1);
        const int d0 = (wn & 1) * 32 + (lane & 7) * 4;
        if (hd >= p.H + 2 * p.Hkv) return;
        const bool rot = hd < p.H + p.Hkv;
#pragma unroll
        for (int it = 0; it < 4 * MT; ++it) {
            const int row = it * 8 + (lane >> 3), m = mrow0 + row;
            const f4 x0 = *(const f4*)(st + row * 64 + (lane & 7) * 4);
            const f4 x1 = *(const f4*)(st + row * 64 + 32 + (lane & 7) * 4);
            if (m >= p.M) continue;
            f4 a = x0, c = x1;
            if (rot) {
                const f4 w01 = *(const f4*)(p.cs + (int64_t)m * 64 + d0);          // (cos, sin) of pairs d0, d0+1
                const f4 w23 = *(const f4*)(p.cs + (int64_t)m * 64 + d0 + 2);      // ... d0+2, d0+3
                const float cs_[4] = {w01[0], w01[2], w23[0], w23[2]}, sn_[4] = {w01[1], w01[3], w23[1], w23[3]};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // q*cos + rotate_half(q)*sin (llama2.py:208): the low half pairs with -high, the high half with +low
                    a[e] = x0[e] * cs_[e] - x1[e] * sn_[e];
                    c[e] = x1[e] * cs_[e] + x0[e] * sn_[e];
                }
            }
            h4 ah, al, ch, cl;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                _Float16 t0, t1, t2, t3;
                pc_split(a[e], t0, t1);
                pc_split(c[e], t2, t3);
                ah[e] = t0; al[e] = t1; ch[e] = t2; cl[e] = t3;
            }
            _Float16* dh;
            _Float16* dl = nullptr;
            if (hd < p.H) {
                const int64_t off = (int64_t)m * p.q_ts + hd * 128 + d0;
                dh = p.q_hi + off;
                if (p.q_lo) dl = p.q_lo + off;
            } else {
                const int b = m / p.q_len, t = m - b * p.q_len;
                const int past = p.past_lens ? p.past_lens[b] : p.past_len;
                const bool is_k = hd < p.H + p.Hkv;
                const int kh = is_k ? hd - p.H : hd - p.H - p.Hkv;
                dh = (is_k ? p.k_arena : p.v_arena) + b * p.a_bs + kh * p.a_hs + (int64_t)(past + t) * 128 + d0;
                if (p.k_lo) dl = (is_k ? p.k_lo : p.v_lo) + b * p.lo_bs + kh * p.lo_hs + (int64_t)(past + t - p.lo_row0) * 128 + d0;
            }
            *(h4*)dh = ah;
            *(h4*)(dh + 64) = ch;
            if (dl) { *(h4*)dl = al; *(h4*)(dl + 64) = cl; }
        }
        return;
    }
    const int n = ni * BN + wn * 64 + (lane & 15) * 4;
#pragma unroll
    for (int it = 0; it < 8 * MT; ++it) {
        const int row = it * 4 + (lane >> 4), m = mrow0 + row;
        f4 v = *(const f4*)(st + row * 64 + (lane & 15) * 4);
        if (m < p.M && n < p.N) {
            if (p.wscale) {
                const f4 sv = *(const f4*)(p.wscale + n);
                v[0] *= sv[0]; v[1] *= sv[1]; v[2] *= sv[2]; v[3] *= sv[3];
            }
            if (p.xscale) {
                const float xs = p.xscale[m];
                v[0] *= xs; v[1] *= xs; v[2] *= xs; v[3] *= xs;
                if (*p.corr_has) {
                    const f4 cv = *(const f4*)(p.corr + (int64_t)m * p.ldc + n);
                    v[0] += cv[0]; v[1] += cv[1]; v[2] += cv[2]; v[3] += cv[3];
                }
            }
            if (EPI == EPI_GELU) {
                h4 hi, lo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float s = 0.5f * v[e] * (1.0f + erff(v[e] * 0.70710678118654752f));   // nn.GELU(), falcon.py:726
                    _Float16 sh, sl;
                    pc_split(s, sh, sl);
                    hi[e] = sh; lo[e] = sl;
                }
                *(h4*)(p.oh + (int64_t)m * p.ldo + n) = hi;
                if (p.ol) *(h4*)(p.ol + (int64_t)m * p.ldo + n) = lo;
            } else {
                float* yp = p.y + (int64_t)blockIdx.y * p.slab_stride + (int64_t)m * p.ldy + n;
                if (EPI == EPI_ADD) {
                    const f4 old = *(const f4*)yp;
                    v[0] += old[0]; v[1] += old[1]; v[2] += old[2]; v[3] += old[3];
                }
                *(f4*)yp = v;
            }
        }
    }
}

template <int WM, int EPI>
int launch(DenseParams& p, hipStream_t s, int kslices) {
    constexpr int BN = 64 * (8 / WM);
    p.mb = pc_ceil_div(p.M, BM);
    p.nb = (EPI == EPI_SILU) ? pc_ceil_div(p.nfeat, BN / 2) : pc_ceil_div(p.N, BN);
    const int nkt = pc_ceil_div(p.K, BK);
    p.kper = pc_ceil_div(nkt, kslices);
    const dim3 grid(8 * p.mb * pc_ceil_div(p.nb, 8), pc_ceil_div(nkt, p.kper)), block(512);
    if (p.xl8) {
        if constexpr (EPI == EPI_GELU) {               // (no caller: the Falcon / MPT stacks keep the fp16 residual plane)
            pc_set_error("pc_gemm_dense_lo8: no GELU instantiation");
            return PC_ERR_ARG;
        } else {
            hipLaunchKernelGGL((lockstep_kernel<WM, EPI, false, false, true>), grid, block, 0, s, p);
        }
    } else if (p.xl) hipLaunchKernelGGL((lockstep_kernel<WM, EPI, true, true>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((lockstep_kernel<WM, EPI, false, true>), grid, block, 0, s, p);
    return pc_check_launch("lockstep_kernel");
}
}  // namespace lockstep
