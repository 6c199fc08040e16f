// Dev builds only (-DPC_DEV_SWEEPS; included by pc_gemm_dense.hip): the many-row projections with the residual activation plane on the
// int8 MFMA (pc_gemm_dense_lo8, tools/dense_lo8_ab.py), eight waves and one barrier per K-step.  Needs K % 64 == 0.
#pragma once

namespace lockstep {
constexpr int BM = 128;
constexpr int kXT = BM * BK * 2;                 // bytes of one activation plane tile (16 KiB)

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));

template <int WM, int EPI>
__global__ __launch_bounds__(512) void lockstep_kernel(const DenseParams p) {
    constexpr int WN = 8 / WM, MT = BM / (32 * WM), NT = 2, BN = 64 * WN;
    constexpr int kWT = BN * BK * 2;             // bytes of the weight tile
    // stage image: Xhi | Xlo8 (64-byte rows) | W | W8 (64-byte rows)
    constexpr int oW = kXT + kXT / 2;
    constexpr int oW8 = oW + kWT;
    constexpr int kStage = oW8 + kWT / 2;
    constexpr int NXI = 2, NWI = BN / 64;        // staging instructions per wave: 2 for the activations, BN/64 for W
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
    const int nkt = p.K / BK;                            // K-steps of the whole product
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
#pragma unroll
    for (int j = 0; j < NXI; ++j) {
        const int r = wave * 16 + j * 8 + srow;
        const int gm = (m0 + r < p.M) ? m0 + r : p.M - 1;
        gx[j] = p.xh + (int64_t)gm * p.ldx + (scp ^ ((r >> 1) & 7)) * 8;
    }
#pragma unroll
    for (int j = 0; j < NWI; ++j) {
        const int r = wave * (BN / 8) + j * 8 + srow;
        int gr = wrow(r);
        gr = gr < 0 ? 0 : gr;
        gw[j] = p.w + (int64_t)gr * p.ldw + (scp ^ ((r >> 1) & 7)) * 8;
    }
    // Codes: one instruction of 16 rows x 64 B per wave for the activation codes, NW8 for the weight codes; lane -> (row, chunk
    // POSITION); position c of row r holds source chunk c ^ ((r >> 2) & 3): the 16 lanes of every ds_read_b128 group then fall
    // into 16 distinct 16-byte bank slots (64-byte rows: slot = 4 (r & 3) + position)
    const signed char* gx8;
    const signed char* gw8[NW8];
    {
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
    auto stage = [&](int tl, char* buf) {
        const int64_t ko = (int64_t)(t0 + tl) * BK;
#pragma unroll
        for (int j = 0; j < NXI; ++j) glds16(gx[j] + ko, buf + (wave * 16 + j * 8) * 128);
#pragma unroll
        for (int j = 0; j < NWI; ++j) glds16(gw[j] + ko, buf + oW + (wave * (BN / 8) + j * 8) * 128);
        glds16((const _Float16*)(gx8 + ko), buf + kXT + wave * 1024);
#pragma unroll
        for (int j = 0; j < NW8; ++j) glds16((const _Float16*)(gw8[j] + ko), buf + oW8 + (wave * (BN / 8) + j * 16) * 64);
    };

    // ---- fragment addressing: lane = (row fr of the 32-row subtile, k-half fh) ----
    const int fr = lane & 31, fh = lane >> 5;
    int foff[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) foff[ks] = fr * 128 + (((2 * ks + fh) ^ ((fr >> 1) & 7)) << 4);
    const int a_base = (wm * 32 * MT) * 128;              // + 32*i rows
    const int b_base = oW + (wn * 64) * 128;              // + 32*j rows
    // A lane's 16 codes of a 32-deep block kb are chunk 2 kb + fh of its row (A and B pair slot by slot, so which sixteen k
    // of the block a lane holds is free as long as both sides agree)
    int foff8[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) foff8[kb] = fr * 64 + (((2 * kb + fh) ^ ((fr >> 2) & 3)) << 4);
    const int a8_base = kXT + (wm * 32 * MT) * 64, b8_base = oW8 + (wn * 64) * 64;
    i16v iacc[MT][NT];
    f16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) { acc[i][j][r] = 0.f; iacc[i][j][r] = 0; }

    // ---- main loop: one barrier per K-step, fragment reads one 16-deep slab ahead of the MFMAs ----
    // Two fragment register sets alternate over the 4 slabs of a K-step.  The reads of slab s+1 are issued in front of
    // the MFMAs of slab s, so their LDS latency passes under 4*MT MFMAs of 32 cycles each; the last slab of K-step t is
    // multiplied AFTER the barrier, next to the first reads of K-step t+1 and the LDS-DMA issue of K-step t+2, so the
    // matrix pipe has work while the workgroup re-synchronises.
    struct Frags { h8 ah[MT], bw[NT]; };
    auto load_frags = [&](Frags& f, const char* buf, int ks) {
#pragma unroll
        for (int i = 0; i < MT; ++i) f.ah[i] = *(const h8*)(buf + a_base + i * 32 * 128 + foff[ks]);
#pragma unroll
        for (int j = 0; j < NT; ++j) f.bw[j] = *(const h8*)(buf + b_base + j * 32 * 128 + foff[ks]);
    };
    auto mfmas = [&](const Frags& f) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.ah[i], f.bw[j], acc[i][j], 0, 0, 0);
    };
    // Pin the issue order of one (reads of the next slab, MFMAs of this slab) pair: one MFMA, then two reads, until the reads run out.
    // Left alone, hipcc sinks the ds_reads next to their first use and waits lgkmcnt(0) right behind them (seen in the ISA: four
    // exposed LDS round trips per K-step).
    {
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
            // (the DMA issue spread between this slab's MFMAs measured slower: 4177 vs 4136 us per layer at 6000 rows,
            // profiles/r05_variants.txt)
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
    if constexpr (EPI == EPI_GELU) {                   // (no caller: the Falcon / MPT stacks keep the fp16 residual plane)
        pc_set_error("pc_gemm_dense_lo8: no GELU instantiation");
        return PC_ERR_ARG;
    } else {
        hipLaunchKernelGGL((lockstep_kernel<WM, EPI>), grid, block, 0, s, p);
    }
    return pc_check_launch("lockstep_kernel");
}
}  // namespace lockstep
