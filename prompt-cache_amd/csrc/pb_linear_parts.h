// Products of a few rows with runs of k side by side (pb_linear.hip, pb_linear_pair.hip).
#pragma once
#include "pb_linear_epi.h"

namespace pcb {

// A k-step's products into a pair of sums, odd parts into the second (fp32: shorter chains of roundings -- against 64 bits 0.7 of one chain's
// error at every size -- and of dependent MFMAs; bf16 has one part); chain: into one, in order of k
template <typename E>
struct Sum;
template <>
struct Sum<bf16_t> {
    f4 c = {0.f, 0.f, 0.f, 0.f};
    __device__ __forceinline__ void add(const Frag<bf16_t>& a, const Frag<bf16_t>& b) { c = mma(a, b, c); }
    __device__ __forceinline__ void chain(const Frag<bf16_t>& a, const Frag<bf16_t>& b) { add(a, b); }
    __device__ __forceinline__ f4 total() const { return c; }
};
template <>
struct Sum<float> {
    f4 c[2] = {f4{0.f, 0.f, 0.f, 0.f}, f4{0.f, 0.f, 0.f, 0.f}};
    __device__ __forceinline__ void add(const Frag<float>& a, const Frag<float>& b) {
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[e], b.v[e], c[e & 1], 0, 0, 0);
    }
    __device__ __forceinline__ void chain(const Frag<float>& a, const Frag<float>& b) { c[0] = mma(a, b, c[0]); }
    __device__ __forceinline__ f4 total() const { return c[0] + c[1]; }
};

// Few rows of a plain or batched launch whose rows can be read in 16-byte pieces, whole k-steps; R = 16 / PARTS rows at most.  PARTS runs of k lie side
// by side in one product: the operands' row (and column) i stands for row i % R of run i / R, so the R x R blocks on the result's diagonal hold the
// runs' sums of R columns each, and what lies beside them is thrown away.  A workgroup then has R columns instead of 16: twice or four times the
// workgroups where 16 columns each would leave CUs idle, and as many more loads under way per column.  Eight waves split k; a wave requests U k-steps
// at a time (a loop of single steps waits for each).
// What bounds it: the launch (2.2 us), then the weights at 6 TB/s where nothing stands beside their stream.  An instruction that reads eight rows of
// 128 bytes (two runs) costs what one that reads a KB in a row does, sixteen rows of 64 bytes 10 to 20 % more (weights alone, 42 MB 8.3 / 8.3 / 9.5 us); the rows
// themselves are as many bytes a workgroup as its weights at eight rows and eight columns, so several blocks of columns share one reading of them.  8 rows, K = 2048,
// before / with both, us: 5136 columns (21 MB) 9.1 / 7.1, 10272 14.1 / 10.8, 32000 34.1 / 24.6 (weights alone 21).
// the waves' sums: lane R i .. of run 0 ends up with what it stores (rows m0 = 4 (lane >> 4) .. + 3 of column lane & 15)
template <int PARTS>
__device__ __forceinline__ f4 parts_total(const f4 (*red)[64], int lane) {
    constexpr int R = 16 / PARTS;
    f4 acc = red[0][lane];
#pragma unroll
    for (int w = 1; w < 8; ++w) acc += red[w][lane];
    // run p of column i: lane R i.. of the rows p R ..: (16 R / 4 + R) lanes further per run
#pragma unroll
    for (int o = PARTS / 2; o > 0; o >>= 1)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += __shfl(acc[r], (lane + o * (4 * R + R)) & 63, 64);
    return acc;
}

// Workgroup `block` of such a launch, 512 threads; red: [G, gated 2 G][8][64].  LATE: where a result goes is worked out behind the products.  G: blocks of
// R columns a workgroup has, which share what it reads of the rows.  NEAR: load_piece().
template <typename E, int EPI, int PARTS, int U, bool LATE, int G, bool ONCE, bool NEAR = false>
__device__ __forceinline__ void parts_block(const pcb_linear_args& a, int block, f4 (*red)[8][64]) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL, ADD = EPI == PCB_EPI_SCALE_ADD;
    constexpr int R = 16 / PARTS, SKW = 8, T = TWO ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = G > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid >> 6, group = lane >> 4, l15 = lane & 15;
    const int K = a.K, N = a.N, n_lo = block * (R * G), g = a.n_batch > 0 ? blockIdx.z : 0;
    const int run = l15 / R, i = l15 % R;
    const int m_a = i < a.M ? i : a.M - 1, at = piece_at<E, NEAR>(run, group);
    const E* X = (const E*)a.x + g * a.x_batch_stride;
    const E* wrow[G * T];
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const int n = n_lo + j * R + i < N ? n_lo + j * R + i : N - 1;
        const int64_t w_at = g * a.w_group_stride + n * a.ldw + at;
        wrow[j * T] = (const E*)a.w + w_at;
        if (TWO) wrow[j * T + T - 1] = (const E*)a.w2 + w_at;
    }
    const E* xrow = X + (int64_t)(a.row_src ? a.row_src[m_a] : m_a) * a.ldx + at;
    // (the lanes that store: rows m0 .. m0 + 3 of column n_b, run 0, of a wave's block)
    const int m0 = 4 * group, mine = n_lo + (G > 1 ? wave * R : 0) + i, n_b = mine < N ? mine : N - 1;
    float bv = 0.0f, bv2 = 0.0f, cs = 0.0f;
    Place to[4] = {};
    const bool stores = wave < G && m0 < R && run == 0;
    auto places = [&] {
        if (a.bias) bv = to_f32(((const E*)a.bias)[n_b]);
        if (TWO && a.bias2) bv2 = to_f32(((const E*)a.bias2)[n_b]);
        if (ADD) cs = a.col_scale[n_b];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (TWO || m0 + r < a.M) to[r] = place<E, EPI>(a, m0 + r < a.M ? m0 + r : a.M - 1, n_b);
    };
    if (!LATE && stores) places();
    Sum<E> sum[G * T];
    const int steps = K / (32 * PARTS);
    for (int s0 = wave; s0 < steps; s0 += U * SKW) {
        Frag<E> fa[U], fb[G * T][U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * SKW < steps) {                                // (uniform over the wave)
                const int k = 32 * PARTS * (s0 + u * SKW);
#pragma unroll
                for (int j = 0; j < G * T; ++j) fb[j][u] = weight_piece<PARTS, ONCE, NEAR>(wrow[j] + k);
                fa[u] = load_piece<PARTS, NEAR>(xrow + k);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * SKW < steps) {
#pragma unroll
                for (int j = 0; j < G * T; ++j) sum[j].add(fa[u], fb[j][u]);
            }
    }
    if (LATE && stores) places();
#pragma unroll
    for (int j = 0; j < G * T; ++j) red[j][wave][lane] = sum[j].total();
    __syncthreads();
    if (wave >= G) return;
    const int at_red = G > 1 ? wave * T : 0;
    const f4 acc = parts_total<PARTS>(red[at_red], lane), acc2 = TWO ? parts_total<PARTS>(red[at_red + T - 1], lane) : f4{};
    if (!stores || mine >= N) return;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (m0 + r < a.M) put<E, EPI>(to[r], finished<E, EPI>(a, to[r], n_b, acc[r], acc2[r], bv, bv2), cs);
}

// ---- the norm in the launch of its products (pb_linear_normed.hip, pb_norm_stream.hip) ----
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }   // (loads stay under way)

// the sum over a row's waves: 8 >> log2 rows of them, row r's from r (8 >> log2 rows) on
__device__ __forceinline__ float row_total(float s, float* part, int wave, int lane, int per, int r) {
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xb1, 0xf, 0xf, true));       // quad_perm [1,0,3,2]
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x4e, 0xf, 0xf, true));       // quad_perm [2,3,0,1]
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x141, 0xf, 0xf, true));      // row_half_mirror
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x140, 0xf, 0xf, true));      // row_mirror
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    if (lane == 0) part[wave] = s;
    lds_barrier();
    const f4 lo = *(const f4*)part, hi = *(const f4*)(part + 4);
    s = 0.0f;
#pragma unroll
    for (int w = 0; w < 8; ++w) s += (unsigned)(w - r * per) < (unsigned)per ? (w < 4 ? lo[w & 3] : hi[w & 3]) : 0.0f;
    return s;
}

}  // namespace pcb

// Whether a launch's weights (K to a row, `rows` rows of es bytes an element) are read past the caches (nontemporal): where they come from a model whose weights
// do not stay in the 256 MB of the Infinity Cache from one step to the next, as rows of 4 KB in matrices of 8 MB do (bf16 of width 2048), in fp32 of 4 MB
// (width 1024).  us, through the caches / past them: from memory, 8 rows, K = 2048, 5136 columns 7.9 / 7.1, 10272 11.8 / 10.8, 2048 5.6 / 5.1; fp32, K = 1024, 2 rows,
// 2568 columns 6.1 / 5.8, a step of two requests 315 without the 4 MB ones, 305 with them; weights that do stay, 1 row, K = 1024 and 4096 added 6.7 / 8.0,
// 32000 x 1024 12.0 / 13.2.
inline bool pcb_weights_once(int64_t rows, int64_t K, int es) { return K * es >= 4096 && rows * K * es >= (es == 2 ? 8000000 : 4000000); }

// How many of `groups` blocks of columns a workgroup has so that the busiest CU has the fewest, the more the better, up to four (deeper k three); how many it then has
struct pcb_blocks {
    int blocks;
    int64_t share;
};
inline pcb_blocks pcb_parts_blocks(int64_t groups, int64_t K) {
    pcb_blocks f{1, 0};
    for (int n = 1; n <= (K <= 2048 ? 4 : 3); ++n) {
        const int64_t share = ((groups + n - 1) / n + 255) / 256 * n;
        if (n == 1 || share <= f.share) f = {n, share};
    }
    return f;
}
// PCB_OK when the arguments are valid (pb_linear.hip)
int pcb_linear_check(const pcb_linear_args* a);
// whether a launch's rows can be read in 16-byte pieces, whole k-steps
inline bool pcb_linear_pieces(const pcb_linear_args& a) {
    const int es = a.dtype == PCB_BF16 ? 2 : 4;
    return a.n_groups == 0 && !a.row_scale && a.K % 32 == 0 && a.ldx * es % 16 == 0 && a.ldw * es % 16 == 0 && a.x_batch_stride * es % 16 == 0 &&
           a.w_group_stride * es % 16 == 0 &&
           ((uintptr_t)a.x | (uintptr_t)a.w | (uintptr_t)(a.epilogue == PCB_EPI_SILU_MUL ? a.w2 : nullptr)) % 16 == 0;
}

// Memory that a launch reads or stores: rows of cols elements of es bytes, ld elements apart (a null pointer: nothing)
struct pcb_span {
    uintptr_t at;
    uint64_t bytes;
};
inline pcb_span pcb_rows_span(const void* p, int64_t rows, int64_t ld, int64_t cols, int es) {
    return {(uintptr_t)p, p && rows > 0 ? (uint64_t)((rows - 1) * ld + cols) * es : 0};
}
inline bool pcb_apart(const pcb_span& p, const pcb_span& q) { return p.bytes == 0 || q.bytes == 0 || p.at + p.bytes <= q.at || q.at + q.bytes <= p.at; }
// Whether what an unbatched product stores lies apart from s -- as far as the host can say: not the rows that tables on the device place (row_dst, row_off2, row_off3)
inline bool pcb_results_apart(const pcb_linear_args& a, const pcb_span& s) {
    const int es = a.epilogue == PCB_EPI_SCALE_ADD || a.out_f32 || a.dtype == PCB_F32 ? 4 : 2;
    const int cols = a.split_n > 0 ? a.split_n : a.split_n3 > 0 ? a.split_n3 : a.N;
    return (a.row_dst || pcb_apart(pcb_rows_span(a.y, a.M, a.ldy, cols, es), s)) &&
           (!a.y2_f32 || a.split_n <= 0 || pcb_apart(pcb_rows_span(a.y2, a.M, a.head_stride2, a.N - a.split_n, 4), s));
}

// What pcb_norm_linear and pcb_norm_stream ask of their arguments (pb_linear_normed.hip): PCB_OK when they are valid; whether their kernels can read and place them;
// whether x_out (results: what the products store) lies apart from what the rows are made of
int pcb_norm_linear_check(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b);
bool pcb_norm_linear_pieces(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b);
bool pcb_norm_linear_apart(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b, bool results);
