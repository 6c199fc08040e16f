// pcb_norm_stream: pcb_norm_linear (pb_linear_normed.hip) for up to eight rows of 2048 elements and any number of columns.
//
// What bounds it: the weights.  A launch of its own for the norm is 4.3 us (8 rows of 2048: launch, rows, two sums, rows), and the products' launch behind it begins with nothing
// under way.  Here every workgroup works out all rows, as there, but there is one workgroup a CU, so that this is done 256 times whatever the columns, and its first two runs of
// weights (8 columns x K, 32 KB each in bf16) are asked for behind the rows: they arrive while the norm is worked out.  Then run after run, the next but one under way (four
// were slower, 0.3 .. 1 us: the rows of workgroups that start later wait behind them), and a run's 8 x 8 results are one wave's, a lane each -- not the four
// rows of 16 lanes, in a chain of four activations: 15.5 / 13.4 us gated -- the waves taking turns.
// us, weights from memory, 8 rows, K = 2048, launches apart / here: behind a sublayer, 5136 columns 11.4 / 10.5, 10240 17.0 / 13.0, 32000 28.2 / 26.6, 2048 and gated 4096 16.0 / 13.7; a
// table's rows, 5136 10.2 / 8.1; fp32, 2 rows, K = 1024, 32000 columns 29.1 / 23.9; five streams, 1 row, K = 1024, 32000 columns (weights from the caches) 14.8 / 13.6.
// (Two workgroups a CU: 22 for 15.7 us, the rows again for each.  Rows waited for before the weights are asked for: +0.2.)
#include <type_traits>

#include "pb_linear_parts.h"

namespace {
using namespace pcb;

constexpr int CHUNK = 2048, MAX_ROWS = 8, PAD = 8, R = 8, SKW = 8, D = 2, CUS = 256;      // (a row in LDS begins 8 elements behind the end of the one before)
enum { TABLE, POST, MIX };                                           // what the rows are made of

// Who has which blocks of R columns.  A workgroup has those b_step or a_step apart: b_each of the second product's, the first b_more one more; a_each of the first's, a_more one
// more, from the workgroup on whom the second's did not reach.  apart > 0 (products of different gains): so many workgroups have the second's, the others the first's.
struct Deal {
    int apart, b_step, b_each, b_more, a_step, a_each, a_more;
};

// What a launch is asked for, in few lines of memory: a workgroup waits for its arguments before anything else
struct Product {
    const void *w, *w2, *bias, *bias2;
    int ldw, N;
    void *y, *y2;
    const int64_t* row_off2;
    int64_t ldy, head_stride2;
    int split_n, head_dim2, out_f32, y2_f32, act, act_split, act2;
    float act_param;
};
struct Launch {
    const float *gain, *gain2, *x;
    const void* gate;                                                // or the table
    const float *y, *post_gain;
    const int* ids;
    const float* coef;
    int64_t x_stride;
    int M, W, ldg, n_terms, vocab;
    float scale, eps;
    Deal deal;
    Product a, b;
    float* x_out;
};
template <typename E, int EPI>
__device__ __forceinline__ void store_result(const Product& p, int m, int col, int64_t off2, float acc, float acc2, float bv, float bv2) {
    pcb_linear_args q;
    q.act = p.act, q.act_split = p.act_split, q.act2 = p.act2, q.act_param = p.act_param, q.split_n = p.split_n, q.split_n3 = 0, q.N = p.N, q.row_gate = nullptr;
    const float f = finished<E, EPI>(q, Place{}, col, acc, acc2, bv, bv2);
    auto put = [&](void* y, int wide, int64_t to) {
        if (wide)
            ((float*)y)[to] = f;
        else
            ((E*)y)[to] = from_f32<E>(f);
    };
    if (p.split_n <= 0 || col < p.split_n)                           // (two stores: a place chosen by lanes is loaded by lanes, and waited for behind the weights)
        put(p.y, p.out_f32, m * p.ldy + col);
    else if (const int d = col - p.split_n; p.y2_f32)
        put(p.y2, 1, m * p.head_stride2 + d);
    else
        put(p.y2, 0, off2 + (int64_t)(d / p.head_dim2) * p.head_stride2 + d % p.head_dim2);
}

// U: k-steps a wave has of a run of columns (or fewer); NC: chunks of four columns a thread works out of the rows; D: runs of weights under way
template <typename E, int EPI, int U, int NC, int KIND>
__global__ __launch_bounds__(512) void norm_stream_kernel(Launch n) {
    constexpr int TB = EPI == PCB_EPI_SILU_MUL ? 2 : 1;
    // (weights past the caches, fp32 and the deepest k.  us, past / through them: fp32, 1 row, K = 768, 5136 columns from memory 8.2 / 9.1, from the Infinity Cache 8.2 / 8.5, 32000
    // from memory 21.7 / 22.8, K = 576 19.7 / 21.0; where 32000 columns stay there, 98 and 74 MB that nothing else displaces, 21.1 / 20.2, 19.6 / 18.7)
    constexpr bool ONCE = U == 4 || sizeof(E) == 4;
    __shared__ f4 red[2][D][SKW][64];
    __shared__ __attribute__((aligned(16))) E rows[NC * CHUNK + MAX_ROWS * PAD];
    __shared__ __attribute__((aligned(16))) float gains[KIND == POST ? 2 : 1][CHUNK];
    __shared__ __attribute__((aligned(16))) float part[2][SKW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = lane >> 4, l15 = lane & 15;
    const int M = n.M, W = n.W, run = l15 / R, i = l15 % R, at = piece_at<E>(run, group), steps = W / 64;
    // ---- what the rows are made of: row r, columns c[k] .. + 3 of this thread
    const int lg = M <= 1 ? 0 : M <= 2 ? 1 : M <= 4 ? 2 : 3, r = wave >> (3 - lg), rm = r < M ? r : M - 1;
    int c[NC];
    bool on[NC];
    f4 v[NC], t[KIND == POST ? NC : 1];
    float gt[KIND == MIX ? 1 : NC][4];
    const int G = gridDim.x, g = blockIdx.x, gc = 4 * tid < W ? 4 * tid : 0;
    const float* gain = g < n.deal.apart ? n.gain2 : n.gain;
    const f4 g4 = *(const f4*)(gain + gc), p4 = *(const f4*)((KIND == POST ? n.post_gain : gain) + gc);
    const E* row = nullptr;
    if constexpr (KIND == TABLE) {
        int id = n.ids[rm];
        id = id < 0 ? 0 : id >= n.vocab ? n.vocab - 1 : id;
        row = (const E*)n.gate + (int64_t)id * W;
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int col = 4 * ((tid & ((512 >> lg) - 1)) + k * (512 >> lg));
        on[k] = r < M && col < W;
        c[k] = col < W ? col : 0;
        const int64_t from = (int64_t)rm * W + c[k];
        if constexpr (KIND == TABLE) {
            load4(row + c[k], true, 4, gt[k]);
        } else if constexpr (KIND == POST) {
            v[k] = *(const f4*)(n.x + from);
            t[k] = *(const f4*)(n.y + from);
            load4((const E*)n.gate + (int64_t)rm * n.ldg + c[k], true, 4, gt[k]);
        } else {
            v[k] = f4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if constexpr (KIND == MIX) {
        constexpr int TERMS = NC <= 2 ? 8 : 16 / NC;
        for (int j = 0; j < n.n_terms; j += TERMS) {                 // (so many streams under way; past the end the last one again, which is not counted)
            f4 h[TERMS][NC];
            float w[TERMS];
#pragma unroll
            for (int q = 0; q < TERMS; ++q) {
                const int jq = j + q < n.n_terms ? j + q : n.n_terms - 1;
                w[q] = n.coef[jq];
#pragma unroll
                for (int k = 0; k < NC; ++k) h[q][k] = *(const f4*)(n.x + jq * n.x_stride + (int64_t)rm * W + c[k]);
            }
#pragma unroll
            for (int q = 0; q < TERMS; ++q)
                if (j + q < n.n_terms) {
#pragma unroll
                    for (int k = 0; k < NC; ++k) v[k] += w[q] * h[q][k];
                }
        }
    }
    const Product &a = n.a, &b = n.b;
    const Deal& deal = n.deal;
    // A result is one lane's: row m, column cl of a block
    const int m = lane >> 3, cl = lane & 7, mc = m < M ? m : M - 1;
    const int64_t off_a = *(a.split_n > 0 && !a.y2_f32 ? a.row_off2 + mc : (const int64_t*)gain), off_b = *(b.split_n > 0 && !b.y2_f32 ? b.row_off2 + mc : (const int64_t*)gain);
    __builtin_amdgcn_sched_barrier(0);
    // ---- this workgroup's runs of weights: its blocks of the second product (both halves of a gated one behind one another), then of the first
    const int turn = g - deal.b_more, first_a = deal.apart ? g - deal.apart : turn < 0 ? turn + G : turn;
    const int ub = deal.apart && g >= deal.apart ? 0 : TB * (deal.b_each + (g < deal.b_more)), total = ub + (g < deal.apart ? 0 : deal.a_each + (first_a < deal.a_more));
    auto block_of = [&](int u) { return u < ub ? g + u / TB * deal.b_step : first_a + (u - ub) * deal.a_step; };
    auto weights = [&](int u, Frag<E> (&f)[U]) {                     // (past the last one a gain, from the caches, which is not counted: a branch would be waited at)
        const bool second = u < ub;
        const int N = second ? b.N : a.N, col = block_of(u) * R + i;
        const int ld = second ? b.ldw : a.ldw;
        const E* w = (const E*)(!second ? a.w : TB == 2 && (u & 1) ? b.w2 : b.w) + (int64_t)(col < N ? col : N - 1) * ld + at;
        if (u >= total) w = (const E*)gain;
#pragma unroll
        for (int s = 0; s < U; ++s) {
            const int k = wave + s * SKW;
            f[s] = weight_piece<2, ONCE>(w + 64 * (k < steps ? k : steps - 1));
        }
    };
    Frag<E> fb[D][U];
#pragma unroll
    for (int d = 0; d < D; ++d) weights(d, fb[d]);
    E bias, bias2;                                                   // of the results that this wave has next, if it has
    auto biases = [&](int u0) {
        const int u = u0 + ((wave - u0) & (D - 1));
        const bool second = u < ub;
        const int N = second ? b.N : a.N, col = block_of(u) * R + cl, n_b = col < N ? col : N - 1;
        const E *p = (const E*)(second ? b.bias : a.bias), *p2 = TB == 2 && second ? (const E*)b.bias2 : nullptr;
        bias = *(p && u < total ? p + n_b : (const E*)gain), bias2 = *(p2 && u < total ? p2 + n_b : (const E*)gain);
    };
    biases(0);
    __builtin_amdgcn_sched_barrier(0);
    // ---- the residual and its norm
    if (4 * tid < W) {
        *(f4*)(gains[0] + gc) = g4;
        if constexpr (KIND == POST) *(f4*)(gains[1] + gc) = p4;
    }
    const int per = SKW >> lg;
    auto scale_of = [&](const f4 (&x)[NC], float* where) {
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < NC; ++k) s += on[k] ? (x[k][0] * x[k][0] + x[k][1] * x[k][1]) + (x[k][2] * x[k][2] + x[k][3] * x[k][3]) : 0.0f;
        return 1.0f / sqrtf(row_total(s, where, wave, lane, per, r) / (float)W + n.eps);
    };
    if constexpr (KIND == TABLE) {
#pragma unroll
        for (int k = 0; k < NC; ++k) v[k] = n.scale * f4{gt[k][0], gt[k][1], gt[k][2], gt[k][3]};
    } else if constexpr (KIND == POST) {
#pragma unroll
        for (int k = 0; k < NC; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) t[k][e] *= gt[k][e];
        const float inv = scale_of(t, part[0]);
#pragma unroll
        for (int k = 0; k < NC; ++k) v[k] += t[k] * inv * *(const f4*)(gains[1] + c[k]);
    }
    const float inv = scale_of(v, part[1]);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const f4 o = v[k] * inv, gn = *(const f4*)(gains[0] + c[k]);
        if (on[k]) store4(rows + r * (W + PAD) + c[k], o[0] * gn[0], o[1] * gn[1], o[2] * gn[2], o[3] * gn[3]);
    }
    if (G >= MAX_ROWS ? g == r : g == 0) {                           // (each row by another workgroup)
#pragma unroll
        for (int k = 0; k < NC; ++k)
            if (on[k]) *(f4*)(n.x_out + (int64_t)r * W + c[k]) = v[k];
    }
    lds_barrier();
    // ---- the products: every wave's part of k of D runs, then the waves' sums
    Frag<E> fa[U];
    const E* xrow = rows + (i < M ? i : M - 1) * (W + PAD) + at;
#pragma unroll
    for (int s = 0; s < U; ++s) {
        const int k = wave + s * SKW;
        fa[s] = load_piece<2>(xrow + 64 * (k < steps ? k : steps - 1));
    }
    auto total_of = [&](const f4 (*w)[64]) {                         // (the waves' sums of each run of k, then the runs': as parts_total() has them, to the bit)
        float s[2] = {0.0f, 0.0f};
#pragma unroll
        for (int v = 0; v < SKW; ++v)
#pragma unroll
            for (int p = 0; p < 2; ++p) s[p] += ((const float*)&w[v][(m + 8 * p) / 4 * 16 + cl + 8 * p])[m & 3];
        return s[0] + s[1];
    };
    for (int u0 = 0, par = 0; u0 < total; u0 += D, par ^= 1) {
        const int slot = (wave - u0) & (SKW - 1), u = u0 + (slot & (D - 1));       // (the waves take turns at the results)
        const bool second = u < ub;
        const E b0 = bias, b1 = bias2;
        const bool more = u0 + D < total;
        if (more) biases(u0 + D);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int d = 0; d < D; ++d) {
            Sum<E> sum;
#pragma unroll
            for (int s = 0; s < U; ++s)
                if (wave + s * SKW < steps && u0 + d < total) sum.add(fa[s], fb[d][s]);       // (uniform over the wave)
            red[par][d][wave][lane] = sum.total();
            __builtin_amdgcn_sched_barrier(0);
            if (more) weights(u0 + D + d, fb[d]);
            __builtin_amdgcn_sched_barrier(0);
        }
        lds_barrier();                                               // (the other half of red is read by waves that come to the next one behind that)
        if (slot >= D || u >= total || (TB == 2 && second && (u & 1))) continue;
        const int N = second ? b.N : a.N, n_b = block_of(u) * R + cl;
        const float acc = total_of(red[par][slot]), acc2 = TB == 2 && second ? total_of(red[par][(slot + 1) & (D - 1)]) : 0.0f;
        if (m >= M || n_b >= N) continue;
        if (second)
            store_result<E, EPI>(n.b, m, n_b, off_b, acc, acc2, b.bias ? to_f32(b0) : 0.0f, TB == 2 && b.bias2 ? to_f32(b1) : 0.0f);
        else
            store_result<E, PCB_EPI_STORE>(n.a, m, n_b, off_a, acc, 0.0f, a.bias ? to_f32(b0) : 0.0f, 0.0f);
    }
}

template <typename E>
int launch(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b, hipStream_t stream) {
    const bool gated = b && b->epilogue == PCB_EPI_SILU_MUL;
    const int na = pcb_ceil_div(a.N, R), nb = b ? pcb_ceil_div(b->N, R) : 0, grid = na + nb < CUS ? na + nb : CUS, runs_b = gated ? 2 * nb : nb;
    int gb = 0;
    if (b && n.gain2 != n.gain) {
        gb = (int)((int64_t)grid * runs_b / (na + runs_b));
        gb = gb < 1 ? 1 : gb > nb ? nb : gb >= grid ? grid - 1 : gb;
    }
    const int sb = gb > 0 ? gb : grid, sa = grid - gb;
    auto product = [](const pcb_linear_args& q) {
        return Product{q.w, q.w2, q.bias, q.bias2, (int)q.ldw, q.N, q.y, q.y2, q.row_off2, q.ldy, q.head_stride2, q.split_n, q.head_dim2, q.out_f32, q.y2_f32, q.act, q.act_split,
                       q.act2, q.act_param};
    };
    const Launch l{n.gain, n.gain2, n.x, n.table ? n.table : n.gate, n.y, n.post_gain, n.ids, n.coef, n.x_stride, a.M, a.K, (int)n.ldg, n.n_terms, n.vocab, n.scale, n.eps,
                   Deal{gb, sb, nb / sb, nb % sb, sa, na / sa, na % sa}, product(a), product(b ? *b : a), n.x_out};
    auto go = [&](auto epi, auto kind, auto u, auto nc) {
        hipLaunchKernelGGL((norm_stream_kernel<E, decltype(epi)::value, decltype(u)::value, decltype(nc)::value, decltype(kind)::value>), dim3(grid), dim3(512), 0, stream, l);
        return pcb_check_launch("norm_stream_kernel");
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Four = std::integral_constant<int, 4>;
    using Eight = std::integral_constant<int, 8>;
    const int64_t elems = (int64_t)a.K << (a.M <= 1 ? 0 : a.M <= 2 ? 1 : a.M <= 4 ? 2 : 3);
    auto sized = [&](auto epi, auto kind) {
        if (a.K <= 1024)
            return elems <= CHUNK ? go(epi, kind, Two{}, One{}) : elems <= 2 * CHUNK ? go(epi, kind, Two{}, Two{}) : go(epi, kind, Two{}, Four{});
        return elems <= CHUNK       ? go(epi, kind, Four{}, One{})
               : elems <= 2 * CHUNK ? go(epi, kind, Four{}, Two{})
               : elems <= 4 * CHUNK ? go(epi, kind, Four{}, Four{})
                                    : go(epi, kind, Four{}, Eight{});
    };
    using Store = std::integral_constant<int, PCB_EPI_STORE>;
    if (n.table) return sized(Store{}, std::integral_constant<int, TABLE>{});
    if (!n.y) return sized(Store{}, std::integral_constant<int, MIX>{});
    using Post = std::integral_constant<int, POST>;
    return gated ? sized(std::integral_constant<int, PCB_EPI_SILU_MUL>{}, Post{}) : sized(Store{}, Post{});
}

// Where this is faster than launches of their own and pcb_norm_linear does not go (its callers ask that one first: a workgroup for each block of columns is 0.5 .. 1.5 us
// faster where there are few of them, and up to K = 512, where a run of weights is less than what finding it costs: bf16 gated, 1 row, K = 384, 72 and 2200 columns 4.2, here 5.8).
// us, launches apart / here, medians of 900 random sizes: K = 576 .. 1024 and 1600 .. 2048 a table or behind a sublayer 0.62 .. 0.97 of it, one fp32 size in 60 1.04; between them
// waves have a third k-step, or not, in registers for four: bf16, 5 rows, K = 1088, 4176 columns 8.5 / 9.8, fp32, 2 rows, 13000 columns 17.2 / 20.2.  The streams' sum is worked
// out by every workgroup: up to 32768 elements of all streams of more than 256 runs of weights 0.75 .. 1.03 (of K = 576 .. 768 up to 20480: 8 rows, five streams, 5136 columns, bf16, K = 576 1.01,
// 16000 1.16, fp32 1.03 and 1.09), of fewer up to 12288 0.8 .. 0.97, beyond 1.05 .. 1.5.  A vocabulary's runs of a short k go by faster in launches of their own, several blocks of columns a
// workgroup: 32000 columns, bf16, 1 row, K = 576 12.1 / 14.6, 768 13.5 / 15.3, 960 1.00, 1024 0.97, 4 rows, K = 576 13.4 / 14.9, 704 1.01, 8 rows 1.05, 0.95, fp32, 1 row 1.01 .. 1.06 and 0.97; 16000 columns, the
// sum of five streams, bf16, 1 row, K = 576 1.12, 704 1.04, 832 0.99.
bool faster(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b) {
    const int64_t elems = (int64_t)a.K << (a.M <= 1 ? 0 : a.M <= 2 ? 1 : a.M <= 4 ? 2 : 3);
    const int64_t runs = pcb_ceil_div(a.N, R) + (b ? (int64_t)pcb_ceil_div(b->N, R) * (b->epilogue == PCB_EPI_SILU_MUL ? 2 : 1) : 0);
    const int least = runs > 3000 ? (a.dtype == PCB_F32 ? 704 : a.M <= 2 ? 960 : a.M <= 4 ? 768 : 704) : runs > 1500 && n.n_terms > 0 && a.dtype == PCB_BF16 ? 768 : 0;
    return (a.K > 1536 || (a.K > 512 && a.K <= 1024)) && a.K >= least && n.n_terms * elems <= (runs <= CUS ? 12288 : a.K <= 768 ? 20480 : 32768);
}

int route(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b) {
    const int rc = pcb_norm_linear_check(n, a, b);
    if (rc != PCB_OK) return rc;
    auto narrow = [](int64_t v) { return v >= 0 && v <= INT32_MAX; };
    const bool can = a->M <= MAX_ROWS && a->K <= CHUNK && narrow(n->ldg) && narrow(a->ldw) && (!b || narrow(b->ldw)) && pcb_norm_linear_pieces(*n, *a, b);
    return can && faster(*n, *a, b) && pcb_norm_linear_apart(*n, *a, b, true) ? PCB_OK : PCB_NOT_TAKEN;
}

}  // namespace

PCB_EXPORT int pcb_norm_stream_takes(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b) { return route(n, a, b); }

PCB_EXPORT int pcb_norm_stream(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b, void* stream) {
    const int rc = route(n, a, b);
    if (rc < 0 || a->M == 0) return rc < 0 ? rc : PCB_OK;
    if (rc != PCB_OK) return rc;
    return a->dtype == PCB_BF16 ? launch<bf16_t>(*n, *a, b, (hipStream_t)stream) : launch<float>(*n, *a, b, (hipStream_t)stream);
}
