// Two products of a few rows in one launch: a step of few requests is a chain of launches of three to five us each, whatever little they do.
//   pcb_linear_pair   two products that do not need one another
//   pcb_linear_add2   two scaled accumulations into the same rows, the second one's input optionally the polynomial norm of fp32 rows
// What they do not take runs as the launches that they stand for.
#include <type_traits>

#include "pb_linear_parts.h"
#include "pb_linear_tiles.h"

namespace {
using namespace pcb;

// ---- side by side: the first na workgroups are the first product's, GA blocks of columns each ----------------------------------------------
template <typename E, int EPI, int PARTS, int U, int GA, bool LATE, bool ONCE>
__global__ __launch_bounds__(512) void linear_pair_kernel(pcb_linear_args a, pcb_linear_args b, int na) {
    __shared__ f4 red[EPI == PCB_EPI_SILU_MUL ? 2 : GA][8][64];
    if ((int)blockIdx.x < na)
        parts_block<E, PCB_EPI_STORE, PARTS, U, true, GA, ONCE>(a, blockIdx.x, red);
    else
        parts_block<E, EPI, PARTS, U, LATE, 1, ONCE>(b, blockIdx.x - na, red);
}

// ---- one behind the other: y = (base + col_scale (x w^T + bias)) + b.col_scale (b.x b.w^T + b.bias) ------------------------------------------
// Workgroups and waves as in pb_linear_parts.h, both products' sums side by side.  POLY: the rows of b.x are polynorm(z), worked out where they are
// used: every workgroup takes the rows' sums itself (eight waves share the rows), beside the first product's loads and with the second's first weights
// under way.
template <typename E, int PARTS, int U, bool POLY, bool ONCE>
__global__ __launch_bounds__(512) void linear_add2_kernel(pcb_linear_args a, pcb_linear_args b, const float* __restrict__ z, const float* __restrict__ coef,
                                                          float eps) {
    constexpr int R = 16 / PARTS, SKW = 8;
    __shared__ f4 red[2][8][64];
    __shared__ float part[8][3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, group = lane >> 4, l15 = lane & 15;
    const int M = a.M, N = a.N, n_lo = blockIdx.x * R, run = l15 / R, i = l15 % R;
    const int n_b = n_lo + i < N ? n_lo + i : N - 1, m_a = i < M ? i : M - 1, at = piece_at<E>(run, group);
    const E* wa = (const E*)a.w + n_b * a.ldw + at;
    const E* wb = (const E*)b.w + n_b * b.ldw + at;
    const E* xa = (const E*)a.x + m_a * a.ldx + at;
    const E* xb = POLY ? nullptr : (const E*)b.x + m_a * b.ldx + at;
    const int steps_a = a.K / (32 * PARTS), steps_b = b.K / (32 * PARTS), ff = b.K;

    // the rows' sums: row tid / (512 / rows), each of its waves a part of the columns
    const int rows = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : 8, tpr = 512 / rows;
    float c[4];
    if (POLY) {
        const int r = tid / tpr;
        const float* zr = z + (int64_t)(r < M ? r : M - 1) * ff;
        float s[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int e = 0; e < 4; ++e) c[e] = coef[e];
#pragma unroll 4
        for (int k = 4 * (tid % tpr); k < ff; k += 4 * tpr) {
            const f4 v = *reinterpret_cast<const f4*>(zr + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = v[e], x2 = x * x, x3 = x2 * x;
                s[0] += x2;
                s[1] += x2 * x2;
                s[2] += x3 * x3;
            }
        }
#pragma unroll
        for (int e = 0; e < 3; ++e) {
            s[e] = wave_sum(s[e]);
            if (lane == 0) part[wave][e] = s[e];
        }
    }
    // (the lanes that store)
    const int m0 = 4 * group;
    const bool stores = wave == 0 && m0 < R && run == 0;
    float bv = 0.0f, cs = 0.0f, bv2 = 0.0f, cs2 = 0.0f;
    Place to[4] = {};
    if (stores) {
        if (a.bias) bv = to_f32(((const E*)a.bias)[n_b]);
        if (b.bias) bv2 = to_f32(((const E*)b.bias)[n_b]);
        cs = a.col_scale[n_b];
        cs2 = b.col_scale[n_b];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (m0 + r < M) to[r] = place<E, PCB_EPI_SCALE_ADD>(a, m0 + r, n_b);
    }
    Sum<E> sum, sum2;
    for (int s0 = wave; s0 < steps_a; s0 += U * SKW) {
        Frag<E> fa[U], fb[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * SKW < steps_a) {                            // (uniform over the wave)
                const int k = 32 * PARTS * (s0 + u * SKW);
                fb[u] = weight_piece<PARTS, ONCE>(wa + k);
                fa[u] = load_piece<PARTS>(xa + k);
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * SKW < steps_a) sum.add(fa[u], fb[u]);
    }
    const float* zrow = z + (int64_t)m_a * ff + at;
    float i1 = 0.0f, i2 = 0.0f, i3 = 0.0f;
    for (int s0 = wave; s0 < steps_b; s0 += U * SKW) {
        Frag<E> fa[U], fb[U];
        f4 zv[POLY ? U : 1][2];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * SKW < steps_b) {
                const int k = 32 * PARTS * (s0 + u * SKW);
                fb[u] = weight_piece<PARTS, ONCE>(wb + k);
                if constexpr (POLY)
                    zv[u][0] = *reinterpret_cast<const f4*>(zrow + k), zv[u][1] = *reinterpret_cast<const f4*>(zrow + k + (sizeof(E) == 2 ? 4 : 16 * PARTS));
                else
                    fa[u] = load_piece<PARTS>(xb + k);
            }
        if constexpr (POLY) {
            if (s0 == wave) {                                        // (every wave comes by exactly once: steps_b >= 8)
                __syncthreads();
                float s[3] = {0.0f, 0.0f, 0.0f};
                for (int w = 0; w < SKW / rows; ++w)
#pragma unroll
                    for (int e = 0; e < 3; ++e) s[e] += part[m_a * (SKW / rows) + w][e];
                i1 = c[0] / sqrtf(s[0] / (float)ff + eps);
                i2 = c[1] / sqrtf(s[1] / (float)ff + eps);
                i3 = c[2] / sqrtf(s[2] / (float)ff + eps);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (s0 + u * SKW < steps_b) {
                    float o[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float x = zv[u][e >> 2][e & 3], x2 = x * x;
                        o[e] = i1 * x + i2 * x2 + i3 * (x2 * x) + c[3];
                    }
                    if constexpr (sizeof(E) == 2) {
                        fa[u].v = u32x4{bf16_pair(o[0], o[1]), bf16_pair(o[2], o[3]), bf16_pair(o[4], o[5]), bf16_pair(o[6], o[7])};
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e) fa[u].v[e] = o[e];
                    }
                }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * SKW < steps_b) sum2.add(fa[u], fb[u]);
    }
    red[0][wave][lane] = sum.total();
    red[1][wave][lane] = sum2.total();
    __syncthreads();
    if (wave != 0) return;
    const f4 acc = parts_total<PARTS>(red[0], lane), acc2 = parts_total<PARTS>(red[1], lane);
    if (!stores || n_lo + i >= N) return;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (m0 + r < M) *(float*)to[r].p = (to[r].base + cs * (acc[r] + bv)) + cs2 * (acc2[r] + bv2);
}

// k in runs of eight k-steps at least, for every wave one
bool splits(const pcb_linear_args& a, int parts) { return a.K % (32 * parts) == 0 && a.K >= 256 * parts; }

template <typename E>
int pair(const pcb_linear_args& a, const pcb_linear_args& b, hipStream_t stream) {
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Four = std::integral_constant<int, 4>;
    const bool once = pcb_weights_once(a.N + (b.epilogue == PCB_EPI_SILU_MUL ? 2 : 1) * (int64_t)b.N, a.K < b.K ? a.K : b.K, sizeof(E));
    auto go = [&](auto epi, auto p, auto u, auto ga, auto late) {
        constexpr int EPI = decltype(epi)::value, P = decltype(p)::value, GA = decltype(ga)::value;
        const int na = pcb_ceil_div(a.N, 16 / P * GA), nb = pcb_ceil_div(b.N, 16 / P);
        if (P > 1 && once)
            hipLaunchKernelGGL((linear_pair_kernel<E, EPI, P, decltype(u)::value, GA, decltype(late)::value, (P > 1)>), dim3(na + nb), dim3(512), 0, stream, a, b, na);
        else
            hipLaunchKernelGGL((linear_pair_kernel<E, EPI, P, decltype(u)::value, GA, decltype(late)::value, false>), dim3(na + nb), dim3(512), 0, stream, a, b, na);
        return pcb_check_launch("linear_pair_kernel");
    };
    // Two runs of k side by side up to eight rows, while the workgroups are not too many for a k of so few steps; results' places behind the products where the second is gated,
    // ahead of them over a k of up to 1536.  Weights from memory, us, one run (as all were that are not marked *) / two: bf16 1 row, 2048 and 4096 gated, K = 2048
    // 12.5 / 9.4, 8 rows 13.7 / 10.9, places ahead 14.3; 2560 and 5120, K = 2560 20.3 / 16.8; 2560 + 8192 columns, K = 2048, 8 rows 15.0 / 14.0, 1 row 10.5 * / 9.6; K = 1024, places ahead, 512
    // and 512 gated, 1 and 8 rows 5.2 / 4.4 and 6.3 / 5.3, 1024 and 1024 5.6 / 4.9 and 6.6 / 5.8, 1024 and 2048 8 rows 6.5 / 6.1 (behind 6.7), 2700 and 2700 8.3 / 9.8, K = 1152, 2048 and 2048, 1 and 8 rows, ahead and behind 5.8 / 6.4 and 6.9 / 7.4, K = 1536 0.98 and 0.99 of it; plain, 8 rows, K = 1024,
    // 3072 + 9216 columns 1.00 / 1.08, 8192 + 24576 1.00 / 1.07, K = 1536 3072 + 9216 1.00 / 1.08, K = 2048 1.00 / 0.97; 512 + 1024 gated, K = 512 3.7 / 3.9; fp32 5.5 / 4.1, 2048 and 2048
    // gated, K = 512 1.00 / 0.92, 2700 and 2700 8.4 / 9.2, 3072 and 3072, K = 512, 8 rows 8.4 / 9.9, 8192 and 8192 14.8 / 20.0, K = 768 20.1 / 25.7, K = 1024, 4 and 8 rows 1.00 / 0.97 and 1.00 / 1.16; 2048 and 4096
    // gated, K = 2048, fp32, 2 rows 18.7 * / 16.8 with one k-step a time and places behind, 8 rows 21.9 * / 19.8; 2560 + 8192 columns, 8 rows 22.8 / 24.4.  The first product's blocks two a
    // workgroup where that is a round of the chip less: 1536 and 3072 gated, K = 1536, 8 rows 9.1 / 8.0, 3072 and 6144 23.4 / 20.9; 2048 and 4096 10.9 / 11.9.
    constexpr bool bf = sizeof(E) == 2;
    const bool gated = b.epilogue == PCB_EPI_SILU_MUL;
    const int K = a.K < b.K ? a.K : b.K;
    const int64_t w_rows = (int64_t)a.N + (gated ? 2 : 1) * (int64_t)b.N;
    const bool few = w_rows <= 7168, two = a.M <= 8 && splits(a, 2) && splits(b, 2) &&
                                           (gated ? (bf ? K > 1024 || (K == 1024 && few) : K > 1024 || few || (K == 1024 && (w_rows <= 16384 || a.M <= 4)))
                                                  : K >= 1024 && (w_rows <= 8192 || a.M <= 4 || (bf && K > 1536)));
    auto yes = std::true_type{};
    auto no = std::false_type{};
    using Plain = std::integral_constant<int, bf ? 4 : 2>;
    if (!gated) {
        std::integral_constant<int, PCB_EPI_STORE> epi;
        return !two ? go(epi, One{}, Plain{}, One{}, yes) : go(epi, Two{}, Plain{}, One{}, std::integral_constant<bool, !bf>{});
    }
    std::integral_constant<int, PCB_EPI_SILU_MUL> epi;
    if (!two) return go(epi, One{}, Plain{}, One{}, no);
    if constexpr (bf) {
        if (K < 1536 && few) return go(epi, Two{}, Four{}, One{}, no);
        const int na = pcb_ceil_div(a.N, 8), nb = pcb_ceil_div(b.N, 8);
        return pcb_ceil_div(nb + (na + 1) / 2, 256) < pcb_ceil_div(nb + na, 256) ? go(epi, Two{}, Four{}, Two{}, yes) : go(epi, Two{}, Four{}, One{}, yes);
    } else {
        return K > 1024 ? go(epi, Two{}, One{}, One{}, yes) : go(epi, Two{}, Two{}, One{}, no);
    }
}

template <typename E>
int add2(const pcb_linear_args& a, const pcb_linear_args& b, const float* z, const float* coef, float eps, int parts, hipStream_t stream) {
    constexpr int U = sizeof(E) == 2 ? 4 : 2;
    const dim3 grid(pcb_ceil_div(a.N, 16 / parts));
    const bool once = pcb_weights_once(2 * (int64_t)a.N, a.K < b.K ? a.K : b.K, sizeof(E));
    auto go = [&](auto p, auto poly) {
        if (once)
            hipLaunchKernelGGL((linear_add2_kernel<E, decltype(p)::value, U, decltype(poly)::value, true>), grid, dim3(512), 0, stream, a, b, z, coef, eps);
        else
            hipLaunchKernelGGL((linear_add2_kernel<E, decltype(p)::value, U, decltype(poly)::value, false>), grid, dim3(512), 0, stream, a, b, z, coef, eps);
        return pcb_check_launch("linear_add2_kernel");
    };
    using Four = std::integral_constant<int, 4>;
    using Two = std::integral_constant<int, 2>;
    if (z) return parts == 4 ? go(Four{}, std::true_type{}) : go(Two{}, std::true_type{});
    return parts == 4 ? go(Four{}, std::false_type{}) : go(Two{}, std::false_type{});
}

}  // namespace

// Whether either product's results lie apart from the other's results and from the rows and gates it reads: in one launch nothing orders the two
static bool pair_apart(const pcb_linear_args& a, const pcb_linear_args& b) {
    auto from = [](const pcb_linear_args& p, const pcb_linear_args& q) {         // p's results from what q reads
        const int es = q.dtype == PCB_BF16 ? 2 : 4;
        return (q.row_src || pcb_results_apart(p, pcb_rows_span(q.x, q.M, q.ldx, q.K, es))) &&
               pcb_results_apart(p, pcb_rows_span(q.row_gate, q.M, q.ld_row_gate, 1, es));
    };
    const int es = b.out_f32 || b.dtype == PCB_F32 ? 4 : 2, cols = b.split_n > 0 ? b.split_n : b.split_n3 > 0 ? b.split_n3 : b.N;
    return from(a, b) && from(b, a) && (b.row_dst || pcb_results_apart(a, pcb_rows_span(b.y, b.M, b.ldy, cols, es))) &&
           (!b.y2_f32 || b.split_n <= 0 || pcb_results_apart(a, pcb_rows_span(b.y2, b.M, b.head_stride2, b.N - b.split_n, 4)));
}

// How a pair goes out: 0 two launches, 1 one of few rows, 2 + shape one grid of tiles
static int pair_form(const pcb_linear_args& a, const pcb_linear_args& b) {
    if (a.dtype != b.dtype || a.M != b.M || a.M <= 0 || a.n_batch != 0 || b.n_batch != 0 || a.epilogue != PCB_EPI_STORE || b.epilogue == PCB_EPI_SCALE_ADD ||
        !pcb_linear_pieces(a) || !pcb_linear_pieces(b) || !pair_apart(a, b))
        return 0;
    // (More than four rows of bf16 with many plain columns as two, where the busiest CU has no more blocks of columns then: each is the faster by itself, with several of them a
    // workgroup.  us, one launch / two, 8 rows, 2560 + 8192 columns, K = 2048 14.0 / 14.6, 5136 + 15408, K = 2048 22.4 / 20.7, 8192 + 24576, K = 1536 26.9 / 23.5, 3840 + 12288, K = 3072
    // 24.9 / 23.8, 2700 + 8100, K = 4096 24.4 / 22.9, 3072 + 9216, K = 4096 (six blocks / two and five) 26.2 / 29.5, 5120 + 16384 42.6 / 37.2; gated 3072 and 6144, K = 3072 20.9 / 25.0, 1 row
    // 17.7 / 20.3, 4096 and 8192 32.2 / 36.6, 16 rows 44.1 / 49.0; fp32 2048 and 4096, 9 and 16 rows 23.6 / 27.5 and 26.5 / 29.1; plain, 2560 + 8192 columns, 9 and 16 rows
    // 15.1 / 18.9 and 17.6 / 20.8.)
    const int ga = pcb_ceil_div(a.N, 8), gb = pcb_ceil_div(b.N, 8);
    const bool heavy = a.dtype == PCB_BF16 && b.epilogue == PCB_EPI_STORE && a.M > 4 && a.M <= 8 && ((int64_t)a.N * a.K + (int64_t)b.N * b.K) * 2 > 80000000 &&
                       pcb_parts_blocks(ga, a.K).share + pcb_parts_blocks(gb, b.K).share <= pcb_ceil_div(ga + gb, 256);
    if (a.M <= 16) return heavy ? 0 : 1;
    const int shape = a.M > 64 ? pcb_linear_tiles_pair_shape(a, b) : -1;
    return shape < 0 ? 0 : 2 + shape;
}

PCB_EXPORT int pcb_linear_pair_form(const pcb_linear_args* a, const pcb_linear_args* b) {
    int rc = pcb_linear_check(a);
    if (rc == PCB_OK) rc = pcb_linear_check(b);
    return rc == PCB_OK ? pair_form(*a, *b) : rc;
}

PCB_EXPORT int pcb_linear_pair(const pcb_linear_args* a, const pcb_linear_args* b, void* stream) {
    const int form = pcb_linear_pair_form(a, b);
    if (form < 0) return form;
    if (form >= 2) return pcb_linear_tiles_pair(*a, *b, form - 2, (hipStream_t)stream);
    if (form == 1) return a->dtype == PCB_BF16 ? pair<pcb::bf16_t>(*a, *b, (hipStream_t)stream) : pair<float>(*a, *b, (hipStream_t)stream);
    const int rc = pcb_linear(a, stream);
    return rc == PCB_OK ? pcb_linear(b, stream) : rc;
}

PCB_EXPORT int pcb_linear_add2(const pcb_linear_args* a, const pcb_linear_args* b, const float* z, const float* coef, float eps, void* stream) {
    int rc = pcb_linear_check(a);
    if (rc == PCB_OK) rc = pcb_linear_check(b);
    if (rc != PCB_OK) return rc;
    PCB_REQUIRE(a->dtype == b->dtype && a->M == b->M && a->N == b->N && a->epilogue == PCB_EPI_SCALE_ADD && b->epilogue == PCB_EPI_SCALE_ADD &&
                    a->y == b->y && a->ldy == b->ldy && !b->base,
                PCB_ERR_ARG, "pcb_linear_add2: two scaled accumulations into the same rows");
    PCB_REQUIRE(!z || (coef && !b->row_src && b->ldx == b->K && b->n_groups == 0), PCB_ERR_ARG, "pcb_linear_add2: normed rows are plain rows of K columns");
    if (a->M == 0) return PCB_OK;
    // Up to eight rows, runs of k as pcb_linear takes them.  As launches of their own / here, us, with the norm: 1 row bf16, 1024 columns, K = 1024 and 4096
    // 11.2 / 7.3, 4 rows 12.7 / 8.9, 8 rows 15.0 / 12.1; 2048 columns, K = 2048 and 8192 18.1 / 14.3, 4 rows 21.7 / 20.7, 8 rows 22.3 / 21.7, fp32 34.0 / 30.2.
    const bool pieces = pcb_linear_pieces(*a) && pcb_linear_pieces(*b) && !a->row_src && !b->row_src && (!z || (uintptr_t)z % 16 == 0);
    const int parts = a->M <= 4 && splits(*a, 4) && splits(*b, 4) && pcb_ceil_div(a->N, 4) <= 768 ? 4 : a->M <= 8 && splits(*a, 2) && splits(*b, 2) ? 2 : 0;
    // In bf16 three rows and more only up to 56 MB of weights: 4 rows, 2048 columns, K = 2048 and 8192 (42 MB) as launches of their own 21.8, here 20.9, 2560 and
    // 10240 (66 MB) 31.6 / 35.7, 4096 and 16384 48.3 / 53.9, 8 rows 56.1 / 68.8; 1 row 24.5 / 23.0, 43.9 / 42.5; 4 rows fp32 48.4 / 47.7, 86.7 / 81.6.
    const bool heavy = a->dtype == PCB_BF16 && a->M > 2 && (int64_t)a->N * ((int64_t)a->K + b->K) * 2 > 56000000;
    if (pieces && parts && !heavy)
        return a->dtype == PCB_BF16 ? add2<pcb::bf16_t>(*a, *b, z, coef, eps, parts, (hipStream_t)stream)
                                    : add2<float>(*a, *b, z, coef, eps, parts, (hipStream_t)stream);
    rc = pcb_linear(a, stream);
    if (rc == PCB_OK && z) rc = pcb_polynorm(z, coef, const_cast<void*>(b->x), b->dtype, eps, b->M, b->K, stream);
    return rc == PCB_OK ? pcb_linear(b, stream) : rc;
}
