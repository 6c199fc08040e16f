// Two products of a few rows in one launch: a step of few requests is a chain of launches of three to five us each, whatever little they do.
//   pcb_linear_pair   two products that do not need one another
//   pcb_linear_add2   two scaled accumulations into the same rows, the second one's input optionally the polynomial norm of fp32 rows
// What they do not take runs as the launches that they stand for.
#include <type_traits>

#include "pb_linear_parts.h"
#include "pb_linear_tiles.h"

namespace {
using namespace pcb;

// ---- side by side: the first na workgroups are the first product's ---------------------------------------------------------------------
template <typename E, int EPI, int PARTS, int U>
__global__ __launch_bounds__(512) void linear_pair_kernel(pcb_linear_args a, pcb_linear_args b, int na) {
    __shared__ f4 red[EPI == PCB_EPI_SILU_MUL ? 2 : 1][8][64];
    if ((int)blockIdx.x < na)
        parts_block<E, PCB_EPI_STORE, PARTS, U, true>(a, blockIdx.x, red);
    else
        parts_block<E, EPI, PARTS, U, EPI == PCB_EPI_STORE>(b, blockIdx.x - na, red);
}

// ---- one behind the other: y = (base + col_scale (x w^T + bias)) + b.col_scale (b.x b.w^T + b.bias) ------------------------------------------
// Workgroups and waves as in pb_linear_parts.h, both products' sums side by side.  POLY: the rows of b.x are polynorm(z), worked out where they are
// used: every workgroup takes the rows' sums itself (eight waves share the rows), beside the first product's loads and with the second's first weights
// under way.
template <typename E, int PARTS, int U, bool POLY>
__global__ __launch_bounds__(512) void linear_add2_kernel(pcb_linear_args a, pcb_linear_args b, const float* __restrict__ z, const float* __restrict__ coef,
                                                          float eps) {
    constexpr int R = 16 / PARTS, SKW = 8;
    __shared__ f4 red[2][8][64];
    __shared__ float part[8][3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, group = lane >> 4, l15 = lane & 15;
    const int M = a.M, N = a.N, n_lo = blockIdx.x * R, run = l15 / R, i = l15 % R;
    const int n_b = n_lo + i < N ? n_lo + i : N - 1, m_a = i < M ? i : M - 1, at = 32 * run + 8 * group;
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
                fb[u] = load8(wa + k);
                fa[u] = load8(xa + k);
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
                fb[u] = load8(wb + k);
                if constexpr (POLY)
                    zv[u][0] = *reinterpret_cast<const f4*>(zrow + k), zv[u][1] = *reinterpret_cast<const f4*>(zrow + k + 4);
                else
                    fa[u] = load8(xb + k);
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
    auto go = [&](auto epi, auto p) {
        constexpr int EPI = decltype(epi)::value, P = decltype(p)::value;
        const int na = pcb_ceil_div(a.N, 16 / P), nb = pcb_ceil_div(b.N, 16 / P);
        hipLaunchKernelGGL((linear_pair_kernel<E, EPI, P, sizeof(E) == 2 ? 4 : 2>), dim3(na + nb), dim3(512), 0, stream, a, b, na);
        return pcb_check_launch("linear_pair_kernel");
    };
    // Two runs of k side by side (up to eight rows) while both products together have no more than 8192 weight rows, beyond that up to four rows, not
    // with a gated bf16 unit.  Weights from memory, us, one run / two: 1 row bf16, 1280 + 4096 columns, K = 1024 5.9 / 5.5, 640 + 2048, K = 512 3.9 / 4.1; 2560 + 8192,
    // K = 2048 12.9 / 11.2, 8 rows 14.7 / 15.5; 1024 and 2048 gated, K = 1024, 8 rows 6.7 / 6.1, fp32 9.9 / 8.8; 2048 and 4096 gated, K = 2048, 1 row
    // 12.1 / 12.3, 2 rows fp32 21.8 / 19.7, 8 rows 13.5 / 14.9.  (Four runs lose 2 to 20 % against two at each of these.)  As launches of their own,
    // the first of each pair: 8.1, 6.4, 13.9, 19.3, 9.9, 13.2, 13.7, 23.3, 16.0.
    const bool gated = b.epilogue == PCB_EPI_SILU_MUL;
    const int64_t w_rows = (int64_t)a.N + (gated ? 2 : 1) * (int64_t)b.N;
    const bool two = a.M <= 8 && a.K >= 1024 && b.K >= 1024 && splits(a, 2) && splits(b, 2) &&
                     (w_rows <= 8192 || (a.M <= 4 && !(gated && sizeof(E) == 2)));
    auto kind = [&](auto epi) { return two ? go(epi, std::integral_constant<int, 2>{}) : go(epi, std::integral_constant<int, 1>{}); };
    return b.epilogue == PCB_EPI_STORE ? kind(std::integral_constant<int, PCB_EPI_STORE>{}) : kind(std::integral_constant<int, PCB_EPI_SILU_MUL>{});
}

template <typename E>
int add2(const pcb_linear_args& a, const pcb_linear_args& b, const float* z, const float* coef, float eps, int parts, hipStream_t stream) {
    constexpr int U = sizeof(E) == 2 ? 4 : 2;
    const dim3 grid(pcb_ceil_div(a.N, 16 / parts));
    auto go = [&](auto p, auto poly) {
        hipLaunchKernelGGL((linear_add2_kernel<E, decltype(p)::value, U, decltype(poly)::value>), grid, dim3(512), 0, stream, a, b, z, coef, eps);
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
    // (A gated unit in bf16 only up to 80 MB of weights: alone it is faster then.  us, two launches / one, 8 rows, residual gate and gated unit of a width:
    // 2048 15.9 / 14.3, 2560 (66 MB) 24.4 / 21.6, 3072 (94 MB) 28.9 / 29.8, 1 row 13.6 / 12.8, 19.4 / 18.9, 23.4 / 26.5.  9 and 16 rows: bf16 2048 18.7 / 14.7 and
    // 20.0 / 16.0, 2560 29.2 / 22.2 and 32.9 / 25.2; fp32 2048 27.5 / 23.6 and 29.1 / 26.5; plain, 2560 + 8192
    // columns, K = 2048, bf16 18.9 / 15.1 and 20.8 / 17.6.)
    const bool heavy = a.dtype == PCB_BF16 && b.epilogue == PCB_EPI_SILU_MUL && ((int64_t)a.N * a.K + 2 * (int64_t)b.N * b.K) * 2 > 80000000;
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
