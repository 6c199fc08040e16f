// pcb_norm_linear: a step's residual row and its norm inside the launch of the products that read the normed row (what pcb_embed_rows, pcb_mix_norm or
// pcb_post_norm and pcb_linear or pcb_linear_pair are in launches of their own).
//
// Workgroups, waves and runs of k as in pb_linear_parts.h.  Every workgroup works out all M rows itself, four or eight columns a thread: it asks for
// what the rows are made of first and for its weights behind them, so the norm's trips -- memory, and one or two sums over the row -- pass while the weights are
// under way.  The normed rows wait in LDS as E.  The first workgroup writes the new residual, into rows that nobody reads in this launch.
// What bounds it: a launch's own way (arguments, rows, sums, products, store: ~6 us), no longer two of them.  us, a decoding step in a graph, apart / here: Fivesun
// bf16 one request, width 512 134 / 113, 2048 236 / 211, two of 1024 166 / 140, four of 512 155 / 135, fp32 two of 1024 203 / 188; Kazolorn bf16 one of 1024
// 108 / 100, four of 512 107 / 96.  (What results need from memory asked for behind the norm, by the wave that stores: 2 us a launch more.)
#include <type_traits>

#include "pb_linear_parts.h"

namespace {
using namespace pcb;

constexpr int CHUNK = 2048, MAX_ROWS = 8, PAD = 8;    // (a row in LDS begins 8 elements behind the end of the one before)
enum { TABLE, POST, MIX };                                           // (MIX + t: a sum whose last t streams, or all of up to t, are under way at a time)

// U: k-steps a wave takes of its run, all under way at a time (fewer count); NC: chunks of four columns a thread works out
template <typename E, int EPI, int PARTS, int U, int NC, int KIND>
__device__ __forceinline__ void normed_block(const pcb_row_norm_args& n, const float* gain, const pcb_linear_args& a, int block, bool keeps, E* rows,
                                             float (*part)[8], f4 (*red)[8][64]) {
    constexpr bool TWO = EPI == PCB_EPI_SILU_MUL;
    constexpr int R = 16 / PARTS, SKW = 8, LG = NC == 1 ? 2 : 3, TERMS = KIND - MIX;     // (one chunk: four rows at most)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), group = lane >> 4, l15 = lane & 15;
    const int M = a.M, W = a.K, N = a.N, n_lo = block * R, run = l15 / R, i = l15 % R;
    const int n_b = n_lo + i < N ? n_lo + i : N - 1, m_a = i < M ? i : M - 1;

    // (the results' bias and offsets too: a load whose branch is not known here would be waited for, so what is not there is read from the gain and not used)
    const float* none = gain;
    const E b0 = *(a.bias ? (const E*)a.bias + n_b : (const E*)none), b1 = *(TWO && a.bias2 ? (const E*)a.bias2 + n_b : (const E*)none);
    const bool tabled = a.split_n > 0 && !a.y2_f32;
    int64_t off2[1 << LG];
#pragma unroll
    for (int q = 0; q < 1 << LG; ++q) off2[q] = *(tabled ? a.row_off2 + (q < M ? q : M - 1) : (const int64_t*)none);
    // ---- what the rows are made of: row r, columns c[k] .. + 3 of this thread
    const int lg = M <= 1 ? 0 : M <= 2 ? 1 : M <= 4 ? 2 : 3, r = wave >> (3 - lg), rm = r < M ? r : M - 1;
    int c[NC];
    bool on[NC];
    f4 gn[NC], v[NC], t[NC], pg[NC], h[KIND > MIX ? TERMS : 1][NC];
    float gt[NC][4];
    int last = 0;
    const E* row = nullptr;
    if constexpr (KIND == TABLE) {
        int id = n.ids[rm];
        id = id < 0 ? 0 : id >= n.vocab ? n.vocab - 1 : id;
        row = (const E*)n.table + (int64_t)id * W;
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const int col = 4 * ((tid & ((512 >> lg) - 1)) + k * (512 >> lg));
        on[k] = r < M && col < W;
        c[k] = col < W ? col : 0;
        gn[k] = *(const f4*)(gain + c[k]);
        v[k] = f4{0.f, 0.f, 0.f, 0.f};
        const int64_t at = (int64_t)rm * W + c[k];
        if constexpr (KIND == TABLE) {
            load4(row + c[k], true, 4, gt[k]);
        } else if constexpr (KIND > MIX) {
            last = n.n_terms < TERMS ? n.n_terms : TERMS;
            const int lead = n.n_terms - last;
            for (int j = 0; j < lead; ++j) v[k] += n.coef[j] * *(const f4*)(n.x + j * n.x_stride + at);
#pragma unroll
            for (int u = 0; u < TERMS; ++u)                          // (past the end the last one again, which is not counted)
                h[u][k] = *(const f4*)(n.x + (lead + (u < last ? u : last - 1)) * n.x_stride + at);
        } else {
            v[k] = *(const f4*)(n.x + at);
            t[k] = *(const f4*)(n.y + at);
            pg[k] = *(const f4*)(n.post_gain + c[k]);
            load4((const E*)n.gate + rm * n.ldg + c[k], true, 4, gt[k]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- this workgroup's weights (past the end the last k-step again, which is not counted)
    const int64_t w_at = n_b * a.ldw + piece_at<E>(run, group);
    // (of several runs of k they are read past the caches.  us, past / through them: weights from memory, bf16, 1 row, K = 1536, 1024 + 2048 gated columns 6.9 / 7.8, 5136
    // 7.8 / 8.6, fp32, K = 576, 1024 + 2048 gated 7.4 / 8.3; weights that have stayed in the 256 MB of the Infinity Cache 6.8 / 7.2, 7.8 / 7.9, 7.5 / 7.7)
    const int steps = W / (32 * PARTS);
    Frag<E> fb[U], fc[TWO ? U : 1];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int s = wave + u * SKW, k = 32 * PARTS * (s < steps ? s : steps - 1);
        fb[u] = weight_piece<PARTS, (PARTS > 1)>((const E*)a.w + w_at + k);
        if (TWO) fc[u] = weight_piece<PARTS, (PARTS > 1)>((const E*)a.w2 + w_at + k);
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- the residual and its norm
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
    } else if constexpr (KIND > MIX) {
#pragma unroll
        for (int u = 0; u < TERMS; ++u)
            if (u < last) {
                const float w = n.coef[n.n_terms - last + u];
#pragma unroll
                for (int k = 0; k < NC; ++k) v[k] += w * h[u][k];
            }
    } else {
#pragma unroll
        for (int k = 0; k < NC; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) t[k][e] *= gt[k][e];
        const float inv = scale_of(t, part[0]);
#pragma unroll
        for (int k = 0; k < NC; ++k) v[k] += t[k] * inv * pg[k];
    }
    const float inv = scale_of(v, part[1]);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const f4 o = v[k] * inv;
        if (on[k]) store4(rows + r * (W + PAD) + c[k], o[0] * gn[k][0], o[1] * gn[k][1], o[2] * gn[k][2], o[3] * gn[k][3]);
    }
    lds_barrier();
    // ---- the products
    Sum<E> sum, sum2;
    const E* xrow = rows + m_a * (W + PAD) + piece_at<E>(run, group);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int s = wave + u * SKW;
        if (s >= steps) break;                                       // (uniform over the wave)
        const Frag<E> fa = load_piece<PARTS>(xrow + 32 * PARTS * s);
        sum.add(fa, fb[u]);
        if (TWO) sum2.add(fa, fc[u]);
    }
    red[0][wave][lane] = sum.total();
    if (TWO) red[1][wave][lane] = sum2.total();
    if (keeps) {
#pragma unroll
        for (int k = 0; k < NC; ++k)
            if (on[k]) *(f4*)(n.x_out + (int64_t)r * W + c[k]) = v[k];
    }
    lds_barrier();
    if (wave != 0) return;
    const f4 acc = parts_total<PARTS>(red[0], lane), acc2 = TWO ? parts_total<PARTS>(red[TWO], lane) : f4{};
    const int m0 = 4 * group;                                        // (lane i of a group and run 0: rows m0 .. m0 + 3 of column n_b)
    if (m0 >= M || run != 0 || n_lo + i >= N) return;
    const float bv = a.bias ? to_f32(b0) : 0.0f, bv2 = TWO && a.bias2 ? to_f32(b1) : 0.0f;
    const bool second = a.split_n > 0 && n_b >= a.split_n, wide = second ? a.y2_f32 : a.out_f32;
    const int d = n_b - a.split_n;
    const int64_t col = !second ? n_b : a.y2_f32 ? d : (int64_t)(d / a.head_dim2) * a.head_stride2 + d % a.head_dim2;
    char* y = (char*)(second ? a.y2 : a.y);
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (m0 + q < M) {
            const int64_t off = NC > 1 && m0 ? off2[(4 + q) & ((1 << LG) - 1)] : off2[q];
            const int64_t to = col + (second ? a.y2_f32 ? (m0 + q) * a.head_stride2 : off : (m0 + q) * a.ldy);
            const float f = finished<E, EPI>(a, Place{}, n_b, acc[q], acc2[q], bv, bv2);
            if (wide)
                ((float*)y)[to] = f;
            else
                ((E*)y)[to] = from_f32<E>(f);
        }
}

// the first na workgroups are the first product's
template <typename E, int EPI, int PARTS, int U, int NC, int KIND>
__global__ __launch_bounds__(512) void norm_linear_kernel(pcb_row_norm_args n, pcb_linear_args a, pcb_linear_args b, int na) {
    __shared__ f4 red[EPI == PCB_EPI_SILU_MUL ? 2 : 1][8][64];
    __shared__ __attribute__((aligned(16))) E rows[NC * CHUNK + MAX_ROWS * PAD];
    __shared__ __attribute__((aligned(16))) float part[2][8];
    if ((int)blockIdx.x < na)
        normed_block<E, PCB_EPI_STORE, PARTS, U, NC, KIND>(n, n.gain, a, blockIdx.x, blockIdx.x == 0, rows, part, red);
    else
        normed_block<E, EPI, PARTS, U, NC, KIND>(n, n.gain2, b, blockIdx.x - na, false, rows, part, red);
}

// Which form takes a launch, and whether one launch is the better one.  us against the launches it stands for, weights from memory, by workgroups.
// Runs of k: bf16 one up to K = 1024, two beyond (1 row, K = 1024, 2592 columns behind a sublayer -1.8 / -1.2, 10272 -0.7 / +0.5); fp32 one up to K = 512, then two
// while that is no more than three workgroups a CU, of more than 2048 elements 192 (1 row, K = 1024, the streams' sum, 5376 columns one run +0.8, two -0.6, 10752
// -0.8 / 0.0; 4 rows 2688 columns -1.2 / -0.1, 1312 behind a sublayer -0.7 / -1.6).
// Taken up to `most` workgroups, each of which works out the rows again -- the more streams they are the sum of, the fewer.  us, launches apart / here, medians of 2060
// sizes (1 .. 8 rows, K = 64 .. 2048, 16 .. 12000 columns): one chunk a thread, a table up to 640 workgroups -0.3 .. -1.5; behind a sublayer, plain -1.0 .. -2.2, gated to
// 1280 -0.4 .. -5; two streams to 768 -0.1 .. -1.3; four bf16 to 512 -0.5 .. -1.3, 768 -0.1, fp32 256 -0.8, 512 +0.2; eight 256 -0.6 / -1.0, 512 +0.3 / +0.5, 768 +1.1 /
// +2.7; twelve bf16 256 -0.7, 640 +1.3, fp32 256 -0.4, 640 +2.6; 24 0.0 .. +5.6.  Two chunks: behind a sublayer -0.7 .. -1.9, four streams 256 -0.3 .. -1.3, eight bf16 192 -0.2,
// fp32 +0.0 .. +0.7, twelve 0.0 .. +0.9.  fp32 beyond K = 1024: more than two streams +0.3 .. +0.8.  Next to no k: 128 x 7200, 450 workgroups, two streams +0.8.  Slower
// than apart by more than 2 % at 61 of the 1418 that are taken (by the workgroups alone, whatever the rows are the sum of, at 403 of 2060, by up to 1.9).
struct Form {
    int parts, chunks;
    bool taken;
};
Form form(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b) {
    const int64_t elems = (int64_t)a.K << (a.M <= 1 ? 0 : a.M <= 2 ? 1 : a.M <= 4 ? 2 : 3);
    Form f{1, elems <= CHUNK && a.M <= 4 ? 1 : 2, false};
    if (a.M > MAX_ROWS || elems > (a.K <= 1024 ? 2 * CHUNK : CHUNK)) return f;
    const bool table = n.table, gated = b && b->epilogue == PCB_EPI_SILU_MUL;
    auto groups = [&](int parts) { return (int64_t)pcb_ceil_div(a.N, 16 / parts) + (b ? pcb_ceil_div(b->N, 16 / parts) : 0); };
    if (a.K > 1024 || (a.dtype == PCB_F32 && a.K > 512 && groups(2) <= (f.chunks == 1 ? 768 : 192))) f.parts = 2;
    const bool bf = a.dtype == PCB_BF16, one = f.chunks == 1;
    const int terms = n.n_terms, few = terms <= 12 ? 16 : 0;
    int most;
    if (table)
        most = one ? 768 : bf ? 384 : 256;
    else if (n.y)
        most = one ? (gated ? 1280 : 768) : gated ? 384 : 256;
    else if (!bf && a.K > 1024 && terms > 2)
        most = few;
    else if (one)
        most = terms <= 2 ? 768 : terms <= 4 ? (bf ? 512 : 256) : terms <= 8 || (bf && terms <= 12) ? 256 : few;
    else
        most = terms <= 4 ? 256 : bf && terms <= 8 ? 192 : few;
    if (a.K < 256 && most > (gated ? 768 : 320)) most = gated ? 768 : 320;
    f.taken = groups(f.parts) <= most;
    return f;
}

template <typename E>
int launch(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b, const Form& f, hipStream_t stream) {
    auto go = [&](auto epi, auto kind, auto parts, auto u, auto nc) {
        constexpr int P = decltype(parts)::value;
        const int na = pcb_ceil_div(a.N, 16 / P), nb = b ? pcb_ceil_div(b->N, 16 / P) : 0;
        hipLaunchKernelGGL((norm_linear_kernel<E, decltype(epi)::value, P, decltype(u)::value, decltype(nc)::value, decltype(kind)::value>), dim3(na + nb),
                           dim3(512), 0, stream, n, a, b ? *b : a, na);
        return pcb_check_launch("norm_linear_kernel");
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Four = std::integral_constant<int, 4>;
    auto sized = [&](auto epi, auto kind) {
        if (a.K > 1024) return go(epi, kind, Two{}, Four{}, One{});
        auto chunks = [&](auto parts, auto u) { return f.chunks == 1 ? go(epi, kind, parts, u, One{}) : go(epi, kind, parts, u, Two{}); };
        if constexpr (sizeof(E) == 4)
            if (f.parts == 2) return chunks(Two{}, Two{});
        return a.K > 512 ? chunks(One{}, Four{}) : chunks(One{}, Two{});
    };
    using Store = std::integral_constant<int, PCB_EPI_STORE>;
    if (n.table) return sized(Store{}, std::integral_constant<int, TABLE>{});
    if (!n.y)
        return n.n_terms <= 2   ? sized(Store{}, std::integral_constant<int, MIX + 2>{})
               : n.n_terms <= 4 ? sized(Store{}, std::integral_constant<int, MIX + 4>{})
                                : sized(Store{}, std::integral_constant<int, MIX + 8>{});
    using Post = std::integral_constant<int, POST>;
    return b && b->epilogue == PCB_EPI_SILU_MUL ? sized(std::integral_constant<int, PCB_EPI_SILU_MUL>{}, Post{}) : sized(Store{}, Post{});
}

}  // namespace

// Every workgroup works out the rows from what they are made of, and nothing orders workgroups: what the products store, and x_out, has to lie apart from that.
bool pcb_norm_linear_apart(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b, bool results) {
    const int64_t M = a.M, W = a.K;
    const pcb_span x_out = pcb_rows_span(n.x_out, M, W, W, 4);
    const pcb_span read[] = {n.table ? pcb_span{} : pcb_rows_span(n.x, 1, 0, (n.n_terms > 0 ? n.n_terms - 1 : 0) * n.x_stride + M * W, 4),
                             pcb_rows_span(n.y, M, W, W, 4), n.y ? pcb_rows_span(n.gate, M, n.ldg, W, a.dtype == PCB_BF16 ? 2 : 4) : pcb_span{}};
    for (const pcb_span& s : read) {
        if (!results && !pcb_apart(x_out, s)) return false;
        if (results && !(pcb_results_apart(a, s) && (!b || pcb_results_apart(*b, s)))) return false;
    }
    return !results || (pcb_results_apart(a, x_out) && (!b || pcb_results_apart(*b, x_out)));
}

// Whether what the rows are made of, and the products, can be read in pieces, and the results go where these kernels put them
bool pcb_norm_linear_pieces(const pcb_row_norm_args& n, const pcb_linear_args& a, const pcb_linear_args* b) {
    const uintptr_t e4 = a.dtype == PCB_BF16 ? 8 : 16;              // (four elements of E)
    auto takes = [](const pcb_linear_args& q) { return q.n_batch == 0 && !q.row_src && !q.row_dst && !q.row_gate && q.split_n3 <= 0 && pcb_linear_pieces(q); };
    return a.epilogue == PCB_EPI_STORE && takes(a) && a.K % 64 == 0 &&
           (!b || (takes(*b) && (b->epilogue == PCB_EPI_STORE || (b->epilogue == PCB_EPI_SILU_MUL && n.y)))) && n.x_stride % 4 == 0 && n.ldg % 4 == 0 &&
           ((uintptr_t)n.x | (uintptr_t)n.y | (uintptr_t)n.post_gain | (uintptr_t)n.gain | (uintptr_t)n.gain2 | (uintptr_t)n.x_out) % 16 == 0 &&
           ((uintptr_t)n.gate | (uintptr_t)n.table) % e4 == 0;
}

int pcb_norm_linear_check(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b) {
    int rc = pcb_linear_check(a);
    if (rc == PCB_OK && b) rc = pcb_linear_check(b);
    if (rc != PCB_OK) return rc;
    PCB_REQUIRE(n && n->struct_bytes == sizeof(pcb_row_norm_args), PCB_ERR_ARG, "pcb_norm_linear: struct size mismatch");
    PCB_REQUIRE(n->x_out && n->gain && (!b || n->gain2) && (n->table ? n->ids && n->vocab > 0 && !n->y : n->x && n->x != n->x_out) &&
                    (n->table || n->y ? n->n_terms == 0 : n->n_terms > 0 && n->coef) && (!n->y || (n->gate && n->post_gain && n->ldg >= a->K)),
                PCB_ERR_ARG, "pcb_norm_linear: rows of a table, a sum of streams, or a residual and a gated sublayer's result; x_out is neither's");
    PCB_REQUIRE(!b || (a->dtype == b->dtype && a->M == b->M && a->K == b->K), PCB_ERR_ARG, "pcb_norm_linear: products of the same rows");
    PCB_REQUIRE(pcb_norm_linear_apart(*n, *a, b, false), PCB_ERR_ARG, "pcb_norm_linear: x_out overlaps the rows that are read");
    return PCB_OK;
}

static int norm_linear_route(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b, Form* f) {
    const int rc = pcb_norm_linear_check(n, a, b);
    if (rc != PCB_OK) return rc;
    *f = form(*n, *a, b);
    return f->taken && pcb_norm_linear_pieces(*n, *a, b) && pcb_norm_linear_apart(*n, *a, b, true) ? PCB_OK : PCB_NOT_TAKEN;
}

PCB_EXPORT int pcb_norm_linear_takes(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b) {
    Form f;
    return norm_linear_route(n, a, b, &f);
}

PCB_EXPORT int pcb_norm_linear(const pcb_row_norm_args* n, const pcb_linear_args* a, const pcb_linear_args* b, void* stream) {
    Form f;
    const int rc = norm_linear_route(n, a, b, &f);
    if (rc < 0 || a->M == 0) return rc < 0 ? rc : PCB_OK;
    if (rc != PCB_OK) return rc;
    return a->dtype == PCB_BF16 ? launch<bf16_t>(*n, *a, b, f, (hipStream_t)stream) : launch<float>(*n, *a, b, f, (hipStream_t)stream);
}
