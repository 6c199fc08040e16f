// The launches of the many-row ring kernel (pc_attn_ring_dev.h).
#include "pc_attn_ring_dev.h"

namespace pca {
namespace {

template <bool KVLO, bool PRE, bool GATHER = false>
__global__ __launch_bounds__(kRingThreads) void attn_ring_kernel(const AttnParams p) {
    __shared__ __attribute__((aligned(16))) char lds[2 * kStage];
    __shared__ __attribute__((aligned(16))) char gtab[GATHER ? kRingThreads * 64 : 16];
    attn_ring_body<KVLO, PRE, GATHER>(p, lds, gtab, RingGrid{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, p.nqblk, p.nbatch, p.xcd_remap, 0});
}

}  // namespace

// Launches the ring kernel takes: head_dim 128, split-precision Q (q_lo), more than 32 query rows, no ALiBi, not the tail /
// small-q modes.  PC_ATTN_NO_RING=1: off (A/B against attn_fwd_kernel).
// fewest query rows the ring kernel takes (PC_ATTN_RING_MIN; pc_attn_workspace_bytes sizes the split-KV workspace with the same number)
int ring_min_rows() {
    static const int min_rows = [] { const char* m = getenv("PC_ATTN_RING_MIN"); return m ? atoi(m) : 33; }();
    return min_rows;
}
bool ring_eligible(const AttnParams& p, int D) {
    const char* e = getenv("PC_ATTN_NO_RING");            // (read per call: tests and probes switch it inside one process)
    const bool off = e && e[0] == '1';
    return !off && D == RD && p.q_lo && p.q_len >= ring_min_rows() && !p.key_pos && !p.tail && !p.small;
}

// KV splits of a ring launch: one workgroup per CU; minimise rounds x (stages per split + 1) + the merge
int ring_nsplit(int B, int H, int q_len, int kv_len) {
    const int units = B * H * pc_ceil_div(q_len, kRingQB);
    if (units >= 256) return 1;             // the grid fills the chip by itself: splits only add partials to merge
    // (rounds 3-4 kept >= 4 stages per split; for 33..128 rows over a 1.7 k cache that left half of the CUs idle: 7b q = 36 / 50 /
    // 66 / 102: 5.10 / 5.41 / 6.05 / 6.65 -> 4.91 / 5.27 / 5.85 / 6.48 ms without the floor, profiles/r04_variants.txt)
    static const int min_stages = [] { const char* e = getenv("PC_RING_MIN_STAGES"); return e ? atoi(e) : 1; }();
    // (Round 5 tried pricing a THIN last q-block -- 259 = 128 + 128 + 3 rows: seven of its eight waves only help
    // with the DMA -- at a third of a full block so that 259 rows take the 3 splits 256 rows take: 360 workgroups instead of 240,
    // the attention launch 155 -> 202 us and the step 21.3 -> 22.8 ms on one box (profiles/r05_variants.txt): the second round of
    // workgroups costs more than the shorter key ranges save.  The count below stands.)
    int best = 1;
    double best_cost = 1e30;
    for (int s = 1; s <= 16; ++s) {
        const int stages = pc_ceil_div(pc_ceil_div(kv_len, s), 2 * kTK);
        if (s > 1 && stages < min_stages) break;
        const int rounds = pc_ceil_div(units * s, 256);
        const double cost = rounds * (stages + 1.0) + (s > 1 ? 2.0 + 0.25 * s : 0.0);
        if (cost < best_cost - 1e-9) { best_cost = cost; best = s; }
    }
    return best;
}

int launch_attn_ring(const AttnParams& p0, int B, hipStream_t stream) {
    AttnParams p = p0;
    static const bool no_remap = [] { const char* e = getenv("PC_ATTN_NO_XCD"); return e && e[0] == '1'; }();
    p.nqblk = pc_ceil_div(p.q_len, kRingQB);
    p.nbatch = B;
    p.xcd_remap = (p.nqblk >= 2 && !no_remap) ? 1 : 0;
    dim3 grid(p.nqblk, p.H, B * p.nsplit);
    if (p.xcd_remap) grid = dim3(8 * p.nqblk * ((p.H * B * p.nsplit + 7) / 8), 1, 1);
    const dim3 block(kRingThreads);
    if (p.pre_k) {
        if (p.k_lo) hipLaunchKernelGGL((attn_ring_kernel<true, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((attn_ring_kernel<false, true>), grid, block, 0, stream, p);
    } else if (p.rows) {         // stage while reading (pc_attn gather_rows)
        if (p.k_lo) hipLaunchKernelGGL((attn_ring_kernel<true, false, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((attn_ring_kernel<false, false, true>), grid, block, 0, stream, p);
    } else if (p.k_lo) hipLaunchKernelGGL((attn_ring_kernel<true, false>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((attn_ring_kernel<false, false>), grid, block, 0, stream, p);
    return pc_check_launch("attn_ring_kernel");
}

}  // namespace pca
