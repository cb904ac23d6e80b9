// delta_inst.hip — the instances of the channel-wise delta rule's kernels (delta.h) and their launches.
#include <algorithm>
#include "delta.h"

namespace nvl {
template <bool FUSED, int ROWS, typename ActT>
static void step(hipStream_t st, const DeltaArgs& p, dim3 grid, int lds) {
    NVL_LDS_ATTR((delta_step_kernel<FUSED, ROWS, ActT>), 128 * 1024);
    hipLaunchKernelGGL((delta_step_kernel<FUSED, ROWS, ActT>), grid, dim3(LR_STEP_THREADS), lds, st, p);
}
template <bool FUSED, typename ActT>
static void step_rows(hipStream_t st, const DeltaArgs& p, int n_seqs) {
    const int lds = delta_step_lds_bytes(p.DK, p.DVp, FUSED ? p.a_rkp + p.g_rkp : 0);
    const dim3 grid(p.H, n_seqs);
    int tv = 1;
    while (tv < p.DVp / 4) tv <<= 1;
    const int rows = cdiv(p.DK, LR_STEP_THREADS / tv);        // state rows per thread
    if (rows <= 4) step<FUSED, 4, ActT>(st, p, grid, lds); else if (rows <= 8) step<FUSED, 8, ActT>(st, p, grid, lds); else step<FUSED, 16, ActT>(st, p, grid, lds);
    NVL_HIP(hipGetLastError());
}
void delta_step_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, bool fused, bool f32) {
    if (!fused) step_rows<false, float>(st, p, n_seqs);
    else if (f32) step_rows<true, float>(st, p, n_seqs);
    else step_rows<true, bf16_t>(st, p, n_seqs);
}
template <int NK>
static void prep(hipStream_t st, const DeltaArgs& p, dim3 grid) {
    constexpr int lds = delta_prep_lds_bytes<NK>();
    NVL_LDS_ATTR((delta_prep_kernel<NK>), lds);
    hipLaunchKernelGGL((delta_prep_kernel<NK>), grid, dim3(512), lds, st, p);
}
void delta_prep_launch(hipStream_t st, const DeltaArgs& p, dim3 grid, int nk) {
    if (nk == 2) prep<2>(st, p, grid); else if (nk == 4) prep<4>(st, p, grid); else if (nk == 8) prep<8>(st, p, grid); else prep<16>(st, p, grid);
}
template <int NK, int KSP>
static void scan(hipStream_t st, const DeltaArgs& p, int n_seqs) {
    constexpr int lds = delta_scan_lds_bytes<NK, KSP>();
    NVL_LDS_ATTR((delta_scan_kernel<NK, KSP>), lds);
    hipLaunchKernelGGL((delta_scan_kernel<NK, KSP>), dim3(p.H, cdiv(p.DV, 16 * DELTA_SCAN_WAVES / KSP), n_seqs), dim3(DELTA_SCAN_WAVES * 64), lds, st, p);
}
// Parts of the key channels (KSP): more parts shorten the chain of a sequence's chunks, whose fp32 products bound a wave, and cost each of them an exchange.
// us, fitted to 1 .. 64 sequences of 100 .. 1900 tokens x 16 heads of 128, good to 20 %: the longest sequence's chain, all chunks at the chip's rate, the larger of them
// and a quarter of the other.  Sequences of several lengths, longest first, fill the chip's gaps with the short ones; of one length they end together.
// One / two / four parts, ms a prompt: 1 x 1900 6.5 / 5.9 / 5.6; 5 x 300..1900 12.5 / 11.9 / 11.7; 12 x 300..1900 22.9 / 22.3 / 23.0; 10 x 100..900 10.0 / 9.7 / 9.9; 16 x 900 25.6 / 26.2 / 27.4.
static double scan_cost(const DeltaArgs& p, int n_seqs, int nk, int ksp, int max_len, int tokens) {
    const double size = nk / 8.0, heads = p.H * cdiv(p.DV, 64) / 2.0;
    const double chain = cdiv(max_len, DELTA_C) * (1.95 + size * 2.55 / ksp);
    const double ragged = n_seqs <= DELTA_ORDERED ? 0.4 + 0.6 * tokens / ((double)n_seqs * max_len) : 1.0;
    const double all = heads * ((double)tokens / DELTA_C + 0.5 * n_seqs) * (size * 0.0225 + 0.0105 * ksp) * ragged;
    return std::max(chain, all) + 0.25 * std::min(chain, all);
}
template <int NK, int... PARTS>
static void scan_shape(hipStream_t st, const DeltaArgs& p, int n_seqs, int max_len, int tokens) {
    int best = 1;
    double t = scan_cost(p, n_seqs, NK, 1, max_len, tokens);
    auto consider = [&](int ksp) { const double c = scan_cost(p, n_seqs, NK, ksp, max_len, tokens); if (c < 0.95 * t) { t = c; best = ksp; } };
    (consider(PARTS), ...);
    if (best == 1) { scan<NK, 1>(st, p, n_seqs); return; }
    ((best == PARTS ? scan<NK, PARTS>(st, p, n_seqs) : void()), ...);
}
void delta_scan_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, int nk, int max_len, int tokens) {
    if (nk == 2) scan<2, 1>(st, p, n_seqs);
    else if (nk == 4) scan_shape<4, 2>(st, p, n_seqs, max_len, tokens);
    else if (nk == 8) scan_shape<8, 2, 4>(st, p, n_seqs, max_len, tokens);
    else scan_shape<16, 2, 4>(st, p, n_seqs, max_len, tokens);
}
}  // namespace nvl
