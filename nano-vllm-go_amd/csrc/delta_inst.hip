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
// Workgroups that the chip holds at once, by their LDS (160 KB a CU, 256 CUs) and by what a CU's registers hold of them; each goes from chunk to chunk.  Heads of 256 have one a CU:
// launched for two, they made two rounds, us a layer 1 x 1900 tokens 98 -> 94, 5 x 300 .. 1900 215 -> 204, 200 x 128 channels, 10 x 400 175 -> 169
template <int NK> constexpr int delta_prep_workgroups() { return 256 * std::min(160 * 1024 / delta_prep_lds_bytes<NK>(), 2); }
static_assert(delta_prep_workgroups<8>() == 512 && delta_prep_workgroups<16>() == 256, "two workgroups a CU, heads of 256 one");
template <int NK, bool VEC, bool VECV>
static void prep_as(hipStream_t st, const DeltaArgs& p, int n_seqs, int tokens) {
    constexpr int lds = delta_prep_lds_bytes<NK>();
    NVL_LDS_ATTR((delta_prep_kernel<NK, VEC, VECV>), lds);
    const int chunks = tokens / DELTA_C + n_seqs, per = delta_prep_workgroups<NK>();          // chunks: at most
    hipLaunchKernelGGL((delta_prep_kernel<NK, VEC, VECV>), dim3(p.H, std::min(chunks, std::max(1, per / p.H))), dim3(512), lds, st, p, n_seqs);
}
template <int NK>
static void prep(hipStream_t st, const DeltaArgs& p, int n_seqs, int tokens) {
    if (p.vec4) { if (p.vec4v) prep_as<NK, true, true>(st, p, n_seqs, tokens); else prep_as<NK, true, false>(st, p, n_seqs, tokens); }
    else if (p.vec4v) prep_as<NK, false, true>(st, p, n_seqs, tokens); else prep_as<NK, false, false>(st, p, n_seqs, tokens);
}
void delta_prep_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, int nk, int tokens) {
    if (nk == 2) prep<2>(st, p, n_seqs, tokens); else if (nk == 4) prep<4>(st, p, n_seqs, tokens); else if (nk == 8) prep<8>(st, p, n_seqs, tokens); else prep<16>(st, p, n_seqs, tokens);
}
template <int NK>
static void scan(hipStream_t st, const DeltaArgs& p, int n_seqs) {
    constexpr int lds = delta_scan_lds_bytes<NK>();
    NVL_LDS_ATTR((delta_scan_kernel<NK>), lds);
    hipLaunchKernelGGL((delta_scan_kernel<NK>), dim3(p.H, cdiv(p.DV, 16 * DELTA_SCAN_WAVES), n_seqs), dim3(DELTA_SCAN_WAVES * 64), lds, st, p);
}
template <int NK, int KSP>
static void scan_parts(hipStream_t st, const DeltaArgs& p, int n_seqs) {
    hipLaunchKernelGGL((delta_scan_parts_kernel<NK, KSP>), dim3(p.H, cdiv(p.DV, 16), n_seqs), dim3(KSP * 64), 0, st, p);
}
// All key channels a wave (64 columns a workgroup, operands shared through LDS), or the channels over the KSP waves of a workgroup of 16 columns: a chunk's step is three
// times as short, and each costs an exchange and its operands four reads from L2.  us: the longest sequence's chain, all chunks at the chip's rate, the larger of them and
// 0.4 of the other; fitted to 1 .. 64 sequences of 100 .. 1900 tokens x 2048 columns of heads of 64, 128 and 256, good to 20 %.
// Heads of 128, whole / parts, us a layer: 1 x 1900 220 / 72; 4 x 900 119 / 71; 8 x 900 145 / 153; 12 x 900 222 / 214; 16 x 900 242 / 280; 32 x 512 272 / 310; 64 x 200 246 / 315;
// 5 x 300..1900 244 / 115; 10 x 100..900 135 / 92; 12 x 300..1900 312 / 235.  Heads of 64: 1 x 1900 135 / 64, 4 x 900 79 / 56, 16 x 900 180 / 227; of 256: 432 / 119, 225 / 137, 495 / 579.
struct ScanCost { double start, step, chunk; };          // of the chain: before the first chunk, a chunk; of all: a chunk of 32 columns' worth of a head
static double scan_cost(const DeltaArgs& p, int n_seqs, const ScanCost& k, int max_len, int tokens) {
    const double chain = k.start + k.step * cdiv(max_len, DELTA_C);
    const double all = k.chunk * p.H * cdiv(p.DV, 64) / 2.0 * ((double)tokens / DELTA_C + n_seqs);
    return std::max(chain, all) + 0.4 * std::min(chain, all);
}
template <int NK, int KSP>
static void scan_shape(hipStream_t st, const DeltaArgs& p, int n_seqs, int max_len, int tokens) {
    constexpr double size = NK / 8.0;
    const ScanCost whole{8.0, 0.4 + 3.3 * size, 0.008 + 0.023 * size};
    const ScanCost parts = KSP == 2 ? ScanCost{5.0, 1.0, 0.029} : KSP == 4 ? ScanCost{5.0, 1.1, 0.036} : ScanCost{8.0, 1.85, 0.075};
    if (scan_cost(p, n_seqs, parts, max_len, tokens) < scan_cost(p, n_seqs, whole, max_len, tokens)) scan_parts<NK, KSP>(st, p, n_seqs);
    else scan<NK>(st, p, n_seqs);
}
void delta_scan_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, int nk, int max_len, int tokens) {
    if (nk == 2) scan<2>(st, p, n_seqs);
    else if (nk == 4) scan_shape<4, 2>(st, p, n_seqs, max_len, tokens);
    else if (nk == 8) scan_shape<8, 4>(st, p, n_seqs, max_len, tokens);
    else scan_shape<16, 8>(st, p, n_seqs, max_len, tokens);
}
}  // namespace nvl
