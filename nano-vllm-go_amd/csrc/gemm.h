// gemm.h — projection GEMMs of the forward path (replaces tensor.MatMul,
// purego/tensor/tensor.go:62-88, at every call site of the layer stack).
//
//   C[M,N] = A[M,K] · W[N,K]^T   (+ fused epilogue)
//
// bf16 path (NVL_PRECISION_BF16).  Both operands live in HBM in the fragment-major layout of
// common.h (fm_index): 16-row x 32-k MFMA operand blocks, 1 KiB contiguous each.  The reference
// keeps weights [in,out] fp32 (generic_loader.go:398-403); nvl_upload_tensor converts once at load,
// and every kernel that produces a GEMM input (norm, attention, SwiGLU/GELU epilogue) writes it
// directly in this layout.
//   * gemm_bf16_pp_kernel (prefill, >= 192 tiles of 256x256): the ping-pong form — two groups of four waves one phase
//     apart, K in 32-wide stages through a 4-slot LDS ring filled by global_load_lds_dwordx4, so one group's fragment
//     reads run beside the other's MFMAs.  MFMA-bound.  Also the grouped launch of the MoE prefill (GemmArgs::tile_map:
//     an m-tile = an expert's 256-row segment of the expert-ordered row buffer).
//   * gemm_bf16_kernel (prefill, fewer tiles; decode-sized MoE expert groups): by default 128x128 tiles with 4 waves
//     (2x2), each wave a 64x64 sub-tile as 4x4 v_mfma_f32_16x16x32_bf16 accumulators; operand blocks go HBM->LDS with
//     global_load_lds_dwordx4 (one contiguous KiB per wave-instruction, no VGPR round trip), a ring of four K tiles of 32; the LDS
//     image is lane-linear so the fragment ds_read_b128s are bank-conflict-free with no swizzle.
//   * gemm_skinny_bf16_kernel / gemm_skinny_wide_bf16_kernel (decode, M <= 64): weight-streaming, HBM-bound (see below);
//     the residual projections also carry the deferred RMSNorm (GemmArgs::rs_out / rs_in); their MOE instantiations run
//     a decode MoE block as two dense projections over all experts with the routing weights as a mask (GemmArgs::moe_gate).
// The MFMA is issued "swapped" (weights as the A operand) so each lane ends up with 4 consecutive N
// elements of one output row: 8/16-byte epilogue accesses, and the bf16 epilogues can write the
// next GEMM's fragment-major operand directly.
//
// f32 path (NVL_PRECISION_F32): plain LDS-tiled fp32 FMA kernel on row-major operands, k ascending —
// the tight-tolerance parity mode, not a performance path.
#pragma once
#include <stdexcept>
#include <algorithm>
#include <cmath>
#include <type_traits>
#include "common.h"

namespace nvl {

enum GemmEpi {
    EPI_STORE = 0,   // C = acc (+bias)
    EPI_RESID = 1,   // X += alpha * (acc (+bias))      X fp32, in place   (generic_model.go:320-326)
    EPI_SWIGLU = 2,  // C[m, f] = silu(gate) * up        W rows interleaved (transformer.go:50-66)
    EPI_GELU = 3,    // C = gelu_tanh(acc + bias)                           (transformer.go:67-78)
    EPI_QKV = 4,     // fused QKV projection epilogue (head_dim 64 / 128): bias, RoPE on Q and K (rope.go:153-205),
                     // Q -> q buffer, K and V -> their KV slabs [pos][hd]  (replaces the fp32 qkv
                     // round trip + rope_kv_kernel in prefill; Concatenate tensor.go:283-321)
    EPI_CLAMP_GLU = 6,   // C[m, f] = g sigmoid(slope g) (u + 1), g = min(gate, limit), u = clamp(up, -limit, limit); W as for EPI_SWIGLU
    EPI_GEGLU = 5,   // C[m, f] = gelu_tanh(gate) * up   W rows interleaved as for EPI_SWIGLU
    EPI_RELU2 = 7,   // C = max(acc, 0)^2
    EPI_GROUPED = 9,     // fused input projection of grouped-query attention (grouped.h): every column range goes where it is used, GroupedEpi
    EPI_GROUPED_RAW = 11,    // ... of attention whose queries and keys are normed or rotated first: those go to fp32 rows, as does what lies behind the gate
    EPI_REGLU = 10,      // C[m, f] = max(gate, 0) * up   W rows interleaved as for EPI_SWIGLU
    EPI_GELU_TOK = 8,    // C[m, n] = gelu_tanh(acc) * tok_table[tok_ids[m]][n]   (an input of the token's own, GemmArgs::tok_*)
    // ... with a deferred layer norm (GemmArgs::ln_s): decode kernels alone
    EPI_LN_STORE = 12, EPI_LN_RESID = 13, EPI_LN_GELU = 14, EPI_LN_QKV = 15,
    EPI_JOINT = 16,      // two projections of one operand: the first joint.n columns are stored to fp32 rows, the others C = gelu_tanh(acc + bias)
};
constexpr bool epi_ln(int epi) { return epi >= 12 && epi <= 15; }
// most waves of a workgroup of the narrow decode form (the pairs of a layer norm take registers, and the routing beside several row tiles)
constexpr int skinny_waves(int epi, bool route_rows = false) { return epi_ln(epi) || route_rows ? 8 : 16; }
constexpr int epi_base(int epi) { return !epi_ln(epi) ? epi : epi == 15 ? 4 : epi == 14 ? 3 : epi - 12; }

constexpr bool epi_moe(int epi) { return epi == 2 || epi == 6; }      // ... with instances for masked experts
constexpr bool epi_glu(int epi) { return epi == 2 || epi == 5 || epi == 6 || epi == 10; }      // gate | up pairs in, one column out

struct QkvEpi {             // EPI_QKV only
    const int32_t* tok_pos;
    const int32_t* tok_tbl;     // per token: where its sequence's block table starts in blk_table
    const int32_t* blk_table;   // KV block ids (slab mode: the slot); Tmax tokens per block
    const float* cos_t;     // [max_seq][64] or NULL (no RoPE)
    const float* sin_t;
    bf16_t* q_out;          // [tokens][nH*64] row-major
    bf16_t* kcache;         // layer base
    bf16_t* vcache;
    int64_t slot_stride;
    int Tmax, nH, nKV, hd;
};

struct GroupedEpi {         // EPI_GROUPED: columns [q | k | v | gate | feed-forward | router], each range ending at a multiple of 32 (all but the last)
    int k0, v0, gate0, ffn0, route0;
    // q and gate -> C, side by side (ldc columns, fragment-major); keys and values -> their cache rows
    const int32_t *tok_pos, *tok_tbl, *blk_table;
    bf16_t* cache; int64_t block_stride; int bs, G, dp, vp;        // this layer's part of block 0 (grouped.h)
    int mix; const float* lambda; float* vfirst; int64_t vfirst_ld;
    bf16_t* ffn; int64_t ffn_ld;                                   // [ffn0, route0): max(., 0)^2 -> the output projection's operand (fragment-major, shifted to its columns)
    float* route; int64_t route_ld;                                // from route0 on: fp32 rows
    // EPI_GROUPED_RAW: queries and keys, and everything from raw0 on, to fp32 rows at their own columns; [raw0, silu1): through silu
    float* raw; int64_t raw_ld; int raw0, silu1;
};

// MoE decode, experts' up projection: routing by the launch's first `wgs` workgroups (set by the launcher), `rows` rows each
struct RouteJob {
    const bf16_t* W;        // router, fragment-major [E][K], or NULL: no routing in this launch
    const float* bias;      // [E] or NULL
    float *gate, *logits;   // [rows][gate_ld]; logits [rows][logits_ld] or NULL
    int E, top_k, gate_ld, logits_ld, n_always;      // columns E .. E + n_always - 1 of the gate are one (experts every token takes), those up to gate_ld zero
    int wgs, rows;
};

struct JointEpi { float* rows; int ld, n; };      // EPI_JOINT; n a multiple of 16

// what a residual projection adds to a row's mean.  w: the mean of W's rows, in bf16 and the rest of it in bf16, [K/32][those two][32] and three K steps that nothing uses; b: the mean of the bias
struct MeanShift { const bf16_t* w; float b; };
struct LnResidEpi { MeanShift added; const float *prev, *mean_in; float* mean_out; };      // EPI_LN_RESID (GemmArgs::ln_s)

struct GemmArgs {
    const void* A;          // bf16: fragment-major [M_pad16][K]; f32: row-major [M][lda]
    int lda;
    const int32_t* a_rows;  // optional gather: logical row r reads A row a_rows[r] (MoE), else NULL
    const void* W;          // bf16: fragment-major [N_pad128][K]; f32: row-major [N_pad128][K]
    void* C;                // fp32 outputs row-major [.][ldc]; bf16 outputs fragment-major [.][ldc]
    int ldc;
    const float* bias;      // [N] or NULL
    float alpha;            // EPI_RESID multiplier
    float glu_limit, glu_slope;     // EPI_CLAMP_GLU
    float glu_limit2; int glu_from2;      // ... masked experts: the limit of output columns from glu_from2 on
    const int32_t* tok_ids; int64_t tok_ld;      // EPI_GELU_TOK: row-major, rows of 4 k entries
    union {
        const bf16_t* tok_table;
        const float* ln_s;      // epi_ln: S of the deferred layer norm, which the last comment here explains
    };
    int M, N, K;            // logical sizes
    const int32_t* seg;     // optional device {start,end}: rows [start,end) of A (via a_rows if set)
                            // and of C; M is then only the grid bound (MoE expert segments)
    int c_row0;             // row offset added to every output row (set from seg inside the kernel)
    // grouped (MoE) launch: m-tile i of the grid is rows [row0, row0+nrows) of expert e, from the device table
    // tile_map[i] = {e, row0, nrows, 0}; blocks with i >= *n_mtiles exit; expert e's weights start at
    // W + e * w_expert_stride.  One launch covers every expert (moe.go:99-120 loops experts per token).
    const int32_t* tile_map;
    const int32_t* n_mtiles;
    int64_t w_expert_stride;
    int x_mask;             // decode kernels: rows >= M of a 16-row activation tile are not fetched (set when M % 16 != 0)
    int grp_bm;             // rows per m-tile of the grouped launch (128, or 256: the 256x128 three-stage instance)
    union {
        QkvEpi qkv;         // EPI_QKV
        RouteJob route;     // masked experts (epi_moe with moe_gate)
        JointEpi joint;     // EPI_JOINT
        LnResidEpi ln;      // EPI_LN_RESID
    };
    GroupedEpi grp;         // EPI_GROUPED
    // decode kernel, EPI_RESID only: K split over gridDim.y = sk_slices workgroups per column block.  Each
    // writes its fp32 partial tile to sk_part[slice][m][n] (ld = N) with plain stores; the NEXT kernel in the
    // stream — the norm that follows every residual add — folds x += alpha * sum(slices) into its read of x.
    // The kernel boundary is the synchronisation: no fences, no atomics, fixed summation order.
    float* sk_part;
    int sk_slices;
    // K split inside a launch: partial tiles and, zero between launches, the tiles' arrival counters (split_finish); NULL: no such split
    float* split_ws;
    int* split_cnt;
    int splits;             // workgroups per tile (set by the launcher)
    // Deferred RMSNorm (decode; RMSNorm + SwiGLU, sequential block): the residual projection that completes x also
    // emits the NEXT projection's operand un-normalised, xn_raw = bf16(x * w_norm) (fragment-major), plus the sums of
    // x^2 over its 16 columns, rs_out[tile][m]; the consumer scales its accumulators by
    // rstd[m] = 1 / sqrt(sum_tiles(rs_in[tile][m]) / H + eps) — (x*w/rms)·W == (1/rms)·((x*w)·W).  The norm launch
    // between the two projections disappears; all sums keep a fixed order.
    int m_split;            // narrow decode kernel: gridDim.y indexes 16-row activation tiles (not K slices): the
                            // workgroups of a weight tile stream the same weights (one XCD: L2 serves the second)
    int m_passes;           // decode kernels, 64 < M: the launch covers m_passes = ceil(M/64) groups of 64 activation rows;
                            // the workgroups of one weight tile sit 8 block ids apart — same XCD, dispatched together —
                            // so the weights cross HBM once and the later groups hit L2 (see launch_gemm_bf16)
    int grid_y;             // decode kernels: gridDim.y of the launch (set by the launcher)
    unsigned long long* stamps;   // diagnostic runs: per-workgroup time stamps (common.h nvl_stamp), else NULL
    int rs_half;            // producer, M <= 16: 8 weight rows per workgroup, x^2 partials per 8 columns (rs_tiles = N / 8)
    const float* nrm_w;     // producer: weight of the norm that follows, [N]
    bf16_t* nrm_xn;         // producer: xn_raw [M_pad16][N] fragment-major
    float* rs_out;          // producer: [64 rows][N/16]
    const float* rs_in;     // consumer: the same buffer
    int rs_tiles;
    float rs_inv_h, rs_eps;
    int split_units;        // size of split_ws in SPLIT_UNITs (for the launchers)
    // MoE decode, "dense-masked" form (decode kernels only, M <= 64).  All experts are ONE projection each way:
    //   up   W = [E * 2I][H] (the experts' interleaved gate|up rows back to back), output column f belongs to expert f / I;
    //   down W = [H][E * I] (the experts concatenated along K), a wave's K range lies inside ONE expert.
    // moe_gate [M][E] holds the renormalised routing weight of (token, expert), 0 when the token did not pick the expert.
    // A workgroup (up) / wave (down) whose expert no token of the batch picked returns before it loads a weight byte, so
    // only the touched experts are streamed; the down projection's waves multiply their sums, one expert each, by moe_gate[m][e],
    // which makes its K reduction the weighted combine itself (moe.go:105-120) — no sort, no plan, no combine launch.
    // Where a batch is expected to pick nearly all experts the up projection streams them all and needs no routing: its first
    // workgroups then do the routing (route) beside it.
    const float* moe_gate;
    int moe_E, moe_I;
    // Deferred layer norm (epi_ln; M <= 64): ((x - mean) w / sd + b) W == rstd ((x - s) w W - (mean - s) S) + B for any s, S[n] = sum_k W[n][k] w[k] and
    // B[n] = bias[n] + sum_k W[n][k] b[k] from the weights alone.  Producer: xn_raw = bf16((x - s) w) and per tile the pair of sums of x - s and
    // (x - s)^2.  The operand's rounding and the variance cost sqrt(1 + d^2) times a norm launch's where s misses the row's mean by d of its deviations, so s is
    // that mean but for rounding: the mean before (ln.prev: the pairs of the norm before, or NULL, where it was a launch of its own, and ln.mean_in) and what
    // the projection adds to it, its operand times ln.added (one more product a K step; a mean that is 100 deviations away: d < 0.01).  Consumer: bias is B.
    // A norm launch is 3.3 us (1 row) to 4.2 (16) and a boundary; the sums cost the four projections of a layer 0.5 to 1.7 us each, finding s
    // the two residual ones 0.2 to 0.45 (GPT-2, a step of 1 sequence: with the mean before in its place 357 us, 361 so; 11 prompt tokens 6.2 -> 6.6 us a projection).  GPT-2, norm launches -> carried, us a step of
    // 1 / 16 / 24 / 40 / 64 sequences: 387 -> 361, 444 -> 427, 494 -> 463, 517 -> 490, 584 -> 562; prompts of 11 / 3 x 11 / 64 tokens 498 -> 461, 583 -> 537, 574 -> 550.
    // Error of the logits against 64 bits over 240 calls: mean log ratio to the norm launches -0.002 +- 0.002.
};
// blockDim lies 12 bytes behind the arguments.  The decode kernels load it with rs_in: a cache line more is 0.2 us of a 3.4 us launch (8 rows of 2048 x 1024)
static_assert(((sizeof(GemmArgs) + 12) >> 6) == (offsetof(GemmArgs, rs_in) >> 6), "arguments that are loaded together");
// the routing weight that row `lane` of the batch (M <= 64) gives expert e
__device__ __forceinline__ float moe_gate_of(const GemmArgs& p, int e) {
    const int lane = threadIdx.x & 63;
    return lane < p.M ? p.moe_gate[lane * p.moe_E + e] : 0.f;
}

// four columns n .. n + 3 of token `row`, inside one column range
__device__ __forceinline__ void epilogue_grouped4(const GemmArgs& p, int64_t row, int n, f32x4 v) {
    const GroupedEpi& e = p.grp;
    if (n < e.k0) { act_store4<bf16_t>((bf16_t*)p.C, row, n, p.ldc, v); return; }
    if (n >= e.route0) {
        float* c = e.route + row * e.route_ld + (n - e.route0);
        if (n + 3 < p.N) { *(f32x4*)c = v; return; }      // (rows of 4 k floats)
#pragma unroll
        for (int r = 0; r < 4; r++) if (n + r < p.N) c[r] = v[r];
        return;
    }
    if (n >= e.ffn0) {
#pragma unroll
        for (int r = 0; r < 4; r++) { const float t = fmaxf(v[r], 0.f); v[r] = t * t; }
        act_store4<bf16_t>(e.ffn, row, n - e.ffn0, e.ffn_ld, v);
        return;
    }
    if (n >= e.gate0) { act_store4<bf16_t>((bf16_t*)p.C, row, e.k0 + n - e.gate0, p.ldc, v); return; }
    int blk, crow;
    kv_locate(e.blk_table, e.tok_tbl[row], e.tok_pos[row], e.bs, blk, crow);
    bf16_t* base = e.cache + (int64_t)blk * e.block_stride;
    if (n < e.v0) {
        const int c = n - e.k0, g = c / e.dp;
        act_store4<bf16_t>(base + (int64_t)g * e.bs * e.dp, grouped_k_row(crow), c - g * e.dp, e.dp, v);
        return;
    }
    const int c = n - e.v0, g = c / e.vp;
    if (e.mix) {
        f32x4* f = (f32x4*)(e.vfirst + row * e.vfirst_ld + c);
        if (e.mix == 1) *f = v;
        else { const float lam = *e.lambda; v = (1.0f - lam) * v + lam * *f; }
    }
    bf16_t* d = base + (int64_t)e.G * e.bs * e.dp + (int64_t)g * e.bs * e.vp + fm_index(c - g * e.vp, crow, e.bs);      // (transposed: neighbouring channels are 8 apart)
#pragma unroll
    for (int r = 0; r < 4; r++) d[8 * r] = (bf16_t)v[r];
}

// EPI_GROUPED_RAW
__device__ __forceinline__ float silu_f(float g);
__device__ __forceinline__ void epilogue_grouped_raw4(const GemmArgs& p, int64_t row, int n, f32x4 v) {
    const GroupedEpi& e = p.grp;
    if (n >= e.v0 && n < e.raw0) { epilogue_grouped4(p, row, n, v); return; }        // values and gates
    if (n < e.silu1 && n >= e.raw0)
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = silu_f(v[r]);
    float* c = e.raw + row * e.raw_ld + n;
    if (n + 3 < p.N) { *(f32x4*)c = v; return; }      // (rows of 4 k floats)
#pragma unroll
    for (int r = 0; r < 4; r++) if (n + r < p.N) c[r] = v[r];
}

__device__ __forceinline__ float silu_f(float g) { return g / (1.0f + __expf(-g)); }
// ... rounded to bf16 right away: the hardware's reciprocal in place of the division, whose ten instructions for each of a lane's 64 values were 28 of 828 us
// (16384 x 16384 x 2048, all CUs in their epilogues at once; 4176 x 28672 x 4096 743 -> 730).  Error of the bf16 product silu(g) u against 64 bits: the
// same to seven digits for |g| <= 0.01 .. 80 (1.64e-3 .. 1.66e-3 in the 2-norm); 4 results of a million round the other way.
// The quarters keep the reciprocal of sums above 2^126 (g < -87.3) out of the denormals, which it returns as zero.  exp2 -> inf gives 0 and -inf NaN, as the division does
__device__ __forceinline__ float silu_bf16_f(float g) {
    return 0.25f * g * __builtin_amdgcn_rcpf(__builtin_fmaf(0.25f, __builtin_amdgcn_exp2f(-1.4426950408889634f * g), 0.25f));
}
__device__ __forceinline__ float deferred_rstd(const GemmArgs& p, int m);

// ------------------------------------------------------------------------------------------
// epilogue shared by all kernels: 4 consecutive n for one row m
// ------------------------------------------------------------------------------------------
template <int EPI, typename OutT>
__device__ __forceinline__ void epilogue4(const GemmArgs& p, int m, int n, f32x4 v, float rstd = 1.0f) {
    if (m >= p.M || n >= p.N) return;
    v *= rstd;                       // deferred RMSNorm of the input row (1 otherwise), before the bias
    const bool full = (n + 3 < p.N);
    if (p.bias) {
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (n + r < p.N) v[r] += p.bias[n + r];
    }
    if (EPI == EPI_JOINT) {
        if (n < p.joint.n) { *(f32x4*)(p.joint.rows + ((int64_t)p.c_row0 + m) * p.joint.ld + n) = v; return; }
        n -= p.joint.n;
    }
    if (EPI == EPI_GELU || EPI == EPI_JOINT) {
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = gelu_tanh_f(v[r]);
    }
    if (EPI == EPI_RELU2) {
#pragma unroll
        for (int r = 0; r < 4; r++) { const float t = fmaxf(v[r], 0.f); v[r] = t * t; }
    }
    const int64_t row = (int64_t)p.c_row0 + m;
    if (EPI == EPI_GROUPED) { epilogue_grouped4(p, row, n, v); return; }
    if (EPI == EPI_GROUPED_RAW) { epilogue_grouped_raw4(p, row, n, v); return; }
    if (EPI == EPI_GELU_TOK) {
        const bf16x4 e = *(const bf16x4*)(p.tok_table + (int64_t)p.tok_ids[row] * p.tok_ld + n);
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = gelu_tanh_f(v[r]) * (float)e[r];
    }
    if (EPI == EPI_RESID) {
        float* x = (float*)p.C + row * p.ldc + n;
        if (full) {
            f32x4 o = *(f32x4*)x;
            o += p.alpha * v;
            *(f32x4*)x = o;
        } else {
            for (int r = 0; r < 4; r++)
                if (n + r < p.N) x[r] += p.alpha * v[r];
        }
        return;
    }
    if (sizeof(OutT) == 4) {
        float* c = (float*)p.C + row * p.ldc + n;
        if (full) *(f32x4*)c = v;
        else
            for (int r = 0; r < 4; r++)
                if (n + r < p.N) c[r] = v[r];
    } else {
        // bf16 activation for the next GEMM: widths are multiples of 64, so the group is always full
        act_store4<bf16_t>((bf16_t*)p.C, row, n, p.ldc, v);
    }
}

// deferred RMSNorm scale of input row m (< 64): the 4 lanes that share a row (same lane & 15) split the tile partials.
// Call with all 64 lanes active; 1 when the projection's operand is already normalised.
__device__ __forceinline__ float deferred_rstd(const GemmArgs& p, int m) {
    if (!p.rs_in) return 1.0f;
    // rs_in is [64 rows][rs_tiles] (rs_tiles % 16 == 0): a lane sums a quarter of its row with independent 16-byte loads
    const int per = p.rs_tiles >> 2;
    const f32x4* src = (const f32x4*)(p.rs_in + (int64_t)m * p.rs_tiles + ((threadIdx.x & 63) >> 4) * per);
    f32x4 a4 = f32x4{0.f, 0.f, 0.f, 0.f};
    // only the lanes of live rows fetch: each of these loads touches one cache line per row, every epilogue wave of every
    // workgroup issues them, and at batch 1 the 15 padding rows were 94 % of the requests queued at the L2 channels that
    // hold these few KiB (batch 1: QKV 5.1 -> 4.6 us, FFN-up 13.3 -> 12.2 us, LM head 45.6 -> 42.8 us per launch,
    // profiles/r03_timeline_b1_rstd.txt; the non-deferred forms take 4.1 / 12.0 / 42.2).  Rows >= M get a finite scale
    // nobody stores with.  (Tried on top: the sums once per workgroup, coalesced, issued ahead of the weight stream — the
    // first weight data came 0.9 us earlier and the stream took 0.9 us longer, same file.)
    if (m < p.M) {
#pragma unroll 8
        for (int q = 0; q < (per >> 2); q++) a4 += src[q];
    }
    float s = (a4[0] + a4[1]) + (a4[2] + a4[3]);
    s += __shfl_xor(s, 16, 64);
    s += __shfl_xor(s, 32, 64);
    return 1.0f / sqrtf(s * p.rs_inv_h + p.rs_eps);
}

// deferred layer norm: a row's pairs of partial sums, `tiles` of them (a multiple of 16), by the four lanes that share the row.  The loads
// leave together and are added where they are needed: a loop of eight and its remainder waited for memory five times, 2 us of a 5 us launch (768 columns).
struct RowPairs {
    static constexpr int NB = 12;
    f32x4 t[NB];
    int n;
    const f32x4* src;
    __device__ __forceinline__ void fetch(const float* pairs, int tiles, int m, bool live) {
        n = tiles >> 3;
        src = (const f32x4*)(pairs + 2 * ((int64_t)m * tiles)) + ((threadIdx.x & 63) >> 4) * n;
#pragma unroll
        for (int j = 0; j < NB; j++) t[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (live) {
#pragma unroll
            for (int j = 0; j < NB; j++) t[j] = src[j < n ? j : n - 1];
        } else n = 0;
    }
    // sums of x - s and of its square, in every lane of the row
    __device__ __forceinline__ f32x2 sum() const {
        f32x4 a4 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NB; j++) a4 += j < n ? t[j] : f32x4{0.f, 0.f, 0.f, 0.f};
        for (int j = NB; j < n; j++) a4 += src[j];
        float s = a4[0] + a4[2], ss = a4[1] + a4[3];
        s += __shfl_xor(s, 16, 64); ss += __shfl_xor(ss, 16, 64);
        s += __shfl_xor(s, 32, 64); ss += __shfl_xor(ss, 32, 64);
        return f32x2{s, ss};
    }
};
// what scales row m's sums, and what then adds ln_s
struct RowNorm { float scale, shift; };
__device__ __forceinline__ RowNorm layer_norm_of(const GemmArgs& p, f32x2 s) {
    const float d = s[0] * p.rs_inv_h, rstd = 1.0f / sqrtf(fmaxf(s[1] * p.rs_inv_h - d * d, 0.f) + p.rs_eps);
    return {rstd, -rstd * d};
}
template <int EPI>
__device__ __forceinline__ RowNorm row_norm(const GemmArgs& p, int m) {
    if constexpr (!epi_ln(EPI)) return {deferred_rstd(p, m), 0.f};
    RowPairs r;
    r.fetch(p.rs_in, p.rs_tiles, m, m < p.M);
    return layer_norm_of(p, r.sum());
}
// ... applied to four columns from n on
template <int EPI>
__device__ __forceinline__ f32x4 normed(const GemmArgs& p, int n, f32x4 v, RowNorm r) {
    if constexpr (epi_ln(EPI)) return v * r.scale + r.shift * *(const f32x4*)(p.ln_s + n);
    else return v * r.scale;
}

template <int EPI, typename OutT, bool MOE = false>
__device__ __forceinline__ void epilogue_glu4(const GemmArgs& p, int m, int f, f32x4 g, f32x4 u, float rstd = 1.0f) {
    // p.N counts fused rows (2F); the output has F = N/2 columns, ldc = F
    if (m >= p.M || f >= (p.N >> 1)) return;
    g *= rstd; u *= rstd;
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if constexpr (EPI == EPI_CLAMP_GLU) v[r] = clamp_glu_f(g[r], u[r], MOE && f >= p.glu_from2 ? p.glu_limit2 : p.glu_limit, p.glu_slope);
        else if constexpr (EPI == EPI_REGLU) v[r] = fmaxf(g[r], 0.f) * u[r];
        else v[r] = (EPI == EPI_GEGLU ? gelu_tanh_f(g[r]) : sizeof(OutT) == 2 ? silu_bf16_f(g[r]) : silu_f(g[r])) * u[r];
    }
    act_store4<OutT>((OutT*)p.C, (int64_t)p.c_row0 + m, f, p.ldc, v);
}

// EPI_RESID of a wave's TM x TN tiles of 16 rows x 16 columns that all lie within N (N % 4 == 0): the old values of eight tiles are fetched ahead of the stores of the eight
// before.  One at a time, a tile waits for its values and, since the counter runs in order, for the store of the tile before: 32 times for a wave of a 256 x 256 tile.
// us, a prompt before -> here:
// Llama-3-8B 6 of 200 .. 1400 tokens 49280 -> 48701 (O 158 -> 152, FFN-down 399 -> 387 by events), Llama-3.2-1B 8 x 512 7574 -> 7528 (32 x 512, whose CUs are all at it at once,
// 137 both), hybrid 8 of 90 .. 600 5190 -> 5143, GPT-2 900 / 8 x 512 1019 -> 978, 1852 -> 1822
template <int TM, int TN>
__device__ __forceinline__ void epilogue_resid_tiles(const GemmArgs& p, int m0, int n0, f32x4 (&acc)[TM][TN]) {      // m0, n0: this lane's first row and column
    constexpr int R = TN >= 8 ? 1 : 8 / TN < TM ? 8 / TN : TM;
    static_assert(TM % R == 0, "whole groups of rows");
    float* x = (float*)p.C + (int64_t)p.c_row0 * p.ldc + n0;
    f32x4 old[2][R][TN], bias[TN];
    if (p.bias)
#pragma unroll
        for (int j = 0; j < TN; j++) bias[j] = *(const f32x4*)(p.bias + n0 + 16 * j);
    auto fetch = [&](int i0, f32x4 (&o)[R][TN]) {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float* from = x + (int64_t)min(m0 + 16 * (i0 + r), p.M - 1) * p.ldc;
#pragma unroll
            for (int j = 0; j < TN; j++) o[r][j] = *(const f32x4*)(from + 16 * j);
        }
    };
    fetch(0, old[0]);
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += R) {
        if (i0 + R < TM) fetch(i0 + R, old[(i0 / R + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int m = m0 + 16 * (i0 + r);
            if (m < p.M)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    f32x4 v = acc[i0 + r][j];
                    if (p.bias) v += bias[j];
                    *(f32x4*)(x + (int64_t)m * p.ldc + 16 * j) = old[(i0 / R) & 1][r][j] + p.alpha * v;
                }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// EPI_QKV: TM wave sub-tiles of 16 rows x TH*16 columns = one head (TH = 4: hd 64, TH = 8: hd 128).  The lane holds, for
// token m, d = 16j + 4fg + r (j = 0..TH-1): the RoPE partner d + hd/2 is tile j + TH/2 of the SAME lane.
// Positions and blocks of all rows are fetched together, a row's angles ahead of the stores of the row before (as epilogue_resid_tiles).  us by events, a row
// after the other -> here: Llama-3.2-1B 32 x 512 / 8 x 512 / 1900 177 -> 169, 57.2 -> 54.4, 37.3 -> 34.9, Granite 16 of 150 .. 900 42.8 -> 38.9, GPT-2 8 x 512 32.9 -> 30.6,
// heads of 128 87.7 -> 85.6 (Llama-3-8B 1500); Falcon-7B 900, 71 of whose 73 heads are query heads, 60.9 -> 61.2 with lookups for all of them, 58.4 -> 58.1 without
template <int TM, int TH>
__device__ __forceinline__ void epilogue_qkv_tiles(const GemmArgs& p, int m0, int head, int fg, f32x4 (&acc)[TM][TH]) {      // m0: this lane's first row
    constexpr int HD = TH * 16;
    const QkvEpi& q = p.qkv;
    const bool rotated = head < q.nH + q.nKV && q.cos_t, cached = head >= q.nH;
    constexpr bool AHEAD = TH <= 4;      // (heads of 128 spill so: QKV of Llama-3-8B 192 -> 196 us; theirs come row by row)
    int pos[TM], tbl[TM], blk[TM], row[TM];
    f32x4 bias[TH], c[2][TH / 2], s[2][TH / 2];
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = min(m0 + 16 * i, p.M - 1);
        pos[i] = q.tok_pos[m];
        tbl[i] = q.tok_tbl[m];
    }
    auto bias_at = [&](int j) { return *(const f32x4*)(p.bias + head * HD + 16 * j + 4 * fg); };
    if (AHEAD && p.bias)
#pragma unroll
        for (int j = 0; j < TH; j++) bias[j] = bias_at(j);
    auto angles = [&](int i) {
        if (rotated)
#pragma unroll
            for (int j = 0; j < TH / 2; j++) {
                c[i & 1][j] = *(const f32x4*)(q.cos_t + (int64_t)pos[i] * HD + 16 * j + 4 * fg);
                s[i & 1][j] = *(const f32x4*)(q.sin_t + (int64_t)pos[i] * HD + 16 * j + 4 * fg);
            }
    };
    if (AHEAD) angles(0);
#pragma unroll
    for (int i = 0; i < TM; i++) blk[i] = row[i] = 0;
    if (!AHEAD || cached)      // (one branch of the whole wave around all rows' lookups, which query heads don't need; for heads of 128 it costs more than they: Llama-3-8B 1500 84.0 -> 84.6)
#pragma unroll
        for (int i = 0; i < TM; i++) kv_locate(q.blk_table, tbl[i], pos[i], q.Tmax, blk[i], row[i]);
#pragma unroll
    for (int i = 0; i < TM; i++) {
        if (!AHEAD) angles(i);
        else if (i + 1 < TM) angles(i + 1);
        __builtin_amdgcn_sched_barrier(0);
        const int m = m0 + 16 * i;
        if (m < p.M) {
            f32x4 t[TH];
#pragma unroll
            for (int j = 0; j < TH; j++) { t[j] = acc[i][j]; if (p.bias) t[j] += AHEAD ? bias[j] : bias_at(j); }
            if (rotated) {
#pragma unroll
                for (int j = 0; j < TH / 2; j++) {
                    const f32x4 x1 = t[j], x2 = t[j + TH / 2], cs = c[i & 1][j], sn = s[i & 1][j];
#pragma unroll
                    for (int r = 0; r < 4; r++) {          // rope.go:196-202 (table halves are duplicates: cos[d+hd/2] == cos[d])
                        t[j][r] = __builtin_fmaf(x1[r], cs[r], -(x2[r] * sn[r]));
                        t[j + TH / 2][r] = __builtin_fmaf(x1[r], sn[r], x2[r] * cs[r]);
                    }
                }
            }
            // Q -> q buffer; K and V -> their slabs, both row-major [pos][hd] (kv_cache.go:5-6)
            bf16_t* dst;
            if (!cached) dst = q.q_out + (int64_t)m * (q.nH * HD) + head * HD + 4 * fg;
            else if (head < q.nH + q.nKV) dst = q.kcache + (int64_t)blk[i] * q.slot_stride + ((int64_t)(head - q.nH) * q.Tmax + row[i]) * HD + 4 * fg;
            else dst = q.vcache + (int64_t)blk[i] * q.slot_stride + ((int64_t)(head - q.nH - q.nKV) * q.Tmax + row[i]) * HD + 4 * fg;
#pragma unroll
            for (int j = 0; j < TH; j++) {
                bf16x4 o;
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = (bf16_t)t[j][r];
                *(bf16x4*)(dst + 16 * j) = o;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ------------------------------------------------------------------------------------------
// bf16 MFMA kernel (prefill), one template, instances chosen per shape by the launcher:
//   <128,128, 2,2, 4, BK 32>  4 waves, wave tile 64x64, a ring of 4 K tiles of 32 (64 KiB, 2 workgroups/CU): what does not fill
//                             256x256 tiles (below); <128,128, 4,2, 4, BK 32> on 8 waves of 32x64 (ring_eight)
//   < 64,128, 2,2, 4 or 6, BK 32>  4 waves, wave tile 32x64: few tiles (ring64_fits)
//   <256,128, 4,2, 6, BK 32>  8 waves, wave tile 64x64, a ring of 6 (144 KiB): where 128x128 tiles would be two on some CUs (ring256_wins)
//   <256,128, 4,2, 3>  8 waves, wave tile  64x64, 3 LDS stages (144 KiB): two K tiles in flight (experts, a tuning option)
//   <256,256, 2,4, 2>  8 waves, wave tile 128x64, 2 LDS stages (128 KiB): least LDS traffic per MFMA
//                      ((8+4) fragment reads per 32 MFMAs instead of (4+4) per 16)
// BK 32: the fragments of a K tile are read, and the loads of another issued, between the products of the tile before.  A lone workgroup's K tile is
// 0.125 us of products; with reads and loads in a row in front of them it took 0.234, between them 0.188 (two workgroups a CU 0.34 and 0.33 for
// both), and three K tiles in flight instead of one cover the weights' way from HBM.  The lock-step loop over two tiles of 64 that was here -> now, us:
// 487 x 3072 x 2048 33.5 -> 22.7, 487 x 2048 x 8192 112 -> 73, 200 x 16384 x 2048 33 -> 24, 974 x 3072 x 2048 26.5 -> 21.0, 600 x 768 x 3072 37.5 -> 26.9,
// 2000 x 2048 x 2048 31.7 -> 26.6, 487 x 16384 x 2048 (two a CU) 40.8 -> 39.5, 900 x 4672 x 4544 60.7 -> 58.2.  Deeper rings of 128x128 tiles are slower.
// Every operand tile is a run of 1-KiB fragment-major blocks, so one
// global_load_lds_dwordx4 per block fills LDS lane-linearly and the fragment ds_read_b128s are
// conflict-free.  Raw s_barrier + counted s_waitcnt vmcnt keep (STAGES-2) later tiles in flight
// across the barrier (never vmcnt(0) in the steady state of the 3-stage instance).
// ------------------------------------------------------------------------------------------
constexpr int G_BK = 64;
__device__ __forceinline__ int cdiv_dev(int a, int b) { return (a + b - 1) / b; }

// XCD-aware block remap (bijective for any grid size): blocks b and b+8 share an XCD, so give
// each XCD a contiguous run of tiles -> neighbouring tiles (same A row panel) hit one L2.
__device__ __forceinline__ int xcd_remap(int bid, int nwg) {
    const int q = nwg >> 3, r = nwg & 7, xcd = bid & 7, k = bid >> 3;
    const int base = (xcd < r) ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
    return base + k;
}

// tile id -> (tm, tn), "grouped" order: ids run down GM row-tiles before moving to the next column
// tile, so the ~32 workgroups an XCD runs at once (a contiguous id range after xcd_remap) cover a
// compact GM x (32/GM) patch: every A row-panel chunk pulled into that XCD's L2 is reused by 32/GM
// column tiles and every W panel chunk by GM row tiles, instead of each tile streaming its own W
// panel from MALL/HBM (tiles advance through K in near lock-step, so the live window is small).
__device__ __forceinline__ void tile_coords(int pid, int tiles_m, int tiles_n, int GM, int& tm, int& tn) {
    const int per_group = GM * tiles_n;
    const int group = pid / per_group, first = group * GM;
    const int gsz = (tiles_m - first) < GM ? (tiles_m - first) : GM;
    const int r = pid - group * per_group;
    tm = first + r % gsz;
    tn = r / gsz;
}

template <int BM, int BN, int STAGES, int BK = G_BK>
constexpr int gemm_lds_bytes() { return STAGES * (BM + BN) * BK * 2; }

// SLICES (EPI_RESID): K tiles dealt over gridDim.y, partial sums to sk_part (beside the residual's epilogue in one instance their launches lose 1 %)
template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int EPI, typename OutT, int BK = G_BK, bool SLICES = false>
__global__ __launch_bounds__(WAVES_M * WAVES_N * 64, (WAVES_M * WAVES_N == 4 && STAGES * BK <= 160) ? 2 : (BK == 32 && BM == 128) ? 4 : 1)
void gemm_bf16_kernel(GemmArgs p) {
    constexpr int NW = WAVES_M * WAVES_N;
    constexpr int TM = BM / WAVES_M / 16, TN = BN / WAVES_N / 16;   // 16x16 accumulator tiles per wave
    constexpr int KS = BK / 32;                                      // MFMA k-steps of a K tile
    constexpr int NA = BM / 16 * KS, NB = BN / 16 * KS;               // 1-KiB blocks per stage (A, W)
    constexpr int PW = (NA + NB) / NW;                               // blocks staged per wave per K tile
    constexpr int STAGE_BYTES = (BM + BN) * BK * 2;
    static_assert((NA + NB) % NW == 0, "blocks must divide evenly over the waves");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_n = (p.N + BN - 1) / BN;
    int tm, tn;
    int row_base = 0;
    if (p.tile_map) {                      // grouped launch: the m-tile index selects (expert, row segment)
        tn = blockIdx.x % tiles_n;
        const int ti = blockIdx.x / tiles_n;
        if (ti >= *p.n_mtiles) return;
        const int e = p.tile_map[4 * ti];
        row_base = p.tile_map[4 * ti + 1];
        p.M = p.tile_map[4 * ti + 2];
        p.c_row0 = row_base;
        p.W = (const bf16_t*)p.W + (int64_t)e * p.w_expert_stride;
        tm = 0;
    } else {
        tile_coords(xcd_remap(blockIdx.x, gridDim.x), gridDim.x / tiles_n, tiles_n, NW == 4 || BK == 32 ? 8 : 4, tm, tn);
        if (p.seg) {
            row_base = p.seg[0];
            p.M = p.seg[1] - row_base;
            p.c_row0 = row_base;
        }
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int fr = lane & 15, fg = lane >> 4;
    if (m0 >= p.M) return;

    // ---- staging sources: wave w moves blocks w*PW .. w*PW+PW-1 of the stage's [A blocks | W blocks] list
    const bf16_t* src[PW];
#pragma unroll
    for (int i = 0; i < PW; i++) {
        const int blk = wave * PW + i;
        if (blk < NA) {
            const int rt = blk / KS, ksb = blk % KS;
            int am = m0 + rt * 16 + fr;
            if (am > p.M - 1) am = p.M - 1;                 // clamp: rows >= M are never stored
            am += row_base;
            if (p.a_rows) am = p.a_rows[am];
            src[i] = (const bf16_t*)p.A + ((((int64_t)(am >> 4) * (p.K >> 5) + ksb) * 64) + (am & 15) + 16 * fg) * 8;
        } else {
            const int wb = blk - NA, rt = wb / KS, ksb = wb % KS;
            src[i] = (const bf16_t*)p.W + (((int64_t)((n0 >> 4) + rt) * (p.K >> 5) + ksb) * 64 + lane) * 8;
        }
    }
    auto stage = [&](int buf, int kt) {
        char* base = smem + buf * STAGE_BYTES + wave * (PW * 1024);
        const int64_t koff = (int64_t)kt * (512 * KS);
#pragma unroll
        for (int i = 0; i < PW; i++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + koff),
                                             (__attribute__((address_space(3))) void*)(base + i * 1024), 16, 0, 0);
    };
    auto stage_one = [&](int buf, int kt, int i) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (int64_t)kt * (512 * KS)),
                                         (__attribute__((address_space(3))) void*)(smem + buf * STAGE_BYTES + wave * (PW * 1024) + i * 1024), 16, 0, 0);
    };
    auto wait_tiles_in_flight = [&](int tiles) {   // s_waitcnt needs an immediate
        if (tiles <= 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if (tiles == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PW) : "memory");
        else if (tiles == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PW) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PW) : "memory");
    };
    static_assert(STAGES <= 8 && 3 * PW < 64, "at most three younger tiles");

    // ---- fragment reads: stage image [A row-tile][k-step][lane][16 B] then [W row-tile][k-step][lane][16 B]
    const int a_blk_off = wm * TM * (1024 * KS) + lane * 16;                 // activation rows -> MFMA B operand (output col m)
    const int w_blk_off = NA * 1024 + wn * TN * (1024 * KS) + lane * 16;     // weight rows     -> MFMA A operand (output row n)

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // K split over gridDim.y workgroups per tile (residual projections of 65..512 rows: N / 128 x M / 128 tiles alone are
    // far too few workgroups): slice y takes K tiles [kt0, kt0 + nt) and leaves an fp32 partial tile in sk_part[y]; the
    // norm that follows sums the slices into x (PendingResid: the kernel boundary is the synchronisation)
    const int nt_all = p.K / BK;
    int nt = nt_all, kt0 = 0;
    if (SLICES) {
        const int per = nt_all / (int)gridDim.y, extra = nt_all - per * (int)gridDim.y;
        kt0 = (int)blockIdx.y * per + ((int)blockIdx.y < extra ? (int)blockIdx.y : extra);
        nt = per + ((int)blockIdx.y < extra ? 1 : 0);
    }
    if constexpr (BK == 32) {
        constexpr bool ONE = TM * TN < 16;      // eight products: a read at each, the loads beside the first; sixteen: reads and loads in turn
        static_assert(TM + TN <= TM * TN / (ONE ? 1 : 2) && PW <= TM * TN / (ONE ? 1 : 2), "reads and loads between the products");
        // a K tile's fragments are read while the products of the one before run; its slot is filled again as soon as every wave holds them
        bf16x8 fa[2][TM], fw[2][TN];
        auto fragments = [&](int slot, bf16x8 (&af)[TM], bf16x8 (&wf)[TN]) {
            const char* sbuf = smem + slot * STAGE_BYTES;
#pragma unroll
            for (int j = 0; j < TN; j++) wf[j] = *(const bf16x8*)(sbuf + w_blk_off + j * 1024);
#pragma unroll
            for (int i = 0; i < TM; i++) af[i] = *(const bf16x8*)(sbuf + a_blk_off + i * 1024);
        };
#pragma unroll
        for (int s = 0; s < STAGES; s++)
            if (s < nt) stage(s, kt0 + s);
        wait_tiles_in_flight((nt < STAGES ? nt : STAGES) - 1);
        __builtin_amdgcn_s_barrier();
        fragments(0, fa[0], fw[0]);
        wait_tiles_in_flight((nt < STAGES ? nt : STAGES) - 2);
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_s_barrier();
        int slot = 0, t = 0;
        // FULL: all of the ring is in flight, so that the wait is an immediate and nothing is asked
        auto step = [&](auto full, int t, bf16x8 (&af)[TM], bf16x8 (&wf)[TN], bf16x8 (&an)[TM], bf16x8 (&wn)[TN]) __attribute__((always_inline)) {
            constexpr bool FULL = decltype(full)::value;
            const int next = slot + 1 == STAGES ? 0 : slot + 1;
            const char* sbuf = smem + next * STAGE_BYTES;
            const bool load = FULL || t + STAGES < nt;
            // reads and loads between the products: issued in a row they hold the products up (0.234 -> 0.188 us a tile of a lone workgroup)
#pragma unroll
            for (int e = 0; e < TM * TN; e++) {
                const int i = e / TN, j = e % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                const int rd = ONE ? e : e % 2 == 0 ? e / 2 : TM + TN, ld = ONE ? e : e % 2 == 1 ? e / 2 : PW;
                if (rd < TN) wn[rd < TN ? rd : 0] = *(const bf16x8*)(sbuf + w_blk_off + rd * 1024);
                else if (rd < TM + TN) an[rd < TM + TN ? rd - TN : 0] = *(const bf16x8*)(sbuf + a_blk_off + (rd - TN) * 1024);
                if (ld < PW && load) stage_one(slot, kt0 + t + STAGES, ld);
                __builtin_amdgcn_sched_barrier(0);
            }
            slot = next;
            // tile t + 2 must have landed; the younger ones stay in flight
            __builtin_amdgcn_s_waitcnt(0xC07F);      // lgkmcnt(0); the builtin, which the compiler counts: behind asm it waits for the reads a second time, in front of the products
            if (FULL) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PW * (STAGES - 2)) : "memory");
            else wait_tiles_in_flight(nt - 3 - t);
            __builtin_amdgcn_s_barrier();
        };
        for (; t + 1 + STAGES < nt; t += 2) {
            step(std::true_type{}, t, fa[0], fw[0], fa[1], fw[1]);
            step(std::true_type{}, t + 1, fa[1], fw[1], fa[0], fw[0]);
        }
        for (; t < nt; t += 2) {
            step(std::false_type{}, t, fa[0], fw[0], fa[1], fw[1]);
            if (t + 1 < nt) step(std::false_type{}, t + 1, fa[1], fw[1], fa[0], fw[0]);
        }
    } else {
#pragma unroll
    for (int s = 0; s < STAGES - 1; s++)
        if (s < nt) stage(s, kt0 + s);
    wait_tiles_in_flight((nt < STAGES - 1 ? nt : STAGES - 1) - 1);
    __builtin_amdgcn_s_barrier();
    int cur = 0;
    for (int t = 0; t < nt; t++) {
        if (t + STAGES - 1 < nt) {
            int nb = cur + STAGES - 1;
            if (nb >= STAGES) nb -= STAGES;
            stage(nb, kt0 + t + STAGES - 1);
        }
        const char* sbuf = smem + cur * STAGE_BYTES;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            bf16x8 af[TM], wf[TN];
#pragma unroll
            for (int j = 0; j < TN; j++) wf[j] = *(const bf16x8*)(sbuf + w_blk_off + j * (1024 * KS) + ks * 1024);
#pragma unroll
            for (int i = 0; i < TM; i++) af[i] = *(const bf16x8*)(sbuf + a_blk_off + i * (1024 * KS) + ks * 1024);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
        }
        // tile t+1 must have landed; up to STAGES-2 younger tiles may stay in flight
        int younger = nt - 2 - t;
        if (younger > STAGES - 2) younger = STAGES - 2;
        wait_tiles_in_flight(younger);
        __builtin_amdgcn_s_barrier();
        cur = cur + 1 == STAGES ? 0 : cur + 1;
    }
    }

    // ---- epilogue: lane holds rows n = 4*fg + r of column m = fr of each 16x16 tile ----
    if constexpr (EPI == EPI_QKV) {      // the wave's columns are exactly one head: TN = 4 <-> head_dim 64, TN = 8 <-> head_dim 128
        const int head = (n0 + wn * (TN * 16)) / (TN * 16);
        if (head * (TN * 16) < p.N) epilogue_qkv_tiles<TM, TN>(p, m0 + wm * (TM * 16) + fr, head, fg, acc);
        return;
    }
    if constexpr (EPI == EPI_RESID)
        if (!SLICES && (p.N & 3) == 0 && n0 + (wn + 1) * (TN * 16) <= p.N) { epilogue_resid_tiles<TM, TN>(p, m0 + wm * (TM * 16) + fr, n0 + wn * (TN * 16) + 4 * fg, acc); return; }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + wm * (TM * 16) + i * 16 + fr;
        if (epi_glu(EPI)) {
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                const int ntile = (n0 + wn * (TN * 16) + j * 16) >> 4;   // even: gate block, +1: up block
                const int f = (ntile >> 1) * 16 + 4 * fg;
                epilogue_glu4<EPI, OutT>(p, m, f, acc[i][j], acc[i][j + 1]);
            }
        } else if (SLICES) {
            GemmArgs q = p;                                   // this slice's partial tile: plain fp32 store, bias with slice 0
            q.C = p.sk_part + (int64_t)blockIdx.y * p.M * p.N; q.ldc = p.N; q.c_row0 = 0;
            if (blockIdx.y != 0) q.bias = nullptr;
#pragma unroll
            for (int j = 0; j < TN; j++)
                epilogue4<EPI_STORE, float>(q, m, n0 + wn * (TN * 16) + j * 16 + 4 * fg, acc[i][j]);
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++)
                epilogue4<EPI, OutT>(p, m, n0 + wn * (TN * 16) + j * 16 + 4 * fg, acc[i][j]);
        }
    }
}

// ------------------------------------------------------------------------------------------
// K split inside one launch.  `parts` workgroups share an output tile; each leaves its fp32 accumulators in split_ws, draws a number
// from the tile's counter, and the one that draws the last adds the parts up in part order (always the same sum) and runs the
// epilogue.  Nobody waits for anybody.  The workgroups may sit on different XCDs, whose L2s are not coherent: the parts are
// written through and read past the L2 (sc0 sc1) instead of fencing, which would write back everything that XCD has dirty
// (4096 x 2048 x 6144 in two parts: 85 us so, 156 us with __threadfence, 94 us unsplit).
// ------------------------------------------------------------------------------------------
constexpr int64_t SPLIT_WS_BYTES = 64ll << 20;      // all a launch can use: 256 parts of 256 x 256 fp32 (gemm_bf16_pp_kernel)
constexpr int64_t SPLIT_MID_BYTES = 8ll << 20;      // ... gemm_mid_bf16_kernel, unless its parts are forced: 256 of 128 x 64 or 64 x 128
constexpr int64_t SPLIT_UNIT = 32 << 10;            // a 128 x 64 fp32 part
constexpr int SPLIT_MAX_TILES = 512;
constexpr int PP_MIN_STAGES = 12;                   // K-steps of 32 that a part of a 256 x 256 tile has at least
constexpr int MID_MAX_PARTS = 8, MID_MIN_STAGES = 2;      // parts of a tile of gemm_mid_bf16_kernel; K-steps of 128 that one has at least
// what the launches of an N x K projection of up to M rows can use of it
static inline int64_t split_need(int64_t M, int64_t N, int64_t K) {
    if (M > 64 && (K >> 5) >= 2 * PP_MIN_STAGES && cdiv(M, 256) * cdiv(N, 256) >= 8) return SPLIT_WS_BYTES;
    if (cdiv(K, 128) < 2 * MID_MIN_STAGES) return 0;
    return std::min(SPLIT_MID_BYTES, (int64_t)MID_MAX_PARTS * 4 * round_up(std::min<int64_t>(M, 512), 128) * round_up(N, 128));
}
constexpr int SPLIT_COHERENT = 0x11;      // buffer cache policy: sc0 | sc1
constexpr int LOAD_NT = 2;                // ... nt: a line read once

// acc: this wave's F fragments; a part takes `bytes` of split_ws (waves one after the other, 1 KiB a fragment).  True in the workgroup
// that holds the sum.  Whole workgroups call it; `flag`: one int of LDS that nothing else uses.
template <int F>
__device__ __forceinline__ bool split_finish(const GemmArgs& p, int tile, int part, int parts, int bytes, int wave, f32x4* acc, int* flag, bool holds = true) {
    const int lane = threadIdx.x & 63, voff = wave * (F * 1024) + lane * 16;
    int* cnt = p.split_cnt + tile;
    char* ws = (char*)p.split_ws + (int64_t)tile * parts * bytes;
    {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(ws + (int64_t)part * bytes, 0, bytes, 0x00020000);
        if (holds) {
#pragma unroll
            for (int f = 0; f < F; f++) {
                union { f32x4 v; u32x4 u; } t; t.v = acc[f];
                __builtin_amdgcn_raw_buffer_store_b128(t.u, rs, voff, f * 1024, SPLIT_COHERENT);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // this wave's stores have reached memory
        __syncthreads();
        if (threadIdx.x == 0) *flag = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (*flag != parts - 1) return false;
    }
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!holds) return true;
    constexpr int B = F > 16 ? 4 : F % 8 == 0 ? 8 : F;      // fragments at a time, of four parts: their loads travel together
    static_assert(B <= 8 && F % B == 0, "registers of the loads in flight");
#pragma unroll
    for (int f0 = 0; f0 < F; f0 += B) {
        f32x4 sum[B];
#pragma unroll
        for (int f = 0; f < B; f++) sum[f] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int c0 = 0; c0 < parts; c0 += 4) {
            union { f32x4 v; u32x4 u; } t[4][B];
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (c0 + c >= parts || c0 + c == part) continue;
                const auto rs = __builtin_amdgcn_make_buffer_rsrc(ws + (int64_t)(c0 + c) * bytes, 0, bytes, 0x00020000);
#pragma unroll
                for (int f = 0; f < B; f++) t[c][f].u = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, (f0 + f) * 1024, SPLIT_COHERENT);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if (c0 + c >= parts) break;
#pragma unroll
                for (int f = 0; f < B; f++) sum[f] += c0 + c == part ? acc[f0 + f] : t[c][f].v;
            }
        }
#pragma unroll
        for (int f = 0; f < B; f++) acc[f0 + f] = sum[f];
    }
    return true;
}

// ------------------------------------------------------------------------------------------
// bf16 MFMA kernel, ping-pong form (prefill, tuning option 5): 256x256 tile, 8 waves as two groups of four (one wave
// of each group per SIMD), K in 32-wide stages through a STAGES-slot LDS ring (4 slots = 128 KiB by default).  A stage is one PHASE for a wave:
//   L: 12 fragment ds_reads of stage s, LDS-DMA issue of stage s+STAGES-1, lgkmcnt(0), counted vmcnt (stage s+1 landed)
//   -- barrier --   C: 32 MFMAs at priority 1   -- barrier --
// Group 1 enters the loop one barrier late, so while one wave of a SIMD issues its MFMAs the other does its LDS reads
// and DMA issue: the fragment reads (384 of every 896 cycles in the lock-step kernel above) move under the MFMAs.
// Hazards (LDS-DMA is ordered only by the issuer's vmcnt + a barrier the reader passes): a slot is re-filled in L(s)
// after its last readers retired their ds_reads before the barrier that ended L(s-1) of the LATE group (WAR);
// stage s+1 is waited for at the end of L(s) by every wave, one barrier before the early group reads it (RAW).
// ------------------------------------------------------------------------------------------
// SPLIT: its own instance, the unsplit loop loses 3 % beside the code of the sum
// ROWS: a grouped launch whose A is row-major, a segment's rows wherever a_rows says.  Against a copy in expert order, us of copy and product ->
// product, 32 experts of 1024 x 512, 8 a row: 900 rows 7 + 30.5 -> 35.5, 3600 18 + 77 -> 85, 6867 32.6 + 118 -> 122, 14400 67 + 215 -> 229 (a line is fetched in two
// k-steps, and the first stage waits for the rows' places).  From a fragment-major operand every 16 bytes would be a line of their own: those are copied.
template <int EPI, typename OutT, int STAGES = 4, int PRIO = 0, int WAVES_N = 4, int BN = 256, bool SPLIT = false, bool ROWS = false>
__global__ __launch_bounds__(512, 1) void gemm_bf16_pp_kernel(GemmArgs p) {
    // BN 256: WAVES_N = 4 -> wave tile 128x64 (a head of 64 per wave), WAVES_N = 2 -> 64x128 (a head of 128 per wave);
    // BN 128 (mid-size M: twice the tiles): WAVES_N = 2 -> wave tile 64x64
    constexpr int BM = 256, WAVES_M = 8 / WAVES_N, TM = BM / WAVES_M / 16, TN = BN / WAVES_N / 16;
    constexpr int NA = BM / 16, NB = BN / 16;            // 1-KiB blocks per stage (one k-step)
    constexpr int PW = (NA + NB) / 8;                    // blocks per wave per stage: 4 (BN 256) or 3 (BN 128)
    constexpr int STAGE_BYTES = (BM + BN) * 32 * 2;      // 32 KiB / 24 KiB
    static_assert((NA + NB) % 8 == 0, "stage blocks must divide over the 8 waves");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_n = (p.N + BN - 1) / BN;
    int tm, tn;
    int row_base = 0, part = 0, split_tile = -1;
    if (p.tile_map) {
        // grouped launch (MoE prefill): m-tile ti = (expert, 256-row segment of its rows in the expert-ordered buffer).
        // After xcd_remap an XCD owns a contiguous range of (ti, tn): whole experts, so an expert's weights and each
        // row segment are re-read from that XCD's L2 by the tiles that share them.
        const int pid = xcd_remap(blockIdx.x, gridDim.x);
        tn = pid % tiles_n;
        const int ti = pid / tiles_n;
        if (ti >= *p.n_mtiles) return;                    // (whole workgroup: before any barrier)
        row_base = p.tile_map[4 * ti + 1];
        p.M = p.tile_map[4 * ti + 2];
        p.c_row0 = row_base;
        p.W = (const bf16_t*)p.W + (int64_t)p.tile_map[4 * ti] * p.w_expert_stride;
        tm = 0;
    } else if (SPLIT) {
        // Each XCD has a contiguous run of tiles, 32 at a time; those of its last, partly filled round are cut along K into p.splits parts
        // (the launcher says when).  All workgroups of the round walk the same K ranges in step, so the panels they share
        // stay in the XCD's L2.
        const int tiles_m = cdiv_dev(p.M, BM), T = tiles_m * tiles_n, xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
        const int first = xcd * (T >> 3) + min(xcd, T & 7), n = (T >> 3) + (xcd < (T & 7) ? 1 : 0), whole = n & ~31, rest = n - whole;
        int i = k;
        if (k >= whole) {
            if (k - whole >= rest * p.splits) return;
            part = (k - whole) / rest;
            i = whole + (k - whole) - part * rest;
            split_tile = xcd * (32 / p.splits) + i - whole;      // (rest * splits <= 32)
        }
        tile_coords(first + i, tiles_m, tiles_n, 4, tm, tn);
    } else {
        tile_coords(xcd_remap(blockIdx.x, gridDim.x), gridDim.x / tiles_n, tiles_n, 4, tm, tn);
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int grp = wave >> 2;                            // the ping-pong group: first / second dispatched half
    const int fr = lane & 15, fg = lane >> 4;
    if (m0 >= p.M) return;

    // K-steps of this workgroup
    const int k_all = p.K >> 5, k0 = !SPLIT || split_tile < 0 ? 0 : (int)((int64_t)part * k_all / p.splits);
    const int nt = !SPLIT || split_tile < 0 ? k_all : (int)((int64_t)(part + 1) * k_all / p.splits) - k0;            // stages
    const bf16_t* src[PW];
#pragma unroll
    for (int i = 0; i < PW; i++) {
        const int blk = wave * PW + i;
        if (blk < NA) {
            int am = m0 + blk * 16 + fr;
            if (am > p.M - 1) am = p.M - 1;
            am += row_base;                               // (a segment may start on any row: per-lane 16-byte sources)
            if constexpr (ROWS) src[i] = (const bf16_t*)p.A + (int64_t)p.a_rows[am] * p.K + 8 * fg;
            else src[i] = (const bf16_t*)p.A + (((int64_t)(am >> 4) * (p.K >> 5) * 64) + (am & 15) + 16 * fg) * 8;
        } else {
            src[i] = (const bf16_t*)p.W + ((int64_t)((n0 >> 4) + blk - NA) * (p.K >> 5) * 64 + lane) * 8;
        }
        src[i] += (int64_t)k0 * 512;
    }
    static_assert(!ROWS || (!SPLIT && NA % PW == 0), "a wave's blocks are all rows or all columns");
    const int step = ROWS && wave * PW < NA ? 32 : 512;      // a k-step further
    auto stage = [&](int buf, int ks) {
        char* base = smem + buf * STAGE_BYTES + wave * (PW * 1024);
#pragma unroll
        for (int i = 0; i < PW; i++)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + (ROWS ? (int64_t)(ks * step) : (int64_t)ks * 512)),
                                             (__attribute__((address_space(3))) void*)(base + i * 1024), 16, 0, 0);
    };
    const int a_off = wm * TM * 1024 + lane * 16;
    const int w_off = NA * 1024 + wn * TN * 1024 + lane * 16;
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int s = 0; s < STAGES - 1; s++)
        if (s < nt) stage(s, s);
    // stage 0 landed (my part); up to STAGES-2 younger stages stay in flight
    auto wait_younger = [&](int younger) {
        if (younger > STAGES - 2) younger = STAGES - 2;
        if (PW == 4) {
            if (younger >= 3) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
            else if (younger == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else if (younger == 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        } else {
            if (younger >= 3) asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
            else if (younger == 2) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
            else if (younger == 1) asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
    };
    static_assert(STAGES >= 3 && STAGES <= 5 && (PW == 4 || PW == 3), "vmcnt immediates above cover up to three stages in flight");
    wait_younger((nt < STAGES - 1 ? nt : STAGES - 1) - 1);
    __builtin_amdgcn_s_barrier();
    if (grp == 1) __builtin_amdgcn_s_barrier();         // the late group: one phase behind from here on
    if (PRIO == 1 && grp == 1) __builtin_amdgcn_s_setprio(1);  // static priority for the second-dispatched half
    int buf = 0;
    for (int s = 0; s < nt; s++) {
        // ---- L phase ----
        bf16x8 af[TM], wf[TN];
        const char* sbuf = smem + buf * STAGE_BYTES;
#pragma unroll
        for (int j = 0; j < TN; j++) wf[j] = *(const bf16x8*)(sbuf + w_off + j * 1024);
#pragma unroll
        for (int i = 0; i < TM; i++) af[i] = *(const bf16x8*)(sbuf + a_off + i * 1024);
        if (s + STAGES - 1 < nt) {
            int nb = buf + STAGES - 1;                   // the slot read in phase s-1
            if (nb >= STAGES) nb -= STAGES;
            stage(nb, s + STAGES - 1);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): my fragment reads are retired
        // stage s+1 landed; stages s+2 .. s+4 (those that exist) may stay in flight
        wait_younger(nt - 2 - s);                        // (stages beyond s+1 that exist)
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        // ---- C phase ----
        // There and back over the columns, in this order: consecutive products share one operand throughout.  With every CU at work the clock follows
        // the power drawn, and operands that stay save some (16384 x 16384 x 2048 838 -> 827 us, 4176 x 28672 x 4096 751 -> 743).
        // Products of 32 x 32 x 16, which move their sums twice as often, draw more: 940 and 845 us
        if (PRIO == 0) __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int jj = 0; jj < TN; jj++) {
                const int j = i & 1 ? TN - 1 - jj : jj;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        if (PRIO == 0) __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        buf = buf + 1 == STAGES ? 0 : buf + 1;
    }
    if (grp == 0) __builtin_amdgcn_s_barrier();         // pairs with the late group's last barrier
    if (SPLIT && split_tile >= 0 && !split_finish<TM * TN>(p, split_tile, part, p.splits, BM * BN * 4, wave, &acc[0][0], (int*)(smem + STAGES * STAGE_BYTES))) return;

    if constexpr (EPI == EPI_QKV) {      // the wave's columns are exactly one head: TN = 4 <-> head_dim 64, TN = 8 <-> head_dim 128
        const int head = (n0 + wn * (TN * 16)) / (TN * 16);
        if (head * (TN * 16) < p.N) epilogue_qkv_tiles<TM, TN>(p, m0 + wm * (TM * 16) + fr, head, fg, acc);
        return;
    }
    if constexpr (EPI == EPI_RESID)
        if ((p.N & 3) == 0 && n0 + (wn + 1) * (TN * 16) <= p.N) { epilogue_resid_tiles<TM, TN>(p, m0 + wm * (TM * 16) + fr, n0 + wn * (TN * 16) + 4 * fg, acc); return; }
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + wm * (TM * 16) + i * 16 + fr;
        if (epi_glu(EPI)) {
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                const int ntile = (n0 + wn * (TN * 16) + j * 16) >> 4;
                epilogue_glu4<EPI, OutT>(p, m, (ntile >> 1) * 16 + 4 * fg, acc[i][j], acc[i][j + 1]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < TN; j++)
                epilogue4<EPI, OutT>(p, m, n0 + wn * (TN * 16) + j * 16 + 4 * fg, acc[i][j]);
        }
    }
}

// ------------------------------------------------------------------------------------------
// bf16 kernel for up to 512 rows (decode batches, short prompts; mid_wins says where): weights still come from HBM once, but the 64-row groups of the
// decode form pull every activation row through every CU for 16 weight rows each (FFN-down of Llama-3.2-1B at 96 rows: 128 workgroups x
// 2 x 1.3 MB, 25 us for 34 MB of weights).  Here a workgroup owns MT x 16 rows by CT x 32 columns, both operands staged through an
// LDS ring by global_load_lds, so an activation row is fetched once per CT x 32 weight rows and the ring keeps a
// fixed amount of weights in flight per CU; K is split over workgroups (split_finish) until the launch fills the chip.
// Eight waves: 2 x 2 over the tile (a wave reads MT / 2 + CT fragments for MT / 2 x CT products) times two halves of every
// 128-wide K stage, added through LDS at the end.
// ------------------------------------------------------------------------------------------
template <int MT, int CT> constexpr int mid_stage_bytes() { return (MT + 2 * CT) * 4096; }
template <int MT, int CT> constexpr int mid_stages() { return 163200 / mid_stage_bytes<MT, CT>() > 5 ? 5 : 163200 / mid_stage_bytes<MT, CT>(); }
template <int MT, int CT> constexpr int mid_lds_bytes() { return mid_stages<MT, CT>() * mid_stage_bytes<MT, CT>() + 16 + MT * 64; }
constexpr int MID_MAX_ROWS = 512;

// one pair of rotated quads (EPI_QKV): x1 at column d of the head, x2 at d + hd / 2
__device__ __forceinline__ void epilogue_qkv_pair(const GemmArgs& p, int m, int head, int d, f32x4 x1, f32x4 x2) {
    if (m >= p.M) return;
    const QkvEpi& q = p.qkv;
    const int HD = q.hd, half = HD >> 1;
    if (p.bias) { x1 += *(const f32x4*)(p.bias + head * HD + d); x2 += *(const f32x4*)(p.bias + head * HD + d + half); }
    const int pos = q.tok_pos[m];
    if (head < q.nH + q.nKV && q.cos_t) {
        const f32x4 c = *(const f32x4*)(q.cos_t + (int64_t)pos * HD + d), s = *(const f32x4*)(q.sin_t + (int64_t)pos * HD + d);
        const f32x4 a = x1, b = x2;
        x1 = a * c + (-b) * s;          // rope.go:196-202
        x2 = b * c + a * s;
    }
    int blk = 0, row = 0;
    if (head >= q.nH) kv_locate(q.blk_table, q.tok_tbl[m], pos, q.Tmax, blk, row);
    bf16_t* dst;
    if (head < q.nH) dst = q.q_out + (int64_t)m * (q.nH * HD) + head * HD + d;
    else if (head < q.nH + q.nKV) dst = q.kcache + (int64_t)blk * q.slot_stride + ((int64_t)(head - q.nH) * q.Tmax + row) * HD + d;
    else dst = q.vcache + (int64_t)blk * q.slot_stride + ((int64_t)(head - q.nH - q.nKV) * q.Tmax + row) * HD + d;
    bf16x4 o1, o2;
#pragma unroll
    for (int r = 0; r < 4; r++) { o1[r] = (bf16_t)x1[r]; o2[r] = (bf16_t)x2[r]; }
    *(bf16x4*)dst = o1;
    *(bf16x4*)(dst + half) = o2;
}

// STREAM: a launch of a single row group of up to 96 rows, which reads each weight once.  The weights then go past what the caches hold: states, keys and values of the
// next launches stay there (without nt a delta-rule scan behind an input projection at 20 rows 31.5 -> 36.0 us, a lightning scan at 32 29.9 -> 34.4),
// and the ring is faster itself (4544 x 18176 at 16 rows 32.5 -> 29.8 us, 4096 x 14336 at 32 26.4 -> 24.9).  Its own instance: as a run-time branch
// around the loads it cost launches of several groups 3 to 11 % (Falcon-7B at 200 rows, its products together, 5.4 -> 5.8 ms).
// Groups of 128 rows gain nothing by it (Falcon-7B, a decode step of 104 sequences 5.61 -> 5.71 ms, a 2048-wide model with a delta rule at 97 1.73 -> 1.75)
template <int MT, int CT, int EPI, typename OutT, bool STREAM>
__global__ __launch_bounds__(512, 1) void gemm_mid_bf16_kernel(GemmArgs p) {
    constexpr int NST = mid_stages<MT, CT>(), SB = mid_stage_bytes<MT, CT>(), NA = 4 * MT, PW = (MT + 2 * CT) / 2, TM = MT / 2;
    static_assert(MT % 2 == 0 && NST >= 3 && PW * (NST - 2) < 64, "two waves share the rows; vmcnt counts to 63");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, fr = lane & 15, fg = lane >> 4;
    const int wave8 = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wave8 & 3, kh = wave8 >> 2, wm = wave >> 1, wn = wave & 1;
    // ids 8 apart share an XCD: the row groups and parts of a column block follow each other there, so its weights cross HBM once
    const int groups = cdiv_dev(p.M, 16 * MT), per = groups * p.splits, nb = cdiv_dev(p.N, 32 * CT);
    const int q = blockIdx.x >> 3, cb = (q / per) * 8 + (blockIdx.x & 7), item = q % per;
    if (cb >= nb) return;
    const int part = item % p.splits, m0 = item / p.splits * (16 * MT), n0 = cb * (32 * CT);
    const int stages = (p.K + 127) >> 7;
    const int k0 = (int)((int64_t)part * stages / p.splits), n = (int)((int64_t)(part + 1) * stages / p.splits) - k0;
    const bool ragged = (p.K & 64) && k0 + n == stages;          // K % 128 == 64: the last stage has its first half only

    // 1-KiB blocks (row tile, k-step) of a stage, PW for each wave: rows first, then columns
    const bf16_t* src[PW];
#pragma unroll
    for (int i = 0; i < PW; i++) {
        const int blk = wave8 * PW + i, rt = (blk < NA ? blk : blk - NA) >> 2, ks = blk & 3;
        if (blk < NA) {
            int am = m0 + rt * 16 + fr;
            if (am > p.M - 1) am = p.M - 1;                     // rows >= M are never stored
            src[i] = (const bf16_t*)p.A + ((((int64_t)(am >> 4) * (p.K >> 5) + ks) * 64) + (am & 15) + 16 * fg) * 8;
        } else src[i] = (const bf16_t*)p.W + (((int64_t)((n0 >> 4) + rt) * (p.K >> 5) + ks) * 64 + lane) * 8;
        src[i] += (int64_t)k0 * 2048;
    }
    auto stage = [&](int buf, int s) {
        char* base = smem + buf * SB + wave8 * (PW * 1024);
        const bool cut = ragged && s == n - 1;
#pragma unroll
        for (int i = 0; i < PW; i++) {
            if (cut && ((wave8 * PW + i) & 2)) continue;        // (k-steps 2 and 3; waited for with vmcnt(0))
            const auto from = (const __attribute__((address_space(1))) void*)(src[i] + (int64_t)s * 2048);
            const auto to = (__attribute__((address_space(3))) void*)(base + i * 1024);
            if (STREAM && wave8 * PW + i >= NA) __builtin_amdgcn_global_load_lds(from, to, 16, 0, LOAD_NT);
            else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
        }
    };
    // a wave's column tiles: neighbours for gate | up pairs, else two apart (a head's rotated halves then lie in one wave)
    constexpr bool PAIRS = epi_glu(EPI);
    int ct[CT];
#pragma unroll
    for (int j = 0; j < CT; j++) ct[j] = PAIRS ? CT * wn + j : wn + 2 * j;
    constexpr bool QKV = EPI == EPI_QKV, BOTH = TM % 2 == 0 || !(PAIRS || QKV), RSTD = PAIRS || EPI == EPI_STORE;
    constexpr int F = TM * CT, H = BOTH ? F / 2 : F;
    f32x4 acc[F];
#pragma unroll
    for (int i = 0; i < F; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NST - 1; s++)
        if (s < n) stage(s, s);
    // the rows' scales of a deferred RMSNorm, once per workgroup and beside the first operands (by every wave for the rows it
    // finishes they were 64 .. 128 KiB of loads: 3 us of a 14 us launch)
    float* rstd = (float*)(smem + NST * SB + 16);
    if (RSTD && p.rs_in && wave8 < MT) {
        const float r = deferred_rstd(p, min(m0 + wave8 * 16 + fr, p.M - 1));
        if (fg == 0) rstd[wave8 * 16 + fr] = r;
    }
    int buf = 0;
    for (int t = 0; t < n; t++) {
        // my pieces of stage t landed; the ring's younger stages stay in flight (a cut stage only ever is the youngest)
        if (n - 1 - t > NST - 2 || (n - 1 - t == NST - 2 && !ragged)) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PW * (NST - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();           // everybody's pieces landed, and everybody is done with the slot that is filled next
        __builtin_amdgcn_sched_barrier(0);
        if (t + NST - 1 < n) stage(buf == 0 ? NST - 1 : buf - 1, t + NST - 1);
        const char* sb = smem + buf * SB + kh * 2048 + lane * 16;
        if (!(kh == 1 && ragged && t == n - 1)) {
            bf16x8 af[2][TM], wf[2][CT];
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
#pragma unroll
                for (int j = 0; j < CT; j++) wf[ks][j] = *(const bf16x8*)(sb + NA * 1024 + ct[j] * 4096 + ks * 1024);
#pragma unroll
                for (int i = 0; i < TM; i++) af[ks][i] = *(const bf16x8*)(sb + (wm * TM + i) * 4096 + ks * 1024);
            }
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < CT; j++)
                        acc[i * CT + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[ks][j], af[ks][i], acc[i * CT + j], 0, 0, 0);
        }
        buf = buf + 1 == NST ? 0 : buf + 1;
        __builtin_amdgcn_s_waitcnt(0xC07F);     // fragment reads retired before the barrier that lets their slot be filled
    }
    // add the K halves: each of the two waves keeps half of the fragments (all of them the first one, where pairs would be cut)
    __syncthreads();
    f32x4* red = (f32x4*)smem + lane;
    f32x4 mine[H];
    if constexpr (BOTH) {
#pragma unroll
        for (int e = 0; e < H; e++) red[(wave8 * H + e) * 64] = kh ? acc[e] : acc[H + e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < H; e++) mine[e] = (kh ? acc[H + e] : acc[e]) + red[((wave8 ^ 4) * H + e) * 64];
    } else {
        if (kh == 1)
#pragma unroll
            for (int e = 0; e < H; e++) red[(wave * H + e) * 64] = acc[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < H; e++) mine[e] = acc[e] + red[(wave * H + e) * 64];
    }
    // residual: the rows' old values and the next norm's weights come under the hand-over (every part fetches them, one uses them)
    f32x4 old[EPI == EPI_RESID ? H : 1], nrm[EPI == EPI_RESID ? H : 1];
    const bool whole = EPI == EPI_RESID && (p.N & 3) == 0;
    if constexpr (EPI == EPI_RESID) {
        if (whole) {
#pragma unroll
            for (int e = 0; e < H; e++) {
                const int idx = (BOTH ? kh * H : 0) + e, i = idx / CT, j = idx - i * CT;
                const int m = min(m0 + (wm * TM + i) * 16 + fr, p.M - 1), nn = min(n0 + (wn + 2 * j) * 16 + 4 * fg, p.N - 4);
                old[e] = *(const f32x4*)((const float*)p.C + (int64_t)m * p.ldc + nn);
                if (p.rs_out) nrm[e] = *(const f32x4*)(p.nrm_w + nn);
            }
        }
    }
    if (p.splits > 1 && !split_finish<H>(p, cb * groups + item / p.splits, part, p.splits, (BOTH ? 8 : 4) * H * 1024, BOTH ? wave8 : wave, mine, (int*)(smem + NST * SB), BOTH || kh == 0)) return;
    if (!BOTH && kh == 1) return;

#pragma unroll
    for (int e = 0; e < H; e += (PAIRS || (QKV && CT == 2) ? 2 : 1)) {
        const int idx = (BOTH ? kh * H : 0) + e, i = idx / CT, j = idx - i * CT;
        const int m = m0 + (wm * TM + i) * 16 + fr, ctile = PAIRS ? CT * wn + j : wn + 2 * j;
        const int nn = n0 + ctile * 16 + 4 * fg;
        const float rs = RSTD && p.rs_in ? rstd[(wm * TM + i) * 16 + fr] : 1.0f;
        if constexpr (QKV) {
            if (CT == 4 && (e & 2)) continue;                        // (pairs are CT / 2 fragments apart)
            epilogue_qkv_pair(p, m, n0 / (32 * CT), 16 * ctile + 4 * fg, mine[e], mine[e + CT / 2]);      // the workgroup's columns are one head
        } else if constexpr (PAIRS) {
            epilogue_glu4<EPI, OutT>(p, m, ((n0 >> 4) + ctile) / 2 * 16 + 4 * fg, mine[e], mine[e + 1], rs);
        } else if (EPI == EPI_RESID && p.rs_out) {                   // deferred RMSNorm producer: as in the decode kernel (N % 16 == 0)
            f32x4 v = mine[e];
            float ss = 0.f;
            if (m < p.M && nn < p.N) {
                if (p.bias) v += *(const f32x4*)(p.bias + nn);
                float* x = (float*)p.C + (int64_t)m * p.ldc + nn;
                const f32x4 o = old[EPI == EPI_RESID ? e : 0] + p.alpha * v;
                *(f32x4*)x = o;
                act_store4<bf16_t>(p.nrm_xn, m, nn, p.N, o * nrm[EPI == EPI_RESID ? e : 0]);
                ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
            }
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            if (fg == 0 && m < p.M && nn < p.N) p.rs_out[(int64_t)m * (p.N >> 4) + (nn >> 4)] = ss;
        } else if (EPI == EPI_RESID && whole) {
            if (m < p.M && nn < p.N) {
                f32x4 v = mine[e];
                if (p.bias) v += *(const f32x4*)(p.bias + nn);
                *(f32x4*)((float*)p.C + (int64_t)m * p.ldc + nn) = old[EPI == EPI_RESID ? e : 0] + p.alpha * v;
            }
        } else epilogue4<EPI, OutT>(p, m, nn, mine[e], rs);
    }
}

// ------------------------------------------------------------------------------------------
// bf16 skinny kernel (decode: M <= 64 rows).  The projection is then a weight-streaming problem
// (HBM-bound: every weight byte is read once, activations are a few hundred KB in L2), so the
// shape of the kernel is set by memory-level parallelism, not by MFMA:
//   * one workgroup owns NTW 16-row weight tiles (16*NTW output columns) over ALL of K;
//   * it runs NTW*KSPLIT waves; wave w streams tile w/KSPLIT over K slice w%KSPLIT straight
//     HBM -> VGPR with non-temporal 16-byte loads — one contiguous KiB per instruction thanks to the
//     fragment-major layout; no LDS round trip, nothing is shared between waves; two register sets
//     keep the next block of k-steps in flight behind the current block's MFMAs;
//   * activations (<= 64 x K bf16, fragment-major too) are read as MFMA fragments from L2;
//   * the K slices are reduced through LDS in fixed wave order (deterministic, no atomics) and the
//     fused epilogue (bias / residual / SwiGLU / GELU) runs once per output element.  For SwiGLU
//     NTW = 2: tile 0 is the gate block, tile 1 the up block of the same 16 features.
// ------------------------------------------------------------------------------------------
// weight fragments are read once per launch: non-temporal.  In the 64-row-group launches the groups of a weight block
// read them side by side, so there they take the regular path and stay in L2 for the other groups.
template <bool KEEP>
__device__ __forceinline__ bf16x8 weight_load(const bf16x8* p) {
    if constexpr (KEEP) return *p;
    else return __builtin_nontemporal_load(p);
}

// ------------------------------------------------------------------------------------------
// MoE routing (moe.go:57-103) of rows first .. first + n - 1 of a 16-row activation tile by a workgroup of `waves` waves: router logits of the tile (E <= 64
// experts, all of K), softmax, top-k, renormalised weights as the dense gate matrix GemmArgs::moe_gate of the expert projections, or the
// chosen experts in rank order (RouteIds).  A wave takes expert tiles over K slices that lie together (fragments straight from L2 / HBM, as the skinny
// kernel), the K slices are summed through LDS in order, then a wave routes a row with a lane per expert.  The slices are those of sixteen waves whatever
// the launch has, so that a row's logits, and with them near ties between experts, depend neither on the batch nor on prompt or step.
// U k-steps of T expert tiles travel together: few waves need more of them (a lone wave, K = 1024, 32 experts: 4 round trips instead of 16; decode steps
// of 20 rows of 1024 +6 % without).
// p: A (fragment-major operand, possibly the deferred-norm raw form with rs_in), M, K.  smem: MOE_ROUTE_LDS
// ------------------------------------------------------------------------------------------
struct RouteIds { int32_t* ids; float* w; };      // [row][top_k], or NULL
// one row's logits, an expert a lane (-inf beyond them) -> its column of the gate matrix, or the chosen experts in rank order
__device__ __forceinline__ void moe_route_row(const RouteJob& r, const RouteIds& out, int m, float v, int lane) {
    const int E = r.E;
    if (r.logits && lane < E) r.logits[(int64_t)m * r.logits_ld + lane] = v;
    float mx = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    const float e = (lane < E) ? expf(v - mx) : 0.f;
    float sum = e;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) sum += __shfl_xor(sum, o, 64);
    const float prob = (lane < E) ? e / sum : -1.f;
    int rank = 0;                                   // larger first, ties to the lower index (moe.go:75-92)
    const int pbits = __builtin_bit_cast(int, prob), key = score_key(prob);
#pragma unroll 8
    for (int j = 0; j < E; j++) {                   // (lanes >= E hold -1: they never outrank an expert)
        const int kj = __builtin_amdgcn_readlane(key, j);
        rank += (kj > key || (kj == key && j < lane)) ? 1 : 0;
    }
    float wsum = 0.f;
    for (int k = 0; k < r.top_k; k++) {             // moe.go:89-92: fp32 sum in rank order
        const int src = __ffsll((unsigned long long)__ballot(rank == k)) - 1;
        wsum += __builtin_bit_cast(float, __builtin_amdgcn_readlane(pbits, src));
    }
    if (out.ids) {
        if (lane < E && rank < r.top_k) { out.ids[(int64_t)m * r.top_k + rank] = lane; out.w[(int64_t)m * r.top_k + rank] = prob / wsum; }
        return;
    }
    if (lane < E) r.gate[(int64_t)m * r.gate_ld + lane] = rank < r.top_k ? prob / wsum : 0.f;      // moe.go:103
    for (int e2 = E + lane; e2 < r.gate_ld; e2 += 64) r.gate[(int64_t)m * r.gate_ld + e2] = e2 < E + r.n_always ? 1.0f : 0.f;
}
// ALONE: sixteen waves, a slice of a tile and a row each: without the loops a launch of its own takes 5.7 us instead of 6.4 (1 row of 1024, 32 experts; code
// that is fetched cold)
template <int U, int T, bool ALONE = false>
__device__ __forceinline__ void moe_route_rows(const GemmArgs& p, const RouteJob& r, RouteIds out, int tile16, int first, int n, int waves, char* smem) {
    f32x4* red = (f32x4*)smem;                                   // [K slices][expert tiles][64]
    const int E = r.E, ET = (E + 15) >> 4, KW = 16 / ET;         // expert tiles (1 .. 4), K slices
    float* lg = (float*)(smem + 16 * 1024);                      // [16][64]
    // (uniform, and known to be: matrix products heed no lane mask, and a step that a wave does not have is to be jumped over)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const int row0 = tile16 * 16;
    const int nks = p.K >> 5, q = nks / KW, rr = nks - q * KW;
    const bool x_live = row0 + fr < p.M;
    const bf16x8 zero = {};
    auto first_step = [&](int kw) { return kw * q + (kw < rr ? kw : rr); };
    if constexpr (ALONE) {
        static_assert(T == 1, "a tile a wave");
        const int tile = wave % ET, kw = wave / ET;
        const int n = kw < KW ? q + (kw < rr ? 1 : 0) : 0, ks0 = first_step(kw);      // (three tiles leave a wave idle)
        const bf16_t* wp = r.W + (((int64_t)tile * nks + ks0) * 64 + lane) * 8;
        const bf16_t* xp = (const bf16_t*)p.A + (((int64_t)tile16 * nks + ks0) * 64 + lane) * 8;
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        int s = 0;
        for (; s + U <= n; s += U) {
            bf16x8 w[U], x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                w[u] = *(const bf16x8*)(wp + (int64_t)(s + u) * 512);
                x[u] = x_live ? *(const bf16x8*)(xp + (int64_t)(s + u) * 512) : zero;
            }
#pragma unroll
            for (int u = 0; u < U; u++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], x[u], acc, 0, 0, 0);
        }
        for (; s < n; s++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(wp + (int64_t)s * 512), x_live ? *(const bf16x8*)(xp + (int64_t)s * 512) : zero, acc, 0, 0, 0);
        red[wave * 64 + lane] = acc;
    } else {
    const int TS = (ET + T - 1) / T, G = waves >= TS ? waves / TS : 1;          // groups of T tiles, which share a row fragment; waves a group
    for (int it = wave; it < TS * G; it += waves) {
        const int t0 = it % TS * T, part = it / TS, last = (part + 1) * KW / G;
        int kw = part * KW / G;
        const int ks0 = first_step(kw), n = first_step(last) - ks0;
        int slice_end = first_step(kw + 1) - ks0;
        const bf16_t* wp[T];
#pragma unroll
        for (int t = 0; t < T; t++) wp[t] = r.W + (((int64_t)min(t0 + t, ET - 1) * nks + ks0) * 64 + lane) * 8;
        const bf16_t* xp = (const bf16_t*)p.A + (((int64_t)tile16 * nks + ks0) * 64 + lane) * 8;
        f32x4 acc[T];
#pragma unroll
        for (int t = 0; t < T; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto finish = [&](int done) {          // the slices that end here (several of them where K has fewer steps than slices)
            while (kw < last && slice_end == done) {
#pragma unroll
                for (int t = 0; t < T; t++) {
                    if (t0 + t < ET) red[(kw * ET + t0 + t) * 64 + lane] = acc[t];
                    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                kw++;
                slice_end = first_step(kw + 1) - ks0;
            }
        };
        finish(0);
        for (int s = 0; s < n; s += U) {
            bf16x8 w[T][U], x[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int64_t at = (int64_t)min(s + u, n - 1) * 512;
#pragma unroll
                for (int t = 0; t < T; t++) w[t][u] = *(const bf16x8*)(wp[t] + at);
                x[u] = x_live ? *(const bf16x8*)(xp + at) : zero;
            }
#pragma unroll
            for (int u = 0; u < U; u++)
                if (s + u < n) {
#pragma unroll
                    for (int t = 0; t < T; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[t][u], x[u], acc[t], 0, 0, 0);
                    finish(s + u + 1);
                }
        }
    }
    }
    // deferred RMSNorm: the x^2 partials of a row, a lane per 16-byte chunk
    auto sum_squares = [&](int m) {
        const f32x4* src = (const f32x4*)(p.rs_in + (int64_t)m * p.rs_tiles);
        f32x4 a4 = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int c = lane; c < (p.rs_tiles >> 2); c += 64) a4 += src[c];
        float t = (a4[0] + a4[1]) + (a4[2] + a4[3]);
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) t += __shfl_xor(t, o, 64);
        return t;
    };
    const int end = min(n, min(16, p.M - row0) - first);          // rows of this workgroup
    float ssq = p.rs_in && wave < end ? sum_squares(row0 + first + wave) : 0.f;
    __syncthreads();
    for (int t = wave; t < ET; t += waves) {        // acc of lane (fr, fg): row fr, experts 16 t + 4 fg .. + 3
        f32x4 v = red[t * 64 + lane];
#pragma unroll 4
        for (int k = 1; k < KW; k++) v += red[(k * ET + t) * 64 + lane];
        *(f32x4*)(lg + fr * 64 + 16 * t + 4 * fg) = v;
    }
    __syncthreads();
    for (int i = wave; i < end; i += ALONE ? 16 : waves) {
        const int row = first + i, m = row0 + row;
        if (!ALONE && p.rs_in && i != wave) ssq = sum_squares(m);
        const float rstd = p.rs_in ? 1.0f / sqrtf(ssq * p.rs_inv_h + p.rs_eps) : 1.0f;
        moe_route_row(r, out, m, lane < E ? lg[row * 64 + lane] * rstd + (r.bias ? r.bias[lane] : 0.f) : -INFINITY, lane);
        if (ALONE) return;
    }
}
// workgroup `id` of the RouteJob of a launch
template <int U, int T>
__device__ __forceinline__ void moe_route_part(const GemmArgs& p, int id, int waves, char* smem) {
    const int per_tile = cdiv_dev(p.M < 16 ? p.M : 16, p.route.rows), t = id / per_tile;
    moe_route_rows<U, T>(p, p.route, RouteIds{nullptr, nullptr}, t, (id - t * per_tile) * p.route.rows, p.route.rows, waves, smem);
}
// Does a decode batch route inside the experts' up launch?  The launch that this saves is some 8 us (16 rows of 1024 and 32 experts; 2048 and 6 rows: 7.4
// and the gap); not knowing the chosen experts, the up projection streams them all, at 6 TB/s.  Either all that a token leaves out costs little more than
// that, or a batch is expected to leave out next to nothing, were its choices even; but rows that choose alike (answers to one prompt) leave out what
// one does, and may not lose more than others gain.  Us a layer of 32 rows, launch -> beside, 32 experts, 8 a token: 512 x 1024 apart 55.1 -> 53.5, alike
// 44.2 -> 47.8; 512 x 2048 80.9 -> 77.7, 59.8 -> 67.5; not 1024 x 4096 223.9 -> 217.2, 132 -> 181
static inline bool moe_streams_all(int M, int E, int k, double expert_bytes) {
    const double out_us = E > k ? (E - k) * expert_bytes / 6e6 : 0.0, expected_us = E > k ? pow(1.0 - (double)k / E, M) * E * expert_bytes / 6e6 : 0.0;
    return (out_us < 17.0 && expected_us < 1.5) || (out_us < 9.0 && expected_us < 6.0);
}
constexpr size_t MOE_ROUTE_LDS = 20 * 1024;
// ... set up for a launch with workgroups of `waves` waves
static inline void moe_route_share(GemmArgs& a, int waves) {
    a.route.rows = waves >= 8 ? 8 : waves >= 4 ? 4 : 2;
    a.route.wgs = cdiv(a.M, 16) * cdiv(a.M < 16 ? a.M : 16, a.route.rows);
}

// split_finish for one 16 x 16 tile held by one wave (a lane: four columns of a row): its parts are 1 KiB each, [part][tiles] in sk_part.
__device__ __forceinline__ bool split_finish_wave(const GemmArgs& p, int tile, int tiles, int part, int parts, f32x4& v) {
    const int lane = threadIdx.x & 63, voff = lane * 16;
    const auto rs = __builtin_amdgcn_make_buffer_rsrc((char*)p.sk_part, 0, parts * tiles * 1024, 0x00020000);
    union { f32x4 v; u32x4 u; } mine; mine.v = v;
    __builtin_amdgcn_raw_buffer_store_b128(mine.u, rs, voff, __builtin_amdgcn_readfirstlane((part * tiles + tile) * 1024), SPLIT_COHERENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the part has reached memory
    int before = 0;
    if (lane == 0) before = __hip_atomic_fetch_add(p.split_cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(before) != parts - 1) return false;
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(p.split_cnt + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < parts; c0 += 4) {
        union { f32x4 v; u32x4 u; } got[4];
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (c0 + c < parts) got[c].u = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, __builtin_amdgcn_readfirstlane(((c0 + c) * tiles + tile) * 1024), SPLIT_COHERENT);
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (c0 + c < parts) sum += got[c].v;
    }
    v = sum;
    return true;
}
// x += alpha * v for four columns of row m, with the operand and the x^2 partials of the deferred norm that follows
__device__ __forceinline__ void resid_norm_tile(const GemmArgs& p, int m, int n, f32x4 v, const f32x4* x_pre) {
    const int fg = (threadIdx.x >> 4) & 3;
    float ss = 0.f;
    if (m < p.M) {
        float* x = (float*)p.C + (int64_t)m * p.ldc + n;
        const f32x4 o = (x_pre ? *x_pre : *(f32x4*)x) + p.alpha * v;
        *(f32x4*)x = o;
        act_store4<bf16_t>(p.nrm_xn, m, n, p.N, o * *(const f32x4*)(p.nrm_w + n));
        ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
    }
    ss += __shfl_xor(ss, 16, 64);
    if (p.rs_half) {      // (partials per 8 columns)
        if (m < p.M && (fg & 1) == 0) p.rs_out[(int64_t)m * (p.N >> 3) + (n >> 3)] = ss;
        return;
    }
    ss += __shfl_xor(ss, 32, 64);
    if (m < p.M && fg == 0) p.rs_out[(int64_t)m * (p.N >> 4) + (n >> 4)] = ss;
}

// m_passes > 1: block id -> (weight block, 64-row activation group).  Ids that differ by 8 share an XCD and are
// dispatched back to back: the groups of one weight block stream the same weights at the same time.
template <int ROWS = 64>
__device__ __forceinline__ void skinny_pass_remap(GemmArgs& p, int& bx) {
    const int slot = bx >> 3, z = slot % p.m_passes;
    bx = (slot / p.m_passes) * 8 + (bx & 7);
    p.A = (const bf16_t*)p.A + (int64_t)z * ROWS * p.K;    // fragment-major: 16-row tiles are contiguous
    p.c_row0 += z * ROWS;
    p.M = min(ROWS, p.M - z * ROWS);                       // the last group may be ragged (operands are padded to 64 rows)
    if (p.rs_in) p.rs_in += (int64_t)z * ROWS * p.rs_tiles;    // deferred RMSNorm: this group's rows of the x^2 partials
    if (p.rs_out) {                                        // ... and on the producer side (its epilogue indexes rows locally)
        p.C = (float*)p.C + (int64_t)z * ROWS * p.ldc;
        p.nrm_xn += (int64_t)z * ROWS * p.N;
        p.rs_out += (int64_t)z * ROWS * (p.N >> 4);
    }
}

// HALF (deferred-norm residual projections of <= 16 rows: O and FFN-down at decode batches 1..16): a workgroup owns 8 of
// a weight tile's 16 rows, so a 2048-column projection runs on 256 workgroups instead of 128 (x must be complete when the
// launch ends — no K split over workgroups —, and with one workgroup per 16-row tile half of the CUs stayed idle while the
// others pulled 256 KB each through one CU).  The other 8 lanes of every 16-lane row group feed zeros (their loads are
// predicated off: 4 x 128-byte lines per k-step instead of 8); only the owned rows are stored; the x^2 partials are per
// 8 columns (rs_tiles = N / 8).
// EXTRA: a residual projection whose input rows carry a deferred scale of their own (rs_in; SCALED), or with MOE one that completes its K slices
// (rs_out; COMPLETES).  Instances of their own: beside it the others lose 1 %, and the experts' slices 16 % at 40 rows (4096 x 32 x 448:
// 43.9 -> 51 us, their registers spill).
// MOE: 1 masked experts, 2 (up) all experts, the launch's first workgroups route.
template <int MT, int NTW, int U, int EPIV, typename OutT, bool PASSES = false, int MOE = 0, bool HALF = false, bool EXTRA = false>
__global__ __launch_bounds__(skinny_waves(EPIV, MOE == 2 && MT > 1) * 64) void gemm_skinny_bf16_kernel(GemmArgs p) {
    constexpr int EPI = epi_base(EPIV);
    constexpr bool LN = epi_ln(EPIV);
    constexpr bool SCALED = EXTRA && MOE == 0, COMPLETES = EXTRA && MOE != 0;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    f32x4* red = (f32x4*)smem;                       // [NTW][ksplit][MT][64]
    const int swg = blockIdx.y * gridDim.x + blockIdx.x;
    NvlStamps stamps(p.stamps, swg);                 // (diagnostic runs; slot 0: workgroup entered)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ksplit = (blockDim.x >> 6) / NTW;
    const int tile = wave / ksplit, kw = wave - tile * ksplit;
    const int fr = lane & 15, fg = lane >> 4;
    int bx = blockIdx.x;
    if constexpr (PASSES) skinny_pass_remap(p, bx);     // (its own instantiation: rewriting the arguments costs the
                                                        // single-group kernels a few scratch dwords otherwise)
    const int half = HALF ? (bx & 1) : 0;
    if constexpr (HALF) bx >>= 1;
    if constexpr (MOE == 2) {
        if (bx < p.route.wgs) { moe_route_part<4, 1>(p, bx, blockDim.x >> 6, smem); return; }
        bx -= p.route.wgs;
    }
    const bool w_live = !HALF || (fr >> 3) == half;  // HALF: this lane's weight row belongs to the workgroup
    const int nt0 = bx * NTW;                        // first 16-row weight tile of this workgroup
    // K/32 k-steps dealt over (gridDim.y slices) x (ksplit waves) as evenly as possible (K need not divide:
    // Falcon's 4544 = 142 steps)
    const int i_off = p.m_split ? blockIdx.y : 0;                  // first 16-row activation tile of this workgroup
    // deferred RMSNorm (consumer side): the scale of the rows of this wave's first epilogue element, fetched under the weight
    // stream instead of after it.  Issued HERE, ahead of the first weight block.  (Round 3 moved it behind the first block on
    // the evidence of in-kernel time stamps — first weight data 0.5 us earlier — and lost 0.5 us per QKV launch and 0.25 us
    // per FFN-up launch at B = 32 by the kernel trace of the unstamped build: the stamp sites themselves had changed the
    // schedule they measured.  profiles/r03_ab_vs_r02.txt)
    const int i_pre = wave % MT;
    // (MT = 4 — batches above 32 and the 64-row groups of larger ones — has no registers to hold it across the stream:
    // 34-54 spilled there, QKV at 128 rows 7.2 -> 10.8 us; those launches are long enough to fetch it in the epilogue)
    constexpr bool RSTD_PRE = MT <= 2;
    constexpr bool NORMED = EPI == EPI_STORE || EPI == EPI_QKV || SCALED || epi_glu(EPI) || (LN && EPI == EPI_GELU);
    // (layer norms have the registers to add the sums up behind the stream)
    constexpr bool LN_LATE = LN && NORMED;
    RowPairs pairs;
    if constexpr (LN_LATE) pairs.fetch(p.rs_in, p.rs_tiles, 16 * i_pre + fr, 16 * i_pre + fr < p.M && wave < NTW * MT);
    RowNorm rn_pre = (!LN_LATE && RSTD_PRE && NORMED && wave < NTW * MT) ? row_norm<EPIV>(p, 16 * (i_pre + (SCALED ? i_off : 0)) + fr) : RowNorm{1.0f, 0.f};   // (only the waves that run an epilogue element)
    const float rstd_pre = LN ? 1.0f : rn_pre.scale;
    auto row_norm_of = [&](int i) { return (RSTD_PRE || LN_LATE) && i == i_pre ? rn_pre : row_norm<EPIV>(p, 16 * i + fr); };
    // (grid_y: gridDim.y as an explicit argument — the built-in lives in the hidden part of the kernarg block and costs a
    // dependent scalar round trip of its own before the first weight load)
    const int nslices = p.m_split ? 1 : p.grid_y, slice = p.m_split ? 0 : blockIdx.y;
    const int nparts = ksplit * nslices, part = slice * ksplit + kw;
    const int nks = p.K >> 5, q = nks / nparts, rr = nks - q * nparts;
    int my_steps = q + (part < rr ? 1 : 0);
    const int ks0 = part * q + (part < rr ? part : rr);   // first k-step of this wave
    // MoE decode (its own instantiation): stream only the experts some token of the batch picked.  Up: a workgroup's rows belong to one
    // expert.  Down: a wave's K range is exactly one expert (launch_gemm_skinny_ntw), of any width; without a token it has nothing to stream.
    // Its rows' routing weights wait in LDS for the sums (in a register they spill others of the instances of several row tiles).
    float* gates = (float*)(smem + NTW * ksplit * MT * 1024) + wave * 64;
    if constexpr (MOE != 0) {
        if (EPI == EPI_RESID) {
            const float g = moe_gate_of(p, part);
            gates[lane] = g;
            my_steps = __builtin_amdgcn_readfirstlane(__any(g != 0.f) ? my_steps : 0);      // (uniform: scalar loops)
        } else if (MOE == 1 && !__any(moe_gate_of(p, (nt0 * 16) / (2 * p.moe_I)) != 0.f)) return;          // (whole workgroup: uniform)
    }

    // EPI_QKV: the workgroup's two tiles are half a head apart (they rotate together)
    const int q_half = EPI == EPI_QKV ? p.qkv.hd >> 5 : 0, q_head = EPI == EPI_QKV ? bx / q_half : 0, q_tile = bx - q_head * q_half;
    const int wt = EPI == EPI_QKV ? q_head * 2 * q_half + q_tile + tile * q_half : nt0 + tile;
    const bf16_t* wp = (const bf16_t*)p.W + (((int64_t)wt * (p.K >> 5) + ks0) * 64 + lane) * 8;
    const bf16_t* xp[MT];
#pragma unroll
    for (int i = 0; i < MT; i++)   // rows >= M of the last 16-row tile exist (padded allocation) and are never stored
        xp[i] = (const bf16_t*)p.A + (((int64_t)(i + i_off) * (p.K >> 5) + ks0) * 64 + lane) * 8;
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Only the lanes of rows < M fetch their activation fragment (the rest feed zeros: their output columns are never
    // stored).  The CU's ingest rate, not HBM, bounds these kernels, and at M = 1 a padded 16-row fragment would be as
    // many bytes as the weight fragment beside it (M <= 4: a quarter of it with the mask, four 64-byte sectors).
    bool x_live[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) x_live[i] = !p.x_mask || 16 * (i + i_off) + fr < p.M;   // (x_mask: the host sets it when M % 16 != 0)
    const bf16x8 x_zero = {};

    // k loop: blocks of U k-steps (U*32 of K), two register sets -> the next block's loads are in
    // flight while the current block's MFMAs issue (the compiler emits counted vmcnt for these).
    const int nblk = my_steps / U;
    bf16x8 wA[U], xA[U][MT], wB[U], xB[U][MT];
    // carried layer norm: the mean row of U steps, and the rest of it, as rows 0, 2, .. and 1, 3, .. of one weight tile.  Step u's product is right in its two
    // rows of an accumulator of its own, and the others are not looked at (a load a step instead, GPT-2, us a step of 1 / 40 sequences: 361 -> 373, 492 -> 498)
    constexpr bool LN_SHIFT = LN && EPI == EPI_RESID;
    static_assert(!LN_SHIFT || (U == 4 && MT == 1), "rows of four steps");
    f32x4 mean_acc[U];
    if constexpr (LN_SHIFT)
#pragma unroll
        for (int u = 0; u < U; u++) mean_acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8* cp = LN_SHIFT ? (const bf16x8*)p.ln.added.w + (int64_t)ks0 * 8 + (fr & 7) * 4 + fg : nullptr;
    bf16x8 cA, cB;
    auto load_blk = [&](bf16x8 (&w)[U], bf16x8 (&x)[U][MT], bf16x8& c, int b) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if constexpr (HALF) w[u] = w_live ? weight_load<PASSES>((const bf16x8*)(wp + (int64_t)(b * U + u) * 512)) : x_zero;
            else w[u] = weight_load<PASSES>((const bf16x8*)(wp + (int64_t)(b * U + u) * 512));
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const bf16x8* src = (const bf16x8*)(xp[i] + (int64_t)(b * U + u) * 512);
                if (p.x_mask) x[u][i] = x_live[i] ? *src : x_zero; else x[u][i] = *src;      // (uniform branch)
            }
        }
        if constexpr (LN_SHIFT) c = cp[b * U * 8];
    };
    auto comp_blk = [&](bf16x8 (&w)[U], bf16x8 (&x)[U][MT], bf16x8& c) {
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int i = 0; i < MT; i++)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], x[u][i], acc[i], 0, 0, 0);
            if constexpr (LN_SHIFT) mean_acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c, x[u][0], mean_acc[u], 0, 0, 0);
        }
    };
    // carried layer norms: the steps behind the last whole block are on their way beside it.  One after the other behind it, GPT-2's six steps a wave waited for memory
    // three times: us by events, 8 rows, 3072 x 768 8.1 -> 7.2; a prompt of 11 tokens 484 -> 453 us, a step of 1 / 8 / 24 / 48 sequences 372 -> 352, 409 -> 380,
    // 461 -> 437, 557 -> 546.  The others have no such widths and lose by the code alone (Falcon-7B, 142 steps a wave, 37.8 -> 40.3 us a launch; Llama-3.2-1B steps
    // 1 %), and spill where they have several row tiles and 128 registers
    constexpr bool TAIL = LN;
    const int tail = TAIL ? __builtin_amdgcn_readfirstlane(my_steps - nblk * U) : 0;      // (uniform: matrix products heed no lane mask)
    auto load_tail = [&](bf16x8 (&w)[U], bf16x8 (&x)[U][MT], bf16x8& c) {
#pragma unroll
        for (int u = 0; u < U - 1; u++)
            if (u < tail) {
                const int64_t at = (int64_t)(nblk * U + u) * 512;
                w[u] = w_live ? weight_load<PASSES>((const bf16x8*)(wp + at)) : x_zero;
#pragma unroll
                for (int i = 0; i < MT; i++) x[u][i] = x_live[i] ? *(const bf16x8*)(xp[i] + at) : x_zero;
            }
        if constexpr (LN_SHIFT) c = cp[nblk * U * 8];
    };
    auto comp_tail = [&](bf16x8 (&w)[U], bf16x8 (&x)[U][MT], bf16x8& c) {
#pragma unroll
        for (int u = 0; u < U - 1; u++)
            if (u < tail) {
#pragma unroll
                for (int i = 0; i < MT; i++) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], x[u][i], acc[i], 0, 0, 0);
                if constexpr (LN_SHIFT) mean_acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c, x[u][0], mean_acc[u], 0, 0, 0);
            }
    };
    if (nblk > 0) load_blk(wA, xA, cA, 0);
    else if (tail) load_tail(wA, xA, cA);
    stamps.mark(1);                     // first block of loads issued
    // the residual operand of this wave's first epilogue element (deferred-norm producer form): fetched under the weight
    // stream, not as a dependent round trip after the K reduction (this launch is the only writer of these elements)
    f32x4 x_pre = f32x4{0.f, 0.f, 0.f, 0.f};
    if (EPI == EPI_RESID && (!MOE || COMPLETES) && p.rs_out && wave < NTW * MT) {
        const int t = wave / MT, i = wave - t * MT;
        const int m = 16 * (i + i_off) + fr, n = (nt0 + t) * 16 + 4 * fg;
        if (m < p.M && n < p.N && (!HALF || (fg >> 1) == half)) x_pre = *(const f32x4*)((const float*)p.C + (int64_t)m * p.ldc + n);
    }
    float ln_shift = 0.f;      // (MT = 1: one row tile)
    if constexpr (LN_SHIFT) {
        static_assert(MT == 1 && NTW == 1, "one epilogue element");
        const int m = 16 * i_off + fr;
        const bool live = wave == 0 && m < p.M;
        if (live) ln_shift = p.ln.mean_in[m];
        pairs.fetch(p.ln.prev, p.rs_tiles, m, live && p.ln.prev);
    }
    if constexpr (MOE != 0 && EPI == EPI_RESID) {
        for (int b = 0; b < nblk; b += 2) {
            if (b + 1 < nblk) load_blk(wB, xB, cB, b + 1);
            comp_blk(wA, xA, cA);
            if (b + 1 >= nblk) break;
            if (b + 2 < nblk) load_blk(wA, xA, cA, b + 2);
            comp_blk(wB, xB, cB);
        }
        if (tail) {
            if (nblk > 0) load_tail(wA, xA, cA);
            comp_tail(wA, xA, cA);
        }
    } else {
    int b = 0;
    for (; b + 2 <= nblk; b += 2) {
        load_blk(wB, xB, cB, b + 1);
        comp_blk(wA, xA, cA);
        if (b == 0) stamps.mark_used(2, acc[0]);       // first block's data arrived and was used
        if (b + 2 < nblk) load_blk(wA, xA, cA, b + 2);
        else if (tail) load_tail(wA, xA, cA);
        comp_blk(wB, xB, cB);
    }
    if (b < nblk) {
        if (tail) load_tail(wB, xB, cB);
        comp_blk(wA, xA, cA);
        if (tail) comp_tail(wB, xB, cB);
    } else if (tail) comp_tail(wA, xA, cA);
    }
    if constexpr (!TAIL)
    for (int s = nblk * U; s < my_steps; s++) {
        const bf16x8 w = w_live ? weight_load<PASSES>((const bf16x8*)(wp + (int64_t)s * 512)) : x_zero;
#pragma unroll
        for (int i = 0; i < MT; i++)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, x_live[i] ? *(const bf16x8*)(xp[i] + (int64_t)s * 512) : x_zero, acc[i], 0, 0, 0);
    }

    if constexpr (MOE != 0 && EPI == EPI_RESID)
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const float g = gates[16 * i + fr];
            acc[i] = g != 0.f ? acc[i] * g : f32x4{0.f, 0.f, 0.f, 0.f};       // (0: not routed, whatever the expert made of the row)
        }
    if constexpr (LN_LATE) rn_pre = layer_norm_of(p, pairs.sum());
    float* mean_red = (float*)(smem + ksplit * 1024);      // [16][8][2]
    if constexpr (LN_SHIFT) {
        ln_shift += pairs.sum()[0] * p.rs_inv_h;
        const f32x4 even = fg ? mean_acc[2] : mean_acc[0], odd = fg ? mean_acc[3] : mean_acc[1];
        if (fg < 2) mean_red[(fr * 8 + kw) * 2 + fg] = (even[0] + even[1]) + (odd[2] + odd[3]);
    }
    // ---- reduce the K slices in wave order ----
#pragma unroll
    for (int i = 0; i < MT; i++) red[((tile * ksplit + kw) * MT + i) * 64 + lane] = acc[i];
    stamps.mark(3);                     // wave 0's stream done
    __syncthreads();
    stamps.mark(4);                     // every wave's stream done
    if constexpr (LN_SHIFT) {
        static_assert(skinny_waves(EPIV) == 8, "four reads a row");
        const f32x4* sums = (const f32x4*)(mean_red + fr * 16);
        float added = 0.f;
#pragma unroll
        for (int w = 0; w < 8; w += 2) {
            const f32x4 v = sums[w >> 1];
            added += w < ksplit ? v[0] + v[1] : 0.f;
            added += w + 1 < ksplit ? v[2] + v[3] : 0.f;
        }
        ln_shift += p.alpha * (added + p.ln.added.b);
        if (blockIdx.x == 0 && wave == 0 && fg == 0 && 16 * i_off + fr < p.M) p.ln.mean_out[16 * i_off + fr] = ln_shift;
    }
    auto ksum = [&](int t, int i) {
        f32x4 s = red[((t * ksplit) * MT + i) * 64 + lane];
        for (int w = 1; w < ksplit; w++) s += red[((t * ksplit + w) * MT + i) * 64 + lane];
        return s;
    };
    if (epi_glu(EPI)) {
        for (int i = wave; i < MT; i += NTW * ksplit) {
            const int f = (nt0 >> 1) * 16 + 4 * fg;    // NTW == 2: tiles [gate 16 | up 16] of features 8*nt0..
            epilogue_glu4<EPI, OutT, MOE != 0>(p, 16 * i + fr, f, ksum(0, i), ksum(NTW - 1, i),
                                        RSTD_PRE && i == i_pre ? rstd_pre : deferred_rstd(p, 16 * i + fr));
        }
    } else if constexpr (EPI == EPI_QKV) {
        for (int i = wave; i < MT; i += NTW * ksplit) {
            const RowNorm rn = row_norm_of(i);
            const int n = q_head * p.qkv.hd + q_tile * 16 + 4 * fg;
            epilogue_qkv_pair(p, 16 * i + fr, q_head, q_tile * 16 + 4 * fg, normed<EPIV>(p, n, ksum(0, i), rn), normed<EPIV>(p, n + (p.qkv.hd >> 1), ksum(NTW - 1, i), rn));
        }
    } else if (EPI == EPI_RESID && nslices > 1) {
        // split-K across workgroups: publish the partial tile (slice 0 carries the bias); the following norm
        // kernel adds the slices into x in slice order
        for (int e = wave; e < NTW * MT; e += NTW * ksplit) {
            const int t = e / MT, i = e - t * MT;
            const int m = 16 * i + fr, n = (nt0 + t) * 16 + 4 * fg;
            if constexpr (COMPLETES) {
                f32x4 v = ksum(t, i);
                const int n16 = p.N >> 4;
                if (nt0 + t < n16 && split_finish_wave(p, i * n16 + nt0 + t, n16 * MT, slice, nslices, v)) resid_norm_tile(p, m, n, v, e == wave ? &x_pre : nullptr);
                continue;
            }
            if (m >= p.M || n >= p.N) continue;
            f32x4 v = ksum(t, i);
            if (p.bias && slice == 0) v += *(const f32x4*)(p.bias + n);    // N % 4 == 0 for residual widths
            *(f32x4*)(p.sk_part + ((int64_t)slice * p.M + m) * p.N + n) = v;
        }
    } else if (EPI == EPI_RESID && p.rs_out) {
        // x += alpha * (acc + bias) in place, and the deferred-RMSNorm operand + x^2 partials for the next projection
        for (int e = wave; e < NTW * MT; e += NTW * ksplit) {
            const int t = e / MT, i = e - t * MT;
            const int m = 16 * (i + i_off) + fr, n = (nt0 + t) * 16 + 4 * fg;      // N % 16 == 0 (hidden width)
            f32x4 v = ksum(t, i);
            if constexpr (SCALED) v *= rstd_pre;      // (MT = 1: one row tile)
            float ss = 0.f, sx = 0.f;
            if (m < p.M && n < p.N && (!HALF || (fg >> 1) == half)) {
                if (p.bias) v += *(const f32x4*)(p.bias + n);
                float* x = (float*)p.C + (int64_t)m * p.ldc + n;
                const f32x4 o = (e == wave ? x_pre : *(f32x4*)x) + p.alpha * v;
                *(f32x4*)x = o;
                if constexpr (LN) {
                    const f32x4 c = o - ln_shift;
                    act_store4<bf16_t>(p.nrm_xn, m, n, p.N, c * *(const f32x4*)(p.nrm_w + n));
                    ss = c[0] * c[0] + c[1] * c[1] + c[2] * c[2] + c[3] * c[3];
                    sx = (c[0] + c[1]) + (c[2] + c[3]);
                } else {
                act_store4<bf16_t>(p.nrm_xn, m, n, p.N, o * *(const f32x4*)(p.nrm_w + n));
                ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
                }
            }
            ss += __shfl_xor(ss, 16, 64);
            if constexpr (LN) {
                sx += __shfl_xor(sx, 16, 64);
                const int tiles = p.N >> (HALF ? 3 : 4), tile = HALF ? 2 * (nt0 + t) + half : nt0 + t;
                if constexpr (!HALF) { ss += __shfl_xor(ss, 32, 64); sx += __shfl_xor(sx, 32, 64); }
                if (fg == (HALF ? 2 * half : 0) && m < p.M && (nt0 + t) * 16 < p.N) *(f32x2*)(p.rs_out + 2 * ((int64_t)m * tiles + tile)) = f32x2{sx, ss};
                continue;
            }
            if constexpr (HALF) {     // the two lane rows (fg = 2 half, 2 half + 1) of this workgroup's 8 columns
                if (fg == 2 * half && (nt0 + t) * 16 < p.N) p.rs_out[(int64_t)m * (p.N >> 3) + 2 * (nt0 + t) + half] = ss;
                continue;
            }
            ss += __shfl_xor(ss, 32, 64);
            if (fg == 0 && (nt0 + t) * 16 < p.N) p.rs_out[(int64_t)m * (p.N >> 4) + (nt0 + t)] = ss;
        }
    } else {
        for (int e = wave; e < NTW * MT; e += NTW * ksplit) {
            const int t = e / MT, i = e - t * MT;
            if constexpr (LN) epilogue4<EPI, OutT>(p, 16 * i + fr, (nt0 + t) * 16 + 4 * fg, normed<EPIV>(p, (nt0 + t) * 16 + 4 * fg, ksum(t, i), row_norm_of(i)));
            else epilogue4<EPI, OutT>(p, 16 * i + fr, (nt0 + t) * 16 + 4 * fg, ksum(t, i),
                                 EPI != EPI_STORE ? 1.0f : (RSTD_PRE && i == i_pre ? rstd_pre : deferred_rstd(p, 16 * i + fr)));
        }
    }
}

#ifndef NVL_GEMM_INST
// ------------------------------------------------------------------------------------------
// MoE routing as a launch of its own (moe_route_rows): prompts, which need the chosen experts before their rows can be sorted, and decode batches that leave
// some experts alone.  grid = 16-row tiles of the batch x ROUTE_ROWS of their rows: the
// logits of a tile are cheap, 96 KiB from L2, and the ranking is serial (at 16 rows all of them in one workgroup 8.4 us, eight 7.2, four 7.0;
// at 6 rows two workgroups lose 0.3).
// ------------------------------------------------------------------------------------------
constexpr int ROUTE_ROWS = 8;
static inline dim3 router_gate_grid(int M) { return dim3(cdiv(M, 16), cdiv(M < 16 ? M : 16, ROUTE_ROWS)); }
// prefill: ids / weights, all 16 rows of a tile in a workgroup (enough workgroups without)
static __global__ __launch_bounds__(1024) void moe_router_gate_kernel(GemmArgs p, RouteJob job, RouteIds out) {
    __shared__ __attribute__((aligned(16))) char smem[MOE_ROUTE_LDS];
    const int rows = out.ids ? 16 : ROUTE_ROWS;
    moe_route_rows<4, 1, true>(p, job, out, blockIdx.x, blockIdx.y * rows, rows, 16, smem);
}
#endif

// ------------------------------------------------------------------------------------------
// fp32 kernel (parity mode): 64x64 tile, BK=16, 256 threads, 4x4 outputs per thread, k ascending.
// The gated epilogues are not instantiated: the f32 path keeps W1 un-interleaved and applies the
// activation with swiglu_kernel.
// ------------------------------------------------------------------------------------------
template <int EPI, typename OutT>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GemmArgs p) {
    __shared__ float As[16][64 + 4];
    __shared__ float Ws[16][64 + 4];
    const int tid = threadIdx.x;
    const int tiles_n = (p.N + 63) / 64;
    const int tn = blockIdx.x % tiles_n, tm = blockIdx.x / tiles_n;
    const int m0 = tm * 64, n0 = tn * 64;
    const int tx = tid & 15, ty = tid >> 4;   // thread -> n = n0 + 4*tx.., m = m0 + 4*ty..
    int row_base = 0;
    if (p.seg) {
        row_base = p.seg[0];
        p.M = p.seg[1] - row_base;
        p.c_row0 = row_base;
    }
    if (m0 >= p.M) return;
    // (the f32 parity path keeps one launch per expert through `seg`; tile_map is bf16-only)

    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.f;

    // each thread stages one float4 of A and one of W per k-step: row = tid/4, k = (tid%4)*4
    const int lrow = tid >> 2, lk = (tid & 3) * 4;
    int am = m0 + lrow;
    if (am > p.M - 1) am = p.M - 1;
    am += row_base;
    if (p.a_rows) am = p.a_rows[am];
    const float* ap = (const float*)p.A + (int64_t)am * p.lda + lk;
    const float* wp = (const float*)p.W + (int64_t)(n0 + lrow) * p.K + lk;   // W has N_pad (x128) rows

    for (int k0 = 0; k0 < p.K; k0 += 16) {
        const f32x4 av = *(const f32x4*)(ap + k0);
        const f32x4 wv = *(const f32x4*)(wp + k0);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            As[lk + r][lrow] = av[r];
            Ws[lk + r][lrow] = wv[r];
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; kk++) {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = Ws[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const f32x4 v = {acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
        epilogue4<EPI, OutT>(p, m0 + ty * 4 + i, n0 + tx * 4, v);
    }
}

// ------------------------------------------------------------------------------------------
// host launchers
// ------------------------------------------------------------------------------------------
// ------------------------------------------------------------------------------------------
// bf16 skinny kernel, wide-N form (decode projections with >= 256 groups of 64 weight rows: FFN up, LM head).
// A wave owns NTB 16-row weight tiles over its K slice, so every activation fragment it fetches from L2 feeds
// NTB MFMAs instead of one: L2->CU traffic per weight byte drops from 1 + MT to 1 + MT/NTB (the activation
// fetches were costing ~15 % of the streaming rate, r01 probe).  8 waves per workgroup (256-VGPR budget): two
// register sets of U k-steps x (NTB weight + MT activation) fragments — for K = 2048 a wave's whole slice is in
// flight at once.  Same deterministic in-LDS K reduction and fused epilogues as the narrow form.  launch_gemm_rows runs it over row groups of 32 .. 64.
// ------------------------------------------------------------------------------------------
template <int MT, int NTB, int U, int EPI, typename OutT, bool PASSES = false, int MOE = 0>
__global__ __launch_bounds__(512) void gemm_skinny_wide_bf16_kernel(GemmArgs p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    f32x4* red = (f32x4*)smem;                       // [ksplit][NTB][MT][64]
    const int swg = blockIdx.x;
    NvlStamps stamps(p.stamps, swg);
    const int tid = threadIdx.x, lane = tid & 63, kw = tid >> 6;
    const int ksplit = blockDim.x >> 6;
    const int fr = lane & 15, fg = lane >> 4;
    int bx = blockIdx.x;
    if constexpr (PASSES) skinny_pass_remap<16 * MT>(p, bx);     // (its own instantiation: rewriting the arguments costs the
                                                        // single-group kernels a few scratch dwords otherwise)
    if constexpr (MOE == 2) {
        if (bx < p.route.wgs) { moe_route_part<8, 2>(p, bx, ksplit, smem); return; }
        bx -= p.route.wgs;
    }
    const int nt0 = bx * NTB;
    if constexpr (MOE == 1) { if (!__any(moe_gate_of(p, (nt0 * 16) / (2 * p.moe_I)) != 0.f)) return; }      // MoE decode: untouched expert (uniform)
    const int nks = p.K >> 5, q = nks / ksplit, rr = nks - q * ksplit;
    const int my_steps = q + (kw < rr ? 1 : 0);
    const int ks0 = kw * q + (kw < rr ? kw : rr);
    const int64_t tile_stride = (int64_t)nks * 512;  // elements between consecutive 16-row weight tiles
    // deferred RMSNorm: the scale of the rows this wave's epilogue elements belong to, fetched under the weight stream
    // (ahead of the first weight block: see the narrow kernel)
    const int i_pre = kw % MT;
    const float rstd_pre = (epi_glu(EPI) || EPI == EPI_STORE) ? deferred_rstd(p, 16 * i_pre + fr) : 1.0f;
    const bf16_t* wp = (const bf16_t*)p.W + (((int64_t)nt0 * nks + ks0) * 64 + lane) * 8;
    const bf16_t* xp = (const bf16_t*)p.A + ((int64_t)ks0 * 64 + lane) * 8;
    f32x4 acc[NTB][MT];
#pragma unroll
    for (int t = 0; t < NTB; t++)
#pragma unroll
        for (int i = 0; i < MT; i++) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // (no row mask here, unlike the narrow kernel: this form runs at 17..64 rows, where at most one tile is ragged, and its
    // 256-register budget is full — the predicated loads cost 6 more spilled registers and 2 us per FFN-up launch at B = 32)
    const int nblk = my_steps / U;
    bf16x8 wA[U][NTB], xA[U][MT], wB[U][NTB], xB[U][MT];
    auto load_blk = [&](bf16x8 (&w)[U][NTB], bf16x8 (&x)[U][MT], int b) {
#pragma unroll
        for (int u = 0; u < U; u++) {
#pragma unroll
            for (int t = 0; t < NTB; t++)
                w[u][t] = weight_load<PASSES>((const bf16x8*)(wp + t * tile_stride + (int64_t)(b * U + u) * 512));
#pragma unroll
            for (int i = 0; i < MT; i++) x[u][i] = *(const bf16x8*)(xp + i * tile_stride + (int64_t)(b * U + u) * 512);
        }
    };
    auto comp_blk = [&](bf16x8 (&w)[U][NTB], bf16x8 (&x)[U][MT]) {
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int t = 0; t < NTB; t++)
#pragma unroll
                for (int i = 0; i < MT; i++)
                    acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][t], x[u][i], acc[t][i], 0, 0, 0);
    };
    if (nblk > 0) load_blk(wA, xA, 0);
    stamps.mark(1);
    // (residual: the old values of this wave's epilogue element come under the stream)
    f32x4 x_pre = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (EPI == EPI_RESID) {
        const int t = kw / MT, m = 16 * (kw - t * MT) + fr, n = (nt0 + t) * 16 + 4 * fg;
        if (t < NTB && m < p.M && n < p.N) x_pre = *(const f32x4*)((const float*)p.C + (int64_t)(p.rs_out ? m : p.c_row0 + m) * p.ldc + n);
    }
    int b = 0;
    for (; b + 2 <= nblk; b += 2) {
        load_blk(wB, xB, b + 1);
        comp_blk(wA, xA);
        if (b == 0) stamps.mark_used(2, acc[0][0]);
        if (b + 2 < nblk) load_blk(wA, xA, b + 2);
        comp_blk(wB, xB);
    }
    if (b < nblk) comp_blk(wA, xA);
    for (int s = nblk * U; s < my_steps; s++) {      // ragged tail
        bf16x8 xs[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) xs[i] = *(const bf16x8*)(xp + i * tile_stride + (int64_t)s * 512);
#pragma unroll
        for (int t = 0; t < NTB; t++) {
            const bf16x8 w = weight_load<PASSES>((const bf16x8*)(wp + t * tile_stride + (int64_t)s * 512));
#pragma unroll
            for (int i = 0; i < MT; i++) acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, xs[i], acc[t][i], 0, 0, 0);
        }
    }

#pragma unroll
    for (int t = 0; t < NTB; t++)
#pragma unroll
        for (int i = 0; i < MT; i++) red[((kw * NTB + t) * MT + i) * 64 + lane] = acc[t][i];
    stamps.mark(3);
    __syncthreads();
    stamps.mark(4);
    auto ksum = [&](int t, int i) {
        f32x4 s = red[(t * MT + i) * 64 + lane];
        for (int w = 1; w < ksplit; w++) s += red[((w * NTB + t) * MT + i) * 64 + lane];
        return s;
    };
    if (epi_glu(EPI)) {
        // tiles come as [gate16 | up16] pairs of the same 16 features
        for (int e = kw; e < (NTB / 2) * MT; e += ksplit) {
            const int j = e / MT, i = e - j * MT;
            const int f = ((nt0 >> 1) + j) * 16 + 4 * fg;
            epilogue_glu4<EPI, OutT, MOE != 0>(p, 16 * i + fr, f, ksum(2 * j, i), ksum(2 * j + 1, i),
                                        i == i_pre ? rstd_pre : deferred_rstd(p, 16 * i + fr));
        }
    } else {
        for (int e = kw; e < NTB * MT; e += ksplit) {
            const int t = e / MT, i = e - t * MT;
            if constexpr (EPI == EPI_RESID) {
                f32x4 v = ksum(t, i);
                const int m = 16 * i + fr, n = (nt0 + t) * 16 + 4 * fg;
                if (p.bias) v += *(const f32x4*)(p.bias + n);
                if (p.rs_out) resid_norm_tile(p, m, n, v, e == kw ? &x_pre : nullptr);
                else if (m < p.M) {
                    float* x = (float*)p.C + (int64_t)(p.c_row0 + m) * p.ldc + n;
                    *(f32x4*)x = (e == kw ? x_pre : *(f32x4*)x) + p.alpha * v;
                }
                continue;
            }
            epilogue4<EPI, OutT>(p, 16 * i + fr, (nt0 + t) * 16 + 4 * fg, ksum(t, i),
                                 EPI != EPI_STORE ? 1.0f : (i == i_pre ? rstd_pre : deferred_rstd(p, 16 * i + fr)));
        }
    }
}

inline int g_chunk_max_m = 512;    // largest M that uses 64-row passes of the decode form at all (nvl_set_tuning key 11; 64 = off)
inline int g_chunk_all_m = 64;     // up to here every projection does; above, only those whose 128x128 tile grid would
                                   // have fewer than g_chunk_min_tiles workgroups (keys 14, 12).  Measured: the mix wins
                                   // from 96 rows on (profiles/r01g_large_decode_batches.txt)
inline int g_pass_interleave = 1;   // 64-row groups of one projection in ONE launch (key 13; 0 = one launch per group)
inline int g_chunk_min_tiles = 160;
inline int g_msplit_ks = 8;         // K split of the deferred-norm residual projections (nvl_set_tuning key 6)
inline int g_narrow_waves = 2048;   // waves per narrow-form launch (nvl_set_tuning key 5).  Round-2 sweep on the final kernels
                                    // (profiles/r02_narrow_waves_sweep.txt): 2048 vs 1024: B=1 +5.4 %, B=8 +5.0 %, B=16 +2.4 %,
                                    // B=32 flat; 4096 = 2048.  (Round 1, before the activation-row mask: 1024 beat 4096 by 3-8 %.)
inline int g_wide_ksplit = 0;   // experiment (nvl_set_tuning key 4): K split of the wide form when groups <= 512
inline int g_x_mask = 1;            // nvl_set_tuning key 24: decode kernels skip the activation fetch of padded rows (M % 16 != 0)
inline int g_force_ntw = 0, g_force_ksplit = 0;   // tuning overrides (nvl_bench_gemm only)
inline int g_force_tile = 0;                      // 0 automatic, 1: 128x128 (ring), 2: 256x128 (ring), 3: 256x256x2st, 5: ping-pong 256x256

template <int EPI, typename OutT>
static inline bool launch_gemm_skinny_bf16(hipStream_t st, const GemmArgs& a);
constexpr int DEFER_MAX_M = 128;    // deferred RMSNorm (decode): rows of the x^2 partial buffer.  Above 64 rows the producer
                                    // runs as 64-row groups like every narrow projection (one workgroup per 16-row tile
                                    // was measured at M = 128: -13 %); above 128 rows FFN-up belongs on the tile kernels
static inline int skinny_rows(const GemmArgs& a) { return a.m_passes > 1 && a.M > 64 ? 64 : a.M; }   // rows a workgroup covers
// the groups of 64 rows as separate launches (weight-block count not a multiple of 8, or key 13 = 0)
template <int EPI, typename OutT>
static inline bool launch_skinny_passes_serial(hipStream_t st, const GemmArgs& a) {
    for (int r0 = 0; r0 < a.M; r0 += 64) {
        GemmArgs c = a;
        c.m_passes = 0;
        c.A = (const bf16_t*)a.A + (int64_t)r0 * a.K;
        c.M = a.M - r0 < 64 ? a.M - r0 : 64;
        c.c_row0 = a.c_row0 + r0;
        if (a.rs_in) c.rs_in = a.rs_in + (int64_t)r0 * a.rs_tiles;
        if (a.rs_out) {
            c.C = (float*)a.C + (int64_t)r0 * a.ldc; c.nrm_xn = a.nrm_xn + (int64_t)r0 * a.N;
            c.rs_out = a.rs_out + (int64_t)r0 * (a.N >> 4);
        }
        if (!launch_gemm_skinny_bf16<EPI, OutT>(st, c)) return false;
    }
    return true;
}

// skinny dispatch: M <= 64, no gather/segments.  Returns false when the shape is not eligible.
template <int NTW, int EPI, typename OutT>
static inline bool launch_gemm_skinny_ntw(hipStream_t st, const GemmArgs& a) {
    const int MT = skinny_rows(a) <= 16 ? 1 : (skinny_rows(a) <= 32 ? 2 : 4);
    if (EPI == EPI_RESID && a.m_split && a.rs_out && NTW == 1 && a.m_passes <= 1 && a.grid_y != 1) {   // (m_split: grid_y unused, keep it defined)
        GemmArgs c = a; c.grid_y = 1; return launch_gemm_skinny_ntw<NTW, EPI, OutT>(st, c);
    }
    const int U = MT <= 2 ? 4 : 2;                       // register budget: (1+MT)*U*2 fragments
    const int nblocks = cdiv(cdiv(a.N, 16), NTW);        // weight rows are padded to 128: all tiles exist
    const int KS = (EPI == EPI_RESID && a.sk_part && a.sk_slices > 1) ? a.sk_slices : 1;
    if (EPI == EPI_RESID && a.m_split && a.rs_out && NTW == 1 && a.m_passes <= 1) {
        // deferred-norm residual projection: one workgroup per (weight tile, 16-row activation tile), all of K each
        int ks = g_msplit_ks;
        while (ks > 1 && (a.K >> 5) / ks < 4) ks >>= 1;
        if (a.K % 32 != 0) return false;
        if constexpr (EPI == EPI_RESID) {
            if (a.rs_in) {        // (the output projection of a Mamba-2 step)
                if (a.rs_half) {
                    if (a.M > 16) return false;
                    hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, NTW, 4, EPI, OutT, false, false, true, true>), dim3(2 * nblocks, 1), dim3(NTW * ks * 64),
                                       (size_t)NTW * ks * 64 * 16, st, a);
                } else {
                    hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, NTW, 4, EPI, OutT, false, false, false, true>), dim3(nblocks, cdiv(a.M, 16)), dim3(NTW * ks * 64),
                                       (size_t)NTW * ks * 64 * 16, st, a);
                }
                return true;
            }
            if (a.rs_half) {      // <= 16 rows: 8 weight rows per workgroup, twice the workgroups (HALF above)
                if (a.M > 16) return false;
                hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, NTW, 4, EPI, OutT, false, false, true>), dim3(2 * nblocks, 1), dim3(NTW * ks * 64),
                                   (size_t)NTW * ks * 64 * 16, st, a);
                return true;
            }
        }
        hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, NTW, 4, EPI, OutT>), dim3(nblocks, cdiv(a.M, 16)), dim3(NTW * ks * 64),
                           (size_t)NTW * ks * 64 * 16, st, a);
        return true;
    }
    if (EPI == EPI_RESID && !a.moe_gate && (a.rs_half || a.rs_in)) return false;      // (half tiles, scaled rows: the form above alone)
    // waves per launch: enough to cover HBM latency on every CU (~2-4 thousand), not more — extra K slices only
    // shorten each wave's stream below the depth of its two-block pipeline (r01 sweeps: LM head, W1)
    int ksplit = 16;
    if (g_force_ksplit) ksplit = g_force_ksplit;
    else {
        // (the MoE gate/up projection counts every expert's workgroups, but those of experts no token picked exit at once:
        //  twice the budget — Granite-1B B=8 decode 6.50 K -> 6.60 K tok/s, profiles/r03_moe_decode_experiments.txt)
        const int64_t budget = (int64_t)g_narrow_waves * ((a.moe_gate && epi_moe(EPI)) ? 2 : 1);
        while (ksplit > 1 && (int64_t)nblocks * KS * NTW * ksplit > budget) ksplit >>= 1;
    }
    while (ksplit > 1 && ((a.K >> 5) / (ksplit * KS) < U || ksplit * NTW > skinny_waves(EPI, a.moe_gate && epi_moe(EPI) && MT > 1))) ksplit >>= 1;   // >= one block of U k-steps per wave
    if (a.moe_gate && EPI == EPI_RESID) {      // MoE down: every wave's K range is exactly one expert (the skip test needs it)
        ksplit = a.moe_E / KS;
        if (ksplit < 1 || ksplit * KS != a.moe_E || ksplit > 16 || (a.moe_I >> 5) < 1) return false;
    }
    if (a.K % 32 != 0) return false;
    size_t lds = (size_t)NTW * ksplit * MT * 64 * 16;
    if (EPI == EPI_RESID && a.moe_gate) lds += (size_t)NTW * ksplit * 256;      // (routing weights, a row a lane of every wave)
    if (a.m_passes > 1 && (nblocks % 8 != 0 || KS != 1)) return launch_skinny_passes_serial<EPI, OutT>(st, a);
    dim3 grid(nblocks * (a.m_passes > 1 ? a.m_passes : 1), KS), block(NTW * ksplit * 64);
    if (a.grid_y != KS) { GemmArgs c = a; c.grid_y = KS; return launch_gemm_skinny_ntw<NTW, EPI, OutT>(st, c); }
#define NVL_SK(MTv, Uv) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MTv, NTW, Uv, EPI, OutT>), grid, block, lds, st, a)
#define NVL_SKM(MTv, Uv, Xv)                                                                                             \
    do {                                                                                                               \
        NVL_LDS_ATTR((gemm_skinny_bf16_kernel<MTv, NTW, Uv, EPI, OutT, false, 1, false, Xv>), 16 * (MTv * 1024 + 256));     \
        hipLaunchKernelGGL((gemm_skinny_bf16_kernel<MTv, NTW, Uv, EPI, OutT, false, 1, false, Xv>), grid, block, lds, st, a); \
    } while (0)
    if constexpr (epi_moe(EPI) || EPI == EPI_RESID) {
        if (a.moe_gate) {                                 // MoE decode instantiation (expert skip + gate weight)
            if (a.m_passes > 1) return false;
            if constexpr (EPI == EPI_RESID) {
                if (a.rs_out) {
                    if (KS < 2) return false;
                    if (MT == 1) NVL_SKM(1, 4, true); else if (MT == 2) NVL_SKM(2, 4, true); else NVL_SKM(4, 2, true);
                    return true;
                }
            }
            if constexpr (epi_moe(EPI)) {
                if (a.route.W) {
                    GemmArgs c = a;
                    moe_route_share(c, NTW * ksplit);
                    grid.x += c.route.wgs;
                    const size_t room = std::max(lds, MOE_ROUTE_LDS);
                    if (MT == 1) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, NTW, 4, EPI, OutT, false, 2>), grid, block, room, st, c);
                    else if (MT == 2) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<2, NTW, 4, EPI, OutT, false, 2>), grid, block, room, st, c);
                    else hipLaunchKernelGGL((gemm_skinny_bf16_kernel<4, NTW, 2, EPI, OutT, false, 2>), grid, block, room, st, c);
                    return true;
                }
            }
            if (MT == 1) NVL_SKM(1, 4, false); else if (MT == 2) NVL_SKM(2, 4, false); else NVL_SKM(4, 2, false);
            return true;
        }
    }
    if (a.m_passes > 1) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<4, NTW, 2, EPI, OutT, true>), grid, block, lds, st, a);
    else if (MT == 1) NVL_SK(1, 4); else if (MT == 2) NVL_SK(2, 4); else NVL_SK(4, 2);
#undef NVL_SK
#undef NVL_SKM
    return true;
}
// Weight tiles per wave of the wide form (nvl_set_tuning key 36: 0 automatic, 2 / 4 forced).  Four tiles per wave quarter the
// activation fetches per weight byte, but an FFN-up launch is then only 256 workgroups of 2 waves — 64 KiB of weights in
// flight per CU.  Two tiles per wave (512 workgroups) for batches of 17..32 rows: Llama-3.2-1B B=32 decode 33.7 K -> 34.5 K
// tok/s (+2.4 %), B=20 +3.1 %, Falcon-7B B=32 +4.7 %, Llama-3-8B / Granite B=32 +0.8 %; the LM head (thousands of groups
// either way) is indifferent, and 64-row launches (MT = 4) lose 2 % (profiles/r03_wide_tiles_per_wave.txt).
inline int g_wide_ntb = 0;
template <int EPI, typename OutT, int NTB = 4>
static inline bool launch_gemm_skinny_wide(hipStream_t st, const GemmArgs& a) {
    if constexpr (NTB == 4) {
        if (g_wide_ntb == 2 || (g_wide_ntb == 0 && skinny_rows(a) <= 32 && a.N < 65536)) return launch_gemm_skinny_wide<EPI, OutT, 2>(st, a);
    }
    if (a.K % 32 != 0 || a.sk_part) return false;
    const int groups = cdiv(cdiv(a.N, 16), NTB);     // weight rows are padded to 256: every tile of a group exists
    const int MT = skinny_rows(a) <= 16 ? 1 : (skinny_rows(a) <= 32 ? 2 : 4);
    const int U = MT <= 2 ? 4 : 2;
    // ~512 waves per launch (256-VGPR waves, each with up to 32 KiB of weights in flight) stream best from HBM: longer
    // per-wave K slices beat more waves (in the model, weights cold: FFN-up ksplit 2 > 4 > 8 > 1; LM head, 8B FFN-up 2)
    int ksplit = 8;
    if (g_force_ksplit) ksplit = g_force_ksplit <= 8 ? g_force_ksplit : 8;
    else if (g_wide_ksplit && groups <= 512) ksplit = g_wide_ksplit;
    else { while (ksplit > 2 && groups * ksplit > 512) ksplit >>= 1; if (groups >= 1024) ksplit = 1; }   // LM head: one wave per group (cold sweep: 96 vs 104 us)
    while (ksplit > 1 && (a.K >> 5) / ksplit < U) ksplit >>= 1;
    const size_t lds = (size_t)ksplit * NTB * MT * 64 * 16;
    if (a.m_passes > 1 && groups % 8 != 0) return launch_skinny_passes_serial<EPI, OutT>(st, a);
    const int wgs = groups * (a.m_passes > 1 ? a.m_passes : 1);
#define NVL_SKW(MTv, Uv, Pv)                                                                                             \
    do {                                                                                                               \
        NVL_LDS_ATTR((gemm_skinny_wide_bf16_kernel<MTv, NTB, Uv, EPI, OutT, Pv>), 8 * NTB * MTv * 64 * 16);            \
        hipLaunchKernelGGL((gemm_skinny_wide_bf16_kernel<MTv, NTB, Uv, EPI, OutT, Pv>), dim3(wgs), dim3(ksplit * 64),      \
                           lds, st, a);                                                                                \
    } while (0)
#define NVL_SKWM(MTv, Uv, Rv, grid, room, args)                                                                          \
    do {                                                                                                               \
        NVL_LDS_ATTR((gemm_skinny_wide_bf16_kernel<MTv, NTB, Uv, EPI, OutT, false, Rv>), std::max<size_t>(8 * NTB * MTv * 1024, MOE_ROUTE_LDS)); \
        hipLaunchKernelGGL((gemm_skinny_wide_bf16_kernel<MTv, NTB, Uv, EPI, OutT, false, Rv>), dim3(grid), dim3(ksplit * 64), \
                           room, st, args);                                                                            \
    } while (0)
    if constexpr (epi_moe(EPI)) {
        if (a.moe_gate) {
            if (a.m_passes > 1) return false;
            if (a.route.W) {
                GemmArgs c = a;
                moe_route_share(c, ksplit);
                const size_t room = std::max(lds, MOE_ROUTE_LDS);
                if (MT == 1) NVL_SKWM(1, 4, 2, wgs + c.route.wgs, room, c); else if (MT == 2) NVL_SKWM(2, 4, 2, wgs + c.route.wgs, room, c); else NVL_SKWM(4, 2, 2, wgs + c.route.wgs, room, c);
                return true;
            }
            if (MT == 1) NVL_SKWM(1, 4, 1, wgs, lds, a); else if (MT == 2) NVL_SKWM(2, 4, 1, wgs, lds, a); else NVL_SKWM(4, 2, 1, wgs, lds, a);
            return true;
        }
    }
    if (a.m_passes > 1) NVL_SKW(4, 2, true); else if (MT == 1) NVL_SKW(1, 4, false); else if (MT == 2) NVL_SKW(2, 4, false); else NVL_SKW(4, 2, false);
#undef NVL_SKW
#undef NVL_SKWM
    return true;
}
template <int EPI, typename OutT>
static inline bool launch_gemm_skinny_bf16(hipStream_t st, const GemmArgs& a0) {
    constexpr int E = epi_base(EPI);
    if (E == EPI_QKV && (a0.qkv.hd % 32 != 0 || a0.m_passes > 1)) return false;
    if (skinny_rows(a0) > 64 || a0.a_rows || a0.seg || a0.tile_map) return false;
    GemmArgs a = a0;
    a.x_mask = (g_x_mask && a0.M % 16 != 0) ? 1 : 0;     // padded rows of the last 16-row activation tile are not fetched
    if constexpr (epi_glu(EPI) || EPI == EPI_STORE || EPI == EPI_GELU || EPI == EPI_RELU2 || EPI == EPI_GROUPED || EPI == EPI_GROUPED_RAW || EPI == EPI_JOINT) {
        // wide-N form once its 64-row groups fill the chip (g_force_ntw: 8 forces it, 1/2/4 force the narrow form)
        const bool wide_ok = skinny_rows(a) > 16 && cdiv(a.N, 64) >= 256 && !a.sk_part;   // M <= 16: the narrow form streams as fast
        if (g_force_ntw == 8 || (g_force_ntw == 0 && wide_ok)) { if (launch_gemm_skinny_wide<EPI, OutT>(st, a)) return true; }
    }
    if constexpr (epi_glu(EPI) || E == EPI_QKV) return launch_gemm_skinny_ntw<2, EPI, OutT>(st, a);      // (pairs: gate | up, the halves of a head)
    if constexpr (epi_ln(EPI)) return launch_gemm_skinny_ntw<1, EPI, OutT>(st, a);
    if (g_force_ntw == 2) return launch_gemm_skinny_ntw<2, EPI, OutT>(st, a);
    if (g_force_ntw == 4) return launch_gemm_skinny_ntw<4, EPI, OutT>(st, a);
    return launch_gemm_skinny_ntw<1, EPI, OutT>(st, a);
}

// a residual projection that carries a layer norm: as one that carries an RMSNorm, a workgroup per (weight tile, 16-row tile) or half of the former
template <typename OutT>
static inline bool launch_gemm_ln_resid(hipStream_t st, const GemmArgs& a0) {
    if (a0.M > 64 || a0.K % 32 != 0 || !a0.rs_out || (a0.rs_half && a0.M > 16)) return false;
    GemmArgs a = a0;
    a.grid_y = 1;
    a.m_split = 1;
    a.x_mask = (g_x_mask && a.M % 16 != 0) ? 1 : 0;
    int ks = skinny_waves(EPI_LN_RESID);
    while (ks > 1 && (a.K >> 5) / ks < 4) ks >>= 1;
    const int tiles = cdiv(a.N, 16);
    const size_t lds = (size_t)ks * 1024 + 1024;      // (the waves' sums of a tile, and of 16 rows' means)
    if (a.rs_half) hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, 1, 4, EPI_LN_RESID, OutT, false, 0, true>), dim3(2 * tiles, 1), dim3(ks * 64), lds, st, a);
    else hipLaunchKernelGGL((gemm_skinny_bf16_kernel<1, 1, 4, EPI_LN_RESID, OutT>), dim3(tiles, cdiv(a.M, 16)), dim3(ks * 64), lds, st, a);
    return true;
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, int EPI, typename OutT, int BK = G_BK>
static inline void launch_gemm_tile(hipStream_t st, const GemmArgs& a) {
    constexpr int lds = gemm_lds_bytes<BM, BN, STAGES, BK>();
    auto launch = [&](auto slices, int n) {
        constexpr bool SLICES = decltype(slices)::value;
        NVL_LDS_ATTR((gemm_bf16_kernel<BM, BN, WAVES_M, WAVES_N, STAGES, EPI, OutT, BK, SLICES>), lds);
        hipLaunchKernelGGL((gemm_bf16_kernel<BM, BN, WAVES_M, WAVES_N, STAGES, EPI, OutT, BK, SLICES>),
                           dim3(cdiv(a.M, BM) * cdiv(a.N, BN), n), dim3(WAVES_M * WAVES_N * 64), lds, st, a);
    };
    if constexpr (EPI == EPI_RESID) if (a.sk_part) { launch(std::true_type{}, a.sk_slices); return; }
    launch(std::false_type{}, 1);
}

// What a projection takes on the two prefill forms, in microseconds: fitted to 200 launches of 300 .. 16384 rows of 768 .. 28672 x 768 .. 22720, good to
// 11 %; the form that they choose is 0.5 % above the faster one in the mean, 18 % at worst.  Ping-pong 256x256 tiles: a K-step is 0.53 us while
// power does not bind (up to half of the CUs busy) and 0.79 with all of them; the last round's tiles (`rest` of 32 per XCD) may be cut into
// parts, which costs 9.3 + 2.4 us a part.
constexpr int PP_LDS = 4 * 32 * 1024 + 16;
inline int g_pp_split = 0;          // nvl_set_tuning key 41: 0 from the grid, 1 never, n parts
static inline double gemm_epilogue_us(int M, int N, int bytes) { return (double)M * N * bytes / 4.5e6; }
static inline double pp_cost(int M, int N, int K, int out_bytes, bool can_split, int& parts) {
    const int T = cdiv(M, 256) * cdiv(N, 256), n = cdiv(T, 8), rest = n & 31, stages = K >> 5;
    parts = 1;
    double best = 0;
    for (int c = 1; c <= 8 && rest * c <= 32; c++) {
        if (c > 1 && (!can_split || !rest || T < 8 || stages / c < PP_MIN_STAGES || (g_pp_split && c != g_pp_split))) continue;
        const double fill = rest * c / 32.0, t = rest ? (stages / c) * (0.525 + (fill > 0.45 ? 0.41 * (fill - 0.45) : 0.0)) + (c > 1 ? 9.3 + 2.4 * c : 0.0) : 0.0;
        if (c == 1 || t < 0.92 * best || g_pp_split == c) { best = t; parts = c; }
    }
    return (n >> 5) * (stages * 0.79 + 3.0) + best + 0.36 * gemm_epilogue_us(M, N, out_bytes) + 13.7;
}
// 128x128 tiles, up to two workgroups a CU; K in `slices` whose sums somebody else adds up
static inline double tile128_cost(int M, int N, int K, int out_bytes, int slices) {
    const double x = (double)cdiv(M, 128) * cdiv(N, 128) * slices / 256.0, per = x <= 1.0 ? 6.7 + x : x <= 2.0 ? 11.6 + 2.0 * (x - 1.0) : 1.1 + 8.3 * x;
    return K / 1024.0 / slices * per + 7.1 + (slices > 1 ? gemm_epilogue_us(M, N, 8 * slices) : 0.44 * gemm_epilogue_us(M, N, out_bytes));
}
// 64x128 tiles of the ring on four waves of 32x64, where each CU has one at most: twice the CUs at work of a launch of few 128x128 tiles.  us, 128x128 -> here (weights from
// HBM): 600 x 3072 x 2048 22.9 -> 20.1, 900 x 2048 x 2048 23.3 -> 21.2, 520 / 2000 x 768 x 768 11.7 -> 9.1, 12.8 -> 10.1, 900 x 768 x 3072 29.2 -> 25.7, 520 x 2304 x 768 10.9 -> 9.2,
// 900 x 1536 x 1024 12.7 -> 10.5, 260 x 6144 x 4096 39.7 -> 33.8; not two a CU (1100 x 2048 x 2048 24.1 / 24.4, 700 x 3072 x 2048 22.7 / 23.5).  Six K tiles deep for a long K
// (6144 x 4096 36.2 -> 33.8, 4096 x 4096 at 260 38.3 -> 36.0; 2048 x 2048 20.6 -> 21.3, 768 x 768 9.1 -> 10.9).  Another wave that touches the weights 12 or 24 K tiles ahead
// makes all forms slower (487 x 16384 x 2048 36 -> 37.6, 39.6)
static inline bool ring64_fits(int M, int N, int slices) { return cdiv(M, 64) * cdiv(N, 128) * slices <= 256; }
static inline double ring64_cost(int M, int N, int K, int out_bytes, int slices) {
    const double fill = cdiv(M, 64) * cdiv(N, 128) * slices / 256.0;
    return 3.7 + (0.235 + 0.05 * fill) * (K >> 5) / slices + (slices > 1 ? gemm_epilogue_us(M, N, 8 * slices) : 0.44 * gemm_epilogue_us(M, N, out_bytes));
}
static inline double tile_cost(int M, int N, int K, int out_bytes, int slices) {
    const double c = tile128_cost(M, N, K, out_bytes, slices);
    return ring64_fits(M, N, slices) ? std::min(c, ring64_cost(M, N, K, out_bytes, slices)) : c;
}
// ... and how many slices cost least, the norm that sums them counted.  Beyond a workgroup a CU more of them only add traffic (487 x 2048 x 8192:
// eight 27.5 us, four 26.0, and half as much for the norm to read)
static inline int tile128_slices(int M, int N, int K, int most, double& cost) {
    int slices = 1;
    cost = tile_cost(M, N, K, 8, 1);
    if (g_chunk_max_m <= 64) {           // (key 11 = 64: sums in one order whatever the rows)
        while (slices < most && cdiv(M, 128) * cdiv(N, 128) * slices < 512 && K / (slices * 2) >= 512) slices *= 2;
        cost = tile_cost(M, N, K, 8, slices);
        return slices;
    }
    for (int s = 2; s <= most && K / s >= 512; s *= 2) {
        const double c = tile_cost(M, N, K, 8, s);
        if (c < 0.97 * cost) { cost = c; slices = s; }
    }
    return slices;
}
// the 64-row groups of the decode form (65 .. 512 rows): every group pulls the weights through the CUs again
static inline double passes_cost(int M, int N, int K) { return 4.0 + 0.3 * cdiv(M, 64) * 2e-6 * N * K; }
// is the ping-pong form the faster one?  (its parts in a.splits)
template <int EPI, typename OutT>
static inline bool pp_wins(GemmArgs& a) {
    a.splits = 1;
    if (a.seg || a.a_rows || a.tile_map || a.sk_part || a.K < 160) return false;
    const int bytes = EPI == EPI_RESID ? 8 : EPI == EPI_GROUPED_RAW ? 4 : epi_glu(EPI) ? (int)sizeof(OutT) / 2 : (int)sizeof(OutT);
    // (key 11 = 64: sums in one order whatever the rows, up to 512.  EPI_GROUPED, whose epilogue is long: not where one round of parts would leave
    // it to a few workgroups, 17424 x 4096 at 140 / 200 rows 82 / 86 us in parts, 74 / 78 on 128x128 tiles)
    const bool parts = a.split_units * SPLIT_UNIT >= SPLIT_WS_BYTES && (a.M > MID_MAX_ROWS || a.M <= std::max(64, g_chunk_max_m)) &&
                       (EPI != EPI_GROUPED || cdiv(a.M, 256) * cdiv(a.N, 256) > 256);
    // (one round of whole tiles with a GLU starts and ends sooner than the fit has it: 520 / 700 x 16384 x 2048 53.4 / 46.2, 57.2 / 47.5 us on 128x128 / large tiles, 700 x 12288 50.5 / 45.2)
    const double cost = pp_cost(a.M, a.N, a.K, bytes, parts, a.splits) - (epi_glu(EPI) && a.splits == 1 && cdiv(a.M, 256) * cdiv(a.N, 256) <= 256 ? 6.0 : 0.0);
    const bool faster = cost < 1.05 * tile_cost(a.M, a.N, a.K, bytes, 1);      // (ties: 4176 x 4096 x 4096 161 / 172, 200 x 18176 x 4544 67 / 79)
    // (whole tiles lose to 128x128 tiles that fit one round of two a CU, which the costs miss at times: 12288 x 2048 at 520 rows 42.6 / 30.2, 16384 x 2048 at 400 42 / 38)
    return faster && (a.splits > 1 || cdiv(a.M, 128) * cdiv(a.N, 128) > 512);
}
// 128x128 tiles on eight waves of 32x64 instead of four of 64x64: twice the waves to cover the way to the operands, half as long an epilogue each, half as many
// products more to read for.  Better while each CU has one tile at most, whatever the K (487 x 2048 x 2048 24.4 -> 22.8 us, 600 x 768 x 3072 27.1 -> 25.4, 700 x 6144 x 4096
// 37.1 -> 36.5), with GELUs always (700 x 3072 x 768 16.8 -> 12.6, 3200 of them 35.9 -> 29.0, 520 x 18176 x 4544 123 -> 103), with fp32 results of a short K (4100 x 2048 x 2048
// 55.7 -> 52.3, 3200 x 3072 36.7 -> 35.8); not two a CU of a long one (1800 x 4096 x 4096 64.1 / 66.0, 900 x 28672 x 4096 221 / 236)
template <int EPI, typename OutT>
static inline bool ring_eight(const GemmArgs& a) {
    const int tiles = cdiv(a.M, 128) * cdiv(a.N, 128) * (a.sk_part ? a.sk_slices : 1);
    return tiles <= 256 || EPI == EPI_GELU || EPI == EPI_GELU_TOK || EPI == EPI_JOINT || (sizeof(OutT) == 4 && a.K <= 2048);
}
// 256x128 tiles of the ring, six K tiles deep, one a CU, where 128x128 tiles would be two on some.  What bounds both is the way from L2 to the CUs (487 x 16384 x 2048
// without its products 37.8 of 39.4 us; some 100 lines a CU on their way, 460 cycles each), and a tile of twice the size asks for a quarter less.  us, 128x128 -> here (weights
// from HBM): 16384 x 2048 at 260 / 350 / 400 / 487 rows 36.7 -> 32.2, 40.2 -> 32.8, 36.4 -> 33.2, 41.1 -> 35.0; 12288 x 2048 at 300 / 450 33.3 -> 29.9, 35.4 -> 32.4; 28672 x 4096 at 130 / 256
// 61.5 -> 55.0, 73.8 -> 63.4; 22848 x 4544 at 140 74.9 -> 65.1; 16384 x 1024 at 300 23.6 -> 19.7.  The cost of up to 512 rows is good to 5 %; large tiles in parts: 18176 x 4544 at 140 / 256
// 65.4 / 69.9, here 62.9 / 73.0.
// More rows, where the 128x128 tiles are 1.2 a CU at least: 8512 x 2048 at 520 / 640 / 768 rows 38.0 -> 34.2, 42.3 -> 35.1, 44.3 -> 38.8; 4096 x 4096 at 1400 / 2048 75.2 -> 60.2, 86.4 -> 69.8
// (large tiles 70.7, 79.3); 4544 x 4544 at 1100 / 1700 80.4 -> 64.7, 84.8 -> 71.9; 3072 x 2048 at 1700 / 2048 / 2560 36.2 -> 33.2, 40.0 -> 34.8, 40.8 -> 36.0; 2048 x 4096 at 2560 / 4096 69.4 -> 60.0,
// 80.8 -> 70.5; 4096 x 1024 at 1100 .. 2048 4 %.  Not 288 tiles (768 x 6144 x 4096 57.7 / 60.8, 2300 x 2048 x 2048 34.2 / 36.4), a K below 1024 (2048 x 3072 x 768 20.5 / 23.5), nor 2048 x 2048 (3000
// rows 35.8 / 38.0, 3500 40.0 / 40.1), nor the long epilogue of raw queries and keys (1600 x 3072 x 2048 42.5 / 46.1); a long K may be better in parts of large tiles (1280 x 4096 x 14336
// 136 / 181, 1900 207 / 210)
template <int EPI, typename OutT>
static inline bool ring256_wins(const GemmArgs& a, bool pp) {
    if (a.seg || a.a_rows || a.sk_part || a.M <= 128) return false;
    const int tiles = cdiv(a.M, 128) * cdiv(a.N, 128), bytes = EPI == EPI_RESID ? 8 : epi_glu(EPI) ? (int)sizeof(OutT) / 2 : (int)sizeof(OutT);
    if (cdiv(a.M, 256) * cdiv(a.N, 128) > 256 || tiles <= 256) return false;
    const double rows = a.M / (256.0 * cdiv(a.M, 256));
    double cost;
    if (a.M <= 512) {
        if (EPI == EPI_RESID || EPI == EPI_QKV || sizeof(OutT) == 4) return false;
        cost = 7.5 + (a.K >> 5) * (0.34 + 0.10 * rows);
    } else {
        if (EPI == EPI_GROUPED_RAW || tiles <= 288 || a.K < 1024 || (a.K < 4096 && a.N < 3072)) return false;
        cost = 7.1 + 0.44 * gemm_epilogue_us(a.M, a.N, bytes) + (a.K >> 5) * (0.30 + 0.12 * rows);
    }
    int parts;
    return !pp || cost < (a.M <= 512 ? 1.0 : 0.93) * pp_cost(a.M, a.N, a.K, bytes, a.splits > 1, parts);
}
template <int EPI, typename OutT, int WAVES_N>
static inline void launch_pp(hipStream_t st, const GemmArgs& a) {
    const int T = cdiv(a.M, 256) * cdiv(a.N, 256), n = cdiv(T, 8);
    if (a.splits > 1) {
        NVL_LDS_ATTR((gemm_bf16_pp_kernel<EPI, OutT, 4, 0, WAVES_N, 256, true>), PP_LDS);
        hipLaunchKernelGGL((gemm_bf16_pp_kernel<EPI, OutT, 4, 0, WAVES_N, 256, true>), dim3(8 * ((n & ~31) + (n & 31) * a.splits)), dim3(512), PP_LDS, st, a);
    } else {
        NVL_LDS_ATTR((gemm_bf16_pp_kernel<EPI, OutT, 4, 0, WAVES_N>), PP_LDS);
        hipLaunchKernelGGL((gemm_bf16_pp_kernel<EPI, OutT, 4, 0, WAVES_N>), dim3(T), dim3(512), PP_LDS, st, a);
    }
}

template <int EPI, typename OutT>
static inline void launch_gemm_grouped(hipStream_t st, const GemmArgs& a, int max_mtiles) {
    if (a.grp_bm == 512) {      // prefill MoE, the default: 256-row m-tiles on the ping-pong kernel
        if constexpr (epi_glu(EPI))
            if (a.a_rows) {
                NVL_LDS_ATTR((gemm_bf16_pp_kernel<EPI, OutT, 4, 0, 4, 256, false, true>), PP_LDS);
                hipLaunchKernelGGL((gemm_bf16_pp_kernel<EPI, OutT, 4, 0, 4, 256, false, true>), dim3(cdiv(a.N, 256) * max_mtiles), dim3(512), PP_LDS, st, a);
                return;
            }
        NVL_LDS_ATTR((gemm_bf16_pp_kernel<EPI, OutT, 4, 0>), PP_LDS);
        hipLaunchKernelGGL((gemm_bf16_pp_kernel<EPI, OutT, 4, 0>), dim3(cdiv(a.N, 256) * max_mtiles), dim3(512), PP_LDS, st, a);
        return;
    }
    if (a.grp_bm == 256) {      // prefill MoE with long expert segments: 256-row m-tiles, three stages
        constexpr int lds3 = gemm_lds_bytes<256, 128, 3>();
        NVL_LDS_ATTR((gemm_bf16_kernel<256, 128, 4, 2, 3, EPI, OutT>), lds3);
        hipLaunchKernelGGL((gemm_bf16_kernel<256, 128, 4, 2, 3, EPI, OutT>), dim3(cdiv(a.N, 128) * max_mtiles), dim3(512),
                           lds3, st, a);
        return;
    }
    // (decode-sized batches too, a handful of rows an expert: us a layer of 1 / 4 / 16 / 64 rows, 32 experts, 8 a token, with four K tiles of 64 in 128 KiB ->
    // four of 32 on four waves: 512 x 2048 75 -> 69.6, 86.6 -> 79.7, 97.2 -> 92.8, 120.2 -> 117.2; 1024 x 4096 128 -> 124, 202 -> 184, 235 -> 229, 271 -> 267; 512 x 1024 3 %.
    // Eight waves of 32x64, us a launch on four -> here, 32 experts, 8 a token: up 1024 x 1024 at 100 / 200 / 255 rows 21.3 -> 20.3, 23.2 -> 21.8, 24.2 -> 22.4, a decode step of
    // 96 21.2 -> 20.4, down 1024 x 512 14.0 -> 13.6, 15.6 -> 15.3, 16.2 -> 16.0, 13.5 -> 13.4; up 1024 x 2048 at 40 / 100 / 200 37.5 / 37.7, 35.8 -> 35.6, 38.9 -> 38.6, down 2048 x 512
    // 27.1 / 27.1, 19.9 -> 19.2, 23.3 -> 23.0, a step of 96 22.5 -> 21.9)
    constexpr int lds = gemm_lds_bytes<128, 128, 4, 32>();
    NVL_LDS_ATTR((gemm_bf16_kernel<128, 128, 4, 2, 4, EPI, OutT, 32>), lds);
    hipLaunchKernelGGL((gemm_bf16_kernel<128, 128, 4, 2, 4, EPI, OutT, 32>), dim3(cdiv(a.N, 128) * max_mtiles), dim3(512),
                       lds, st, a);
}

// What a projection of up to MID_MAX_ROWS rows takes on gemm_mid_bf16_kernel, in microseconds, and into how many parts its K goes (fitted to 8 .. 512
// rows of 2048 .. 4544-wide models, good to 15 %): a stage of a CU moves at some 56 GB/s, all weights together at 6.6 TB/s; a part
// more costs the hand-over 0.45 us and every round of workgroups beyond the first its ramp.
static inline int mid_row_tiles(int M) { return cdiv(cdiv(M, cdiv(M, 128)), 32) * 2; }      // 16-row tiles of a row group: 2, 4, 6 or 8
static inline double mid_cost(int M, int N, int K, int mt, int ct, bool can_split, int& parts) {
    const int tiles = cdiv(N, 32 * ct) * cdiv(M, 16 * mt), stages = cdiv(K, 128);
    const double stage_us = 0.0178 * 4.0 * (mt + 2 * ct), hbm_us = 2e-6 * N * K / 6.6;
    double best = 0;
    parts = 1;
    for (int c = 1; c <= MID_MAX_PARTS; c++) {
        if (c > 1 && (!can_split || tiles * c > 256 || stages / c < MID_MIN_STAGES)) break;
        const double rounds = cdiv(tiles * c, 256), t = std::max(rounds * cdiv(stages, c) * stage_us, hbm_us) + (c > 1 ? 2.5 + 0.45 * c : 0.0) + 2.0 * (rounds - 1);
        if (c == 1 || t < best) { best = t; parts = c; }
    }
    return best + 4.0;
}
// ... and on the narrow decode form (M <= 64), where the activations come beside the weights once per 16 of their rows.  us a MB of weights with every
// CU at work, from the activation rows that a launch fetches (whole row tiles, or the live rows: x_mask), over the share of its last round of
// workgroups that is at work, and not faster than 6.56 TB/s.  Fitted to 1 .. 64 rows of 1024 .. 15360 x 2048 .. 18176, good to 20 %.
// `blocks`: workgroups of one row tile; tile_split: each row tile has its own workgroups (GemmArgs::m_split)
static inline double narrow_cost(int M, int N, int K, int blocks, int waves, bool tile_split) {
    const double mb = 2e-6 * N * K;
    if (tile_split) {
        const double rate = 11.5 * std::min(1.0, blocks * cdiv(M, 16) / 256.0) * (waves >= 2048 ? 1.0 : pow(waves / 2048.0, 0.6));
        return std::max(mb / 5.9, mb * 2.0 * cdiv(M, 16) / rate) + 2.5;
    }
    const double rows = M > 32 && blocks > 512 ? 4.0 : M % 16 ? M / 16.0 : M <= 32 ? M / 16 : 4.0;
    double full = blocks / (256.0 * cdiv(blocks, 256));
    if (blocks > 512 && M <= 32) full = std::max(full, 0.88);      // (of one or two waves each: they even out)
    return std::max(mb / 6.56, mb * (M <= 16 ? 0.113 + 0.03 * rows : 0.14 + 0.032 * rows) / full) + 3.6;
}
inline int g_mid = 1;               // nvl_set_tuning key 38: 0 never, 2 wherever it applies
inline int g_mid_splits = 0;        // nvl_set_tuning key 39: parts of K (0: from the cost)
template <int MT, int CT, int EPI, typename OutT>
static inline void launch_gemm_mid_rows(hipStream_t st, const GemmArgs& a0) {
    GemmArgs a = a0;
    const int nb = cdiv(a.N, 32 * CT), groups = cdiv(a.M, 16 * MT);
    mid_cost(a.M, a.N, a.K, MT, CT, a.split_units > 0, a.splits);
    if (a.split_units > 0 && g_mid_splits) a.splits = std::min(g_mid_splits, std::max(1, a.K >> 7));
    while (a.splits > 1 && (nb * groups > SPLIT_MAX_TILES || (int64_t)nb * groups * a.splits * MT * CT * 2048 > a.split_units * SPLIT_UNIT)) a.splits--;
    auto launch = [&](auto stream) {
        NVL_LDS_ATTR((gemm_mid_bf16_kernel<MT, CT, EPI, OutT, decltype(stream)::value>), (mid_lds_bytes<MT, CT>()));
        hipLaunchKernelGGL((gemm_mid_bf16_kernel<MT, CT, EPI, OutT, decltype(stream)::value>), dim3(cdiv(nb, 8) * 8 * groups * a.splits), dim3(512), (mid_lds_bytes<MT, CT>()), st, a);
    };
    if constexpr (MT < 8) if (groups == 1) { launch(std::true_type{}); return; }
    if constexpr (MT > 4 || CT > 2) launch(std::false_type{});
    else throw std::runtime_error("gemm_mid: several groups of few rows");      // (narrower tiles hold all rows: mid_row_tiles)
}
// does the kernel take this projection, and is it the one to take it?
template <int EPI, typename OutT>
static inline bool mid_wins(const GemmArgs& a) {
    if (!g_mid || a.M > MID_MAX_ROWS || a.M > std::max(64, g_chunk_max_m) || a.K % 64 != 0 || a.a_rows || a.seg || a.tile_map || a.sk_part || a.moe_gate || a.c_row0 || g_force_tile ||
        g_force_ntw || a.rs_half || ((EPI == EPI_RESID || EPI == EPI_QKV) && a.rs_in)) return false;
    if (EPI == EPI_QKV && a.qkv.hd == 128) return a.M > 64 && cdiv(a.N, 128) * cdiv(a.M, 64) <= 512;
    if (EPI == EPI_QKV && a.qkv.hd != 64) return false;
    if (g_mid == 2) return true;
    if (a.M <= 64) {
        // (pairs and wide projections: the decode forms; below some 16 MB of weights, or with few rows of a short K, a launch is all ramp:
        // 5120 x 2048 at 19 rows 12.0 us there, 13.9 here; 8512 x 2048 at 24 13.1 and 15.6, at 48 19.0 and 17.4)
        if (EPI == EPI_QKV || epi_glu(EPI) || cdiv(a.N, 64) >= 256 || (int64_t)a.N * a.K < (8 << 20) || (a.M <= 32 && a.K < 4096)) return false;
        const bool split = EPI == EPI_RESID && a.m_split && a.rs_out;
        const int blocks = cdiv(a.N, 16);
        int ks = split ? 8 : 16, mid_parts;                       // (waves of a workgroup: launch_gemm_skinny_ntw)
        if (!split) while (ks > 1 && blocks * ks > g_narrow_waves) ks >>= 1;
        // a small step in favour of the form that is there.  Decode form -> here, us, weights from HBM: 4544 x 18176 at 5 / 16 / 32 rows 37.1 -> 29.4,
        // 46.4 -> 29.8, 62.9 -> 31.5; 2560 x 8192 at 40 / 64 16.7 -> 13.6, 20.7 -> 14.2; not 4096 x 14336 at 5 / 16 19.8 / 22.8, 22.4 / 23.3 here,
        // 8192 x 4096 at 17 / 32 16.7 / 16.8, 17.9 / 18.1 here.  Row tiles apart, at 24 / 32 / 64 rows: 4096 x 14336 43 -> 28.6, 55 -> 29.9,
        // 85.7 -> 32.6; 2048 x 8192 stays at 15.3 up to 32 rows, 23.1 -> 18.4 at 64
        return mid_cost(a.M, a.N, a.K, mid_row_tiles(a.M), 2, a.split_units > 0, mid_parts) <
               (split ? 0.92 : 0.98) * narrow_cost(a.M, a.N, a.K, blocks, blocks * ks * (split ? cdiv(a.M, 16) : 1), split);
    }
    // (GPT-2's projections at 96 .. 104 rows: 768 x 768 12.7 us here and 8.8 in groups of the decode form, 768 x 3072 14.7 and 13.6)
    if (EPI != EPI_QKV && (a.K < 2048 || (int64_t)a.N * a.K < (4 << 20))) return false;
    // One row group reads the weights once at any width up to a few rounds of workgroups (a workgroup per CU: each round has its own
    // ramp; LM head at 128 rows 168 us against 152 on the tiles, 28672 x 4096 72 against 74).  Several groups pay while one round holds
    // them (3072 x 2048: 192 rows 12.5 against 17.4 us, 512 rows 18.3 against 29; 16384 x 2048 at 512 rows 68 against 43).
    // Long K: parts of large tiles (4544 x 22720 at 140 / 300 rows 117 / 154 us here, 94 / 128 there; not 4096 x 14336 at 300, 92 and 95).
    if (a.M > 128 && a.split_units * SPLIT_UNIT >= SPLIT_WS_BYTES && EPI == EPI_RESID) {
        int parts, mid_parts;
        if (1.05 * pp_cost(a.M, a.N, a.K, 8, true, parts) < mid_cost(a.M, a.N, a.K, mid_row_tiles(a.M), 2, true, mid_parts)) return false;
    }
    return cdiv(a.N, 64) * cdiv(a.M, 128) <= (a.M <= 128 ? 512 : 256);
}
template <int EPI, typename OutT>
static inline bool launch_gemm_mid(hipStream_t st, const GemmArgs& a) {
    if (!mid_wins<EPI, OutT>(a)) return false;
    const int mt = mid_row_tiles(a.M);
    if constexpr (EPI == EPI_QKV) {
        if (a.qkv.hd == 128) {
            launch_gemm_mid_rows<4, 4, EPI, OutT>(st, a);      // (a head of 128 columns per workgroup: 64 rows leave room for three stages)
            return true;
        }
    }
    if (mt <= 2) launch_gemm_mid_rows<2, 2, EPI, OutT>(st, a);
    else if (mt <= 4) launch_gemm_mid_rows<4, 2, EPI, OutT>(st, a);
    else if (mt <= 6) launch_gemm_mid_rows<6, 2, EPI, OutT>(st, a);
    else launch_gemm_mid_rows<8, 2, EPI, OutT>(st, a);
    return true;
}

// Projections of 33 .. 256 rows whose K is short (launch_gemm_rows): groups of 32, 48 or 64 rows by 16 or 32 columns on the wide decode form, all of K in each workgroup
// and one round of them.  Up to eight k-steps of 32 a wave (K = 2048) are all in flight at once, four at a time above: nothing is handed over between workgroups, which is
// what gemm_mid_bf16_kernel's parts of K spend 4 us on, and the groups of 64 rows on the narrow form, two k-steps at a time, wait for memory four times.
// us by events, weights from HBM, before -> here: 3072 x 2048 at 70 / 96 / 128 rows 14.2 -> 11.1, 14.6 -> 11.8, 16.7 -> 13.6; 2048 x 2048 at 70 / 96 / 128 / 190 / 250
// 12.8 -> 10.4, 13.1 -> 10.4, 14.4 -> 11.1, 13.3 -> 11.3, 14.9 -> 12.8; 1536 x 1024 at 96 / 190 8.4 -> 7.4, 12.2 -> 8.0; 2304 x 768 at 70 / 96 / 190 8.6 -> 7.8, 9.4 -> 7.5, 10.0 -> 8.9;
// 768 x 768 8.5 -> 6.8, 768 x 3072 at 70 / 96 / 250 12.8 -> 9.8, 14.7 -> 10.0, 15.5 -> 12.1.  Not a longer K, where the hand-over is the smaller part: 2048 x 8192 at 96 / 150 / 250
// 20.2 / 21.4, 20.8 / 24.1, 24.6 / 29.7, 2048 x 6144 at 96 17.1 / 18.4.
inline int g_rows = 1;              // nvl_set_tuning key 46: 0 never, 1 by cost unless keys 38 or 39 ask for the kernel of parts, 2 wherever it applies
static inline double rows_cost(int N, int K, int tiles) { return 1.3 + K / 256.0 * 0.14 * tiles + 0.14e-6 * N * K; }      // (in mid_cost's terms; tiles: of rows and columns)
// row and column tiles of a workgroup: the fewest bytes that one round of workgroups allows (rows are padded to whole groups of 64)
static inline bool rows_shape(int M, int N, int& mt, int& nt) {
    mt = nt = 0;
    for (int g = 1; g <= 8; g++)
        for (int t = 1; t <= 2; t++) {
            const int r = std::max(2, cdiv(cdiv(M, g), 16));
            if (r > 4 || 16 * r * (g - 1) >= M || 16 * r * g > round_up(M, 64) || N % (128 * t) != 0 || N / (16 * t) * g > 256) continue;
            if (!mt || r + t < mt + nt) { mt = r; nt = t; }
        }
    return mt > 0;
}
// ... of 33 to 64 rows, residual (others gain nothing: 3072 x 2048 at 40 rows 10.6 / 10.6).  Below 48 rows the narrow decode form leaves out what lies beyond them, and is as fast or
// faster wherever it has workgroups for the whole chip.  us by events, that form / here, at 33, 47, 48 and 60 rows:
//   1024 x 2048 7.2 / 5.9 at 34, 7.9 / 6.0 at 64   1024 x 1280 -7, -9, -15, -15 %   1024 x 1088 -2, -4, -9, -9 %
//   2048 x 2048 -15, -17, -23, -23 %   x 1792 -9, -13, -21, -20 %   x 1536 +1, -2, -9, -8 %   x 1280 +5, +2, -5, -5 %   x 1088 +11, +8, +1, +2 %
//   3072 x 2048 +7, +4, -5, -7 %   x 1536 +8, +5, -2, -4 %   4096 x 2048 +5, +1, -8, -9 %   x 1536 +4, +2, -5, -7 %   x 1088 +2, 0, -6, -2 %   1536 x 1088 +9, +7, 0, +1 %
static inline bool rows_pay_few(int M, int N, int K) { return K > 1024 && K <= 2048 && (N <= 1024 || (M >= 48 ? K >= 1280 : N <= 2048 && K >= 1792)); }
template <int MT, int NTB, int EPI, typename OutT>
static inline void launch_gemm_rows_of(hipStream_t st, const GemmArgs& a) {
    GemmArgs c = a;
    c.m_passes = cdiv(a.M, 16 * MT);
    const int nks = a.K >> 5;
    int waves = std::min(8, std::max(1, nks / 4));
    for (int w = waves; w >= 5; w--) if (nks % (4 * w) == 0) { waves = w; break; }      // (whole blocks of four steps)
    NVL_LDS_ATTR((gemm_skinny_wide_bf16_kernel<MT, NTB, 4, EPI, OutT, true>), 8 * NTB * MT * 1024);
    hipLaunchKernelGGL((gemm_skinny_wide_bf16_kernel<MT, NTB, 4, EPI, OutT, true>), dim3(a.N / (16 * NTB) * c.m_passes), dim3(waves * 64), waves * NTB * MT * 1024, st, c);
}
template <int EPI, typename OutT>
static inline bool launch_gemm_rows(hipStream_t st, const GemmArgs& a) {
    int mt, nt, parts;
    if (!g_rows || a.M <= 32 || a.M > 256 || a.M > std::max(64, g_chunk_max_m) || a.K % 32 != 0 || a.a_rows || a.seg || a.sk_part || a.moe_gate || a.c_row0 || a.m_passes > 1 || g_force_tile || g_force_ntw ||
        a.rs_half || (EPI == EPI_RESID && a.rs_in) || !rows_shape(a.M, a.N, mt, nt)) return false;
    if (g_rows == 1) {
        if (g_mid == 2 || g_mid_splits) return false;
        // (a short K leaves nothing to gain: measured from 768 on)
        // (where the 64-row groups would be taken there is nothing to weigh: 18 sizes of 128 .. 4096 x 768 .. 16384 at 66 .. 250 rows, as they are and residual, +2 .. -46 %, most -10 .. -40)
        if (a.K < 768) return false;
        if (a.M <= 64) { if (EPI != EPI_RESID || !rows_pay_few(a.M, a.N, a.K)) return false; }
        else if (mid_wins<EPI, OutT>(a) && rows_cost(a.N, a.K, mt + nt) > mid_cost(a.M, a.N, a.K, mid_row_tiles(a.M), 2, a.split_units > 0, parts)) return false;
    }
#define NVL_RW(MT, NT) if (mt == MT && nt == NT) launch_gemm_rows_of<MT, NT, EPI, OutT>(st, a)
    NVL_RW(2, 1); NVL_RW(2, 2); NVL_RW(3, 1); NVL_RW(3, 2); NVL_RW(4, 1); NVL_RW(4, 2);
#undef NVL_RW
    return true;
}

template <int EPI, typename OutT>
void launch_gemm_bf16(hipStream_t st, const GemmArgs& a) {
    if constexpr (epi_ln(EPI)) {
        bool ok = a.M <= 64;
        if constexpr (EPI == EPI_LN_RESID) ok = ok && launch_gemm_ln_resid<OutT>(st, a);
        else ok = ok && launch_gemm_skinny_bf16<EPI, OutT>(st, a);
        if (!ok) throw std::runtime_error("gemm: a deferred layer norm did not fit the decode kernels");
        return;
    } else {
    if (a.tile_map) { launch_gemm_grouped<EPI, OutT>(st, a, a.M); return; }   // a.M carries the m-tile bound
    if constexpr (EPI == EPI_RESID || (EPI == EPI_STORE && std::is_same_v<OutT, float>)) if (launch_gemm_rows<EPI, OutT>(st, a)) return;
    if (launch_gemm_mid<EPI, OutT>(st, a)) return;
    if (launch_gemm_skinny_bf16<EPI, OutT>(st, a)) return;
    if constexpr (EPI != EPI_QKV) {
        // 64 < M <= g_chunk_max_m (large decode batches): the tile kernels would launch only N/128 * M/128 workgroups, far
        // too few to stream the weights at HBM rate.  Run the decode form over ceil(M/64) groups of 64 activation rows
        // in one launch instead (GemmArgs::m_passes): the groups of a weight block run side by side on one XCD, so the
        // weights cross HBM once.  Only the narrow projections (QKV, O, FFN-down) do; FFN-up and the LM head have enough
        // tiles (g_chunk_all_m: below it every projection would).
        // (us, groups / tiles: 768 x 768 at 300 rows 5.5 / 12.3, 2304 x 768 10.3 / 11.0, 6144 x 4096 62.8 / 39.4, 8512 x 2048 at 140 41.2 / 22.9.  With GELUs: 3072 x 768 at
        // 300 / 350 / 400 / 512 rows 11.9 / 13.2, 14.7 / 13.6, 16.2 / 13.3, 17.4 / 13.9; 4096 x 1024 at 200 / 260 / 350 12.2 / 15.4, 16.1 / 15.1, 19.2 / 15.7; 6144 x 1024 at 200 14.5 / 16.1)
        const bool few_tiles = cdiv(a.M, 128) * cdiv(a.N, 128) < g_chunk_min_tiles &&
                               passes_cost(a.M, a.N, a.K) < tile_cost(a.M, a.N, a.K, EPI == EPI_RESID ? 8 : (int)sizeof(OutT), 1) + (EPI == EPI_GELU || EPI == EPI_JOINT ? 1.0 : 0.0);
        if (a.M > 64 && a.M <= g_chunk_max_m && (a.M <= g_chunk_all_m || few_tiles || a.rs_in || a.rs_out) && !a.a_rows && !a.seg && !a.sk_part && a.K % 32 == 0 &&
            g_force_tile == 0) {
            GemmArgs c = a;
            c.m_passes = cdiv(a.M, 64);
            const bool ok = g_pass_interleave ? launch_gemm_skinny_bf16<EPI, OutT>(st, c)
                                              : launch_skinny_passes_serial<EPI, OutT>(st, c);
            if (ok) return;
        }
    }
    if (a.rs_in || a.rs_out) throw std::runtime_error("gemm: a deferred-RMSNorm projection did not fit the decode kernels");
    if constexpr (EPI == EPI_QKV) {
        if (a.qkv.hd == 128) {     // a wave must own a whole 128-column head: 256x256 tile as 4x2 waves of 64x128
            if (g_force_tile == 0 && a.K >= 160 && !a.seg && !a.a_rows) {
                GemmArgs as = a;
                pp_wins<EPI, OutT>(as);                   // (for its parts: the lock-step form below is never the faster one)
                launch_pp<EPI, OutT, 2>(st, as);                  // wave tile 64x128
                return;
            }
            launch_gemm_tile<256, 256, 4, 2, 2, EPI, OutT>(st, a);
            return;
        }
    }
    int tile = g_force_tile;
    GemmArgs as = a;
    as.splits = 1;
    // 5: the ping-pong form; 2: 256x128 tiles on the ring; else 128x128 tiles (the lock-step 256-wide forms and a ping-pong 256x128 variant with wave
    // tiles of 64x64 never win, profiles/r01e_gemm_sweep_mid.txt)
    if (tile == 0) { tile = pp_wins<EPI, OutT>(as) ? 5 : 1; if (ring256_wins<EPI, OutT>(as, tile == 5)) tile = 2; }
    else if (tile == 5) pp_wins<EPI, OutT>(as);
    if (tile == 5 && !a.seg && !a.a_rows) { launch_pp<EPI, OutT, 4>(st, as); return; }      // (4-slot ring: 5 slots -3 %, 3 slots -3 %, r01 sweep)
    if (tile == 3) launch_gemm_tile<256, 256, 2, 4, 2, EPI, OutT>(st, a);
    else if (tile == 2) launch_gemm_tile<256, 128, 4, 2, 6, EPI, OutT, 32>(st, a);
    else if (ring64_fits(a.M, a.N, a.sk_part ? a.sk_slices : 1) && !a.seg && !a.a_rows) {
        if (a.K >= 4096) launch_gemm_tile<64, 128, 2, 2, 6, EPI, OutT, 32>(st, a);
        else launch_gemm_tile<64, 128, 2, 2, 4, EPI, OutT, 32>(st, a);
    } else if (ring_eight<EPI, OutT>(a)) launch_gemm_tile<128, 128, 4, 2, 4, EPI, OutT, 32>(st, a);
    else launch_gemm_tile<128, 128, 2, 2, 4, EPI, OutT, 32>(st, a);
    }
}

template <int EPI, typename OutT>
void launch_gemm_f32(hipStream_t st, const GemmArgs& a) {
    const int tiles = cdiv(a.M, 64) * cdiv(a.N, 64);
    hipLaunchKernelGGL((gemm_f32_kernel<EPI, OutT>), dim3(tiles), dim3(256), 0, st, a);
}

// The projections' kernels are compiled per epilogue, side by side (gemm_inst.hip): (epilogue, output type)
#define NVL_GEMM_BF16_INSTANCES(X)                                                                                              \
    X(EPI_STORE, float) X(EPI_STORE, bf16_t) X(EPI_RESID, float) X(EPI_SWIGLU, bf16_t) X(EPI_GELU, bf16_t) X(EPI_GEGLU, bf16_t) \
    X(EPI_CLAMP_GLU, bf16_t) X(EPI_QKV, bf16_t) X(EPI_GROUPED, bf16_t) X(EPI_RELU2, bf16_t) X(EPI_GELU_TOK, bf16_t) \
    X(EPI_REGLU, bf16_t) X(EPI_GROUPED_RAW, bf16_t) X(EPI_LN_STORE, float) X(EPI_LN_RESID, float) X(EPI_LN_GELU, bf16_t) X(EPI_LN_QKV, bf16_t) \
    X(EPI_JOINT, bf16_t)
#define NVL_GEMM_F32_INSTANCES(X) X(EPI_STORE) X(EPI_RESID) X(EPI_GELU)
#ifndef NVL_GEMM_INST
#define NVL_X(E, T) extern template void launch_gemm_bf16<E, T>(hipStream_t, const GemmArgs&);
NVL_GEMM_BF16_INSTANCES(NVL_X)
#undef NVL_X
#define NVL_X(E) extern template void launch_gemm_f32<E, float>(hipStream_t, const GemmArgs&);
NVL_GEMM_F32_INSTANCES(NVL_X)
#undef NVL_X
#endif

}  // namespace nvl
