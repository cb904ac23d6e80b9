// mamba.h — Mamba2 (selective state-space) blocks of the Granite-4 hybrid models: the element / scan kernels between
// the two projections of Mamba2Layer.Forward (purego/tensor/mamba2.go:74-181).  The projections themselves
// (in_proj, out_proj) are the GEMMs of gemm.h.
//
//   in_proj GEMM -> proj [tokens][gate EH | xBC conv_dim | dt nh]   (fp32)
//   mamba_conv_kernel      causal conv1d + bias + SiLU on xBC, softplus(dt + bias)        mamba2.go:107-131, 183-254, 360-376
//   mamba_scan_kernel      per (sequence, head): state = abar*state + dt*B*u; y = C·state + D*u   mamba2.go:256-351
//   mamba_gate_norm_kernel y *= SiLU(gate); RMS norm over EH (eps 1e-5); * norm weight -> out_proj operand   :135-170
//   out_proj GEMM (+ residual)
//
// State: the reference keeps SSMState ON THE LAYER (mamba2.go:29-30), i.e. one state for whatever sequence ran last —
// wrong for more than one live sequence.  Here every KV slot (sequence) owns its state,
// [slot][mamba layer][head][head_dim][state] fp32 in HBM, zeroed when the sequence (re)starts at position 0.
// The reference carries NO convolution state across calls (ConvCache is never used): a decode call convolves its one
// token with zeros.  That is mirrored — the conv window never reaches before the call's first token of a sequence.
#pragma once
#include "common.h"

namespace nvl {

struct MambaArgs {
    const float* proj;       // [tokens][P]  P = EH + conv_dim + nh
    int P, EH, conv_dim, nh, hd, ss, ng, K;
    const float* conv_w;     // [conv_dim][K]
    const float* conv_b;     // [conv_dim] or NULL
    const float* a_log;      // [nh] or NULL
    const float* Dskip;      // [nh] or NULL
    const float* dt_bias;    // [nh] or NULL
    const float* norm_w;     // [EH] or NULL
    float* xbc;              // [tokens][conv_dim]  SiLU(conv(xBC))
    float* delta;            // [tokens][nh]
    float* y;                // [tokens][EH]
    float* state;            // this layer's states: slot s at state + s * state_slot_stride
    int64_t state_slot_stride;
    const int32_t* tok_pos;        // per token: absolute position
    const int32_t* tok_seq;        // per token: index of its sequence in the batch
    const int32_t* seq_tok_start;  // per sequence
    const int32_t* seq_len;
    const int32_t* seq_pos;        // first position of the sequence in this call
    const int32_t* seq_slot;       // KV slot of the sequence (blk_table in slab mode)
    // A history longer than max_batch_tokens is prefilled in chunks by the runner (nvllm.hip runner_impl); the reference
    // runs it as ONE Forward whose convolution window spans the whole history.  For those chunks only, the raw xBC rows of
    // the last K-1 tokens of the previous chunk are kept per (slot, Mamba2 layer) and stand in for the zero padding:
    // chain 0 = off (every other call: the reference's zero padding), 1 = first chunk (save the tail), 2 = later chunk
    // (use the saved tail, then save the new one).
    float* tail;                   // this layer's tails: slot s at tail + s * tail_slot_stride, [K-1][conv_dim]
    int64_t tail_slot_stride;
    int chain;
    // chunk-parallel SSD scan (mamba_ssd_kernel MODE 1 / 2): per (sequence, chunk, head) state scratch and chunk decay
    float* ssd_z;                  // [sequences][max_chunks][nh][hd][ss]
    float* ssd_decay;              // [sequences][max_chunks][nh]
};

__device__ __forceinline__ float silu_ref(float x) { return x / (1.0f + __expf(-x)); }
__device__ __forceinline__ float softplus_ref(float x) { return x > 20.f ? x : log1pf(__expf(x)); }    // mamba2.go:370-376

// grid (tokens), 256 threads over channels (+ the nh dt values)
__global__ __launch_bounds__(256) void mamba_conv_kernel(MambaArgs p) {
    const int t = blockIdx.x;
    const int j = p.tok_pos[t] - p.seq_pos[p.tok_seq[t]];      // tokens of this sequence before t IN THIS CALL
    const float* row = p.proj + (int64_t)t * p.P + p.EH;        // xBC of token t
    for (int c = threadIdx.x; c < p.conv_dim; c += blockDim.x) {
        float sum = 0.f;
        for (int k = 0; k < p.K; k++) {                         // out[t] = sum_k x[t - (K-1) + k] * w[c][k], zero before the call
            const int back = p.K - 1 - k;
            if (back <= j) sum = fmaf(row[c - (int64_t)back * p.P], p.conv_w[(int64_t)c * p.K + k], sum);
            else if (p.chain == 2)     // continued chunk: the window reaches into the previous chunk's last K-1 tokens
                sum = fmaf(p.tail[(int64_t)p.seq_slot[p.tok_seq[t]] * p.tail_slot_stride + (int64_t)(p.K - 1 - (back - j)) * p.conv_dim + c],
                           p.conv_w[(int64_t)c * p.K + k], sum);
        }
        if (p.conv_b) sum += p.conv_b[c];
        p.xbc[(int64_t)t * p.conv_dim + c] = silu_ref(sum);
    }
    for (int h = threadIdx.x; h < p.nh; h += blockDim.x) {
        float v = p.proj[(int64_t)t * p.P + p.EH + p.conv_dim + h];
        if (p.dt_bias) v += p.dt_bias[h];
        p.delta[(int64_t)t * p.nh + h] = softplus_ref(v);
    }
}

// The same for four taps on 16-byte rows: a thread convolves four channels over MAMBA_CONV_RUN tokens, each row fetched once per run (a
// workgroup per token re-read the three rows before it from another XCD's memory: 2326 x 4352 took 81 us, 25 here).  The last
// column of workgroups has the dt values.
constexpr int MAMBA_CONV_RUN = 8;
static inline bool mamba_conv_run_ok(const MambaArgs& p) { return p.K == 4 && p.P % 4 == 0 && p.EH % 4 == 0 && p.conv_dim % 4 == 0 && p.tail_slot_stride % 4 == 0; }
__global__ __launch_bounds__(256) void mamba_conv_run_kernel(MambaArgs p, int tokens) {
    constexpr int T = MAMBA_CONV_RUN;
    const int t0 = blockIdx.x * T, n = min(T, tokens - t0);
    if (blockIdx.y == gridDim.y - 1) {
        for (int i = threadIdx.x; i < n * p.nh; i += 256) {
            const int h = i % p.nh;
            const int64_t t = t0 + i / p.nh;
            float v = p.proj[t * p.P + p.EH + p.conv_dim + h];
            if (p.dt_bias) v += p.dt_bias[h];
            p.delta[t * p.nh + h] = softplus_ref(v);
        }
        return;
    }
    const int c = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (c >= p.conv_dim) return;
    const float* col = p.proj + p.EH + c;
    f32x4 x[T + 3], w[4];
#pragma unroll
    for (int i = 0; i < T + 3; i++) {
        const int t = t0 + i - 3;
        x[i] = t >= 0 && t < tokens ? *(const f32x4*)(col + (int64_t)t * p.P) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int r = 0; r < 4; r++) w[r] = *(const f32x4*)(p.conv_w + (int64_t)(c + r) * 4);
    const f32x4 b = p.conv_b ? *(const f32x4*)(p.conv_b + c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < T; i++) {
        if (i >= n) break;
        const int t = t0 + i, seq = p.tok_seq[t], j = p.tok_pos[t] - p.seq_pos[seq];
        f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int back = 3 - k;
            f32x4 v;
            if (back <= j) v = x[i + k];
            else if (p.chain == 2) v = *(const f32x4*)(p.tail + (int64_t)p.seq_slot[seq] * p.tail_slot_stride + (int64_t)(3 - (back - j)) * p.conv_dim + c);
            else continue;
#pragma unroll
            for (int r = 0; r < 4; r++) sum[r] = fmaf(v[r], w[r][k], sum[r]);
        }
        if (p.conv_b) sum += b;
#pragma unroll
        for (int r = 0; r < 4; r++) sum[r] = silu_ref(sum[r]);
        *(f32x4*)(p.xbc + (int64_t)t * p.conv_dim + c) = sum;
    }
}

// grid (sequences), 256 threads over channels: after the convolution of a chunk of a chained prefill (chain >= 1), keep the
// raw xBC rows of the sequence's last K-1 tokens for the next chunk (a chunk shorter than K-1 keeps the newest old rows).
__global__ __launch_bounds__(256) void mamba_tail_kernel(MambaArgs p) {
    const int seq = blockIdx.x;
    const int t0 = p.seq_tok_start[seq], n = p.seq_len[seq];
    float* tl = p.tail + (int64_t)p.seq_slot[seq] * p.tail_slot_stride;
    const bool have_old = p.chain == 2 && p.seq_pos[seq] > 0;
    for (int c = threadIdx.x; c < p.conv_dim; c += blockDim.x) {
        float old[8], nw[8];
        for (int i = 0; i < p.K - 1; i++) old[i] = have_old ? tl[(int64_t)i * p.conv_dim + c] : 0.f;
        for (int i = 0; i < p.K - 1; i++) {
            const int rel = n - (p.K - 1) + i;              // token of this call that lands in tail row i
            nw[i] = rel >= 0 ? p.proj[(int64_t)(t0 + rel) * p.P + p.EH + c] : old[i + n];
        }
        for (int i = 0; i < p.K - 1; i++) tl[(int64_t)i * p.conv_dim + c] = nw[i];
    }
}

// grid (nh, sequences), 256 threads = head_dim x SG state groups; PER = ss / SG states per thread in registers.
// Sequential over the sequence's tokens of this call (the recurrence); everything else is parallel.
template <int PER>
__global__ __launch_bounds__(256) void mamba_scan_kernel(MambaArgs p) {
    const int h = blockIdx.x, seq = blockIdx.y;
    const int SG = 256 / p.hd;                       // host: hd | 256, SG a power of two <= 64, SG * PER == ss (nvllm.hip mamba_states)
    const int d = threadIdx.x / SG, sg = threadIdx.x % SG;
    const int t0 = p.seq_tok_start[seq], n = p.seq_len[seq];
    float* st = p.state + (int64_t)p.seq_slot[seq] * p.state_slot_stride + ((int64_t)h * p.hd + d) * p.ss + sg * PER;
    float s[PER];
    if (p.seq_pos[seq] == 0) {                       // a sequence that (re)starts: zero state (ResetState, generic_model.go:285-292)
#pragma unroll
        for (int i = 0; i < PER; i++) s[i] = 0.f;
    } else {
#pragma unroll
        for (int i = 0; i < PER; i++) s[i] = st[i];
    }
    const float A = p.a_log ? -__expf(p.a_log[h]) : 0.f;          // mamba2.go:286
    const float Dh = p.Dskip ? p.Dskip[h] : 0.f;
    int g = h * p.ng / p.nh;                                      // :301-304
    if (g >= p.ng) g = p.ng - 1;
    for (int i = 0; i < n; i++) {
        const int t = t0 + i;
        const float dt = p.delta[(int64_t)t * p.nh + h];
        const float abar = p.a_log ? __expf(A * dt) : 1.0f;       // :287
        const float* xr = p.xbc + (int64_t)t * p.conv_dim;
        const float u = xr[h * p.hd + d];
        const float* Bt = xr + p.EH + g * p.ss + sg * PER;
        const float* Ct = Bt + p.ng * p.ss;
        float acc = 0.f;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const float v = fmaf(abar, s[q], (dt * Bt[q]) * u);   // :325
            s[q] = v;
            acc = fmaf(Ct[q], v, acc);                            // :333-336
        }
        for (int msk = 1; msk < SG; msk <<= 1) acc += __shfl_xor(acc, msk, 64);
        if (sg == 0) p.y[(int64_t)t * p.EH + h * p.hd + d] = acc + Dh * u;      // :339-345
    }
#pragma unroll
    for (int i = 0; i < PER; i++) st[i] = s[i];
}

// One token per sequence (a decode step), bf16 mode: convolution, softplus, recurrence, gate and the row's share of the gated norm in one
// launch instead of three (8 sequences, 64 heads of 64 x 128 states: 16.4 + 14.9 + 8.7 us).  Bound by the states, read and written once
// (33.5 MB); they are asked for before anything else.  The norm over the whole row is deferred: the operand leaves as bf16(y silu(z) w) with
// the head's sum of squares in rs[token][head], and the output projection multiplies its sums by the row's scale (GemmArgs::rs_in).
// grid (nh, sequences), 256 threads = head_dim x SG state groups; lane group sg holds states 4 (q SG + sg) + 0 .. 3, so that a row's
// lanes read 16 SG contiguous bytes.
template <int PER>
__global__ __launch_bounds__(256) void mamba_step_kernel(MambaArgs p, bf16_t* __restrict__ yn, float* __restrict__ rs) {
    __shared__ __attribute__((aligned(16))) float bc[512], yv[64];
    const int h = blockIdx.x, seq = blockIdx.y, t = p.seq_tok_start[seq];
    const int SG = 256 / p.hd, d = threadIdx.x / SG, sg = threadIdx.x % SG;      // (host: hd | 256, SG * PER == ss <= 256, hd <= 64: nvllm.hip mamba_states)
    f32x4* st = (f32x4*)(p.state + (int64_t)p.seq_slot[seq] * p.state_slot_stride + ((int64_t)h * p.hd + d) * p.ss) + sg;
    f32x4 s[PER / 4];
    if (p.seq_pos[seq] == 0) {
#pragma unroll
        for (int q = 0; q < PER / 4; q++) s[q] = f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
        for (int q = 0; q < PER / 4; q++) s[q] = st[q * SG];
    }
    const float* row = p.proj + (int64_t)t * p.P;
    // (a step's convolution sees its own token only: mamba_conv_kernel)
    auto conv = [&](int c) {
        float v = row[p.EH + c] * p.conv_w[(int64_t)c * p.K + p.K - 1];
        if (p.conv_b) v += p.conv_b[c];
        return silu_ref(v);
    };
    int g = h * p.ng / p.nh;
    if (g >= p.ng) g = p.ng - 1;
    for (int i = threadIdx.x; i < 2 * p.ss; i += 256) bc[i] = conv(p.EH + (i < p.ss ? g * p.ss + i : (p.ng + g) * p.ss + i - p.ss));
    const float u = conv(h * p.hd + d), z = row[h * p.hd + d];
    const float dt = softplus_ref(row[p.EH + p.conv_dim + h] + (p.dt_bias ? p.dt_bias[h] : 0.f));
    const float abar = p.a_log ? __expf(-__expf(p.a_log[h]) * dt) : 1.0f;
    __syncthreads();
    float acc = 0.f;
    const f32x4 *B = (const f32x4*)bc + sg, *C = (const f32x4*)(bc + p.ss) + sg;
#pragma unroll
    for (int q = 0; q < PER / 4; q++) {
        const f32x4 b = B[q * SG], c = C[q * SG];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float v = fmaf(abar, s[q][r], (dt * b[r]) * u);
            s[q][r] = v;
            acc = fmaf(c[r], v, acc);
        }
    }
#pragma unroll
    for (int q = 0; q < PER / 4; q++) st[q * SG] = s[q];
    for (int msk = 1; msk < SG; msk <<= 1) acc += __shfl_xor(acc, msk, 64);
    const float y = (acc + (p.Dskip ? p.Dskip[h] : 0.f) * u) * silu_ref(z);
    float ss = sg == 0 ? y * y : 0.f;
    if (sg == 0) yv[d] = p.norm_w ? y * p.norm_w[h * p.hd + d] : y;
    __shared__ float red[4];
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    if (threadIdx.x == 0) rs[(int64_t)t * p.nh + h] = red[0] + red[1] + red[2] + red[3];
    if ((int)threadIdx.x < p.hd / 4) act_store4<bf16_t>(yn, t, h * p.hd + 4 * threadIdx.x, p.EH, ((const f32x4*)yv)[threadIdx.x]);
}

// ------------------------------------------------------------------------------------------
// Chunked ("SSD") form of the same recurrence for prefill-sized calls in the bf16 mode: one workgroup of four waves per
// (sequence, head) walks its tokens in chunks of Q = 64 and does each chunk with MFMA products instead of 64 dependent
// steps (mamba2.go:256-351 is the sequential statement; this is its algebra).  With a_j = A dt_j, s_t = sum_{j<=t} a_j
// (inclusive, inside the chunk) and S_in the state entering the chunk:
//     state_t = exp(s_t) S_in + sum_{j<=t} exp(s_t - s_j) dt_j  u_j (x) B_j
//     y_t     = exp(s_t) (C_t . S_in) + sum_{j<=t} [exp(s_t - s_j) dt_j (C_t . B_j)] u_j + D u_t
//     S_out   = exp(s_Q) S_in + sum_j [exp(s_Q - s_j) dt_j u_j] (x) B_j
// i.e. four products per chunk, all v_mfma_f32_16x16x32_bf16 with fp32 accumulation:
//     G = C B^T (Q x Q, k = state);  Y_intra = (G o L) U (k = token);  Y_inter = C S_in^T (k = state);  S += (U o w)^T B (k = token)
// Every decay factor is exp of a NON-POSITIVE fp32 number (s decreases), the state lives in fp32 accumulators across the
// chunks and is rounded to bf16 only as the Y_inter operand; u, B, C and the masked decay matrix G o L are rounded to bf16 as
// MFMA operands — the same kind of rounding point the projections around this kernel already have; the
// fp32 parity mode keeps mamba_scan_kernel.  Operands sit in LDS K-contiguous ([row][k], rows padded by 16 bytes: the
// fragment reads are conflict-free), B and U additionally transposed.  A ragged last chunk runs with dt = 0 for the missing
// tokens: they neither decay nor feed the state, and their rows are not stored.
// ------------------------------------------------------------------------------------------
template <int HD, int SS>
constexpr int mamba_ssd_lds_bytes() {
    return 2 * ((64 * (SS + 8)) * 2 + SS * (64 + 8) + 2 * HD * (64 + 8) + 64 * (64 + 8) + HD * (SS + 8)) + 64 * 4 * 2;
}
// MODE 0: one workgroup per (sequence, head) walks the chunks in order (the state stays in its accumulators).
// With few (sequence, head) pairs and long prompts that leaves most of the chip idle, so the chunks can run in parallel:
// MODE 1: grid.z = chunks; each workgroup computes only ITS chunk's contribution to the state from a zero state,
//         Z_c = (U o w)^T B, and the chunk's total decay exp(s_Q) -> scratch;
// mamba_ssd_prefix_kernel: per (sequence, head) the short recurrence S_{c+1} = decay_c S_c + Z_c over the chunks (elementwise),
//         leaving S_c (the state ENTERING chunk c) in the scratch slot of chunk c and the final state in the slot state;
// MODE 2: grid.z = chunks; each workgroup loads the state entering its chunk and computes the chunk's outputs.
template <int HD, int SS, int MODE = 0>
__global__ __launch_bounds__(256) void mamba_ssd_kernel(MambaArgs p) {
    constexpr int Q = 64, DT = HD / 16, NT = SS / 16, NP = 4 / DT, NTW = NT / NP;     // d tiles, state tiles, state parts, state tiles per wave
    constexpr int LC = SS + 8, LQ = Q + 8;                                             // padded row lengths (elements)
    static_assert(HD == 32 || HD == 64, "head_dim 32 / 64");
    static_assert(NT % NP == 0, "state tiles must divide over the waves");
    extern __shared__ __attribute__((aligned(16))) char smem_m[];
    bf16_t* Cs = (bf16_t*)smem_m;                 // [Q][LC]    C_t[n]
    bf16_t* Bs = Cs + Q * LC;                     // [Q][LC]    B_j[n]
    bf16_t* Bt = Bs + Q * LC;                     // [SS][LQ]   B^T
    bf16_t* Ut = Bt + SS * LQ;                    // [HD][LQ]   U^T
    bf16_t* Uw = Ut + HD * LQ;                    // [HD][LQ]   (w_j u_j)^T
    bf16_t* Ms = Uw + HD * LQ;                    // [Q][LQ]    G o L
    bf16_t* Sb = Ms + Q * LQ;                     // [HD][LC]   bf16 copy of the state entering the chunk
    float* s_cum = (float*)(Sb + HD * LC);        // [Q] inclusive prefix sums of a_j
    float* s_dt = s_cum + Q;                      // [Q] dt_j
    const int h = blockIdx.x, seq = blockIdx.y;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int fr = lane & 15, fg = lane >> 4;
    const int t0 = p.seq_tok_start[seq], n = p.seq_len[seq];
    if (MODE != 0 && (int)blockIdx.z * Q >= n) return;          // (uniform: before any barrier)
    const float A = p.a_log ? -__expf(p.a_log[h]) : 0.f;
    const float Dh = p.Dskip ? p.Dskip[h] : 0.f;
    int g = h * p.ng / p.nh;
    if (g >= p.ng) g = p.ng - 1;
    // ---- the state: wave w owns d tile w % DT and state tiles [(w / DT) * NTW, +NTW) in fp32 accumulators ----
    const int sd = wave % DT, sn0 = (wave / DT) * NTW;
    float* st = p.state + (int64_t)p.seq_slot[seq] * p.state_slot_stride + (int64_t)h * HD * SS;
    // chunk-parallel modes: this (sequence, head, chunk)'s scratch slot
    float* zs = MODE != 0 ? p.ssd_z + (((int64_t)seq * gridDim.z + blockIdx.z) * p.nh + h) * (HD * SS) : nullptr;
    f32x4 sacc[NTW];
    const bool fresh = p.seq_pos[seq] == 0;
#pragma unroll
    for (int j = 0; j < NTW; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int64_t o = (int64_t)(16 * sd + 4 * fg + r) * SS + 16 * (sn0 + j) + fr;
            sacc[j][r] = MODE == 1 ? 0.f : (MODE == 2 ? zs[o] : (fresh ? 0.f : st[o]));
        }

    // A chunk's operands travel in registers while the chunk before it is worked on (98 KiB of LDS leave one workgroup a CU: nothing else hides
    // them).  A thread has four tokens of four columns: the transposed copies go to LDS four tokens at a time, in whole rows of banks
    // (token by token they were 2-byte stores, eight to a bank).  2326 tokens x 64 heads, longest 600: 133 us before, 103 now.
    constexpr int BI = 16 * (SS / 4), NBI = (BI + 255) / 256, UI = 16 * (HD / 4);      // (UI <= 256)
    f32x4 rb[NBI][4], rc[NBI][4], ru[4];
    float rdt = 0.f;
    auto fetch = [&](int c0) {
        const int nv = min(Q, n - c0);
        const float* x0 = p.xbc + (int64_t)(t0 + c0) * p.conv_dim;
        rdt = lane < nv ? p.delta[(int64_t)(t0 + c0 + lane) * p.nh + h] : 0.f;
#pragma unroll
        for (int k = 0; k < NBI; k++) {
            const int i = tid + 256 * k, t = 4 * (i & 15), q4 = (min(i, BI - 1) >> 4) * 4;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                // (tokens past the end: the last one's values, replaced below.  With the loads under a condition instead some of these registers lay in scratch memory)
                const float* xr = x0 + (int64_t)min(t + e, nv - 1) * p.conv_dim + p.EH + g * SS + q4;
                rb[k][e] = *(const f32x4*)xr;
                if (MODE != 1) rc[k][e] = *(const f32x4*)(xr + p.ng * SS);
            }
        }
        const int t = 4 * (tid & 15), d4 = (min(tid, UI - 1) >> 4) * 4;
#pragma unroll
        for (int e = 0; e < 4; e++) ru[e] = *(const f32x4*)(x0 + (int64_t)min(t + e, nv - 1) * p.conv_dim + h * HD + d4);
    };
    const int c_first = MODE == 0 ? 0 : (int)blockIdx.z * Q, c_end = MODE == 0 ? n : c_first + 1;
    fetch(c_first);
    for (int c0 = c_first; c0 < c_end; c0 += Q) {
        const int nv = min(Q, n - c0);                          // valid tokens of this chunk
        __syncthreads();                                        // the previous chunk's LDS readers are done
        // ---- decay bookkeeping: every wave scans a_j = A dt_j (lane j), wave 0 leaves it in LDS ----
        float s = A * rdt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const float v = __shfl_up(s, o, 64); if (lane >= o) s += v; }
        const float wj = __expf(__shfl(s, 63, 64) - s) * rdt;
        if (wave == 0) { s_cum[lane] = s; s_dt[lane] = rdt; }
        // ---- the state entering the chunk, as the bf16 operand of Y_inter ----
        if (MODE != 1) {
#pragma unroll
            for (int j = 0; j < NTW; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) Sb[(16 * sd + 4 * fg + r) * LC + 16 * (sn0 + j) + fr] = (bf16_t)sacc[j][r];
        }
        // ---- u, B, C of the chunk as bf16, K-contiguous; B and u also transposed ----
        {
            const int t = 4 * (tid & 15);
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (t + e >= nv) {
                    ru[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int k = 0; k < NBI; k++) { rb[k][e] = f32x4{0.f, 0.f, 0.f, 0.f}; if (MODE != 1) rc[k][e] = f32x4{0.f, 0.f, 0.f, 0.f}; }
                }
        }
#pragma unroll
        for (int k = 0; k < NBI; k++) {
            const int i = tid + 256 * k, t = 4 * (i & 15), q4 = (i >> 4) * 4;
            if (i < BI) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    bf16x4 bb, cc, bt;
#pragma unroll
                    for (int r = 0; r < 4; r++) { bb[r] = (bf16_t)rb[k][e][r]; cc[r] = (bf16_t)rc[k][e][r]; bt[r] = (bf16_t)rb[k][r][e]; }
                    if (MODE != 1) { *(bf16x4*)(Bs + (t + e) * LC + q4) = bb; *(bf16x4*)(Cs + (t + e) * LC + q4) = cc; }
                    if (MODE != 2) *(bf16x4*)(Bt + (q4 + e) * LQ + t) = bt;
                }
            }
        }
        {
            const int t = 4 * (tid & 15), d4 = (tid >> 4) * 4;
            float w[4];
#pragma unroll
            for (int r = 0; r < 4; r++) w[r] = __shfl(wj, 4 * (lane & 15) + r, 64);
            if (tid < UI) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    bf16x4 ut, uw;
#pragma unroll
                    for (int r = 0; r < 4; r++) { ut[r] = (bf16_t)ru[r][e]; uw[r] = (bf16_t)(ru[r][e] * w[r]); }
                    if (MODE != 1) *(bf16x4*)(Ut + (d4 + e) * LQ + t) = ut;
                    if (MODE != 2) *(bf16x4*)(Uw + (d4 + e) * LQ + t) = uw;
                }
            }
        }
        // D u of this wave's rows, then the next chunk (loads return in order)
        float du[4][DT];
        if (MODE != 1) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int t = min(16 * wave + 4 * fg + r, nv - 1);
                const float* ur = p.xbc + (int64_t)(t0 + c0 + t) * p.conv_dim + h * HD;
#pragma unroll
                for (int d = 0; d < DT; d++) du[r][d] = ur[16 * d + fr];
            }
        }
        if (MODE == 0 && c0 + Q < n) fetch(c0 + Q);
        __syncthreads();
        if (MODE != 1) {
            // ---- G = C B^T for this wave's 16 tokens (row tile `wave`), causal column tiles only; M = G o L -> LDS ----
            {
                const int tt = wave;
                float srow[4];
#pragma unroll
                for (int r = 0; r < 4; r++) srow[r] = s_cum[16 * tt + 4 * fg + r];
                for (int jt = 0; jt < 4; jt++) {
                    f32x4 gacc = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (jt <= tt) {
#pragma unroll
                        for (int ks = 0; ks < SS / 32; ks++) {
                            const bf16x8 af = *(const bf16x8*)(Cs + (16 * tt + fr) * LC + ks * 32 + fg * 8);      // A: rows t, k = state
                            const bf16x8 bf = *(const bf16x8*)(Bs + (16 * jt + fr) * LC + ks * 32 + fg * 8);      // B: cols j, k = state
                            gacc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, gacc, 0, 0, 0);
                        }
                    }
                    const int j = 16 * jt + fr;                       // this lane's column (token j), rows t = 16 tt + 4 fg + r
                    const float sj = s_cum[j], dj = s_dt[j];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int t = 16 * tt + 4 * fg + r;
                        const float v = (j <= t) ? gacc[r] * (__expf(srow[r] - sj) * dj) : 0.f;
                        Ms[t * LQ + j] = (bf16_t)v;
                    }
                }
            }
            __syncthreads();
            // ---- y rows of this wave: Y_intra = M U (k = token) and Y_inter = C S_in^T (k = state) ----
            {
                const int tt = wave;
                f32x4 yi[DT], ye[DT];
#pragma unroll
                for (int d = 0; d < DT; d++) { yi[d] = f32x4{0.f, 0.f, 0.f, 0.f}; ye[d] = yi[d]; }
#pragma unroll
                for (int ks = 0; ks < Q / 32; ks++) {
                    if (ks * 32 > 16 * tt + 15) continue;             // tokens beyond this tile's last row: M is zero there
                    const bf16x8 af = *(const bf16x8*)(Ms + (16 * tt + fr) * LQ + ks * 32 + fg * 8);
#pragma unroll
                    for (int d = 0; d < DT; d++) {
                        const bf16x8 bf = *(const bf16x8*)(Ut + (16 * d + fr) * LQ + ks * 32 + fg * 8);
                        yi[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, yi[d], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int ks = 0; ks < SS / 32; ks++) {
                    const bf16x8 af = *(const bf16x8*)(Cs + (16 * tt + fr) * LC + ks * 32 + fg * 8);
#pragma unroll
                    for (int d = 0; d < DT; d++) {
                        const bf16x8 bf = *(const bf16x8*)(Sb + (16 * d + fr) * LC + ks * 32 + fg * 8);
                        ye[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, ye[d], 0, 0, 0);
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int t = 16 * tt + 4 * fg + r;
                    if (t >= nv) continue;
                    const float es = __expf(s_cum[t]);
                    float* yr = p.y + (int64_t)(t0 + c0 + t) * p.EH + h * HD;
#pragma unroll
                    for (int d = 0; d < DT; d++) yr[16 * d + fr] = yi[d][r] + es * ye[d][r] + Dh * du[r][d];
                }
            }
        }
        if (MODE != 2) {
            // ---- S_out = exp(s_Q) S_in + (U o w)^T B  (k = token) ----
            const float eq = __expf(s_cum[Q - 1]);
#pragma unroll
            for (int j = 0; j < NTW; j++) sacc[j] *= eq;
#pragma unroll
            for (int ks = 0; ks < Q / 32; ks++) {
                const bf16x8 af = *(const bf16x8*)(Uw + (16 * sd + fr) * LQ + ks * 32 + fg * 8);              // A: rows d, k = token
#pragma unroll
                for (int j = 0; j < NTW; j++) {
                    const bf16x8 bf = *(const bf16x8*)(Bt + (16 * (sn0 + j) + fr) * LQ + ks * 32 + fg * 8);   // B: cols n, k = token
                    sacc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, sacc[j], 0, 0, 0);
                }
            }
            if (MODE == 1 && tid == 0) p.ssd_decay[((int64_t)seq * gridDim.z + blockIdx.z) * p.nh + h] = eq;
        }
    }
    if (MODE == 2) return;
    float* dst = MODE == 1 ? zs : st;
#pragma unroll
    for (int j = 0; j < NTW; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) dst[(int64_t)(16 * sd + 4 * fg + r) * SS + 16 * (sn0 + j) + fr] = sacc[j][r];
}

// the chunk recurrence of the chunk-parallel form: grid (nh, sequences, state_elems / 1024), one f32x4 of the head's hd x ss
// state per thread; the chunks are walked four at a time so that four slots' loads are in flight per round trip
__global__ __launch_bounds__(256) void mamba_ssd_prefix_kernel(MambaArgs p, int max_chunks, int state_elems) {
    const int h = blockIdx.x, seq = blockIdx.y;
    const int e = (blockIdx.z * 256 + threadIdx.x) * 4;
    if (e >= state_elems) return;
    const int nc = (p.seq_len[seq] + 63) / 64;
    float* st = p.state + (int64_t)p.seq_slot[seq] * p.state_slot_stride + (int64_t)h * state_elems + e;
    f32x4 run = p.seq_pos[seq] == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : *(const f32x4*)st;
    const int64_t slot0 = (int64_t)seq * max_chunks * p.nh + h;          // slot of chunk c: slot0 + c * nh
    for (int c0 = 0; c0 < nc; c0 += 4) {
        f32x4 z[4];
        float dc[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int c = min(c0 + i, nc - 1);
            z[i] = *(const f32x4*)(p.ssd_z + (slot0 + (int64_t)c * p.nh) * state_elems + e);
            dc[i] = p.ssd_decay[slot0 + (int64_t)c * p.nh];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (c0 + i >= nc) break;
            *(f32x4*)(p.ssd_z + (slot0 + (int64_t)(c0 + i) * p.nh) * state_elems + e) = run;      // the state entering chunk c
            run = dc[i] * run + z[i];
        }
    }
    *(f32x4*)st = run;
}

// grid (tokens), 256 threads: y *= SiLU(gate); rms over EH; * norm weight; written as the out_proj GEMM's operand
template <typename ActT>
__global__ __launch_bounds__(256) void mamba_gate_norm_kernel(MambaArgs p, ActT* __restrict__ out) {
    __shared__ float red[4];
    const int t = blockIdx.x;
    const float* gate = p.proj + (int64_t)t * p.P;
    float* yr = p.y + (int64_t)t * p.EH;
    float ss = 0.f;
    for (int c = threadIdx.x; c < p.EH; c += 256) {
        const float v = yr[c] * silu_ref(gate[c]);
        yr[c] = v;
        ss = fmaf(v, v, ss);
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    const float rms = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)p.EH + 1e-5f);      // eps fixed in mamba2.go:147
    for (int c = threadIdx.x * 4; c < p.EH; c += 1024) {       // EH % 4 == 0 (host)
        f32x4 v = *(const f32x4*)(yr + c) * rms;
        if (p.norm_w) v *= *(const f32x4*)(p.norm_w + c);
        act_store4<ActT>(out, t, c, p.EH, v);
    }
}

// Prefill-sized bf16 batches, EH <= 4096: a wave holds a row in registers (y is read once and not written back), eight rows a workgroup, so
// that the operand leaves in whole 128-byte lines (row by row each lane's 8 bytes were a line of their own: 2326 x 4096 48 us, 34
// here).  Below 512 rows too few workgroups: a prompt of 24 layers of 4096 columns, here -> row by row, 130 / 200 / 300 / 400 tokens 1343 -> 1310, 1433 -> 1401, 1681 -> 1658, 1885 -> 1872 us;
// 600 as long either way, 1000 / 1900 2952 -> 2982, 4754 -> 4863.  us a launch, row by row / in tiles, at 130, 300, 512, 600, 1000 and 1900 rows: 4096 columns 11.6 / 15.0, 13.3 / 15.4,
// 15.8 / 15.9, 16.8 / 16.1, 20.5 / 17.6, 33.5 / 21.2; 3072 9.7 / 12.3, 11.0 / 12.7, 11.5 / 12.8, 12.4 / 13.0, 15.3 / 14.9, 26.0 / 17.8; 2048 8.2 / 11.3, 8.7 / 11.2, 9.6 / 11.3, 9.8 / 11.3,
// 11.5 / 12.0, 16.4 / 14.1; 1024 6.5 / 10.0, 7.1 / 10.3, 7.3 / 10.2, 7.5 / 10.3, 8.1 / 10.3, 10.4 / 11.5; 512 6.6 / 9.5, 6.9 / 10.0, 7.0 / 10.4, 6.7 / 9.8, 6.8 / 10.1, 7.8 / 10.6.  So up to 512 rows
// no width is better off in tiles; narrower ones would be row by row for some more.
constexpr int MAMBA_GATE_TILE_ROWS = 512;
static inline constexpr int mamba_gate_tile_lds_bytes(int EH) { return 8 * (EH + 8) * 2; }
static __global__ __launch_bounds__(512) void mamba_gate_norm_tile_kernel(MambaArgs p, bf16_t* __restrict__ out, int tokens) {
    constexpr int CH = 16;
    extern __shared__ __attribute__((aligned(16))) char smem_g[];
    bf16_t* tile = (bf16_t*)smem_g;                       // [8][EH + 8]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, LT = p.EH + 8;
    const int64_t t = (int64_t)blockIdx.x * 8 + wave;
    if (t < tokens) {
        const float *gate = p.proj + t * p.P, *yr = p.y + t * p.EH;
        f32x4 v[CH];
        float ss = 0.f;
#pragma unroll
        for (int c0 = 0; c0 < CH; c0 += 8) {
            f32x4 g[8];
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const int j = (lane + (c0 + c) * 64) * 4;
                const bool in = j < p.EH;
                v[c0 + c] = in ? *(const f32x4*)(yr + j) : f32x4{0.f, 0.f, 0.f, 0.f};
                g[c] = in ? *(const f32x4*)(gate + j) : f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int c = 0; c < 8; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float a = v[c0 + c][r] * silu_ref(g[c][r]);
                    v[c0 + c][r] = a;
                    ss = fmaf(a, a, ss);
                }
        }
        const float rms = 1.0f / sqrtf(wave_sum(ss) / (float)p.EH + 1e-5f);
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int j = (lane + c * 64) * 4;
            if (j >= p.EH) continue;
            f32x4 a = v[c] * rms;
            if (p.norm_w) a *= *(const f32x4*)(p.norm_w + j);
            bf16x4 o;
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = (bf16_t)a[r];
            *(bf16x4*)(tile + wave * LT + j) = o;
        }
    }
    __syncthreads();
    // 32 columns of eight rows: lane (row, 8 columns) of half an operand block, two blocks a wave
    const int nkb = p.EH >> 5, row = lane & 7, q = (lane >> 3) & 3;
    const int64_t r0 = (int64_t)blockIdx.x * 8;
    if (r0 + row < tokens)
        for (int kb = 2 * wave + (lane >> 5); kb < nkb; kb += 16)
            *(bf16x8*)(out + fm_index(r0 + row, kb * 32 + 8 * q, p.EH)) = *(const bf16x8*)(tile + row * LT + kb * 32 + 8 * q);
}

}  // namespace nvl
