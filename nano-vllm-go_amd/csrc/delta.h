// delta.h — gated delta rule with a decay per key channel, in fp32 throughout.  Per head, S [DK][DV]:
//     S <- diag(a_t) S,  u_t = beta_t (v_t - S^T k_t),  S <- S + k_t u_t^T,  o_t = S^T q_t
// q and k are unit vectors (q also times q_scale); a_t = exp(-exp(A_log) softplus(z_t + bias)), z_t a projection; a group of heads
// shares q and k, decays and values are a head's own.
//
//   delta_step_kernel   token by token, the state streamed once per token (decode).  FUSED (one token per sequence): the short
//                       convolutions, the low-rank decay and gate projections, the head norm and the output gate in the same launch.
//   delta_prep_kernel   32 tokens of one head, independent of the state that enters them (prefill; a workgroup goes from chunk to chunk).
//   delta_scan_kernel, delta_scan_parts_kernel   carry the state through the chunks of a sequence: three products per chunk.
//
// Chunk form.  With b_t = the inclusive sum of log a inside the chunk and S_in the state that enters it:
//     u_t = beta_t (v_t - (k_t e^{b_t})^T S_in - sum_{s<t} M[t][s] u_s),      M[t][s] = sum_c k_t[c] k_s[c] e^{b_t[c] - b_s[c]}
//     o_t = (q_t e^{b_t})^T S_in + sum_{s<=t} A[t][s] u_s,                    A[t][s] = sum_c q_t[c] k_s[c] e^{b_t[c] - b_s[c]}
//     S_out = diag(e^{b_end}) S_in + sum_s (k_s e^{b_end - b_s}) u_s^T
// With T = (I + diag(beta) M)^-1 diag(beta):  U = U0 - W S_in,  U0 = T V,  W = T (K e^b);  O = O0 + Q' S_in,  O0 = (A T) V,
// Q' = Q e^b - (A T) (K e^b).  prep leaves -W, Q', (K e^{b_end - b})^T and e^{b_end} in scratch, U0 in the place of v and O0 in the place of o.
// Every exponent that is evaluated is <= 0: a decay per channel cannot be split into e^{b_t} e^{-b_s}, so the four 8 x 8 diagonal
// blocks of A and M are summed pair by pair, and the blocks below take the sums of the token before their rows (7, 15, 23) as their reference.  T is built
// block by block from exact inverses: the powers of M that a series would need can be far larger than T itself.
// Products are v_mfma_f32_16x16x4_f32: operand element i of lane group g stands for k = 16 n + 4 g + i on both sides, so that an
// accumulator (lane = column, rows 4 g + r) is the B operand of the next product as it stands.
#pragma once
#include "common.h"
#include "linrec.h"

namespace nvl {

constexpr float DELTA_UNIT_EPS = 1e-6f;

struct DeltaArgs {
    int H, G, DK, DV, DVp;             // G: heads of q and k; DVp: row pitch of the state (DV padded to 4)
    const float *q, *k; float* v;      // after convolution and silu; row pitch ld; v: prep leaves U0 there
    int64_t ld;
    float q_scale;
    const float* z; int64_t z_ld;      // [token][H * DK] decay projections before the bias
    const float *a_log, *dt_bias;      // [H], [H * DK]
    const float* beta; int64_t beta_ld;        // raw step sizes (before sigmoid), one column per head
    float* o; int64_t o_ld;            // [token][H * DV]
    float* state; int64_t slot_stride; // slot s: state + s * slot_stride, [H][DK][DVp]
    const int32_t *seq_tok_start, *seq_len, *seq_pos, *seq_slot;
    int vec4, vec4v;                   // q, k / v, o rows may be accessed 16 bytes at a time
    int len_lo, len_hi;                // sequences with len_lo <= tokens of this call <= len_hi are served, the others skipped
    float* ws;                         // chunk c of sequence i is (seq_tok_start / 32 + i + c); per chunk and head delta_ws_floats
    // FUSED step: raw [q | k | v] columns before the convolution, a ring of the last `taps` raw rows per slot
    const float* raw; int64_t raw_ld; const float* conv_w; int taps, channels; float* ring; int64_t ring_slot_stride;
    const float *a1, *g1; int64_t lr_ld; int a_rank, g_rank, a_rkp, g_rkp;       // [token][rank]; ranks padded
    const void *a2, *g2;               // [H * DK][a_rkp], [H * DV][g_rkp], row-major
    const float* norm_w; float eps; void* out; int64_t out_ld;
};

constexpr int DELTA_C = 32;            // tokens per chunk
constexpr int DELTA_ORDERED = 64;       // sequences that the scan takes in the order of their lengths, at most
constexpr int DELTA_SCAN_WAVES = 4;    // of a workgroup of the scan
// A chunk of a head in scratch: -W, Q' and (K e^{b_end - b})^T as operands of the scan's products, a KiB each of its 64 lanes' 16 bytes: per 16 key channels
// tokens 0 .. 15 and 16 .. 31 of -W, of Q' and of K.  Then e^{b_end}.
static inline __host__ __device__ int64_t delta_ws_floats(int dkp) { return (int64_t)dkp * (3 * DELTA_C + 1); }
static inline __host__ __device__ constexpr int delta_piece(int i, int x) { return (6 * i + x) * 64; }
__device__ __forceinline__ int64_t delta_chunk(const DeltaArgs& p, int seq, int c) { return p.seq_tok_start[seq] / DELTA_C + seq + c; }

// log(1 + e^x) from the hardware's base-2 exponential and logarithm; what 1 + y rounds away is added back
__device__ __forceinline__ float delta_softplus(float x) {
    const float y = ex2(-1.4426950408889634f * fabsf(x)), u = 1.0f + y;
    return fmaxf(x, 0.f) + fmaf(0.6931471805599453f, __builtin_amdgcn_logf(u), (y - (u - 1.0f)) * __builtin_amdgcn_rcpf(u));
}

// Rows of a chunk, from its first.  The descriptor ends with the sequence and columns beyond a head lie outside it (OUTSIDE): what is read there is zero, and what is
// written there is dropped.
struct DeltaRows { char* base; uint32_t pitch; };
constexpr uint32_t DELTA_OUTSIDE = 1u << 31;
// (a chunk's rows are below 2^31 bytes.  readfirstlane: the compiler doesn't see that these are uniform, and loops over the lanes' descriptors)
__device__ __forceinline__ auto delta_rows(const DeltaRows& w, int64_t row, int rows) {
    const uint64_t at = (uint64_t)(w.base + row * w.pitch);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at), hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    return __builtin_amdgcn_make_buffer_rsrc((void*)((uint64_t)hi << 32 | lo), 0, __builtin_amdgcn_readfirstlane(max(min(rows, DELTA_C), 0) * (int)w.pitch), 0x00020000);
}
template <typename Rsrc> __device__ __forceinline__ float buffer_f32(Rsrc rs, uint32_t at) { return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0)); }
template <typename Rsrc> __device__ __forceinline__ f32x4 buffer_f32x4(Rsrc rs, int lane_off, int off) {
    union { f32x4 f; u32x4 u; } t;
    t.u = __builtin_amdgcn_raw_buffer_load_b128(rs, lane_off, off, 0);
    return t.f;
}
template <typename Rsrc> __device__ __forceinline__ void buffer_put(Rsrc rs, uint32_t at, float x) { __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, x), rs, at, 0, 0); }
template <typename Rsrc> __device__ __forceinline__ void buffer_put4(Rsrc rs, int lane_off, int off, f32x4 x) {
    union { f32x4 f; u32x4 u; } t; t.f = x;
    __builtin_amdgcn_raw_buffer_store_b128(t.u, rs, lane_off, off, 0);
}
template <typename Rsrc> __device__ __forceinline__ f32x4 delta_rows_get(Rsrc rs, uint32_t at, uint32_t pitch) {       // a column of four rows
    f32x4 x;
#pragma unroll
    for (int r = 0; r < 4; r++) x[r] = buffer_f32(rs, at + r * pitch);
    return x;
}

// ------------------------------------------------------------------------------------------
// prep: grid (heads, workgroups that share its chunks), 8 waves.  Bound by the chain of a chunk, six barriers with little for most waves between some of them, of which two
// workgroups a CU hide a part: no unit is full.  5 x 300 .. 1900 tokens x 16 heads of 128, 106 us: 147 KB a chunk (q, k, v, z in, five operands out) are 3.9 TB/s, 3.1 of them
// HBM's (a copy reaches 5.0); vector ALUs 43 % of the time, LDS 32 (12 of it bank conflicts), matrix cores 20.  Loads are no part of the chain because a chunk's leave when the
// one before has read its registers; pairs are summed one by one inside blocks of 8 tokens only (of 16: 8500 of 46000 cycles a chunk, and two of eight waves had the products as well).
// us a layer, a workgroup per chunk and blocks of 16 -> here: 5 x 300 .. 1900 tokens x 16 heads 143 -> 109, 10 x 100 .. 900 134 -> 90, 16 x 900 370 -> 290.
// ------------------------------------------------------------------------------------------
template <int NK> constexpr int delta_prep_lds_bytes() { return 4 * (3 * DELTA_C * (NK * 16 + 4) + 2 * DELTA_C * 36 + DELTA_C + 512); }
// The chunks of all sequences that a launch serves, from the last to the first: the scan begins with those that were written last
struct DeltaChunk { int seq, tok0, rows; int64_t at; };       // sequence, first token, tokens; place in scratch
struct DeltaChunks {
    const int *seq_len, *seq_tok_start;
    int n_seqs, len_lo, len_hi;
    int first, len, tok0, count, end;    // 64 sequences from `first` on: this lane's, its chunks, and all from there on
    __device__ __forceinline__ DeltaChunks(const DeltaArgs& p, int n) : seq_len(p.seq_len), seq_tok_start(p.seq_tok_start), n_seqs(n), len_lo(p.len_lo), len_hi(p.len_hi) { load((n - 1) & ~63, 0); }
    __device__ __forceinline__ void load(int f, int behind) {
        const int lane = threadIdx.x & 63;
        len = f + lane < n_seqs ? seq_len[f + lane] : 0;
        tok0 = f + lane < n_seqs ? seq_tok_start[f + lane] : 0;
        first = f;
        count = len >= len_lo && len <= len_hi ? (len + DELTA_C - 1) / DELTA_C : 0;
        end = count;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int v = __shfl_down(end, o, 64); if (lane + o < 64) end += v; }
        end += behind;
    }
    __device__ __forceinline__ bool find(int j, DeltaChunk& k) {         // chunk j, or false: there are no more (j grows from call to call)
        for (;;) {
            const unsigned long long m = __ballot(end > j);
            if (m) {
                const int l = 63 - __builtin_clzll(m), c = __builtin_amdgcn_readlane(end, l) - 1 - j, t = __builtin_amdgcn_readlane(tok0, l);
                k.seq = first + l;
                k.tok0 = t + c * DELTA_C;
                k.rows = min(DELTA_C, __builtin_amdgcn_readlane(len, l) - c * DELTA_C);
                k.at = t / DELTA_C + k.seq + c;
                return true;
            }
            if (first == 0) return false;
            load(first - 64, __builtin_amdgcn_readlane(end, 0));
        }
    }
};

// VEC, VECV: DeltaArgs::vec4, vec4v, each for its own rows.  Where the values' width ruled both, keys that could come 16 bytes at a time came 4 at a time: 16 x 900 tokens,
// 128 x 130 / 66 x 64 channels 404 -> 372, 285 -> 247 us a layer
template <int NK, bool VEC, bool VECV>
__global__ __launch_bounds__(512, NK > 8 ? 2 : 4) void delta_prep_kernel(DeltaArgs p, int n_seqs) {
    constexpr int C = DELTA_C, DKP = NK * 16, LQ = DKP + 4, LA = 36, NT = 512, NW = NT / 64;
    constexpr float LOG2E = 1.4426950408889634f;
    const int h = blockIdx.x;
    DeltaChunks chunks(p, n_seqs);
    DeltaChunk now, next;
    if (!chunks.find(blockIdx.y, now)) return;                   // (uniform: before any barrier)
    extern __shared__ __attribute__((aligned(16))) float dl_sm[];
    float* qs = dl_sm;                   // [C][LQ]  q, later q e^b
    float* ks = qs + C * LQ;             // [C][LQ]  k, later k e^b
    float* bs = ks + C * LQ;             // [C][LQ]  inclusive sums of log2 a
    float* As = bs + C * LQ;             // [C][LA]  A, later A T
    float* Ms = As + C * LA;             // [C][LA]  M, later X = (I + diag(beta) M)^-1
    float* be = Ms + C * LA;             // [C]
    float* aux = be + C;                 // [512]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = h / (p.H / p.G);
    // the loads of a chunk: q and k (DKP / 4 lanes hold a row), z (a channel per thread, NG groups share the tokens), beta and the
    // first value channels of this wave
    constexpr int LR = DKP / 4, R = NT / LR, NQ = (C + R - 1) / R, NG = NT / DKP, TPG = C / NG;
    const int nvb = (p.DV + 15) >> 4;
    // (a thread's number anew for each part of a chunk, or everything that follows from it is kept in registers all along)
    auto thread = [&]() __attribute__((always_inline)) { int t = threadIdx.x; asm volatile("" : "+v"(t)); return t; };
    f32x4 q4[NQ], k4[NQ], v4[2];
    float pre[TPG], be_raw = 0.f;
    const DeltaRows qr{(char*)(p.q + (int64_t)g * p.DK), 4 * (uint32_t)p.ld}, kr{(char*)(p.k + (int64_t)g * p.DK), qr.pitch}, vr{(char*)(p.v + (int64_t)h * p.DV), qr.pitch};
    const DeltaRows zr{(char*)(p.z + (int64_t)h * p.DK), 4 * (uint32_t)p.z_ld}, br{(char*)(p.beta + h), 4 * (uint32_t)p.beta_ld}, orow{(char*)(p.o + (int64_t)h * p.DV), 4 * (uint32_t)p.o_ld};
    auto ld4 = [&](auto rs, int qd, uint32_t at) __attribute__((always_inline)) {
        if (VEC) return buffer_f32x4(rs, qd < p.DK ? at : DELTA_OUTSIDE, 0);
        f32x4 x;
#pragma unroll
        for (int r = 0; r < 4; r++) x[r] = buffer_f32(rs, qd + r < p.DK ? at + 4 * r : DELTA_OUTSIDE);
        return x;
    };
    auto ldv = [&](int64_t tb, int nv, int i, f32x4 (&v)[2]) __attribute__((always_inline)) {       // 16 value channels as the A operand of a transposed product
        const auto rs = delta_rows(vr, tb, nv);
        const int lane = thread() & 63, fr = lane & 15, fg = lane >> 4, c = 16 * i + fr;
        const uint32_t at = 4 * fg * vr.pitch + (c < p.DV ? 4 * c : DELTA_OUTSIDE);
        v[0] = delta_rows_get(rs, at, vr.pitch); v[1] = delta_rows_get(rs, at + 16 * vr.pitch, vr.pitch);
    };
    auto load_qk = [&](int64_t tb, int nv) __attribute__((always_inline)) {
        const int tid = thread(), qt = tid / LR, qd = tid % LR * 4;
        const auto rq = delta_rows(qr, tb, nv), rk = delta_rows(kr, tb, nv);
        const uint32_t at_q = qt * qr.pitch + 4 * qd;
#pragma unroll
        for (int i = 0; i < NQ; i++) { q4[i] = ld4(rq, qd, at_q + i * R * qr.pitch); k4[i] = ld4(rk, qd, at_q + i * R * qr.pitch); }
    };
    auto load_z = [&](int64_t tb, int nv) __attribute__((always_inline)) {
        const int tid = thread(), zd = tid % DKP, grp = tid / DKP;
        const auto rz = delta_rows(zr, tb, nv);
        const uint32_t at_z = grp * TPG * zr.pitch + (zd < p.DK ? 4 * zd : DELTA_OUTSIDE);
#pragma unroll
        for (int j = 0; j < TPG; j++) pre[j] = buffer_f32(rz, at_z + j * zr.pitch);
        be_raw = buffer_f32(delta_rows(br, tb, nv), (tid & (C - 1)) * br.pitch);
    };
    auto barrier = [&]() __attribute__((always_inline)) {            // (without the wait for the next chunk's loads)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const float A = -expf(p.a_log[h]) * LOG2E, bias = (int)threadIdx.x % DKP < p.DK ? p.dt_bias[h * p.DK + threadIdx.x % DKP] : 0.f;
    load_qk(now.tok0, now.rows);
    load_z(now.tok0, now.rows);
    __builtin_amdgcn_sched_barrier(0);
    ldv(now.tok0, now.rows, wave, v4);                           // (beyond DV: zeros)
    for (int job = blockIdx.y;;) {
    const auto ws = __builtin_amdgcn_make_buffer_rsrc(p.ws + (now.at * p.H + h) * delta_ws_floats(DKP), 0, 4 * (int)delta_ws_floats(DKP), 0x00020000);
    // the chunk behind this one, whose loads go out as soon as this one's registers are read
    job += gridDim.y;
    const bool more = chunks.find(job, next);
    if (!more) next = now;                                       // (the last one's are fetched again instead of a branch)
    const int nv = now.rows, tb = now.tok0;
    int tid = thread();
    const int qt = tid / LR, qd = tid % LR * 4, zd = tid % DKP, grp = tid / DKP;
#pragma unroll
    for (int i = 0; i < NQ; i++) {               // unit vectors
        const f32x4 q = q4[i], k = k4[i];
        float sq = (q[0] * q[0] + q[1] * q[1]) + (q[2] * q[2] + q[3] * q[3]), sk = (k[0] * k[0] + k[1] * k[1]) + (k[2] * k[2] + k[3] * k[3]);
#pragma unroll
        for (int o = 1; o < LR; o <<= 1) { sq += __shfl_xor(sq, o, 64); sk += __shfl_xor(sk, o, 64); }
        if (C % R && qt + i * R >= C) continue;
        *(f32x4*)(qs + (qt + i * R) * LQ + qd) = q * (p.q_scale / sqrtf(sq + DELTA_UNIT_EPS));
        *(f32x4*)(ks + (qt + i * R) * LQ + qd) = k * (1.0f / sqrtf(sk + DELTA_UNIT_EPS));
    }
    __builtin_amdgcn_sched_barrier(0);
    load_qk(next.tok0, next.rows);
    __builtin_amdgcn_sched_barrier(0);
    {   // decays
        float s[TPG];
#pragma unroll
        for (int j = 0; j < TPG; j++) s[j] = zd < p.DK && grp * TPG + j < nv ? A * delta_softplus(pre[j] + bias) : 0.f;
        if (tid < C) be[tid] = tid < nv ? lr_sigmoid(be_raw) : 0.f;
        __builtin_amdgcn_sched_barrier(0);
        load_z(next.tok0, next.rows);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 1; j < TPG; j++) s[j] += s[j - 1];
        aux[grp * DKP + zd] = s[TPG - 1];
        barrier();
        float off = 0.f;
        for (int j = 0; j < grp; j++) off += aux[j * DKP + zd];
#pragma unroll
        for (int j = 0; j < TPG; j++) bs[(grp * TPG + j) * LQ + zd] = off + s[j];
    }
    for (int i = tid; i < 2 * C * LA; i += NT) As[i] = 0.f;      // (what lies above the diagonals stays zero)
    barrier();
    tid = thread();
    // ---- A (s <= t) and M (s < t): 112 pairs of the four 8 x 8 diagonal blocks, four threads each; the last wave takes A's diagonal ----
    if (tid < 448) {
        const int pr = tid >> 2, blk = pr / 28, x = pr - 28 * blk;
        int t = (int)((sqrtf(8.f * (float)x + 1.f) - 1.f) * 0.5f);
        if ((t + 1) * (t + 2) / 2 <= x) t++;
        if (t * (t + 1) / 2 > x) t--;
        const int s = x - t * (t + 1) / 2, tr = (8 * blk + t + 1) * LQ, sr = (8 * blk + s) * LQ;
        f32x4 aq = f32x4{0.f, 0.f, 0.f, 0.f}, ak = aq;
#pragma unroll 2
        for (int d = 4 * (tid & 3); d < DKP; d += 16) {
            const f32x4 q4 = *(const f32x4*)(qs + tr + d), k4 = *(const f32x4*)(ks + tr + d), k2 = *(const f32x4*)(ks + sr + d);
            const f32x4 bt = *(const f32x4*)(bs + tr + d), b2 = *(const f32x4*)(bs + sr + d);
#pragma unroll
            for (int r = 0; r < 4; r++) { const float e = ex2(bt[r] - b2[r]) * k2[r]; aq[r] = fmaf(q4[r], e, aq[r]); ak[r] = fmaf(k4[r], e, ak[r]); }
        }
        const int at = (8 * blk + t + 1) * LA + 8 * blk + s;
        float sa = (aq[0] + aq[1]) + (aq[2] + aq[3]), sm = (ak[0] + ak[1]) + (ak[2] + ak[3]);
        sa += __shfl_xor(sa, 1, 64); sm += __shfl_xor(sm, 1, 64);
        sa += __shfl_xor(sa, 2, 64); sm += __shfl_xor(sm, 2, 64);
        if ((tid & 3) == 0) As[at] = sa; else if ((tid & 3) == 1) Ms[at] = sm;
    } else {
        const int t = (tid - 448) >> 1;
        f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
        for (int d = 4 * (tid & 1); d < DKP; d += 8) a += *(const f32x4*)(qs + t * LQ + d) * *(const f32x4*)(ks + t * LQ + d);
        float s = (a[0] + a[1]) + (a[2] + a[3]);
        s += __shfl_xor(s, 1, 64);
        if ((tid & 1) == 0) As[t * LA + t] = s;
    }
    int lane = tid & 63, fr = lane & 15, fg = lane >> 4;
    if (wave < 4) {                                              // wave 0: A, 1: M of tokens 16..31 against 0..15; 2, 3: of 8..15 against 0..7 and of 24..31 against 16..23
        const float* x = wave & 1 ? ks : qs;
        const int half = 16 * (fr >> 3), ta = wave < 2 ? 16 + fr : half + 8 + (fr & 7), ts = wave < 2 ? fr : half + (fr & 7), tref = wave < 2 ? 15 : half + 7;
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f}, odd = acc;
#pragma unroll 2
        for (int i = 0; i < NK; i++) {
            const int c = 16 * i + 4 * fg;
            const f32x4 ref = *(const f32x4*)(bs + tref * LQ + c);
            const f32x4 a = *(const f32x4*)(x + ta * LQ + c), b = *(const f32x4*)(ks + ts * LQ + c);
            const f32x4 ba = *(const f32x4*)(bs + ta * LQ + c), bb = *(const f32x4*)(bs + ts * LQ + c);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                f32x4& d = r & 1 ? odd : acc;
                d = mfma_f32(a[r] * ex2(ba[r] - ref[r]), b[r] * ex2(ref[r] - bb[r]), d);
            }
        }
        acc += odd;
        float* dst = wave & 1 ? Ms : As;
        // (waves 2 and 3: rows of one half against columns of the other are of no use)
        if (wave < 2 || fg >> 1 == fr >> 3) {
            const int row = wave < 2 ? 16 + 4 * fg : half + 8 + 4 * (fg & 1);
#pragma unroll
            for (int r = 0; r < 4; r++) dst[(row + r) * LA + ts] = acc[r];
        }
    }
    barrier();
    tid = thread(); lane = tid & 63; fr = lane & 15; fg = lane >> 4;
    if (wave < 2) {
        // inverses of the two diagonal blocks of I + N, N = diag(beta) M, from 1 x 1 blocks upwards: with X the inverse of the part inside
        // b x b blocks and N_b the part that a 2b x 2b block adds, X - X N_b X is the inverse inside 2b x 2b blocks
        const int o = 16 * wave;
        float* xt = aux + 256 * wave;                            // X's turn from accumulator to A operand
        const f32x4 na = *(const f32x4*)(Ms + (o + fr) * LA + o + 4 * fg) * be[o + fr];
        f32x4 xa, xd;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int c = 4 * fg + r;                            // (row fr, column c) as an A operand, (row c, column fr) as an accumulator
            xa[r] = fr == c ? 1.f : ((fr ^ c) == 1 ? -na[r] : 0.f);
            xd[r] = fr == c ? 1.f : ((fr ^ c) == 1 ? -Ms[(o + c) * LA + o + fr] * be[o + c] : 0.f);
        }
#pragma unroll
        for (int lb = 1; lb < 4; lb++) {                         // b = 2, 4, 8
            f32x4 y = f32x4{0.f, 0.f, 0.f, 0.f}, z = y;
#pragma unroll
            for (int r = 0; r < 4; r++) y = mfma_f32(((fr ^ (4 * fg + r)) >> lb) == 1 ? na[r] : 0.f, xd[r], y);
#pragma unroll
            for (int r = 0; r < 4; r++) z = mfma_f32(xa[r], y[r], z);
            xd -= z;
            if (lb == 3) break;
#pragma unroll
            for (int r = 0; r < 4; r++) xt[(4 * fg + r) * 16 + fr] = xd[r];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            xa = *(const f32x4*)(xt + fr * 16 + 4 * fg);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) Ms[(o + 4 * fg + r) * LA + o + fr] = xd[r];
    } else {
        // (K e^{b_end - b})^T and e^{b_end}
#pragma unroll
        for (int j = 0; j < (2 * NK * 64 + NT - 129) / (NT - 128); j++) {      // (as often for each thread: the compiler counts the stores behind the next chunk's loads)
            const int i = min(tid - 128 + j * (NT - 128), 2 * NK * 64 - 1);
            const int l = i & 63, sb = (i >> 6) & 1, d = 16 * (i >> 7) + (l & 15), t = 16 * sb + 4 * (l >> 4);
            const float b_end = bs[31 * LQ + d];
            f32x4 x;
#pragma unroll
            for (int r = 0; r < 4; r++) x[r] = ks[(t + r) * LQ + d] * ex2(b_end - bs[(t + r) * LQ + d]);
            buffer_put4(ws, 16 * (delta_piece(i >> 7, 4 + sb) + l), 0, x);
        }
        const int d = min(tid - 128, DKP - 1);
        buffer_put(ws, 4 * (3 * C * DKP + d), ex2(bs[31 * LQ + d]));
    }
    barrier();
    tid = thread(); lane = tid & 63; fr = lane & 15; fg = lane >> 4;
    if (wave == 0) {
        // the block below the diagonal: -X22 N21 X11; then A T, T = X diag(beta), in A's place
        const f32x4 n21 = *(const f32x4*)(Ms + (16 + fr) * LA + 4 * fg) * be[16 + fr], x22 = *(const f32x4*)(Ms + (16 + fr) * LA + 16 + 4 * fg);
        f32x4 x11, y = f32x4{0.f, 0.f, 0.f, 0.f}, w = y, aa[3], at[3];
#pragma unroll
        for (int x = 0; x < 3; x++) {
            aa[x] = *(const f32x4*)(As + (16 * (x > 0) + fr) * LA + 16 * (x > 1) + 4 * fg);
            at[x] = w;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) { x11[r] = Ms[(4 * fg + r) * LA + fr]; y = mfma_f32(n21[r], x11[r], y); }
#pragma unroll
        for (int r = 0; r < 4; r++) w = mfma_f32(x22[r], y[r], w);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float t00 = x11[r] * be[fr], t10 = -w[r] * be[fr], t11 = Ms[(16 + 4 * fg + r) * LA + 16 + fr] * be[16 + fr];
            at[0] = mfma_f32(aa[0][r], t00, at[0]); at[1] = mfma_f32(aa[1][r], t00, at[1]);
            at[1] = mfma_f32(aa[2][r], t10, at[1]); at[2] = mfma_f32(aa[2][r], t11, at[2]);
            Ms[(16 + 4 * fg + r) * LA + fr] = -w[r];
        }
#pragma unroll
        for (int x = 0; x < 3; x++)
#pragma unroll
            for (int r = 0; r < 4; r++) As[(16 * (x > 0) + 4 * fg + r) * LA + 16 * (x > 1) + fr] = at[x][r];
    } else {
#pragma unroll 2
        for (int i = tid - 64; i < C * DKP / 4; i += NT - 64) {  // q e^b, k e^b in place
            const int t = i / (DKP / 4), d = i % (DKP / 4) * 4;
            const f32x4 b = *(const f32x4*)(bs + t * LQ + d);
            f32x4 q = *(const f32x4*)(qs + t * LQ + d), k = *(const f32x4*)(ks + t * LQ + d);
#pragma unroll
            for (int r = 0; r < 4; r++) { const float e = ex2(b[r]); q[r] *= e; k[r] *= e; }
            *(f32x4*)(qs + t * LQ + d) = q;
            *(f32x4*)(ks + t * LQ + d) = k;
        }
    }
    barrier();
    tid = thread(); lane = tid & 63; fr = lane & 15; fg = lane >> 4;
    // rows of T and of A T, blocks (0,0), (1,0), (1,1): B operands of the transposed products, whose accumulators hold four channels of a token
    f32x4 ta[3], ba[3];
#pragma unroll
    for (int x = 0; x < 3; x++) {
        const int at = (16 * (x > 0) + fr) * LA + 16 * (x > 1) + 4 * fg;
        ta[x] = *(const f32x4*)(Ms + at) * *(const f32x4*)(be + 16 * (x > 1) + 4 * fg);
        ba[x] = *(const f32x4*)(As + at);
    }
    auto times = [&](const f32x4 (&x)[2], const f32x4 (&m)[3], f32x4 (&d)[2]) {          // d += (m x)^T
#pragma unroll
        for (int r = 0; r < 4; r++) { d[0] = mfma_f32(x[0][r], m[0][r], d[0]); d[1] = mfma_f32(x[0][r], m[1][r], d[1]); }
#pragma unroll
        for (int r = 0; r < 4; r++) d[1] = mfma_f32(x[1][r], m[2][r], d[1]);
    };
#pragma unroll
    for (int i0 = 0; i0 < NK; i0 += NW) {                        // 16 key channels: -W and Q'
        const int i = i0 + wave;
        if (NK % NW && i >= NK) break;
        f32x4 k[2], w[2], q[2];
#pragma unroll
        for (int sb = 0; sb < 2; sb++) {
#pragma unroll
            for (int r = 0; r < 4; r++) k[sb][r] = -ks[(16 * sb + 4 * fg + r) * LQ + 16 * i + fr];
            w[sb] = f32x4{0.f, 0.f, 0.f, 0.f};
            q[sb] = *(const f32x4*)(qs + (16 * sb + fr) * LQ + 16 * i + 4 * fg);
        }
        times(k, ta, w);
        times(k, ba, q);
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            buffer_put4(ws, 16 * lane, 16 * delta_piece(i, tt), w[tt]);
            buffer_put4(ws, 16 * lane, 16 * delta_piece(i, 2 + tt), q[tt]);
        }
    }
    auto values = [&](int i, const f32x4 (&v)[2]) __attribute__((always_inline)) {       // 16 value channels: U0 and O0
        f32x4 u[2], o[2];
        u[0] = u[1] = o[0] = o[1] = f32x4{0.f, 0.f, 0.f, 0.f};
        times(v, ta, u);
        times(v, ba, o);
        const auto ru = delta_rows(vr, tb, nv), ro = delta_rows(orow, tb, nv);
        const int c = 16 * i + 4 * fg;
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            const uint32_t at_u = (16 * tt + fr) * vr.pitch + 4 * c, at_o = (16 * tt + fr) * orow.pitch + 4 * c;
            if (VECV) { buffer_put4(ru, c < p.DV ? at_u : DELTA_OUTSIDE, 0, u[tt]); buffer_put4(ro, c < p.DV ? at_o : DELTA_OUTSIDE, 0, o[tt]); }
            else
#pragma unroll
                for (int r = 0; r < 4; r++) { buffer_put(ru, c + r < p.DV ? at_u + 4 * r : DELTA_OUTSIDE, u[tt][r]); buffer_put(ro, c + r < p.DV ? at_o + 4 * r : DELTA_OUTSIDE, o[tt][r]); }
        }
    };
    values(wave, v4);                                            // (beyond DV: nothing is stored)
    for (int i = wave + NW; i < nvb; i += NW) {
        f32x4 v[2];
        ldv(tb, nv, i, v);
        values(i, v);
    }
    if (!more) return;
    ldv(next.tok0, next.rows, wave, v4);
    barrier();                                                   // the last readers of this chunk are done
    now = next;
    }
}

// ------------------------------------------------------------------------------------------
// scan: grid (heads, slices of value columns, sequences).  A wave keeps 16 columns of the state in accumulators: of all key channels (delta_scan_kernel), or of a part
// of them (delta_scan_parts_kernel).
// ------------------------------------------------------------------------------------------
// Which sequence a workgroup takes: the shortest first, then the longest to the second shortest.  The chain of the longest one is what a launch lasts; started early it has
// its CU to itself until workgroups have to share, and shares with the start of the shortest.  us a layer, order of the call -> here: 5 sequences of 300 .. 1900 tokens 125 -> 114,
// 12 of them 274 -> 234, 24 of 100 .. 900 220 -> 194; equal lengths keep their order.
// (Beyond 64 sequences, more than the lanes that rank them, the order of the call: there are chains enough to even out)
__device__ __forceinline__ int delta_scan_seq(const int* seq_len, int i, int n_seqs) {
    if (n_seqs == 1 || n_seqs > DELTA_ORDERED) return i;
    const int lane = threadIdx.x & 63, mine = lane < n_seqs ? seq_len[lane] : -1;
    int rank = 0;
    for (int j = 0; j < n_seqs; j++) {
        const int other = __builtin_amdgcn_readlane(mine, j);
        rank += other > mine || (other == mine && j < lane) ? 1 : 0;
    }
    return __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(rank == (i == 0 ? n_seqs - 1 : i - 1) && lane < n_seqs)));
}
template <int N>      // key channels ch0 .. ch0 + 16 N - 1 of a lane's column
__device__ __forceinline__ void delta_state_in(const DeltaArgs& p, const float* st, int ch0, int fg, int col, bool fresh, f32x4 (&S)[N]) {
    const int sc = min(col, p.DVp - 1);              // (clamped addresses instead of branches)
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = ch0 + 16 * i + 4 * fg + r;
            const float x = st[min(row, p.DK - 1) * p.DVp + sc];
            S[i][r] = !fresh && col < p.DVp && row < p.DK ? x : 0.f;
        }
}
template <int N>
__device__ __forceinline__ void delta_state_out(const DeltaArgs& p, float* st, int ch0, int fg, int col, const f32x4 (&S)[N]) {
    int so = 4 * fg * p.DVp + col;
    asm volatile("" : "+v"(so));                     // (or addresses are kept in registers all along)
    st += ch0 * p.DVp;
#pragma unroll
    for (int i = 0; i < N; i++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (col < p.DVp && ch0 + 16 * i + 4 * fg + r < p.DK) (st + (16 * i + r) * p.DVp)[so] = S[i][r];
}

// All key channels of 16 columns a wave: a chunk's operands are in LDS for the workgroup's 64 columns, as they lie in scratch (three workgroups a CU; with padded rows
// two: 16 x 900 tokens 250 -> 242 us a layer, 32 x 512 322 -> 272).  192 products of 32 cycles a chunk bound a wave.
template <int NK> constexpr int delta_scan_lds_bytes() { return 4 * NK * 16 * (3 * DELTA_C + 1); }

template <int NK>
__global__ __launch_bounds__(DELTA_SCAN_WAVES * 64, NK > 8 ? 1 : 3) void delta_scan_kernel(DeltaArgs p) {
    constexpr int NW = DELTA_SCAN_WAVES, C = DELTA_C, DKP = NK * 16, NT = NW * 64;
    const int h = blockIdx.x, seq = delta_scan_seq(p.seq_len, (int)blockIdx.z, (int)gridDim.z);
    const int n = p.seq_len[seq];
    if (n < p.len_lo || n > p.len_hi) return;
    extern __shared__ __attribute__((aligned(16))) float dl_sm[];
    f32x4* ol = (f32x4*)dl_sm;           // the chunk as it lies in scratch
    float* dl = dl_sm + 3 * C * DKP;     // [DKP]     e^{b_end}
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int fr = lane & 15, fg = lane >> 4;
    const int col = (blockIdx.y * NW + wave) * 16 + fr;
    float* st = p.state + (int64_t)p.seq_slot[seq] * p.slot_stride + (int64_t)h * p.DK * p.DVp;
    f32x4 S[NK];
    delta_state_in(p, st, 0, fg, col, p.seq_pos[seq] == 0, S);
    constexpr int E = 3 * C * DKP / 4, NL = E / NT;              // 16-byte pieces of a chunk's operands, per thread
    static_assert(E % NT == 0 && NT >= DKP, "whole pieces, one decay per thread");
    const int64_t stride = p.H * delta_ws_floats(DKP);
    const float* src = p.ws + (delta_chunk(p, seq, 0) * p.H + h) * delta_ws_floats(DKP);
    f32x4 rg[NL], u[2], o[2];
    float rd = 0.f;
    const int64_t tok0 = p.seq_tok_start[seq];
    const DeltaRows vr{(char*)(p.v + tok0 * p.ld + (int64_t)h * p.DV), 4 * (uint32_t)p.ld}, orow{(char*)(p.o + tok0 * p.o_ld + (int64_t)h * p.DV), 4 * (uint32_t)p.o_ld};
    const uint32_t cb = col < p.DV ? 4 * col : DELTA_OUTSIDE;
    constexpr int Q = NK / 2;                                    // a chunk's loads go out in as many portions, between the products of two state tiles each
    auto fetch = [&](int c0, int part) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NL; i++) if (i * Q / NL == part) rg[i] = ((const f32x4*)src + i * NT)[tid];
        if (part == 0) {
            const auto rv = delta_rows(vr, c0, n - c0);
            rd = src[3 * C * DKP + min(tid, DKP - 1)];
#pragma unroll
            for (int tt = 0; tt < 2; tt++) u[tt] = delta_rows_get(rv, (16 * tt + 4 * fg) * vr.pitch + cb, vr.pitch);
        }
        if (part == Q - 1) {
            const auto ro = delta_rows(orow, c0, n - c0);
#pragma unroll
            for (int tt = 0; tt < 2; tt++) o[tt] = delta_rows_get(ro, (16 * tt + 4 * fg) * orow.pitch + cb, orow.pitch);
        }
    };
#pragma unroll
    for (int i = 0; i < Q; i++) fetch(0, i);
    for (int c0 = 0; c0 < n; c0 += C) {
        __syncthreads();                                         // the previous chunk's readers are done
#pragma unroll
        for (int i = 0; i < NL; i++) ol[i * NT + tid] = rg[i];
        if (tid < DKP) dl[tid] = rd;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NK; i++) {
            f32x4 a[4];
#pragma unroll
            for (int x = 0; x < 4; x++) a[x] = ol[delta_piece(i, x) + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                u[0] = mfma_f32(a[0][r], S[i][r], u[0]); u[1] = mfma_f32(a[1][r], S[i][r], u[1]);
                o[0] = mfma_f32(a[2][r], S[i][r], o[0]); o[1] = mfma_f32(a[3][r], S[i][r], o[1]);
            }
            if (i & 1) __builtin_amdgcn_sched_barrier(0);        // (or all reads are hoisted to the front, and registers spill)
        }
        const auto ro = delta_rows(orow, c0, n - c0);
#pragma unroll
        for (int tt = 0; tt < 2; tt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                buffer_put(ro, (16 * tt + 4 * fg + r) * orow.pitch + cb, o[tt][r]);
            }
        f32x4 ub[2] = {u[0], u[1]};
        __builtin_amdgcn_sched_barrier(0);
        const bool more = c0 + C < n;                            // (the last chunk is fetched once more instead of a branch)
        src += more ? stride : 0;
#pragma unroll
        for (int i = 0; i < NK; i += 2) {
            f32x4 a[2][2];
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int sb = 0; sb < 2; sb++) a[x][sb] = ol[delta_piece(i + x, 4 + sb) + lane];
            S[i] *= *(const f32x4*)(dl + 16 * i + 4 * fg);
            S[i + 1] *= *(const f32x4*)(dl + 16 * (i + 1) + 4 * fg);
            fetch(more ? c0 + C : c0, i / 2);
#pragma unroll
            for (int sb = 0; sb < 2; sb++)
#pragma unroll
                for (int r = 0; r < 4; r++) { S[i] = mfma_f32(a[0][sb][r], ub[sb][r], S[i]); S[i + 1] = mfma_f32(a[1][sb][r], ub[sb][r], S[i + 1]); }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    delta_state_out(p, st, 0, fg, col, S);
}

// Key channels over the KSP waves of a workgroup that has 16 columns: a chunk's operands belong to one wave each and go from scratch to its registers, a chunk ahead and
// between the products (in front of them the workgroup's 52 KB kept its waves from their first product for 360 .. 1070 cycles).  The waves' sums of U and O meet in LDS:
// U's on their way while O is multiplied, O's a chunk later.  Bound by the chain of a sequence: a chunk of a head of 128 is 48 products of 32 cycles in 2600 .. 2800 (1.1 us),
// the rest the exchange (150 to write and meet, 140 to add) and what is issued beside the products.  With operands through LDS and their loads behind the products of U
// and O it was 2.6 us: 1 x 1900 tokens 157 -> 72 us a layer, 5 x 300 .. 1900 195 -> 115.
template <int NK, int KSP>
__global__ __launch_bounds__(KSP * 64, 2) void delta_scan_parts_kernel(DeltaArgs p) {
    constexpr int C = DELTA_C, DKP = NK * 16, N = NK / KSP;
    const int h = blockIdx.x, seq = delta_scan_seq(p.seq_len, (int)blockIdx.z, (int)gridDim.z);
    const int n = p.seq_len[seq];
    if (n < p.len_lo || n > p.len_hi) return;
    __shared__ f32x4 xb[2][KSP][4][64];      // [chunk & 1][part][U, U, O, O]
    const int lane = threadIdx.x & 63, kq = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, fg = lane >> 4, col = blockIdx.y * 16 + fr, ch0 = kq * N * 16;
    float* st = p.state + (int64_t)p.seq_slot[seq] * p.slot_stride + (int64_t)h * p.DK * p.DVp;
    f32x4 S[N];
    delta_state_in(p, st, ch0, fg, col, p.seq_pos[seq] == 0, S);
    const int64_t stride = p.H * delta_ws_floats(DKP), tok0 = p.seq_tok_start[seq];
    const float* src = p.ws + (delta_chunk(p, seq, 0) * p.H + h) * delta_ws_floats(DKP);
    const DeltaRows vr{(char*)(p.v + tok0 * p.ld + (int64_t)h * p.DV), 4 * (uint32_t)p.ld}, orow{(char*)(p.o + tok0 * p.o_ld + (int64_t)h * p.DV), 4 * (uint32_t)p.o_ld};
    const uint32_t cb = col < p.DV ? 4 * col : DELTA_OUTSIDE;
    // what U and O start from is dealt over the parts: U's two pieces to the first two, O's to the next two or the same
    constexpr int NI = KSP >= 4 ? 1 : 2;
    const int stt = kq & 1;
    const DeltaRows first = NI == 2 || kq < 2 ? vr : orow;
    const uint32_t at_v = (16 * stt + 4 * fg) * first.pitch + cb, at_o = (16 * stt + 4 * fg) * orow.pitch + cb;
    // ... and what becomes of O: two parts store 16 tokens each, or four 8
    constexpr int NS = KSP == 2 ? 4 : 2;
    const int ott = KSP == 2 ? kq : (kq >> 1) & 1, or0 = KSP == 2 ? 0 : 2 * (kq & 1);
    const uint32_t at_s = KSP <= 4 || kq < 4 ? (16 * ott + 4 * fg + or0) * orow.pitch + cb : DELTA_OUTSIDE;
    struct Chunk { f32x4 op[N][6], d[N], start[NI]; };
    auto fetch_start = [&](Chunk& k, int c0) __attribute__((always_inline)) {
        k.start[0] = delta_rows_get(delta_rows(first, c0, n - c0), at_v, first.pitch);
        if constexpr (NI == 2) k.start[1] = delta_rows_get(delta_rows(orow, c0, n - c0), at_o, orow.pitch);
    };
    auto fetch_op = [&](Chunk& k, int j) __attribute__((always_inline)) {      // load j of 7 N
        const auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, 4 * (int)delta_ws_floats(DKP), 0x00020000);
        const int x = j / N, i = j % N;
        if (x < 6) k.op[i][x] = buffer_f32x4(rs, lane * 16, 16 * delta_piece(kq * N + i, x));
        else if (x == 6) k.d[i] = buffer_f32x4(rs, fg * 16, 4 * (3 * C * DKP + ch0 + 16 * i));
    };
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    auto barrier = [&]() __attribute__((always_inline)) {      // (without the wait for loads on their way)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    float oq[KSP][NS];
    auto read_o = [&](int turn) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < KSP; q++)
#pragma unroll
            for (int r = 0; r < NS; r++) oq[q][r] = ((const float*)&xb[turn][q][2 + ott][lane])[or0 + r];
    };
    auto store_o = [&](int c0) __attribute__((always_inline)) {      // (c0 < 0: none)
        const auto ro = delta_rows(orow, c0, c0 < 0 ? 0 : n - c0);
#pragma unroll
        for (int r = 0; r < NS; r++) {
            float y = oq[0][r];
#pragma unroll
            for (int q = 1; q < KSP; q++) y += oq[q][r];
            buffer_put(ro, at_s + r * orow.pitch, y);
        }
    };
    auto step = [&](Chunk& k, Chunk& next, int c0, int turn) __attribute__((always_inline)) {
        const bool more = c0 + C < n;
        src += more ? stride : 0;                                // (the last chunk is fetched once more instead of a branch)
        f32x4 u[2], o[2], uq[KSP][2];
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            u[tt] = (NI == 2 || kq < 2) && stt == tt ? k.start[0] : zero;
            o[tt] = NI == 2 ? (stt == tt ? k.start[NI - 1] : zero) : (kq == 2 + tt ? k.start[0] : zero);
        }
#pragma unroll
        for (int i = 0; i < N; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                u[0] = mfma_f32(k.op[i][0][r], S[i][r], u[0]); u[1] = mfma_f32(k.op[i][1][r], S[i][r], u[1]);
                if (i == 0 && r == 1) fetch_start(next, more ? c0 + C : c0);
                if (r % 2 == 0) fetch_op(next, 2 * i + r / 2);
                __builtin_amdgcn_sched_barrier(0);
            }
        xb[turn][kq][0][lane] = u[0]; xb[turn][kq][1][lane] = u[1];
        barrier();                                               // (one a chunk: who writes this half of xb again has passed the next)
#pragma unroll
        for (int q = 0; q < KSP; q++) { uq[q][0] = xb[turn][q][0][lane]; uq[q][1] = xb[turn][q][1][lane]; }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < N; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                o[0] = mfma_f32(k.op[i][2][r], S[i][r], o[0]); o[1] = mfma_f32(k.op[i][3][r], S[i][r], o[1]);
                if (r % 2 == 0) fetch_op(next, 2 * N + 2 * i + r / 2);
                if (i == N - 1 && r == 1) read_o(turn ^ 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        u[0] = uq[0][0]; u[1] = uq[0][1];
#pragma unroll
        for (int q = 1; q < KSP; q++) { u[0] += uq[q][0]; u[1] += uq[q][1]; }
#pragma unroll
        for (int i = 0; i < N; i++) S[i] *= k.d[i];
#pragma unroll
        for (int sb = 0; sb < 2; sb++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
#pragma unroll
                for (int i = 0; i < N; i++) S[i] = mfma_f32(k.op[i][4 + sb][r], u[sb][r], S[i]);
#pragma unroll
                for (int j = 0; j < 3 * N; j++) if (j * 8 / (3 * N) == 4 * sb + r) fetch_op(next, 4 * N + j);
                if (sb == 0 && r == 1) { xb[turn][kq][2][lane] = o[0]; xb[turn][kq][3][lane] = o[1]; }
                if (sb == 0 && r == 3) store_o(c0 - C);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    Chunk a, b;
    fetch_start(a, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 7 * N; j++) fetch_op(a, j);
    int c0 = 0;
    for (;;) {
        step(a, b, c0, 0);
        if (c0 + C >= n) { barrier(); read_o(0); break; }
        c0 += C;
        step(b, a, c0, 1);
        if (c0 + C >= n) { barrier(); read_o(1); break; }
        c0 += C;
    }
    store_o(c0);
    delta_state_out(p, st, ch0, fg, col, S);
}

// ------------------------------------------------------------------------------------------
// token by token.  grid (H, sequences), 512 threads: tv threads side by side on a state row (4 columns each), 512 / tv rows at a time.
// With S' = diag(a) S both S'^T k and S'^T q come from one pass over the state: o = S'^T q + (k . q) u.
// ------------------------------------------------------------------------------------------
static inline int delta_step_lds_bytes(int DK, int DVp, int ranks) {
    int tv = 1;
    while (tv < DVp / 4) tv <<= 1;
    const int nred = tv >= 64 ? LR_STEP_THREADS / tv : LR_STEP_THREADS / 64;
    return 4 * (3 * ((DK + 3) & ~3) + 2 * DVp + 2 * nred * DVp + ranks);
}
template <typename WT> __device__ __forceinline__ float delta_dot16(const WT* w, const float* x);       // 16 bytes of weights
template <> __device__ __forceinline__ float delta_dot16<float>(const float* w, const float* x) {
    const f32x4 a = *(const f32x4*)w, b = *(const f32x4*)x;
    return fmaf(a[3], b[3], fmaf(a[2], b[2], fmaf(a[1], b[1], a[0] * b[0])));
}
template <> __device__ __forceinline__ float delta_dot16<bf16_t>(const bf16_t* w, const float* x) {
    const bf16x8 a = *(const bf16x8*)w;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) s = fmaf((float)a[i], x[i], s);
    return s;
}

template <bool FUSED, int ROWS, typename ActT>           // ROWS: state rows a thread keeps in registers; ActT: type of `out` and of a2 / g2
__global__ __launch_bounds__(LR_STEP_THREADS, ROWS <= 8 ? 4 : 2) void delta_step_kernel(DeltaArgs p) {
    constexpr int NT = LR_STEP_THREADS, NW = NT / 64;
    const int h = blockIdx.x, seq = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = FUSED ? 1 : p.seq_len[seq];
    if (n < p.len_lo || n > p.len_hi) return;
    extern __shared__ __attribute__((aligned(16))) float dl_sm[];
    const int DK4 = (p.DK + 3) & ~3;
    float* sq = dl_sm;                   // [DK]
    float* sk = sq + DK4;                // [DK]
    float* sa = sk + DK4;                // [DK]   decays
    float* sv = sa + DK4;                // [DVp]
    float* sg = sv + p.DVp;              // [DVp]  output gates (FUSED)
    const int nv4 = p.DVp >> 2;
    int tv = 1;
    while (tv < nv4) tv <<= 1;           // host: nv4 <= NT
    const int rg = tid / tv, tc = tid - rg * tv, RG = NT / tv, NRED = tv >= 64 ? RG : NW;
    float* red = sg + p.DVp;             // [NRED][2][DVp]
    float* lr = red + 2 * NRED * p.DVp;  // [a_rkp + g_rkp] (FUSED)
    __shared__ float s_red[NW], s_sum[3];
    const bool live = tc < nv4;
    const int t0 = p.seq_tok_start[seq], pos0 = p.seq_pos[seq], slot = p.seq_slot[seq];
    const int g = h / (p.H / p.G);
    float* st = p.state + (int64_t)slot * p.slot_stride + (int64_t)h * p.DK * p.DVp;
    int so = rg * p.DVp + 4 * tc;        // this thread's place in a pass of RG rows
    const int pass = RG * p.DVp;
    f32x4 s[ROWS];                       // the first ROWS rows of this thread, fetched before anything else is known
#pragma unroll
    for (int i = 0; i < ROWS; i++) {
        const bool ok = live && rg + i * RG < p.DK;
        const f32x4 x = *(const f32x4*)(st + (ok ? i * pass + so : 0));
#pragma unroll
        for (int r = 0; r < 4; r++) s[i][r] = ok && pos0 > 0 ? x[r] : 0.f;
    }
    asm volatile("" : "+v"(so));         // (or the addresses of these loads are kept in registers for the stores)
    for (int i = tid; i < p.DVp; i += NT) { sv[i] = 0.f; sg[i] = 0.f; }
    __syncthreads();
    const float ea = expf(p.a_log[h]);
    for (int it = 0; it < n; it++) {
        const int64_t t = t0 + it;
        if constexpr (FUSED) {
            // causal convolution + silu of this head's channels (n == 1)
            const float* rw = p.raw + t * p.raw_ld;
            float* ring = p.ring + (int64_t)slot * p.ring_slot_stride;
            const int KD = p.G * p.DK;
#pragma unroll 1
            for (int i = tid; i < 2 * p.DK + p.DV; i += NT) {
                const int c = i < p.DK ? g * p.DK + i : (i < 2 * p.DK ? KD + g * p.DK + i - p.DK : 2 * KD + h * p.DV + i - 2 * p.DK);
                const float cur = rw[c];
                float acc = 0.f;
                for (int b = p.taps - 1; b >= 1; b--)
                    if (pos0 - b >= 0) acc = fmaf(ring[(int64_t)((pos0 - b) % p.taps) * p.channels + c], p.conv_w[(int64_t)c * p.taps + p.taps - 1 - b], acc);
                acc = fmaf(cur, p.conv_w[(int64_t)c * p.taps + p.taps - 1], acc);
                ring[(int64_t)(pos0 % p.taps) * p.channels + c] = cur;      // (heads of a group write the same values; nobody reads this row now)
                const float y = lr_silu(acc);
                if (i < p.DK) sq[i] = y;
                else if (i < 2 * p.DK) sk[i - p.DK] = y;
                else sv[i - 2 * p.DK] = y;
            }
            for (int i = tid; i < p.a_rkp + p.g_rkp; i += NT) {
                const int j = i - p.a_rkp;
                lr[i] = j < 0 ? (i < p.a_rank ? p.a1[t * p.lr_ld + i] : 0.f) : (j < p.g_rank ? p.g1[t * p.lr_ld + j] : 0.f);
            }
            __syncthreads();
            // decay and gate projections: four lanes per output
            constexpr int CH = 16 / (int)sizeof(ActT);
#pragma unroll 1
            for (int i = tid >> 2; i < p.DK + p.DV; i += NT / 4) {
                const bool dec = i < p.DK;
                const int rkp = dec ? p.a_rkp : p.g_rkp;
                const ActT* w = dec ? (const ActT*)p.a2 + (int64_t)(h * p.DK + i) * rkp : (const ActT*)p.g2 + (int64_t)(h * p.DV + i - p.DK) * rkp;
                const float* x = dec ? lr : lr + p.a_rkp;
                float a = 0.f;
                for (int e = (tid & 3) * CH; e < rkp; e += 4 * CH) a += delta_dot16<ActT>(w + e, x + e);
                a += __shfl_xor(a, 1, 64);
                a += __shfl_xor(a, 2, 64);
                if ((tid & 3) == 0) {
                    if (dec) sa[i] = expf(-ea * delta_softplus(a + p.dt_bias[h * p.DK + i]));
                    else sg[i - p.DK] = lr_sigmoid(a);
                }
            }
        } else {
            for (int i = tid; i < p.DK; i += NT) {
                sq[i] = p.q[t * p.ld + (int64_t)g * p.DK + i];
                sk[i] = p.k[t * p.ld + (int64_t)g * p.DK + i];
                sa[i] = expf(-ea * delta_softplus(p.z[t * p.z_ld + (int64_t)h * p.DK + i] + p.dt_bias[h * p.DK + i]));
            }
            for (int i = tid; i < p.DV; i += NT) sv[i] = p.v[t * p.ld + (int64_t)h * p.DV + i];
        }
        __syncthreads();
        if (wave < 3) {                  // q . q, k . k, k . q
            const float *x = wave == 1 ? sk : sq, *y = wave == 0 ? sq : sk;
            float a = 0.f;
            for (int i = lane; i < p.DK; i += 64) a = fmaf(x[i], y[i], a);
            a = wave_sum(a);
            if (lane == 0) s_sum[wave] = a;
        }
        __syncthreads();
        const float iq = p.q_scale / sqrtf(s_sum[0] + DELTA_UNIT_EPS), ik = 1.0f / sqrtf(s_sum[1] + DELTA_UNIT_EPS), kq = s_sum[2] * iq * ik;
        const float beta = lr_sigmoid(p.beta[t * p.beta_ld + h]);
        f32x4 ra = f32x4{0.f, 0.f, 0.f, 0.f}, pa = ra;      // S'^T k, S'^T q
#pragma unroll
        for (int i = 0; i < ROWS; i++) {
            const int row = rg + i * RG;
            const bool ok = live && row < p.DK;
            const int rr = ok ? row : 0;
            const float al = sa[rr], kk = ok ? sk[rr] : 0.f, qq = ok ? sq[rr] : 0.f;
#pragma unroll
            for (int r = 0; r < 4; r++) { s[i][r] *= al; ra[r] = fmaf(kk, s[i][r], ra[r]); pa[r] = fmaf(qq, s[i][r], pa[r]); }
        }
#pragma unroll 1
        for (int row = rg + ROWS * RG; live && row < p.DK; row += RG) {     // (a state larger than the registers: streamed)
            f32x4 w = f32x4{0.f, 0.f, 0.f, 0.f};
            if (pos0 + it > 0) w = *(const f32x4*)(st + (int64_t)row * p.DVp + 4 * tc);
            w *= sa[row];
            ra += sk[row] * w; pa += sq[row] * w;
        }
        for (int o = tv; o < 64; o <<= 1)
#pragma unroll
            for (int r = 0; r < 4; r++) { ra[r] += __shfl_xor(ra[r], o, 64); pa[r] += __shfl_xor(pa[r], o, 64); }
        if (live && (tv >= 64 || lane < tv)) {
            float* d = red + (int64_t)(tv >= 64 ? rg : wave) * 2 * p.DVp + 4 * tc;
            *(f32x4*)d = ra;
            *(f32x4*)(d + p.DVp) = pa;
        }
        __syncthreads();
        f32x4 u = f32x4{0.f, 0.f, 0.f, 0.f}, ov = u;
        if (live) {
            ra = u; pa = u;
#pragma unroll 4
            for (int r = 0; r < NRED; r++) { ra += *(const f32x4*)(red + (int64_t)r * 2 * p.DVp + 4 * tc); pa += *(const f32x4*)(red + (int64_t)r * 2 * p.DVp + p.DVp + 4 * tc); }
            u = beta * (*(const f32x4*)(sv + 4 * tc) - ra * ik);
            ov = pa * iq + kq * u;
        }
#pragma unroll
        for (int i = 0; i < ROWS; i++) {
            const int row = rg + i * RG;
            const bool ok = live && row < p.DK;
            const float kk = ok ? sk[ok ? row : 0] * ik : 0.f;
#pragma unroll
            for (int r = 0; r < 4; r++) s[i][r] = fmaf(kk, u[r], s[i][r]);
            if (ok && it == n - 1) *(f32x4*)(st + i * pass + so) = s[i];
        }
#pragma unroll 1
        for (int row = rg + ROWS * RG; live && row < p.DK; row += RG) {
            float* sr = st + (int64_t)row * p.DVp + 4 * tc;
            f32x4 w = f32x4{0.f, 0.f, 0.f, 0.f};
            if (pos0 + it > 0) w = *(const f32x4*)sr;
            *(f32x4*)sr = w * sa[row] + sk[row] * ik * u;
        }
        if constexpr (FUSED) {
            // (columns beyond DV: v, S and hence o are zero)
            float ss = rg == 0 ? (ov[0] * ov[0] + ov[1] * ov[1]) + (ov[2] * ov[2] + ov[3] * ov[3]) : 0.f;
            ss = wave_sum(ss);
            if (lane == 0) s_red[wave] = ss;
            __syncthreads();
            float tot = 0.f;
#pragma unroll
            for (int i = 0; i < NW; i++) tot += s_red[i];
            const float inv = 1.0f / sqrtf(tot / (float)p.DV + p.eps);
            if (live && rg == 0)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (4 * tc + r < p.DV)
                        ActIO<ActT>::st((ActT*)p.out + act_index<ActT>(t, (int64_t)h * p.DV + 4 * tc + r, p.out_ld), ov[r] * inv * p.norm_w[4 * tc + r] * sg[4 * tc + r]);
        } else if (live && rg == 0) {
#pragma unroll
            for (int r = 0; r < 4; r++) if (4 * tc + r < p.DV) p.o[t * p.o_ld + (int64_t)h * p.DV + 4 * tc + r] = ov[r];
        }
        __syncthreads();
    }
}

// ---- columns [0, n) and [off2, off2 + n2) of fp32 rows as the operands of two projections (padded with zeros): grid (tokens) ----
struct PackArgs { const float* src; int64_t ld; int n1, np1, n2, np2, off2; void *d1, *d2; };
template <typename ActT>
__global__ __launch_bounds__(64) void pack_rows_kernel(PackArgs p) {
    const int64_t t = blockIdx.x;
    const float* x = p.src + t * p.ld;
    for (int i = threadIdx.x * 4; i < p.np1 + p.np2; i += 256) {
        const bool a = i < p.np1;
        const int c = a ? i : i - p.np1, n = a ? p.n1 : p.n2;
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = c + r < n ? x[(a ? 0 : p.off2) + c + r] : 0.f;
        act_store4<ActT>((ActT*)(a ? p.d1 : p.d2), t, c, a ? p.np1 : p.np2, v);
    }
}

// launches (delta_inst.hip); nk: template argument of the chunk kernels
void delta_step_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, bool fused, bool f32);
void delta_prep_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, int nk, int tokens);
void delta_scan_launch(hipStream_t st, const DeltaArgs& p, int n_seqs, int nk, int max_len, int tokens);

}  // namespace nvl
