// readback.h — logits on their way to the caller's memory (host code, included by nvllm.hip).
#pragma once

#include <system_error>
#include <thread>

namespace {

// A caller's buffer is ordinary memory, mostly fresh from the allocator: the runtime copies into it with one thread, through a staging buffer
// of its own and a page fault at a time.  Here the card writes pinned memory of the model's own in pieces and threads carry the pieces
// over while the next ones arrive.  What bounds it is the first touch of the caller's pages, which several threads share; the
// pieces cross the bus at 55 GB/s.  96 rows of 128256 logits (49 MB) 4.9 -> 1.6 ms, 32 rows 1.0 -> 0.5 ms, 16 rows of 49155 0.25 -> 0.13 ms.
constexpr int64_t RB_PIECE = 1 << 20;
constexpr int RB_SLOTS = 8;              // pieces in flight; a multiple of every number of threads below
static inline int rb_threads(int64_t pieces) { return pieces >= 32 ? 8 : pieces >= 8 ? 4 : pieces >= 3 ? 2 : 1; }

// (a kernel and not a copy engine: the engine's first use costs the process 6 ms, and a hand-over to it 10 us each)
__global__ __launch_bounds__(256) void to_host_kernel(const u32x4* __restrict__ src, u32x4* __restrict__ dst, int n) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) dst[i] = __builtin_nontemporal_load(src + i);
}

void init_readback(nvl_model* m) {
    const int64_t bytes = std::max<int64_t>(m->logit_rows, 1) * m->Vpad * 4;
    m->rb_slots = (int)std::min<int64_t>(RB_SLOTS, (bytes + RB_PIECE - 1) / RB_PIECE);
    m->rb_bytes = std::min<int64_t>(bytes, RB_SLOTS * RB_PIECE);
    NVL_HIP(hipHostMalloc((void**)&m->rb_host, (size_t)m->rb_bytes, hipHostMallocDefault));
    memset(m->rb_host, 0, (size_t)m->rb_bytes);          // (its pages fault in on the host's first touch, a microsecond each)
    m->rb_ev.resize((size_t)m->rb_slots);
    for (auto& e : m->rb_ev) NVL_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
}
void free_readback(nvl_model* m) {
    for (auto e : m->rb_ev) if (e) (void)hipEventDestroy(e);
    m->rb_ev.clear();
    if (m->rb_host) (void)hipHostFree(m->rb_host);
    m->rb_host = nullptr;
}

// memory that the runtime knows (pinned, device, managed) takes the plain copy
bool rb_ordinary_memory(const void* p) {
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, p) != hipSuccess) { (void)hipGetLastError(); return true; }
    return at.type == hipMemoryTypeUnregistered;
}

// the logits of `rows` rows, behind all that the stream holds; returns when they are in `out`
void read_logits(nvl_model* m, float* out, int rows) {
    if (!rb_ordinary_memory(out)) {
        NVL_HIP(hipMemcpy2DAsync(out, (size_t)m->V * 4, m->logits, (size_t)m->Vpad * 4, (size_t)m->V * 4, (size_t)rows, hipMemcpyDeviceToHost, m->stream));
        return;
    }
    const int64_t pitch = (int64_t)m->Vpad * 4, width = (int64_t)m->V * 4, total = (rows - 1) * pitch + width;
    const int64_t piece = std::min(RB_PIECE, m->rb_bytes), pieces = (total + piece - 1) / piece;
    const int64_t slots = std::max<int64_t>(1, m->rb_bytes / piece);
    auto issue = [&](int64_t c) {
        const int n = (int)((std::min(piece, total - c * piece) + 15) / 16);          // (a row's padding covers the last one)
        hipLaunchKernelGGL(to_host_kernel, dim3(std::min(cdiv(n, 256), 128)), dim3(256), 0, m->stream, (const u32x4*)((const char*)m->logits + c * piece), (u32x4*)(m->rb_host + c % slots * piece), n);
        NVL_HIP(hipGetLastError());
        NVL_HIP(hipEventRecord(m->rb_ev[(size_t)(c % slots)], m->stream));
    };
    for (int64_t c = 0; c < std::min(slots, pieces); c++) issue(c);
    int threads = rb_threads(pieces);
    while (slots % threads) threads >>= 1;          // (a slot's pieces are one thread's, which fills it again)
    // pieces first, first + threads, ...: the card's bytes [a, b) without the padding between rows
    auto carry = [&](int64_t first) {
        for (int64_t c = first; c < pieces; c += threads) {
            NVL_HIP(hipEventSynchronize(m->rb_ev[(size_t)(c % slots)]));
            const int64_t a = c * piece, b = std::min(total, a + piece);
            const char* from = m->rb_host + c % slots * piece;
            for (int64_t r = a / pitch; r * pitch < b; r++) {
                const int64_t x = std::max(a, r * pitch), y = std::min(b, r * pitch + width);
                if (x < y) memcpy((char*)out + r * width + (x - r * pitch), from + (x - a), (size_t)(y - x));
            }
            if (c + slots < pieces) issue(c + slots);
        }
    };
    NVL_HIP(hipEventSynchronize(m->rb_ev[0]));       // the pass is over: now threads have something to do
    std::vector<std::exception_ptr> failed((size_t)threads);
    auto guarded = [&](int t) {
        try { NVL_HIP(hipSetDevice(m->device)); carry(t); } catch (...) { failed[(size_t)t] = std::current_exception(); }
    };
    std::vector<std::thread> team;
    team.reserve((size_t)threads);
    int started = 1;
    try { for (; started < threads; started++) team.emplace_back(guarded, started); } catch (const std::system_error&) {}
    guarded(0);
    for (int t = started; t < threads; t++) guarded(t);      // (those that could not be started)
    for (auto& t : team) t.join();
    for (auto& e : failed) if (e) std::rethrow_exception(e);
}

}  // namespace
