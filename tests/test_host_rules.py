"""Rules of the host code that no result shows, compiled from the headers and run without a device."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")


def run(tmp_path, source):
    src, exe = tmp_path / "rule.hip", tmp_path / "rule"
    src.write_text(source)
    subprocess.run([HIPCC, "-std=c++17", "--offload-arch=gfx950", "-w", "-DNVL_GEMM_INST=0", "-I", os.path.join(ROOT, "nano-vllm-go_amd", "csrc"), str(src), "-o", str(exe)], check=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


# tiles: columns a workgroup covers, 16 .. 64 in the decode and ring kernels, 128 and 256 in the tile kernels
@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_tiles_of_joint_matrices_stay_inside(tmp_path):
    run(tmp_path, r"""
#include "common.h"
int main() {
    const int tiles[] = {16, 32, 64, 128, 256};
    auto last = [](int64_t first, int64_t n, int bn) { return first + (n + bn - 1) / bn * bn; };
    for (int64_t a = 16; a <= 5120; a += 16)
        for (int64_t b = 64; b <= 20480; b += 64)
            for (int bn : tiles) {
                const int64_t rows = nvl::joint_weight_rows(a, b);
                if (last(0, a + b, bn) > rows || last(a, b, bn) > rows || last(0, a, bn) > rows) { printf("%lld + %lld rows: tiles of %d read past %lld\n", (long long)a, (long long)b, bn, (long long)rows); return 1; }
            }
    return 0;
}
""")


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_all_experts_are_streamed_only_at_little_cost(tmp_path):
    """Rows that choose the same experts, answers to one prompt for instance, leave the others alone however many rows there are: what streaming them costs then
    stays within twice the launch that it saves (8 us; 17 at 6 TB/s), so that they lose no more than rows that choose apart gain."""
    run(tmp_path, r"""
#include "gemm.h"
int main() {
    for (int M = 1; M <= 64; M++)
        for (int E = 2; E <= 64; E++)
            for (int k = 1; k <= E; k++)
                for (double bytes = 1 << 14; bytes < 1 << 29; bytes *= 1.5)
                    if (nvl::moe_streams_all(M, E, k, bytes) && (E - k) * bytes / 6e6 > 17.0) { printf("%d rows, %d of %d experts of %.0f bytes\n", M, k, E, bytes); return 1; }
    return 0;
}
""")


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_every_attention_layer_finds_its_buffers(tmp_path):
    """Layers of different widths in one model: those whose heads fit the short kernel have partial records, and tickets for a second mixer's recurrence that rides,
    whatever the others take; a launch whose keys are split stays inside the records."""
    run(tmp_path, r"""
#include "grouped.h"
using namespace nvl;
struct Layer { int dp, vp; bool second; };
int main() {
    const int widths[] = {32, 64, 128, 256, 320, 2048};
    std::vector<Layer> all;
    for (int dp : widths) for (int vp : widths) for (bool second : {false, true}) all.push_back({dp, vp, second});
    for (const Layer& a : all)
        for (const Layer& b : all) {
            GroupedBuffers g;
            for (const Layer& l : {a, b}) g.layer(l.dp, l.vp, l.second);
            for (const Layer& l : {a, b}) {
                const bool served = l.dp <= 256 && l.vp <= 256;
                if (served != grouped_fits(l.dp, l.vp)) { printf("form of %d x %d\n", l.dp, l.vp); return 1; }
                if (!served) continue;
                const char* bad = g.vp < l.vp || g.cap() <= 0 ? "no room for its records" : nullptr;
                for (int dk : {16, 128, 256}) for (int dv : {16, 128}) if (l.second && grouped_takes_recurrence(l.dp, l.vp, dk, dv) && !g.tickets) bad = "no tickets";
                for (int wgs = 1; wgs <= 1024; wgs++)
                    for (int tiles = 1; tiles <= 1024; tiles *= 2)
                        for (int force : {0, 3, 16}) {
                            const int z = grouped_key_splits(wgs, g.cap(), tiles, 8, force);
                            if (z < 1 || z > GROUPED_SPLITS || (z > 1 && (int64_t)wgs * z > g.cap())) bad = "parts past the records";
                            if (z > 1 && grouped_key_splits(wgs, 0, tiles, 8, force) != 1) bad = "parts without records";
                        }
                if (bad) { printf("%d x %d%s beside %d x %d: %s\n", l.dp, l.vp, l.second ? " and another mixer" : "", a.dp == l.dp ? b.dp : a.dp, a.vp == l.vp ? b.vp : a.vp, bad); return 1; }
            }
        }
    return 0;
}
""")


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_contexts_are_sorted_wherever_a_step_takes_them_by_length(tmp_path):
    """The sort of a call's first step serves all its steps, and is left out where none of them can ask for it."""
    run(tmp_path, r"""
#include "attn.h"
int main() {
    unsigned seed = 1;
    auto rnd = [&](int n) { seed = seed * 1664525u + 1013904223u; return (int)((seed >> 8) % n); };
    int sorted = 0, left = 0;
    for (int t = 0; t < 20000; t++) {
        const int n = 33 + rnd(200), spread = 1 + rnd(t % 2 ? 60 : 1500), least = rnd(1500);
        int longest = 0; double sum = 0;
        for (int i = 0; i < n; i++) { const int pos = least + rnd(spread); longest = longest > pos ? longest : pos; sum += pos; }
        const bool possible = nvl::attn_order_possible(longest, sum / n);
        (possible ? sorted : left)++;
        for (int s = 0; s < 200; s++) {
            const int keys = longest + s + 1;
            if (nvl::attn_order_pays((keys - 1) / 64 + 1, (sum / n + s + 1) / 64) && !possible) { printf("%d sequences, longest %d, mean %f, step %d\n", n, longest, sum / n, s); return 1; }
        }
    }
    printf("%d sorted, %d not\n", sorted, left);
    return sorted < 1000 || left < 1000;
}
""")


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_few_rows_in_one_piece(tmp_path):
    """Residual projections of 33 .. 64 rows: where the narrow form measured faster it is kept, where it measured slower it is not."""
    run(tmp_path, r"""
#include "gemm.h"
int main() {
    struct { int M, N, K; bool pays; } m[] = {{33, 4096, 2048, false}, {47, 4096, 1536, false}, {40, 3072, 1536, false}, {33, 2048, 1088, false}, {47, 2048, 1280, false}, {60, 2048, 1088, false},
        {40, 1536, 1088, false}, {64, 1024, 1024, false}, {33, 2048, 2304, false}, {33, 2048, 2048, true}, {47, 2048, 1792, true}, {33, 1024, 1088, true}, {40, 512, 2048, true}, {48, 4096, 2048, true},
        {60, 3072, 1536, true}, {48, 2048, 1280, true}};
    for (auto& c : m) if (nvl::rows_pay_few(c.M, c.N, c.K) != c.pays) { printf("%d rows of %d x %d\n", c.M, c.N, c.K); return 1; }
    return 0;
}
""")
