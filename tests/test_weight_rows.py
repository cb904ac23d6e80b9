"""Rows that weight matrices are allocated with, against the rows that whole tiles of the projections' kernels read (host code of common.h, no device)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")

# columns a workgroup covers: 8 .. 64 decode kernels and ring kernel, 128 and 256 tile kernels
SOURCE = r"""
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
"""


@pytest.mark.skipif(HIPCC is None, reason="no hipcc")
def test_tiles_of_joint_matrices_stay_inside(tmp_path):
    src, exe = tmp_path / "rows.hip", tmp_path / "rows"
    src.write_text(SOURCE)
    subprocess.run([HIPCC, "-std=c++17", "--offload-arch=gfx950", "-I", os.path.join(ROOT, "nano-vllm-go_amd", "csrc"), str(src), "-o", str(exe)], check=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
