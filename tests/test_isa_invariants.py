"""ISA invariants of the hand-scheduled prefill attention kernel (scripts/check_isa.sh): hipcc cross-compiles without a
GPU, so this runs in the CPU suite.  What it pins: M0 is written only by the LDS-DMA inline assembly (it cannot be
declared as a clobber), the compiler has put no `s_waitcnt vmcnt(0)` into the tile loop (that serialises the LDS-DMA
ring: the kernel then still computes the right thing, only ~25 % slower, so no numerical test would notice), no spills.
And the register budgets of the decode kernels (two waves per SIMD for the hd-64 decode attention, bounded spills in the
decode projections): once lost were 5-14 % of decode throughput on GPT-2, Llama-3-8B and the 64-row-group projections to
changes measured only on the headline config — no numerical test notices those either."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc") and shutil.which("hipcc") is None, reason="no hipcc")
def test_prefill_attention_isa_invariants(tmp_path):
    env = dict(os.environ, TMPDIR=str(tmp_path))
    r = subprocess.run(["bash", os.path.join(ROOT, "scripts", "check_isa.sh")], capture_output=True, text=True, env=env,
                       timeout=900)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "attn_prefill<64>" in r.stdout and "attn_prefill<128>" in r.stdout
    assert "BAD" not in r.stdout and r.stdout.count("\nok  ") >= 60


def _registers(operand):
    m = re.match(r"^-?\|?([av])(?:\[(\d+):(\d+)\]|(\d+))\|?$", operand)
    if not m:
        return set()
    lo = int(m[2] or m[4])
    return {(m[1], r) for r in range(lo, int(m[3] or lo) + 1)}


def product_readers(asm):
    """(kernel, wait states, line) of the instructions of an assembly that read the result of a v_mfma_f32_16x16x4_f32, by way of the code as it stands (not over
    an unconditional branch): an instruction is a wait state, s_nop n is n + 1, inline assembly's own instructions count as what they are."""
    kernel, past, found = None, [], []
    for line, text in enumerate(asm.split("\n"), 1):
        m = re.match(r"^(_ZN\w+):", text)
        if m:
            kernel, past = m[1], []
            continue
        code = text.split(";")[0].split(None, 1)
        if not code or code[0].startswith(".") or code[0].endswith(":"):
            continue
        op, args = code[0], [a.split()[0] if a.split() else "" for a in (code[1] if len(code) > 1 else "").split(",")]
        if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
            past = []
            continue
        stores = re.match(r"(buffer|global|flat|scratch)_store|ds_write|ds_bpermute", op)
        product = op.startswith("v_mfma")
        reads = set().union(*(_registers(a) for a in (args if stores else args[1:3] if product else args[1:])), set())
        waits = 0
        for was, wrote, states in reversed(past[-40:]):
            if not reads or waits > 40:
                break
            if wrote & reads:
                if was == "v_mfma_f32_16x16x4_f32":
                    found.append((kernel, waits, line))
                reads = reads - wrote
            waits += states
        past.append((op, set() if stores else _registers(args[0]), int(args[0], 0) + 1 if op == "s_nop" else 1))
    return found


@pytest.mark.skipif(not os.path.exists("/opt/rocm/bin/hipcc") and shutil.which("hipcc") is None, reason="no hipcc")
def test_results_of_fp32_products_are_read_in_time(tmp_path):
    """A result of eight passes may be read ten wait states behind its product (the two passes beyond its own that the architecture asks for).  The compiler
    counts them; the kernels whose products are fp32 have no spacing of their own, so that what it leaves has to hold on every path to a store, to LDS and to a lane."""
    csrc = os.path.join(ROOT, "nano-vllm-go_amd", "csrc")
    jobs, prep = [], {}
    for unit, macro in [("delta", None), ("linrec", 1), ("linrec", 2)]:
        out = tmp_path / f"{unit}{macro}.s"
        cmd = ["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-mllvm", "-amdgpu-kernarg-preload-count=6", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               "--cuda-device-only", "-S", "-o", str(out), os.path.join(csrc, unit + "_inst.hip")] + ([] if macro is None else [f"-DNVL_LINREC_INST={macro}"])
        jobs.append((out, subprocess.Popen(cmd, stderr=subprocess.DEVNULL)))
    seen = set()
    for out, job in jobs:
        assert job.wait(timeout=600) == 0
        asm = out.read_text()
        found = product_readers(asm)
        assert found
        for m in re.finditer(r"^_ZN3nvl17delta_prep_kernelILi(\d+)ELb(\d)ELb(\d)EEE\w*:.*?s_endpgm\n\t\.section", asm, re.M | re.S):
            prep[m.groups()] = len(re.findall(r"buffer_load_dwordx4", m[0])), len(re.findall(r"buffer_load_dword ", m[0]))
        seen |= {k for k, _, _ in found}
        early = [f for f in found if f[1] < 10]
        assert not early, early[:5]
    # the preparation reads keys 16 bytes at a time by their own width, whatever the values' is
    assert len(prep) == 16
    for (nk, keys, values), (wide, narrow) in prep.items():
        assert wide == (prep[nk, "1", "1"][0] if keys == "1" else 0) and (narrow == prep[nk, "1", "1"][1] if keys == "1" else narrow > prep[nk, "1", "1"][1]), (nk, keys, values, wide, narrow)
    assert prep["8", "1", "1"][0] > 0
    assert {n for n in ("delta_prep_kernel", "delta_scan_kernel", "delta_scan_parts_kernel") if any(n in k for k in seen)} == {"delta_prep_kernel", "delta_scan_kernel", "delta_scan_parts_kernel"}


def test_readers_of_products_are_found():
    head = "_ZN1kE:\n\tv_mfma_f32_16x16x4_f32 v[4:7], v1, v2, v[4:7]\n"
    assert product_readers(head + "\ts_nop 8\n\tbuffer_store_dwordx4 v[4:7], v9, s[0:3], 0 offen\n") == [("_ZN1kE", 9, 4)]
    assert product_readers(head + "\ts_nop 3\n\tds_write_b32 v9, v8\n\ts_nop 4\n\tv_add_f32_e32 v8, v7, v8\n") == [("_ZN1kE", 10, 6)]
    assert product_readers(head + "\tv_mov_b32_e32 v4, v9\n\tv_add_f32_e32 v8, v4, v8\n") == []
    assert product_readers(head + "\tv_mfma_f32_16x16x4_f32 v[8:11], v1, v2, v[4:7]\n") == []
