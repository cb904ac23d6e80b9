"""Where does the bf16 mode's per-layer error come from?  CPU only: tests/bf16_emulator.py (float64 with a bf16 rounding at
each point where the HIP path rounds an MFMA operand) on the bench model's weights and prompt, one rounding point at a time
and all together, then the whole stack.  The "all together" curve is what tests/test_depth_parity_gpu.py measures on the
device: they are equal to two digits at every one of the 16 layers.
usage: python scripts/bf16_error_budget.py [tokens] [layers]"""
import importlib
import sys
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT))
sys.path.insert(0, str(ROOT / "tests"))
import bf16_emulator as E          # noqa: E402

synth = importlib.import_module("nano-vllm-go_amd").synth


def rel(got, ref):
    return float(np.sqrt(((got - ref) ** 2).mean()) / np.sqrt((ref ** 2).mean()))


def main():
    S = int(sys.argv[1]) if len(sys.argv) > 1 else 24
    L = int(sys.argv[2]) if len(sys.argv) > 2 else 16
    cfg = dict(synth.FULL_CONFIGS["llama-3.2-1b"], num_layers=L)
    w = synth.make_weights(cfg, seed=42, scale=0.02)
    prompt = np.random.default_rng(1234 + 1).integers(0, cfg["vocab_size"], S)
    x0 = w[("tok_emb", 0)][prompt].astype(np.float64)
    ref = E.layer(x0, w, 0, cfg, set())
    points = [p for p in E.ALL if p != "xl"]
    print(f"layer 0, {S} tokens: RMS(error) / RMS(stream) with ONE rounding point on")
    tot = 0.0
    for p in points:
        e = rel(E.layer(x0, w, 0, cfg, {p}), ref)
        tot += e * e
        print(f"  {p:4s} {e:.2e}")
    print(f"  quadrature sum {tot ** 0.5:.2e};  all eight on: {rel(E.layer(x0, w, 0, cfg, set(points)), ref):.2e}")
    print(f"  (unit roundoff of bf16 2^-8 = {2.0 ** -8:.2e}; one rounding's relative RMS error ~ 2^-8 / sqrt(3) / 1.39 = {2.0 ** -8 / 3 ** 0.5 / 1.39:.2e})")
    h_ref, lg_ref = E.forward(cfg, w, prompt, sw=())
    h_emu, lg_emu = E.forward(cfg, w, prompt, sw=E.ALL)
    print(f"{L} layers, all points on, per layer: " + " ".join(f"{rel(h_emu[l], h_ref[l]):.1e}" for l in range(L)))
    print("closed form 1.5 * 2^-8 * (l+1)^(1/3): " + " ".join(f"{1.5 * 2.0 ** -8 * (l + 1) ** (1 / 3):.1e}" for l in range(L)))
    print("stream RMS per layer: " + " ".join(f"{np.sqrt((h_ref[l] ** 2).mean()):.2f}" for l in range(L)))
    print(f"last-row logits: RMS(error)/RMS(logits) {rel(lg_emu, lg_ref):.2e}, max|error|/max|logit| {np.abs(lg_emu - lg_ref).max() / np.abs(lg_ref).max():.2e}")


if __name__ == "__main__":
    main()
