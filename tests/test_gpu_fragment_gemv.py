"""GPU parity of the fragment-ordered batched decode GEMVs (gemv_frag.hip), through the C-ABI.

With 3..8 sequences and bf16 weights the decode step's O, gate/up and down projections read
copies of the matrices in MFMA fragment order, split evenly over every wavefront, and the gate/up
RMSNorm takes its sums of squares from the per-16-row partials that the O projection publishes.
Checked here:

* the C5 layer shape (d 2560, 32 Q / 8 KV heads, F 9728), batch 8: the same greedy decode with the
  fragment GEMVs and with the row-major MFMA GEMVs (ar_hip_qwen3_use_fragment_gemv(m, 0)) agree
  within float rounding (logits 1e-5 relative, every token equal), over a 24-token prompt fed one
  token per step and 16 generated tokens;
* the Qwen3-0.6B layer shape with bf16 weights at batch 3 (sequences 3..7 of the MFMA columns
  unused, most tiles shared by several wavefronts) against the FP32 oracle run on the same bf16-rounded
  weights: logits within 2e-2 and the greedy tokens equal where the reference's top-2 margin is
  above that tolerance (the bar of the other bf16 workload tests);
* widths whose row-major products hold 13 to 16 k-steps a wavefront (the 8B shape's 4,096 among them), three
  sequences, with and without the fragment GEMVs, against the FP64 oracle.
"""
import dataclasses

import numpy as np
import pytest

import oracle
from common_amd import config as C
from common_amd import synthetic
from common_amd.qwen3 import Qwen3
from conftest import rel_err

pytestmark = pytest.mark.gpu
BF16_TOL = 2e-2


def _decode(am, prompts, steps):
    am.reset()
    for b, p in enumerate(prompts):
        am.set_prompt(p, seq=b)
    toks, lgs = [], []
    for _ in range(len(prompts[0]) + steps):
        t, lg = am.next(return_logits=True)
        toks.append(t)
        lgs.append(lg)
    return np.stack(toks, axis=1), np.stack(lgs, axis=1)


def test_fragment_gemv_matches_row_major_c5_shape_batch8(ctx):
    cfg = dataclasses.replace(C.C5_4B, layer_count=2, vocab_size=4096, shared_weights=False, seq_len=64, max_batch=8)
    sd = synthetic.state_dict(cfg, seed=31)
    prompts = synthetic.prompt_ids(24, cfg.vocab_size, seed=32, batch=8)
    print(f"fragment GEMV vs row-major: C5 layer shape, batch 8, 24 + 16 steps", flush=True)
    with Qwen3(cfg, sd, ctx) as m:
        am = m.model
        assert am.fragment_gemv, "the C5 shape at batch 8 should use the fragment-ordered GEMVs"
        tf, lf = _decode(am, prompts, 16)
        am.use_fragment_gemv(False)
        assert not am.fragment_gemv
        tr, lr = _decode(am, prompts, 16)
        am.use_fragment_gemv(True)
        assert am.fragment_gemv
        tf2, lf2 = _decode(am, prompts, 4)  # switching back after the row-major steps
    assert np.array_equal(tf, tr), (tf, tr)
    err = rel_err(lf, lr)
    print(f"  logits max rel err {err:.2e}, distinct tokens per sequence "
          f"{[len(set(t.tolist())) for t in tf]}", flush=True)
    assert err <= 1e-5, err
    assert np.array_equal(tf2, tf[:, :tf2.shape[1]])
    assert rel_err(lf2, lf[:, :lf2.shape[1]]) <= 1e-5


def test_fragment_gemv_batch3_vs_oracle(ctx):
    cfg = dataclasses.replace(C.C3_0_6B, layer_count=2, vocab_size=4096, shared_weights=False, seq_len=64,
                              max_batch=3, weight_dtype=C.DTYPE_BF16)
    sd = synthetic.state_dict(cfg, seed=33)
    prompts = synthetic.prompt_ids(12, cfg.vocab_size, seed=34, batch=3)
    steps = 12
    with Qwen3(cfg, sd, ctx) as m:
        am = m.model
        assert am.fragment_gemv, "d1024 / F3072 bf16 at batch 3 should use the fragment-ordered GEMVs"
        toks, lgs = _decode(am, prompts, steps)
    cfg1 = dataclasses.replace(cfg, max_batch=1)
    for b in range(3):
        ref = oracle.OracleQwen3(cfg1, sd, precision="fp32")
        fed, rl = ref.generate(prompts[b], steps)
        ref.close()
        n = len(prompts[b])
        margins = np.sort(rl, axis=-1)[..., -2:]
        margins = (margins[..., 1] - margins[..., 0]) / np.abs(margins[..., 1])
        compared = 0
        for s in range(n + steps):
            assert rel_err(lgs[b, s], rl[s]) <= BF16_TOL, (b, s, rel_err(lgs[b, s], rl[s]))
            if s + 1 < n + steps and toks[b, s + 1] != fed[s + 1]:
                assert margins[s] < BF16_TOL, (b, s, margins[s])
                break
            compared += 1
        print(f"  seq {b}: {compared} steps equal to the oracle", flush=True)
        assert compared >= n + 2


@pytest.mark.parametrize("dim", [3328, 3616, 4096])
def test_wide_row_major_products_vs_oracle(ctx, dim):
    """QKV (6,144 rows) and the head (4,352) read operand planes and the RMSNorm's raw input in the packed
    row-major form; with the fragment GEMVs off so does the 4,096-wide O product where the model is as wide.
    Two bf16 planes carry 16 bits of an input (2^-17 relative), through four products and a residual stream:
    1e-4."""
    cfg = C.Qwen3Config(dim=dim, hidden_dim=512, layer_count=1, head_count=32, kv_head_count=8, vocab_size=4352,
                        seq_len=16, head_size=128, max_batch=3, weight_dtype=C.DTYPE_BF16, kv_dtype=C.DTYPE_F32)
    sd = synthetic.state_dict(cfg, seed=dim)
    prompts = synthetic.prompt_ids(3, cfg.vocab_size, seed=35, batch=3)
    with Qwen3(cfg, sd, ctx) as m:
        runs = []
        for frag in (True, False):
            m.model.use_fragment_gemv(frag)
            runs.append(_decode(m.model, prompts, 1))
    for b in range(3):
        ref = oracle.OracleQwen3(dataclasses.replace(cfg, max_batch=1), sd, precision="fp64")
        _, rl = ref.generate(prompts[b], 1)
        ref.close()
        for _, lgs in runs:
            for s in range(len(prompts[b])):
                assert rel_err(lgs[b, s], rl[s]) <= 1e-4, (b, s, rel_err(lgs[b, s], rl[s]))
