"""GPU parity of the prompt attention (attn_split_kernel, steps of 64 tokens and more) on the tiny model against the oracle:
row blocks that end inside a tile, steps that end inside a 32-cell block and inside a 16-cell unit, ranges shared with
another sequence's blocks, and blocks that lie in the cache in another order than their positions.

Bar: the forward pass's own (test_gpu_forward.py), which the oracle's reordered sums set.
"""
import numpy as np
import pytest

import oracle
from test_gpu_forward import LOGITS_TOL, RMS_TOL, build, prompt, run, weights

pytestmark = pytest.mark.gpu


def _check(ref, model, seq, toks, hp, dev, what):
    rl = ref.decode(toks)
    gl, _ = run(model, seq, toks, hp, dev)
    err, rms, ra, ga = oracle.diff_logits(rl, gl)
    print(f"[{what}] max|dlogit| {err:.2e} rms {rms:.2e} top1 {ga}/{ra}", flush=True)
    assert err <= LOGITS_TOL and rms <= RMS_TOL and ga == ra, what


@pytest.mark.parametrize("steps", [(64, 65, 97), (79, 130, 64), (129, 64, 1, 66)], ids=lambda s: "-".join(map(str, s)))
@pytest.mark.parametrize("shared", [False, True])
def test_prompt_steps_match_oracle(lstk, dev, steps, shared):
    hp, w = weights("tiny")
    _, model = build(lstk, dev, hp, w, n_batch=130, kv_size=1024)
    ref = oracle.Qwen3(hp, w, 512)
    if shared:  # seq 0's blocks come from a removed sequence's, last released first, between two others'
        for seq, n in ((5, 300), (6, 70), (7, 130)):
            model.fill_context(seq, n, seed=seq)
        model.remove_seq(5)
        model.truncate_seq(7, 33)
    for i, n in enumerate(steps):
        _check(ref, model, 0, prompt(100 * i + n, n, hp["n_vocab"]), hp, dev, f"shared {shared} step {i} of {n}")


def test_block_whose_first_cells_were_never_written(lstk, dev):
    """32 tokens, then 5 cells reserved by a prepare whose forward never ran, then a 91-token step: the second block's first
    cells hold no position, and the step sees its other cells and the first block as steps of 30 tokens do (attn_rows_kernel;
    f32 orders apart, so the bar is the forward pass's own)."""
    hp, w = weights("tiny")
    toks, lg = prompt(3, 32 + 91, hp["n_vocab"]), []
    for steps in ((91,), (30, 30, 31)):
        _, model = build(lstk, dev, hp, w, n_batch=96, kv_size=512)
        run(model, 0, toks[:32], hp, dev)
        model.prepare(0, toks[:5])
        at = 32
        for n in steps:
            out, _ = run(model, 0, toks[at:at + n], hp, dev)
            at += n
        lg.append(out)
    err, rms, ra, ga = oracle.diff_logits(*lg)
    print(f"[hole] max|dlogit| {err:.2e} rms {rms:.2e} top1 {ga}/{ra}", flush=True)
    assert err <= LOGITS_TOL and rms <= RMS_TOL and ga == ra
