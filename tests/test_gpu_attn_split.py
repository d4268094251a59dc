"""GPU parity of the attention of many-token steps (64 tokens and more).

Short chunks (attn_rows_kernel): the tiny model against the oracle, row blocks that end inside a tile, steps that end inside a
32-cell block and inside a 16-cell unit, ranges shared with another sequence's blocks, and blocks that lie in the cache in
another order than their positions. Bar: the forward pass's own (test_gpu_forward.py), which the oracle's reordered sums set.

Long chunks (attn_split_kernel, which kernel a launch takes is asserted): one-layer models of head sizes 64 and 128 and query
groups of 1, 3, 4, 5 and 8, whose attention update (the residual entering the MoE block minus the embedding) is compared with
64-bit attention over the same fp16 q, K and V. Chunks of 192 to 1280 cells give every wavefront one to ten units; one and several
chunks per row block; blocks out of order; a range past the block map; a cache too large for the order by position.
Bar: 1e-3 of the largest update (measured up to 2.7e-4). The device rounds the attention rows to fp16 before the output product and q, k and v to
fp16 after products in f32, 2^-11 each, and a last-place flip of one of them moves an output by its share of the row; a
16-cell unit left out of 1280 moves the update by more than a tenth.
"""
import numpy as np
import pytest

import oracle
from localstack_amd import synth
from test_gpu_forward import LOGITS_TOL, RMS_TOL, build, prompt, run, weights
from test_gpu_long_attention import synthetic_kv

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


ATTN_TOL = 1e-3
_models = {}


def _one_layer(n_head, n_kv, hd):
    """hp and weights of a one-layer model with these heads (dense weights of standard deviation 0.05)."""
    key = (n_head, n_kv, hd)
    if key not in _models:
        hp = dict(n_layer=1, n_embd=256, n_head=n_head, n_head_kv=n_kv, head_dim=hd, n_vocab=512, n_expert=8, n_expert_used=2,
                  n_ff_exp=512, n_ctx_train=1 << 18, rms_eps=1e-6, rope_freq_base=1e6)
        _models[key] = hp, synth.qwen3_weights(np.random.default_rng(n_head + hd), hp, std=0.05)
    return _models[key]


def _qkv(hp, w, tokens, pos):
    """fp16 q [T, n_head, hd], k and v [T, n_kv, hd] of the tokens at these positions, as float64."""
    hd, L = hp["head_dim"], w["layers"][0]
    r16 = lambda a: a.astype(np.float32).astype(np.float16).astype(np.float64)
    norm = lambda a: a / np.sqrt((a * a).mean(-1, keepdims=True) + hp["rms_eps"])
    x = w["tok_embd"][tokens].astype(np.float64)
    hn = r16(norm(x))
    q, k, v = ((hn @ L[m].astype(np.float64).T).reshape(len(tokens), -1, hd) for m in ("wq", "wk", "wv"))
    scale = np.power(np.float32(hp["rope_freq_base"]), np.float32(-2.0) / np.float32(hd))  # ggml: the position times this, again and again
    ang = [np.asarray(pos, np.float32)]
    while len(ang) < hd // 2:
        ang.append(ang[-1] * scale)
    ang = np.stack(ang, 1).astype(np.float64)
    c, s = np.cos(ang)[:, None], np.sin(ang)[:, None]
    rope = lambda a: np.concatenate([a[..., :hd // 2] * c - a[..., hd // 2:] * s, a[..., :hd // 2] * s + a[..., hd // 2:] * c], -1)
    return r16(rope(norm(q))), r16(rope(norm(k))), r16(v)


def _update(hp, w, q, pos, k, v, kpos):
    """The attention block's update of the residual [T, n_embd] in 64 bits."""
    T, n_head, hd = q.shape
    grp = n_head // k.shape[1]
    hide = np.asarray(kpos)[None, :] > np.asarray(pos)[:, None]
    a = np.empty((T, n_head, hd))
    for i in range(n_head):
        s = q[:, i] @ k[:, i // grp].T / np.sqrt(hd)
        s[hide] = -np.inf
        e = np.exp(s - s.max(1, keepdims=True))
        a[:, i] = (e / e.sum(1, keepdims=True)) @ v[:, i // grp]
    return a.reshape(T, -1).astype(np.float32).astype(np.float16).astype(np.float64) @ w["layers"][0]["wo"].astype(np.float64).T


def _device_update(model, hp, w, seq, toks, dev):
    import torch
    mid = torch.zeros(1, len(toks), hp["n_embd"], device=dev)
    model.debug_capture_moe_in(mid)
    run(model, seq, toks, hp, dev)
    model.debug_capture_moe_in(None)
    return mid[0].cpu().numpy().astype(np.float64) - w["tok_embd"][toks].astype(np.float64)


def _compare(got, ref, what):
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"[{what}] attention update rel max err {err:.2e}", flush=True)
    assert err <= ATTN_TOL, what


# heads, head size, tokens, context, cache cells, (cells per chunk, chunks) in the plain layout
LONG = [((128, 32), 64, 113, 100, 2048, (256, 1)), ((128, 32), 64, 128, 900, 2048, (1280, 1)), ((80, 16), 64, 193, 523, 2048, (768, 1)),
        ((80, 16), 64, 204, 60, 2048, (512, 1)), ((128, 32), 64, 70, 3300, 4096, (896, 4)),
        ((48, 16), 128, 321, 900, 2048, (1280, 1)), ((48, 16), 128, 341, 3, 2048, (512, 1)), ((64, 8), 128, 250, 0, 2048, (256, 1)),
        ((64, 8), 128, 255, 600, 2048, (1024, 1)), ((48, 16), 128, 200, 2300, 4096, (640, 4)), ((8, 8), 128, 64, 6000, 8192, (192, 32)),
        ((128, 32), 64, 128, 900, 132096, (1280, 1))]


@pytest.mark.parametrize("heads,hd,T,ctx,kv_size,want", LONG, ids=lambda v: "-".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_long_chunks_match_64_bits(lstk, dev, heads, hd, T, ctx, kv_size, want):
    """In order, and with the blocks out of order between two other sequences' (bit for bit the same where a row block is one
    chunk, whose sums are taken in the order of the positions)."""
    hp, w = _one_layer(*heads, hd)
    cells = (ctx + T + 255) // 256 * 256
    assert lstk.attn_plan(T, *heads, hd, kv_size, cells)[2:4] == want and lstk.attn_split(T, *heads, hd, kv_size, cells, 0, ctx + T)
    toks, pos = prompt(T + ctx, T, hp["n_vocab"]), np.arange(ctx, ctx + T)
    q, k, v = _qkv(hp, w, toks, pos)
    kc, vc = (a.astype(np.float64).reshape(ctx, heads[1], hd) for a in synthetic_kv(9, 0, 0, ctx, heads[1], hd))
    ref = _update(hp, w, q, pos, np.concatenate([kc, k]), np.concatenate([vc, v]), np.arange(ctx + T))
    got = []
    for shared in (False, True):
        store, model = build(lstk, dev, hp, w, n_batch=T, kv_size=kv_size)
        if shared:  # seq 0 takes seq 7's freed blocks, then seq 5's last to first, then what lies above
            for seq, n in ((5, 300), (6, 70), (7, 130)):
                model.fill_context(seq, n, seed=seq)
            model.remove_seq(5)
            model.truncate_seq(7, 33)
        if ctx:
            model.fill_context(0, ctx, seed=9)
        got.append(_device_update(model, hp, w, 0, toks, dev))
        _compare(got[-1], ref, f"{heads} x {hd} T {T} ctx {ctx} kv {kv_size} shared {shared}")
        model.close()
        store.close()
    # (fewer blocks end above cell 0, where the launch has other chunks; a larger cache orders its blocks by cell)
    if want[1] == 1 and ctx + T >= 13 * 32 and kv_size <= 131072:
        assert np.array_equal(*got)


def test_block_whose_first_cells_were_never_written(lstk, dev):
    """96 tokens, then 5 cells reserved by a prepare whose forward never ran, then a 120-token step: the fourth block's first
    cells hold no position, and the step sees its other cells and the blocks before it."""
    heads, hd, T, n = (128, 32), 64, 120, 96
    hp, w = _one_layer(*heads, hd)
    assert lstk.attn_split(T, *heads, hd, 512, 256, 0, n + 5 + T)
    toks = prompt(3, n + T, hp["n_vocab"])
    pos = np.concatenate([np.arange(n), n + 5 + np.arange(T)])
    q, k, v = _qkv(hp, w, toks, pos)
    ref = _update(hp, w, q[n:], pos[n:], k, v, pos)
    store, model = build(lstk, dev, hp, w, n_batch=T, kv_size=512)
    run(model, 0, toks[:n], hp, dev)
    model.prepare(0, toks[:5])
    _compare(_device_update(model, hp, w, 0, toks[n:], dev), ref, "hole")
    model.close()
    store.close()


def test_range_past_the_block_map(lstk, dev):
    """A sequence whose first block lies 131072 cells below the others: 2052 passes, more than the map of live blocks holds, so
    every cell of the range is visited in order, in a cache too large for the order by position."""
    heads, hd, T, other, kv_size, n = (128, 32), 64, 113, 131072, 132096, 96
    hp, w = _one_layer(*heads, hd)
    cells = (n + other + T + 255) // 256 * 256
    assert lstk.attn_plan(T, *heads, hd, kv_size, cells)[2:4] == (cells, 1) and cells > 64 * 2048
    assert lstk.attn_split(T, *heads, hd, kv_size, cells, 0, n + T)
    toks, pos = prompt(8, n + T, hp["n_vocab"]), np.arange(n + T)
    q, k, v = _qkv(hp, w, toks, pos)
    ref = _update(hp, w, q[n:], pos[n:], k, v, pos)
    store, model = build(lstk, dev, hp, w, n_batch=T, kv_size=kv_size)
    run(model, 0, toks[:n], hp, dev)
    model.fill_context(5, other, seed=5)
    _compare(_device_update(model, hp, w, 0, toks[n:], dev), ref, "past the map")
    model.close()
    store.close()
