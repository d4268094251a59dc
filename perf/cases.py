"""Timed cases of the Qwen3-MoE path: MoE layers through ExpertStore.block and forward passes through Qwen3Model.forward.

Listed cases (what each stands for in real use):
  decode_q8_t1        one token through four MoE layers of Qwen3-30B-A3B with Q8_0 experts: single-user decode
  decode_q2k_t1       the same with Q2_K gate / up and Q3_K down, the mix of a UD-Q2_K_XL file
  decode_235b_t1      one token through two MoE layers of Qwen3-235B-A22B with Q4_K experts
  batch_q8_t8         eight tokens (a short speculative or chat turn) through Q8_0 experts
  batch_q2k_t64       a 64-token prompt through the UD-Q2_K_XL mix
  chunk_q4km_t203     an odd prompt remainder through a Q4_K_M file's layer (Q4_K gate / up, Q6_K down)
  prefill_q4_t512     a full 512-token prompt step, Q4_K experts, Zipf-skewed routing
  prefill_q8_t512     the same through Q8_0 experts with an even router
  model_t1_4k         whole forward pass (two 30B-shaped layers, full vocabulary head), one token after 4095
  model_t32_4k        32 tokens of one sequence in one step after 4064
  model_prompt_3584   the last 512-token step of a 4096-token prompt
  tiny_t1             the smallest call: a two-layer test-size model, one token, no graph
A forward pass also returns its router ids (the engine's routing trace). Steps of up to 32 tokens are captured once in a HIP graph and replayed, as a serving loop does; longer ones and
tiny_t1 are launched call by call.

Weights are drawn as GGUF blocks on the GPU and handed over as host arrays, as a GGUF file would be; a stack's
layers hold the same values at their own addresses. The 64-bit results dequantize the same blocks and follow
ggml's definition of the path: F16 products take fp16-rounded rows, expert products take rows quantized to Q8_0
(for Q8_0 experts) or Q8_K (for k-quants).
"""
import functools
import math

import numpy as np
import torch

import localstack_amd as L

Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K = 8, 10, 11, 12, 13, 14
BLOCK_BYTES = {Q8_0: 34, Q2_K: 84, Q3_K: 110, Q4_K: 144, Q5_K: 176, Q6_K: 210}
# expert types (gate and up, down) of files in use
MIXES = {"q8": (Q8_0, Q8_0), "q4": (Q4_K, Q4_K), "q4km": (Q4_K, Q6_K), "q5km": (Q5_K, Q6_K), "q2kxl": (Q2_K, Q3_K)}
SHAPES = {"30b": dict(h=2048, f=768, E=128, k=8, heads=32, kv=4, hd=128),
          "235b": dict(h=4096, f=1536, E=128, k=8, heads=64, kv=4, hd=128),
          "tiny": dict(h=256, f=512, E=8, k=2, heads=4, kv=2, hd=64)}
N_BATCH = 512  # largest step of the pools and models
EPS, ROPE_BASE = 1e-6, 1e6
DEV = "cuda:0"


def _moe(name, mix, T, layers, shape="30b", skew=0.0, gate="f16"):
    return {"name": name, "kind": "moe", "shape": shape, "mix": mix, "T": T, "layers": layers, "skew": skew, "gate": gate,
            "graph": T <= 32}


def _model(name, T, ctx, mix="q4", shape="30b", vocab=151936, graph=None):
    return {"name": name, "kind": "model", "shape": shape, "mix": mix, "T": T, "ctx": ctx, "layers": 2, "vocab": vocab,
            "skew": 0.0, "gate": "f16", "graph": T <= 32 if graph is None else graph}


def listed():
    return [_moe("decode_q8_t1", "q8", 1, 4),
            _moe("decode_q2k_t1", "q2kxl", 1, 4),
            _moe("decode_235b_t1", "q4", 1, 2, shape="235b"),
            _moe("batch_q8_t8", "q8", 8, 2),
            _moe("batch_q2k_t64", "q2kxl", 64, 2),
            _moe("chunk_q4km_t203", "q4km", 203, 2),
            _moe("prefill_q4_t512", "q4", 512, 2, skew=1.1),
            _moe("prefill_q8_t512", "q8", 512, 2),
            _model("model_t1_4k", 1, 4095),
            _model("model_t32_4k", 32, 4064),
            _model("model_prompt_3584", 512, 3584),
            _model("tiny_t1", 1, 15, mix="q8", shape="tiny", vocab=1024, graph=False)]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    if rng.random() < 0.7:
        shape = rng.choice(["30b", "30b", "30b", "30b", "235b", "tiny"])
        T = _log_int(rng, 1, 64 if shape == "235b" else 512)
        mix = "q4" if shape == "235b" else rng.choice(sorted(MIXES))
        c = _moe("", mix, T, 1 if shape == "235b" or T > 32 else 2, shape, rng.choice([0.0, 1.1]), rng.choice(["f16", "f16", "f32"]))
    else:
        shape = rng.choice(["30b", "30b", "30b", "tiny"])
        T = _log_int(rng, 1, 512)
        c = _model("", T, _log_int(rng, 16, 4096 - T), rng.choice(["q4", "q8", "q4km"]), shape, 1024 if shape == "tiny" else 32768)
    del c["name"]
    return c


# ---- inputs ------------------------------------------------------------------------------------

def _f16_bytes(x):
    return x.half().view(torch.uint8).reshape(*x.shape, 2)


def _blocks(g, wtype, n, std):
    """n GGUF blocks of wtype (uint8 [n, bytes]) whose values are about zero-mean with a spread near std."""
    dev = g.device
    unit = lambda *s: torch.rand(*s, generator=g, device=dev)
    if wtype == Q8_0:
        out = torch.empty(n, 34, dtype=torch.uint8, device=dev)
        out[:, 2:] = (torch.randn(n, 32, generator=g, device=dev) * 45.0).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        out[:, :2] = _f16_bytes((0.8 + 0.4 * unit(n)) * (std / 45.0))
        return out
    out = torch.randint(0, 256, (n, BLOCK_BYTES[wtype]), generator=g, device=dev, dtype=torch.uint8)
    if wtype == Q4_K:  # sub-block scales 4 .. 8 and mins round(7.5 sc): every sub-block centred on zero
        sc = torch.randint(4, 9, (n, 8), generator=g, device=dev, dtype=torch.int32)
        m = (sc * 15 + 1) // 2
        d = _f16_bytes((0.8 + 0.4 * unit(n)) * (std / (4.61 * 6.0)))
        out[:, 0:2], out[:, 2:4] = d, d
        out[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
        out[:, 8:12] = (m[:, :4] | ((m[:, 4:] >> 4) << 6)).to(torch.uint8)
        out[:, 12:16] = ((sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)).to(torch.uint8)
        return out
    # random quants and scales; (offset of d, of dmin, d for std 0.02, dmin / d)
    od, om, d0, mf = {Q2_K: (80, 82, 1.3e-3, 1.5), Q3_K: (108, None, 5e-4, 0), Q5_K: (0, 2, 3.7e-5, 15.5),
                      Q6_K: (208, None, 1.5e-5, 0)}[wtype]
    d = (0.5 + unit(n)) * (d0 * std / 0.02)
    out[:, od:od + 2] = _f16_bytes(d)
    if om is not None:
        out[:, om:om + 2] = _f16_bytes(d * mf)
    return out


def _expert_tensor(g, wtype, n_expert, rows, cols, std=0.02):
    per = 32 if wtype == Q8_0 else 256
    return _blocks(g, wtype, n_expert * rows * (cols // per), std).view(n_expert, rows, -1)


def _router(g, c, s):
    w = torch.randn(s["E"], s["h"], generator=g, device=DEV) * 0.02
    if c["skew"]:  # Zipf popularity as a per-expert logit bias on a constant column of the rows
        rank = torch.randperm(s["E"], generator=g, device=DEV) + 1
        p = rank.double() ** -c["skew"]
        w[:, 0] = (p / p.sum()).log().float()
    return w.half() if c["gate"] == "f16" else w


def _inputs(c, seed):
    """Everything a case holds, as device tensors, from the seed alone."""
    s = SHAPES[c["shape"]]
    g = torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)
    tg, td = MIXES[c["mix"]]
    d = {"gate": _expert_tensor(g, tg, s["E"], s["f"], s["h"]), "up": _expert_tensor(g, tg, s["E"], s["f"], s["h"]),
         "down": _expert_tensor(g, td, s["E"], s["h"], s["f"])}
    if c["kind"] == "moe":
        d["router"] = [_router(g, c, s) for _ in range(c["layers"])]
        d["x"] = torch.randn(c["layers"], c["T"], s["h"], generator=g, device=DEV)
        d["resid"] = torch.randn(c["layers"], c["T"], s["h"], generator=g, device=DEV)
        if c["skew"]:
            d["x"][:, :, 0] = 1.0
        return d
    f16 = lambda rows, cols, std=0.02: (torch.randn(rows, cols, generator=g, device=DEV) * std).half()
    norm = lambda n: 1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)
    hq, hk = s["heads"] * s["hd"], s["kv"] * s["hd"]
    d["tok_embd"], d["output_norm"] = f16(c["vocab"], s["h"], 1.0), norm(s["h"])  # a residual stream that outweighs one layer's update
    d["layers"] = [{"attn_norm": norm(s["h"]), "wq": f16(hq, s["h"]), "wk": f16(hk, s["h"]), "wv": f16(hk, s["h"]),
                    "wo": f16(s["h"], hq), "q_norm": norm(s["hd"]), "k_norm": norm(s["hd"]), "ffn_norm": norm(s["h"]),
                    "gate_inp": _router(g, c, s)} for _ in range(c["layers"])]
    d["tokens"] = torch.randint(0, c["vocab"], (c["T"],), generator=g, device=DEV, dtype=torch.int32).cpu().numpy()
    d["kv_seed"] = seed + 1
    return d


def prepare(case, seed):
    c, s = case, SHAPES[case["shape"]]
    d = _inputs(c, seed)
    host = {m: d[m].cpu().numpy().reshape(-1) for m in ("up", "gate", "down")}
    tg, td = MIXES[c["mix"]]
    store = L.ExpertStore(c["layers"], s["h"], s["f"], s["E"], s["k"], N_BATCH,
                          [((tg, tg, td), host["up"], host["gate"], host["down"])] * c["layers"])
    T, n = c["T"], c["layers"]
    if c["kind"] == "moe":
        st = {"store": store, "router": d["router"], "x": d["x"], "resid": d["resid"],
              "gate_type": L.TYPE_F16 if c["gate"] == "f16" else L.TYPE_F32, "n": n,
              "out": torch.zeros(n, T, s["h"], device=DEV), "ids": torch.zeros(n, T, s["k"], dtype=torch.int32, device=DEV),
              "w": torch.zeros(n, T, s["k"], device=DEV)}
        step = functools.partial(_moe_step, st)
    else:
        cpu = lambda t: t.cpu().numpy()
        weights = {"tok_embd": cpu(d["tok_embd"]), "output_norm": cpu(d["output_norm"]), "output": None,
                   "layers": [{k: cpu(v) for k, v in lw.items()} for lw in d["layers"]]}
        hp = dict(n_layer=n, n_embd=s["h"], n_head=s["heads"], n_head_kv=s["kv"], head_dim=s["hd"], n_vocab=c["vocab"],
                  n_expert=s["E"], n_expert_used=s["k"], n_ff_exp=s["f"], n_ctx_train=32768, rms_eps=EPS, rope_freq_base=ROPE_BASE)
        model = L.Qwen3Model(hp, weights, store, (c["ctx"] + T + 255) // 256 * 256, N_BATCH, device=DEV)
        model.fill_context(0, c["ctx"], seed=d["kv_seed"])
        st = {"store": store, "model": model, "T": T, "ids": torch.zeros(n, T, s["k"], dtype=torch.int32, device=DEV)}
        st["cells"] = model.prepare(0, d["tokens"])
        step = functools.partial(_model_step, st)
    st["step"] = step
    if c["graph"]:
        step()
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            step()
    torch.cuda.synchronize()
    return st


def _moe_step(st):
    for l in range(st["n"]):
        st["store"].block(l, st["x"][l], st["router"][l], st["gate_type"], st["resid"][l], st["out"][l], st["ids"][l], st["w"][l])


def _model_step(st):
    # the step's kernels over the inputs prepare() uploaded; its cells and logits are written again each time
    st["model"].forward(0, st["T"], st["cells"], trace=st["ids"])


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        state["step"]()
    if "model" in state:
        return state["model"].logits, state["ids"]
    return state["out"], state["ids"], state["w"]


# ---- what a pass cannot do without -------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _distinct(E, k, T, skew):
    """Expected distinct experts of T tokens under the cases' routers (logit noise of standard deviation 0.9)."""
    r = np.random.default_rng(5)
    p = (np.arange(1, E + 1) ** -skew) if skew else np.ones(E)
    lg = np.log(p / p.sum()) + 0.9 * r.standard_normal((T, E))
    return len(np.unique(np.argpartition(-lg, k - 1, axis=1)[:, :k])) if k < E else E


def _moe_work(c, s, T):
    tg, td = MIXES[c["mix"]]
    per = lambda t: BLOCK_BYTES[t] / (32 if t == Q8_0 else 256)
    wbytes = s["f"] * s["h"] * (2 * per(tg) + per(td))
    nb = _distinct(s["E"], s["k"], T, c["skew"]) * wbytes + s["E"] * s["h"] * (2 if c["gate"] == "f16" else 4)
    return nb, 2.0 * T * s["k"] * 3 * s["h"] * s["f"] + 2.0 * T * s["E"] * s["h"]


def work(case):
    c, s = case, SHAPES[case["shape"]]
    T = c["T"]
    if c["kind"] == "moe":
        nb, fl = _moe_work(c, s, T)
        return {"bytes": int(c["layers"] * (nb + T * s["h"] * 12 + T * s["k"] * 8)), "flops": int(c["layers"] * fl)}
    hq, hk, cells = s["heads"] * s["hd"], s["kv"] * s["hd"], c["ctx"] + T
    nb = c["vocab"] * s["h"] * 2 + T * s["h"] * 2 + c["vocab"] * 4
    fl = 2.0 * c["vocab"] * s["h"]
    for l in range(c["layers"]):
        last = l == c["layers"] - 1  # its MoE block runs on the output row only
        mb, mf = _moe_work(c, s, 1 if last else T)
        nb += (2 * hq + 2 * hk) * s["h"] * 2 + cells * hk * 4 + mb
        # causal attention: token t of the step sees ctx + t + 1 cells
        fl += 2.0 * T * s["h"] * (2 * hq + 2 * hk) + 4.0 * hq * (T * c["ctx"] + T * (T + 1) / 2) + mf
    return {"bytes": int(nb), "flops": int(fl)}


def tolerance(case):
    # Against 64 bits a MoE layer measures 3e-8 to 4.3e-5 (an expert activation whose rounding to 8 bits goes the other
    # way now and then) and a forward pass 7e-8 to 2.1e-3 (such a flip travels on, and may swap two near-equal experts).
    return {"rel": 2e-4, "differ": 0.002} if case["kind"] == "moe" else {"rel": 1e-2, "differ": 0.01}


# ---- the same results in 64 bits ---------------------------------------------------------------

def _h(b, o):
    return b[:, o:o + 2].contiguous().view(torch.float16).double()  # [n, 1]


def _scale_min(b):
    """Eight 6-bit scales and mins of Q4_K / Q5_K (12 bytes at 4) as int64 [n, 8] each."""
    q = b[:, 4:16].long()
    lo, mid, hi = q[:, 0:4], q[:, 4:8], q[:, 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1)
    return sc, torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1)


def _dequant(wtype, b):
    """GGUF blocks [n, bytes] as float64 values [n, 32 or 256]."""
    n = b.shape[0]
    if wtype == Q8_0:
        return b[:, 2:].view(torch.int8).double() * _h(b, 0)
    if wtype in (Q4_K, Q5_K):
        sc, m = _scale_min(b)
        qs = b[:, 16 if wtype == Q4_K else 48:].long().view(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2)  # [n, 4, 2, 32]
        if wtype == Q5_K:
            bit = torch.arange(8, device=b.device).view(1, 4, 2, 1)
            q = q + 16 * ((b[:, 16:48].long().view(n, 1, 1, 32) >> bit) & 1)
        return (_h(b, 0) * sc).view(n, 8, 1).mul(q.view(n, 8, 32)).sub((_h(b, 2) * m).view(n, 8, 1)).view(n, 256)
    shift = torch.tensor([0, 2, 4, 6], device=b.device).view(1, 1, 4, 1)
    if wtype == Q6_K:
        ql, qh = b[:, 0:128].long().view(n, 2, 2, 32), b[:, 128:192].long().view(n, 2, 1, 32)
        q = (torch.cat([ql & 15, ql >> 4], 2) | (((qh >> shift) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _h(b, 208)
        return sc.view(n, 16, 1).mul(q.view(n, 16, 16)).view(n, 256)
    if wtype == Q2_K:
        q = (b[:, 16:80].long().view(n, 2, 1, 32) >> shift) & 3
        sc = b[:, 0:16].long()
        return (_h(b, 80) * (sc & 15)).view(n, 16, 1).mul(q.view(n, 16, 16)).sub((_h(b, 82) * (sc >> 4)).view(n, 16, 1)).view(n, 256)
    bit = torch.arange(8, device=b.device).view(1, 2, 4, 1)  # Q3_K
    q = ((b[:, 32:96].long().view(n, 2, 1, 32) >> shift) & 3) - 4 + 4 * ((b[:, 0:32].long().view(n, 1, 1, 32) >> bit) & 1)
    p = b[:, 96:108].long()
    low = torch.cat([p[:, 0:8] & 15, p[:, 0:8] >> 4], 1)
    sc = (low | (torch.cat([(p[:, 8:12] >> s) & 3 for s in (0, 2, 4, 6)], 1) << 4)) - 32
    return (_h(b, 108) * sc).view(n, 16, 1).mul(q.view(n, 16, 16)).view(n, 256)


def _quantized(x, wtype):
    """Rows as ggml quantizes them for weights of wtype (Q8_0 or Q8_K, in 32 bits), dequantized to 64."""
    v = x.float()
    if wtype == Q8_0:
        v = v.reshape(*x.shape[:-1], -1, 32)
        amax = v.abs().amax(-1, keepdim=True)
        q = torch.round(v * torch.where(amax > 0, 127.0 / amax, torch.zeros_like(amax)))
        d = (amax / 127.0).half().double()
    else:
        v = v.reshape(*x.shape[:-1], -1, 256)
        mx = v.gather(-1, v.abs().argmax(-1, keepdim=True))
        iscale = torch.where(mx != 0, -127.0 / mx, torch.zeros_like(mx))
        q = torch.round(iscale * v).clamp_(max=127.0)
        d = torch.where(mx != 0, 1.0 / iscale, torch.zeros_like(mx)).double()
    return (q.double() * d).reshape(x.shape)


def _exact_moe(c, s, d, x, router, resid):
    """One MoE block: (out, ids, weights) of rows x [T, h] (float32 values), router [E, h], residual rows."""
    T, k, (tg, td) = x.shape[0], s["k"], MIXES[c["mix"]]
    xr = x.half().double() if c["gate"] == "f16" else x.double()
    p = torch.softmax(xr @ router.double().T, -1)
    top, ids = torch.sort(p, dim=-1, descending=True, stable=True)
    top, ids = top[:, :k], ids[:, :k]
    w = top / top.sum(-1, keepdim=True).clamp_min(2.0 ** -14)
    xq = _quantized(x, tg)
    y = torch.zeros(T, k, s["h"], dtype=torch.float64, device=x.device)
    for e in torch.unique(ids).tolist():
        t, j = torch.nonzero(ids == e, as_tuple=True)
        mat = lambda name, ty, rows: _dequant(ty, d[name][e].reshape(-1, BLOCK_BYTES[ty])).view(rows, -1)
        gv = xq[t] @ mat("gate", tg, s["f"]).T
        a = gv * torch.sigmoid(gv) * (xq[t] @ mat("up", tg, s["f"]).T)
        y[t, j] = (_quantized(a, td) @ mat("down", td, s["h"]).T) * w[t, j, None]
    return resid.double() + y.sum(1), ids.int(), w


def _mix64(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _context(layer, n, hk, seed):
    """K and V of fill_context: fp16 values in [-1, 1) hashed from (seed, layer, position, element)."""
    with np.errstate(over="ignore"):
        at = (np.uint64(layer) << np.uint64(48)) ^ (np.arange(n, dtype=np.uint64)[:, None] << np.uint64(20)) ^ np.arange(hk, dtype=np.uint64)
        z = _mix64(np.uint64(seed) ^ _mix64(at))
    val = lambda b: torch.from_numpy((b & np.uint64(0xFFFFFF)).astype(np.float32) * np.float32(2.0 / 16777216.0) - np.float32(1.0))
    return tuple(val(b).to(DEV).half().double() for b in (z, z >> np.uint64(24)))


def _exact_model(c, s, d):
    T, ctx, hd = c["T"], c["ctx"], s["hd"]
    norm = lambda x, w: x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    r16 = lambda x: x.float().half().double()
    x = d["tok_embd"][torch.from_numpy(d["tokens"]).to(DEV).long()].double()
    # RoPE angles as ggml defines them: the position times theta_scale again and again, in 32 bits
    pos = torch.arange(ctx, ctx + T, device=DEV)
    scale = np.power(np.float32(ROPE_BASE), np.float32(-2.0) / np.float32(hd))
    ang = [np.arange(ctx, ctx + T).astype(np.float32)]
    while len(ang) < hd // 2:
        ang.append(ang[-1] * scale)
    ang = torch.from_numpy(np.stack(ang, 1)).to(DEV).double()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    rope = lambda v: torch.cat([v[..., :hd // 2] * cos - v[..., hd // 2:] * sin, v[..., :hd // 2] * sin + v[..., hd // 2:] * cos], -1)
    trace = torch.full((len(d["layers"]), T, s["k"]), -1, dtype=torch.int32, device=DEV)
    for l, w in enumerate(d["layers"]):
        hn = r16(norm(x, w["attn_norm"]))
        q, k, v = ((hn @ w[m].double().T).view(T, -1, hd) for m in ("wq", "wk", "wv"))
        q, k, v = r16(rope(norm(q, w["q_norm"]))), r16(rope(norm(k, w["k_norm"]))), r16(v)
        kc, vc = (t.view(ctx, s["kv"], hd) for t in _context(l, ctx, s["kv"] * hd, d["kv_seed"]))
        k, v = torch.cat([kc, k]), torch.cat([vc, v])
        hide = torch.arange(ctx + T, device=DEV)[None] > pos[:, None]
        a = torch.empty(T, s["heads"], hd, dtype=torch.float64, device=DEV)
        for i in range(s["heads"]):
            g = i // (s["heads"] // s["kv"])
            sc = (q[:, i] @ k[:, g].T.contiguous()) / math.sqrt(hd)
            a[:, i] = torch.softmax(sc.masked_fill(hide, -math.inf), -1) @ v[:, g]
        x = x + r16(a.view(T, -1)) @ w["wo"].double().T
        if l == len(d["layers"]) - 1:
            x = x[-1:]
        x, trace[l, T - x.shape[0]:], _ = _exact_moe(c, s, d, norm(x, w["ffn_norm"]).float(), w["gate_inp"], x)
    return (r16(norm(x, d["output_norm"])) @ d["tok_embd"].double().T)[0], trace


def exact(case, seed):
    c, s = case, SHAPES[case["shape"]]
    d = _inputs(c, seed)
    if c["kind"] == "model":
        return _exact_model(c, s, d)
    outs = [_exact_moe(c, s, d, d["x"][l], d["router"][l], d["resid"][l]) for l in range(c["layers"])]
    return tuple(torch.stack(v) for v in zip(*outs))
