"""What a user of this framework has it do, as cases that can be timed.

Four kinds of call, each through the public entry points:

* ``linear``: one packed linear at inference, ``PackedLinear(store)(x)``:
  one decoded token (m = 1), a small decode batch, a prompt;
* ``train``: one packed linear in a compressed-state fine-tune step
  (``make_trainable``: fp32 codebook and group scales that learn): its
  forward, and the gradients of the activations, the codebook and the scales;
* ``experts``: the expert-indexed linear of a mixture layer,
  ``PackedExperts(store)(x, ids)``, every token sent to its top-k experts;
* ``decode``: a whole call, ``Decoder.generate(prompt, n_new)``: the prompt
  and the greedy tokens after it of a decoder with random weights.

Sizes are those of the benchmark's configurations (the Llama-3-8B, Qwen3-1.7B
and Qwen3-30B-A3B expert shapes) and of the decoder list in ``epure.decode``.
Weights: uniform indices, sorted N(0, 1) codebook (fp16 values), fp16 group
scales |N(0, 0.02)| + 1e-3; activations N(0, 1); upstream gradients N(0, 1e-2).
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "epure-runtime_amd"))

from epure import PackedExperts, PackedLinear, PackedWeight, make_trainable  # noqa: E402
from epure import decode as ed  # noqa: E402

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ------------------------------------------------------------------ the cases
def _linear(name, bits, m, n, k, dtype="bf16", group=128):
    return {"name": name, "kind": "linear", "bits": bits, "m": m, "n": n, "k": k, "dtype": dtype,
            "group": group}


def _train(name, m, n, k, group=128):
    return {"name": name, "kind": "train", "bits": 4, "m": m, "n": n, "k": k, "dtype": "bf16",
            "group": group}


def _experts(name, bits, tokens, topk, e, n, k, dtype="bf16", group=128):
    return {"name": name, "kind": "experts", "bits": bits, "tokens": tokens, "topk": topk, "e": e,
            "n": n, "k": k, "dtype": dtype, "group": group}


def _decode(name, model, prompt, new):
    return {"name": name, "kind": "decode", "model": model, "prompt": prompt, "new": new}


def listed():
    return [
        # one token through an attention projection of an 8B model: the
        # smallest call, latency and launches
        _linear("token_4096x4096_4bit", 4, 1, 4096, 4096),
        # the same token through a tied packed lm_head (Qwen3-1.7B)
        _linear("token_head_151936x2048_4bit", 4, 1, 151936, 2048, "fp16"),
        # small decode batches of a server, 8-bit and 4-bit weights
        _linear("batch4_14336x4096_8bit", 8, 4, 14336, 4096),
        _linear("batch16_4096x14336_4bit", 4, 16, 4096, 14336, "fp16"),
        # a larger batch, or a short prompt
        _linear("batch64_4096x4096_8bit", 8, 64, 4096, 4096),
        # a prompt of no round length through a decoder of no power-of-two size
        _linear("prompt333_6656x2560_4bit", 4, 333, 6656, 2560),
        # a long prompt (or several at once) through an MLP matrix: the
        # largest linear
        _linear("prompt2048_14336x4096_8bit", 8, 2048, 14336, 4096),
        # fine-tune steps on the MLP matrices of a 1.7B model: a full batch of
        # tokens, and one short ragged sequence
        _train("train2048_6144x2048", 2048, 6144, 2048),
        _train("train201_2048x6144", 201, 2048, 6144),
        # a mixture layer's gate/up matrices for a prompt of 512 tokens
        _experts("experts512_128x768x2048_4bit", 4, 512, 8, 128, 768, 2048),
        # whole calls: a prompt and twice as many greedy tokens
        _decode("generate_llama3_8b", "llama3-8b", 32, 64),
        _decode("generate_qwen3_1.7b", "qwen3-1.7b", 32, 64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more call of the same ranges: rows (tokens) from 1 to 2048, weights
    from 512 x 512 up to the head's size, output widths of any parity for
    inference, prompts and decoders of the list."""
    kind = rng.choice(["linear"] * 6 + ["train"] * 2 + ["experts", "decode"])
    if kind == "linear":
        m = rng.choice([1, 1, _log(rng, 2, 16), _log(rng, 17, 64), _log(rng, 65, 512),
                        _log(rng, 512, 2048)])
        k = 64 * _log(rng, 8, 224)
        n = _log(rng, 512, 16384)
        if rng.random() < 0.7:
            n = n // 64 * 64
        return {"kind": kind, "bits": rng.choice([4, 8]), "m": m, "n": n, "k": k,
                "dtype": rng.choice(["bf16", "bf16", "fp16"]),
                "group": rng.choice([128, 128, 128, 64])}
    if kind == "train":
        return {"kind": kind, "bits": 4, "m": _log(rng, 32, 2048), "n": 128 * _log(rng, 8, 64),
                "k": 128 * _log(rng, 8, 64), "dtype": "bf16",
                "group": rng.choice([128, 128, 64])}
    if kind == "experts":
        return {"kind": kind, "bits": rng.choice([4, 4, 8]), "tokens": _log(rng, 1, 2048),
                "topk": rng.choice([2, 4, 8]), "e": rng.choice([8, 32, 64, 128]),
                "n": 128 * _log(rng, 4, 16), "k": 128 * _log(rng, 8, 24), "dtype": "bf16",
                "group": 128}
    # at most the listed calls' steps, so that none costs more than the largest
    prompt = _log(rng, 4, 32)
    return {"kind": kind, "model": rng.choice(sorted(ed.CONFIGS)), "prompt": prompt,
            "new": _log(rng, 8, 64)}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _raw_weight(g, rows, k, bits, group):
    """(packed, scale, codebook) of a packed weight of ``rows`` x ``k``."""
    packed = torch.randint(0, 256, (rows * k * bits // 8,), generator=g, device=DEV,
                           dtype=torch.uint8)
    cb = torch.sort(torch.randn(16 if bits == 4 else 256, generator=g, device=DEV)).values
    cb = cb.half().float()
    scale = (torch.randn(rows, -(-k // group), generator=g, device=DEV).abs() * 0.02 + 1e-3).half()
    return packed, scale, cb


def _inputs(case, seed):
    """The tensors of a linear, train or experts case."""
    g = _gen(seed)
    dt = DTYPES[case["dtype"]]
    n, k, bits, group = case["n"], case["k"], case["bits"], case["group"]
    if case["kind"] == "experts":
        packed, scale, cb = _raw_weight(g, case["e"] * n, k, bits, group)
        x = torch.randn(case["tokens"], k, generator=g, device=DEV).to(dt)
        x = x.repeat_interleave(case["topk"], 0)
        ids = torch.rand(case["tokens"], case["e"], generator=g, device=DEV) \
            .topk(case["topk"], dim=1).indices.reshape(-1)
        return {"packed": packed, "scale": scale, "cb": cb, "x": x, "ids": ids}
    packed, scale, cb = _raw_weight(g, n, k, bits, group)
    x = torch.randn(case["m"], k, generator=g, device=DEV).to(dt)
    t = {"packed": packed, "scale": scale, "cb": cb, "x": x}
    if case["kind"] == "train":
        t["gy"] = (torch.randn(case["m"], n, generator=g, device=DEV) * 1e-2).to(dt)
    return t


def _weights(case, seed):
    return ed.random_weights(ed.CONFIGS[case["model"]], seed=int(seed), device=DEV)


def _prompt(case, seed):
    g = torch.Generator()
    g.manual_seed(int(seed) + 1)
    return torch.randint(0, ed.CONFIGS[case["model"]].vocab, (case["prompt"],), generator=g).tolist()


def prepare(case, seed):
    if case["kind"] == "decode":
        w = _weights(case, seed)
        # room for the prompt, the new tokens and the next position
        dec = ed.Decoder(w, max_pos=case["prompt"] + case["new"] + 1)
        return {"kind": "decode", "dec": dec, "prompt": _prompt(case, seed), "new": case["new"]}
    t = _inputs(case, seed)
    shape = (case["n"], case["k"])
    levels = 16 if case["bits"] == 4 else 256
    if case["kind"] == "experts":
        store = PackedWeight((case["e"],) + shape, t["packed"], t["scale"], t["cb"], case["group"],
                             levels)
        return {"kind": "experts", "mod": PackedExperts(store), "x": t["x"], "ids": t["ids"]}
    lin = PackedLinear(PackedWeight(shape, t["packed"], t["scale"], t["cb"], case["group"], levels))
    s = {"kind": case["kind"], "mod": lin, "x": t["x"]}
    if case["kind"] == "train":
        make_trainable(lin, "both", verbose=False)
        s["x"].requires_grad_(True)
        s["gy"] = t["gy"]
    return s


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state["kind"]
    if kind == "linear":
        with torch.no_grad():
            return state["mod"](state["x"])
    if kind == "experts":
        with torch.no_grad():
            return state["mod"](state["x"], state["ids"])
    if kind == "train":
        x, lin = state["x"], state["mod"]
        y = lin(x)
        gx, gcb, gsc = torch.autograd.grad(y, (x, lin.store.cb, lin.store.scale), state["gy"])
        return {"y": y.detach(), "grad_x": gx, "grad_cb": gcb, "grad_scale": gsc}
    dec = state["dec"]
    tokens, _ = dec.generate(state["prompt"], state["new"])
    n = len(tokens) - 1
    return {"logits": dec.logits, "k": dec.kcache[:, :, :n], "v": dec.vcache[:, :, :n],
            "tokens": torch.tensor(tokens)}


# ------------------------------------------------------------------ its cost
def _weight_bytes(rows, k, bits, group, scale_bytes=2):
    return rows * k * bits // 8 + rows * -(-k // group) * scale_bytes


def work(case):
    """Weights, inputs and outputs once each, and the products' operations."""
    if case["kind"] == "decode":
        cfg = ed.CONFIGS[case["model"]]
        per = sum(_weight_bytes(n, k, 4, cfg.group) for _, n, k in cfg.packed_linear_shapes())
        params = sum(n * k for _, n, k in cfg.packed_linear_shapes())
        head = cfg.vocab * cfg.hidden
        new, prompt = case["new"], case["prompt"]
        # the prompt's tokens share one read of the weights; a decoded token
        # reads all of them and the cache before it
        passes = new
        kv = 2 * cfg.n_kv * cfg.head_dim * 4 * cfg.layers
        cache = kv * (prompt + sum(prompt + i for i in range(1, new)))
        return {"bytes": passes * (cfg.layers * per + head * 2) + cache,
                "flops": 2 * (prompt + new - 1) * (cfg.layers * params + head)}
    n, k, bits, group = case["n"], case["k"], case["bits"], case["group"]
    if case["kind"] == "experts":
        rows = case["tokens"] * case["topk"]
        used = min(case["e"], rows)
        return {"bytes": used * _weight_bytes(n, k, bits, group) + rows * (k + n) * 2 + rows * 8,
                "flops": 2 * rows * n * k}
    m = case["m"]
    if case["kind"] == "linear":
        return {"bytes": _weight_bytes(n, k, bits, group) + m * (k + n) * 2, "flops": 2 * m * n * k}
    # forward, gradient of the activations, and the weight gradient that the
    # codebook and scale gradients reduce
    sc = n * -(-k // group) * 4
    return {"bytes": 2 * (n * k * bits // 8 + sc) + sc + 2 * m * (2 * k + 2 * n), "flops": 6 * m * n * k}


def tolerance(case):
    """About four times the largest error against 64 bits that was measured
    over the listed and drawn cases (in brackets)."""
    if case["kind"] == "decode":
        # float32 semantics throughout, some thirty layers deep (1.9e-6)
        return {"rel": 8e-6, "max": 3e-4, "differ": 0.0}
    if case["kind"] == "train":
        # 16-bit y and grad_x (1.7e-3); the fp32 sums stay within 4e-7
        return {"rel": 7e-3, "max": 0.05}
    if case["dtype"] == "fp16":
        # fp16 outputs and weights rounded to fp16 (2.9e-4)
        return {"rel": 1.2e-3, "max": 0.02}
    return {"rel": 7e-3, "max": 0.05}  # bf16 outputs (1.8e-3)


# ------------------------------------------------------------------ 64 bits
def _dense(packed, scale, cb, rows, k, group):
    """cb[idx] * scale in float64, ``[rows, k]``."""
    if cb.numel() <= 16:
        idx = torch.stack((packed & 15, packed >> 4), dim=-1).reshape(rows, k)
    else:
        idx = packed.reshape(rows, k)
    w = cb.double()[idx.long()]
    s = scale.double().repeat_interleave(group, dim=1)[:, :k]
    return w.mul_(s)


def _exact_train(t, case):
    n, k, group = case["n"], case["k"], case["group"]
    w = _dense(t["packed"], t["scale"], t["cb"], n, k, group)
    x, gy = t["x"].double(), t["gy"].double()
    y, gx = x @ w.T, gy @ w
    del w
    gw = gy.T.contiguous() @ x
    idx = torch.stack((t["packed"] & 15, t["packed"] >> 4), dim=-1).reshape(n, k).long()
    ng = -(-k // group)
    s = t["scale"].double().repeat_interleave(group, dim=1)[:, :k]
    gcb = torch.zeros(16, device=DEV, dtype=torch.float64)
    gws = gw * s
    for level in range(16):
        gcb[level] = torch.where(idx == level, gws, torch.zeros_like(gws)).sum()
    gsc = gw.mul_(t["cb"].double()[idx])
    gsc = torch.nn.functional.pad(gsc, (0, ng * group - k)).view(n, ng, group).sum(-1)
    return {"y": y, "grad_x": gx, "grad_cb": gcb, "grad_scale": gsc}


def _norm(v, w, eps):
    return v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps) * w.double()


def _rope(v, pos, theta):
    # the angles are the model's own float32 values
    d = v.shape[-1]
    inv = 1.0 / (theta ** (torch.arange(0, d, 2).float() / d))
    ang = (pos.float()[:, None] * inv[None]).to(DEV).float()
    c, s = ang.cpu().cos().double().to(DEV), ang.cpu().sin().double().to(DEV)
    a, b = v[..., :d // 2], v[..., d // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _exact_decode(case, seed):
    w, cfg = _weights(case, seed), ed.CONFIGS[case["model"]]
    D, hq, hkv = cfg.head_dim, cfg.n_heads, cfg.n_kv
    ids, n_new = _prompt(case, seed), case["new"]
    ks = [torch.zeros(hkv, 0, D, dtype=torch.float64, device=DEV) for _ in w.layers]
    vs = [k.clone() for k in ks]
    dense = {}

    def weight(li, name):
        # the small models' float64 weights are kept from token to token; the
        # large ones' (8 bytes a weight) fit the card too
        if (li, name) not in dense:
            s = w.layers[li].lin[name]
            dense[li, name] = _dense(s.packed, s.scale, s.cb, s.out_features, s.in_features, s.group)
        return dense[li, name]

    head = w.lm_head.double()
    tokens, fresh, logits = list(ids), list(ids), None
    for step in range(n_new):
        base = ks[0].shape[1]
        t = len(fresh)
        pos = torch.arange(base, base + t)
        h = w.embed[torch.tensor(fresh, device=DEV)].double()
        seen = torch.arange(base + t, device=DEV)[None] <= pos.to(DEV)[:, None]
        for li, L in enumerate(w.layers):
            a = _norm(h, L.attn_norm, cfg.rms_eps)
            q = (a @ weight(li, "q").T).view(t, hq, D).transpose(0, 1)
            k = (a @ weight(li, "k").T).view(t, hkv, D).transpose(0, 1)
            v = (a @ weight(li, "v").T).view(t, hkv, D).transpose(0, 1)
            if L.q_norm is not None:
                q, k = _norm(q, L.q_norm, cfg.rms_eps), _norm(k, L.k_norm, cfg.rms_eps)
            q, k = _rope(q, pos, cfg.rope_theta), _rope(k, pos, cfg.rope_theta)
            ks[li] = torch.cat((ks[li], k), 1)
            vs[li] = torch.cat((vs[li], v), 1)
            kk = ks[li].repeat_interleave(hq // hkv, 0)
            vv = vs[li].repeat_interleave(hq // hkv, 0)
            p = torch.matmul(q, kk.transpose(1, 2).contiguous()) / math.sqrt(D)
            p = p.masked_fill(~seen, float("-inf")).softmax(-1)
            o = torch.matmul(p, vv).transpose(0, 1).reshape(t, hq * D)
            h = h + o @ weight(li, "o").T
            a = _norm(h, L.mlp_norm, cfg.rms_eps)
            g = a @ weight(li, "gate").T
            h = h + (g * torch.sigmoid(g) * (a @ weight(li, "up").T)) @ weight(li, "down").T
        logits = (_norm(h[-1:], w.final_norm, cfg.rms_eps) @ head.T)[0]
        fresh = [int(logits.argmax())]
        tokens += fresh
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs), "tokens": None}


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "decode":
            return _exact_decode(case, seed)
        t = _inputs(case, seed)
        if case["kind"] == "train":
            return _exact_train(t, case)
        n, k, group = case["n"], case["k"], case["group"]
        if case["kind"] == "linear":
            w = _dense(t["packed"], t["scale"], t["cb"], n, k, group)
            return t["x"].double() @ w.T
        y = torch.empty(t["x"].shape[0], n, dtype=torch.float64, device=DEV)
        rb = n * k * case["bits"] // 8
        for e in range(case["e"]):
            rows = (t["ids"] == e).nonzero().reshape(-1)
            if rows.numel():
                w = _dense(t["packed"][e * rb:(e + 1) * rb], t["scale"][e * n:(e + 1) * n], t["cb"], n, k,
                           group)
                y[rows] = t["x"][rows].double() @ w.T
        return y
