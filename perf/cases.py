"""The work whose speed this repository is held to, through the package's public entry points.

Six kinds of work, each over a range of sizes (`draw`), of which `listed` holds the usual ones:

  train    one LoRA step (forward, loss, backward, clipping, AdamW): 16 .. 2048 rows in 1 .. 8 sequences of any length, Qwen3 and
           Gemma3 widths and the tiny shape, F16 and Q8_0 weights, 1 .. 36 layers
  policy   the update half of a GRPO step on all parameters: groups of 2 .. 8 completions of ragged lengths
  prompt   a prompt of 8 .. 768 tokens into an empty cache, logits of its last token, F16 and Q8_0
  reply    one sequence token by token, with the logits of every token on the host (a caller that samples) or with the
           argmax from the GPU (greedy), behind a short prompt
  batch    2 .. 32 sequences in lock step, each with its own token, logits of every step
  layered  a prompt of 16 .. 2048 tokens and some further tokens on models whose layers are listed one by one

Widths are those of the package's configurations (configs.py).  Where a case holds fewer layers than the model, the vocabulary
is cut too, so that the head keeps about its share of the weights.  Weights are random: one pool of normal values per state,
of which every matrix is a window at a place of its own, rounded so that F16 (or Q8_0) holds the values exactly.
"""
import math
import os
import tempfile

import numpy as np
import torch

from llm_metal_amd import configs, synth
from llm_metal_amd.sft import InferenceState, SFTState

BASES = {"tiny": configs.C1, "gemma3_1b": configs.C2, "qwen3_4b": configs.C3}
LAYERED = {"nevurax_1k": configs.NEVURAX_SIZES["1k"], "paposun_1k": configs.PAPOSUN_SIZES["1k"], "paposun_2k": configs.PAPOSUN_SIZES["2k"]}
LR = 1e-4
POLICY_LR = 3e-4


def listed():
    quarter = {"model": "qwen3_4b", "layers": 9, "vocab": 32768}           # a quarter of the layers, head in proportion
    return [
        # fine-tuning a model small enough that launches and waits are all there is
        {"name": "train_tiny_1x64", "kind": "train", "model": "tiny", "layers": 2, "vocab": 4096, "format": "f16", "batch": 1, "seq": 64},
        # the two steps the reference publishes rates for, whole models
        {"name": "train_gemma3_1b_1x64", "kind": "train", "model": "gemma3_1b", "layers": 26, "vocab": 262144, "format": "f16", "batch": 1, "seq": 64},
        {"name": "train_qwen3_4b_1x64", "kind": "train", "model": "qwen3_4b", "layers": 36, "vocab": 151936, "format": "f16", "batch": 1, "seq": 64},
        # one example of everyday length, ragged against every tile
        {"name": "train_qwen3_4b_1x250", "kind": "train", "format": "f16", "batch": 1, "seq": 250, **quarter},
        # a full batch on quantised weights, whole model: the largest case
        {"name": "train_qwen3_4b_q8_4x512", "kind": "train", "model": "qwen3_4b", "layers": 36, "vocab": 151936, "format": "q8_0", "batch": 4, "seq": 512},
        # GRPO on all parameters: four sampled completions of one prompt
        {"name": "policy_gemma3_1b_4x160", "kind": "policy", "model": "gemma3_1b", "layers": 8, "vocab": 262144, "group": 4, "prompt": 32, "completion": 128},
        # reading a document before the first token comes out
        {"name": "prompt_qwen3_4b_500", "kind": "prompt", "format": "f16", "tokens": 500, **quarter},
        # sampling a completion on the CPU: a short question and an answer
        {"name": "reply_qwen3_4b", "kind": "reply", "format": "f16", "tokens": 32, "steps": 48, "greedy": False, **quarter},
        # greedy decoding on quantised weights, whole model
        {"name": "greedy_gemma3_1b_q8", "kind": "reply", "model": "gemma3_1b", "layers": 26, "vocab": 262144, "format": "q8_0", "tokens": 1, "steps": 128, "greedy": True},
        # sampling a group of completions together
        {"name": "batch8_qwen3_4b", "kind": "batch", "format": "f16", "batch": 8, "steps": 40, **quarter},
        # models described layer by layer: a long prompt, a short one with an answer
        {"name": "layered_nevurax_1k_2000", "kind": "layered", "model": "nevurax_1k", "tokens": 2000, "steps": 4},
        {"name": "layered_paposun_2k_300", "kind": "layered", "model": "paposun_2k", "tokens": 300, "steps": 32},
    ]


def _log_uniform(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(("train", "train", "policy", "prompt", "reply", "batch", "layered"))
    if kind == "layered":
        return {"kind": kind, "model": rng.choice(sorted(LAYERED)), "tokens": _log_uniform(rng, 16, 2048), "steps": rng.randint(1, 32)}
    if kind == "policy":
        return {"kind": kind, "model": "gemma3_1b", "layers": rng.randint(2, 8), "vocab": 4 * rng.randint(8192, 65536), "group": rng.randint(2, 8),
                "prompt": rng.randint(8, 64), "completion": rng.randint(16, 128)}
    model = rng.choice(("gemma3_1b", "qwen3_4b", "qwen3_4b"))
    layers = rng.randint(3, 9)
    c = {"kind": kind, "model": model, "layers": layers, "vocab": 4 * rng.randint(2048, 2048 * layers), "format": rng.choice(("f16", "f16", "q8_0"))}
    if kind == "train":
        if rng.random() < 0.15:
            c.update(model="tiny", layers=rng.randint(1, 4), vocab=4 * rng.randint(512, 2048))
        c["batch"] = rng.choice((1, 1, 2, 4, 8))
        c["seq"] = max(8, min(1024, _log_uniform(rng, 16, 2048) // c["batch"]))
    elif kind == "prompt":
        c["tokens"] = _log_uniform(rng, 8, 768)
    elif kind == "reply":
        c.update(tokens=_log_uniform(rng, 1, 128), steps=rng.randint(8, 48), greedy=rng.random() < 0.5)
    else:
        c.update(format="f16", batch=_log_uniform(rng, 2, 32), steps=rng.randint(8, 40))
    return c


# ---------------------------------------------------------------- inputs

def _config(case):
    kw = {"NL": case["layers"], "V": case["vocab"], "weight_format": case.get("format", "f16")}
    if case["kind"] == "train":
        kw.update(batch=case["batch"], seq=case["seq"])
    elif case["kind"] == "policy":
        kw.update(batch=case["group"], seq=case["prompt"] + case["completion"], R=0)
    return BASES[case["model"]].with_(name=case["kind"], **kw)


class _Weights:
    """The matrices of a model as windows of one pool: `matrix` gives the place of each.  Places are multiples of 32 (a
    block of Q8_0) and none of them a multiple of a row, so no two matrices share rows."""

    def __init__(self, c, seed):
        self.c, emb, self.sizes = c, c.V * c.D, synth.mat_shapes(c)
        largest = max(r * k for r, k in self.sizes.values())
        n = max(emb, largest) + (1 << 22)
        n += -n % 32
        self.span, self.head_at = n, (1 << 21) + 1312
        self.head_at += 32 if self.head_at % c.D == 0 else 0
        g = torch.Generator("cuda").manual_seed(1_000_003 * seed + 17)
        x = torch.randn(n, generator=g, device="cuda").mul_(0.02)
        if c.weight_format == "q8_0":                     # blocks of 32: int8 codes times a scale that is a half
            b = x.view(-1, 32)
            d = (b.abs().amax(1, keepdim=True) / 127.0).half().float()
            x = (b / d).round_().clamp_(-127, 127).mul_(d).view(-1)
        else:
            x = x.half().float()
        self.pool = x
        r = torch.Generator("cuda").manual_seed(1_000_003 * seed + 29)
        self.gammas = {}
        for key, dim in (("g_in", c.D), ("g_post_attn", c.D), ("g_pre_ff", c.D), ("g_post_ff", c.D), ("g_q", c.hd), ("g_k", c.hd)):
            self.gammas[key] = 1.0 + 0.1 * torch.randn(c.NL, dim, generator=r, device="cuda")
        self.g_final = 1.0 + 0.1 * torch.randn(c.D, generator=r, device="cuda")
        qd, kd = c.Hq * c.hd, c.Hkv * c.hd
        lora = []
        for _ in range(c.NL if c.R else 0):
            for rows, cols, down in ((c.R, c.D, True), (qd, c.R, False), (c.R, c.D, True), (kd, c.R, False)):
                a = torch.rand(rows * cols, generator=r, device="cuda") * 2 - 1
                lora.append(a / math.sqrt(c.D) if down else torch.randn(rows * cols, generator=r, device="cuda") * 0.01)
        self.lora = torch.cat(lora) if lora else torch.zeros(0, device="cuda")

    def matrix(self, pool, layer, key):
        rows, cols = self.sizes[key]
        n = rows * cols
        at = (layer * 7 + list(self.sizes).index(key)) * 12_582_944 % (self.span - n + 32) // 32 * 32
        return pool[at:at + n].reshape(rows, cols)

    def embedding(self, pool):
        return pool[:self.c.V * self.c.D].reshape(self.c.V, self.c.D)

    def head(self, pool):
        at = 0 if self.c.tied else self.head_at
        return pool[at:at + self.c.V * self.c.D].reshape(self.c.V, self.c.D)

    def model(self):
        """The dictionary of host arrays that the package's states are created from."""
        c, pool = self.c, self.pool.cpu().numpy()
        m = {k: [self.matrix(pool, L, k) for L in range(c.NL)] for k in self.sizes}
        m["token_emb"] = self.embedding(pool)
        m["lm_head"] = m["token_emb"] if c.tied else self.head(pool)
        for k, g in self.gammas.items():
            gemma_only = k in ("g_pre_ff", "g_post_ff") and c.model_type != configs.GEMMA3
            m[k] = [None] * c.NL if gemma_only else list(g.cpu().numpy())
        m["g_final"] = self.g_final.cpu().numpy()
        m["lora"] = self.lora.cpu().numpy()
        return m


def _tokens(case, seed):
    """Token ids of a case, uniform over the vocabulary."""
    rng = np.random.default_rng([seed, 5])
    kind = case["kind"]
    if kind == "layered":
        shape, V = case["tokens"] + case["steps"], LAYERED[case["model"]]["vocab"]
    else:
        V = case["vocab"]
        shape = {"train": lambda: (case["batch"], case["seq"]), "policy": lambda: (case["group"], case["prompt"] + case["completion"]),
                 "prompt": lambda: case["tokens"], "reply": lambda: case["tokens"] + case["steps"],
                 "batch": lambda: (case["batch"], case["steps"])}[kind]()
    t = rng.integers(0, V, size=shape, dtype=np.int64)
    if kind == "policy":
        t[:, :case["prompt"]] = t[0, :case["prompt"]]
    return t


def _group(case, seed, w):
    """Completions of a group: lengths, advantages, and log-probabilities as the sampling policy had them (a little off)."""
    rng = np.random.default_rng([seed, 6])
    c, t = w.c, _tokens(case, seed)
    P, L = case["prompt"], case["completion"]
    lens = rng.integers(L - L // 4, L + 1, size=case["group"])
    adv = rng.standard_normal(case["group"])
    adv = ((adv - adv.mean()) / (adv.std() + 1e-6)).astype(np.float32)
    valid = np.arange(c.seq)[None, :] < P + lens[:, None]
    action = np.where(valid & (np.arange(c.seq)[None, :] >= P), t, 0)
    with torch.no_grad():
        logits = _decoder64(c, w, torch.from_numpy(t).cuda(), rows=torch.from_numpy(valid).cuda())
        lp = (logits.gather(-1, torch.from_numpy(action).cuda()[..., None])[..., 0] - logits.logsumexp(-1)).cpu().numpy()
    old = (lp + 0.05 * rng.standard_normal(lp.shape)).astype(np.float32)
    return t, lens, adv, action, valid, old


def _layered_weights(case, seed):
    """Every tensor of a layer-by-layer model, bfloat16 on the GPU, with the spreads the package's own random models have."""
    g = torch.Generator("cuda").manual_seed(1_000_003 * seed + 41)
    out = {}
    for name, shape in synth.stack_shapes(LAYERED[case["model"]]).items():
        leaf = name.rsplit(".", 1)[-1]

        def normal():
            return torch.randn(shape, generator=g, device="cuda")

        def uniform(low, high):
            return low + (high - low) * torch.rand(shape, generator=g, device="cuda")
        if leaf in ("norm", "norm1", "norm1b", "norm2", "norm2b"):
            x = 1.0 + 0.1 * normal()
        elif leaf == "b" and len(shape) == 1:
            x = uniform(1.0, 6.0) if name.endswith(".f.b") else 0.3 * normal()
        elif leaf == "conv":
            x = normal() / math.sqrt(shape[1])
        elif leaf == "A_log":
            x = uniform(-3.0, 0.5)
        elif leaf == "dt_bias":
            x = uniform(-3.0, 0.0)
        elif leaf == "embed":
            x = normal()
        else:
            x = normal() * ((0.5 if leaf in ("down", "o") else 1.0) / math.sqrt(shape[-1]))
        out[name] = x.bfloat16()
    return out


def _write_checkpoint(folder, cfg, weights):
    import json
    import struct
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump(cfg, f)
    header, at = {}, 0
    for name, x in weights.items():
        header[name] = {"dtype": "BF16", "shape": list(x.shape), "data_offsets": [at, at + 2 * x.numel()]}
        at += 2 * x.numel()
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(folder, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        f.write(torch.cat([x.reshape(-1) for x in weights.values()]).view(torch.int16).cpu().numpy())


class _Owner:
    """Frees a state of the package with the last reference to it."""

    def __init__(self, state):
        self.state = state

    def __del__(self):
        self.state.free()


class _DeviceArray:
    """A device buffer of a state, for torch to look at in place; keeps the state alive."""

    def __init__(self, owner, pointer, shape, kind):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (int(pointer), False), "version": 2}


def _view(owner, pointer, shape, kind="<f4"):
    return torch.as_tensor(_DeviceArray(owner, pointer, shape, kind), device="cuda")


def prepare(case, seed):
    kind, t = case["kind"], _tokens(case, seed)
    if kind == "layered":
        with tempfile.TemporaryDirectory() as folder:
            _write_checkpoint(folder, LAYERED[case["model"]], _layered_weights(case, seed))
            st = InferenceState(path=folder, model_type=None, max_seq=len(t), weight_format="f16")
        return {"kind": kind, "owner": _Owner(st), "prompt": t[:case["tokens"]], "rest": [int(i) for i in t[case["tokens"]:]],
                "rows": np.zeros((1 + case["steps"], st.V), np.float32)}
    c = _config(case)
    w = _Weights(c, seed)
    if kind == "train":
        st = SFTState(c, w.model())
        owner, L = _Owner(st), st.L
        logits = _view(owner, L.hip_buf_device_ptr(L.sft_get_logits(st.h)), (c.BN, c.V))
        adapters = _view(owner, L.hip_buf_device_ptr(L.sft_get_lora_weight_buf(st.h, 0, 0)), (L.sft_lora_numel(st.h),))
        return {"kind": kind, "owner": owner, "tok": t.astype(np.uint32).reshape(-1), "tgt": np.roll(t, -1, 1).astype(np.uint32).reshape(-1),
                "logits": logits, "adapters": adapters}
    if kind == "policy":
        t, lens, adv, action, _, old = _group(case, seed, w)
        st = SFTState(c, w.model())
        P = case["prompt"]
        return {"kind": kind, "owner": _Owner(st), "prompt": t[0, :P].astype(np.uint32), "adv": adv,
                "gen": [t[i, P:P + n].astype(np.uint32) for i, n in enumerate(lens)], "old": [old[i, P:P + n].copy() for i, n in enumerate(lens)]}
    length = {"prompt": lambda: case["tokens"], "reply": lambda: case["tokens"] + case["steps"], "batch": lambda: case["steps"]}[kind]()
    st = InferenceState(c, w.model(), max_seq=length, use_fp16=c.weight_format == "f16")
    s = {"kind": kind, "owner": _Owner(st)}
    if kind == "batch":
        s["steps"] = [np.ascontiguousarray(t[:, i], dtype=np.int32) for i in range(case["steps"])]
    else:
        s.update(prompt=t[:case["tokens"]].astype(np.int32), greedy=case.get("greedy", False), rest=[int(i) for i in t[case["tokens"]:]])
        s["rows"] = np.zeros((1 if s["greedy"] else 1 + len(s["rest"]), c.V), np.float32)
    return s


# ---------------------------------------------------------------- one pass

def _weight_views(owner):
    """The weights of a training state as it hands them out (row-major F16), matrix by matrix."""
    st = owner.state
    L, out = st.L, {}
    layers = L.sft_get_layers(st.h)
    head = L.sft_get_lm_head(st.h).contents
    L.metal_flush()
    for i in range(st.c.NL):
        for k, field in zip(synth.MATS, ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")):
            m = getattr(layers[i], field).contents
            out[f"{k}{i}"] = _view(owner, L.hip_buf_device_ptr(m.mbuf), (m.rows, m.cols), "<f2")
    out["head"] = _view(owner, L.hip_buf_device_ptr(head.mbuf), (head.rows, head.cols), "<f2")
    return out


def run(s):
    st, kind = s["owner"].state, s["kind"]
    if kind == "train":
        st.train_step(s["tok"], s["tgt"], LR)
        return {"losses": st.losses(), "logits": s["logits"], "adapters": s["adapters"]}
    if kind == "policy":
        lp = st.grpo_apply_completions(s["prompt"], s["gen"], s["old"], s["adv"], 0.2, POLICY_LR)
        return {"logprobs": lp, "weights": _weight_views(s["owner"])}
    if kind == "batch":
        return [st.step_batch(t, i) for i, t in enumerate(s["steps"])]
    st.reset()
    first = st.forward_tokens(s["prompt"], [len(s["prompt"]) - 1])
    if kind == "prompt":
        return first
    if s.get("greedy"):
        ids = [st.forward_token_argmax(t) for t in s["rest"][:-1]]
        return {"first": first, "ids": np.asarray(ids, np.int64), "last": st.forward_token(s["rest"][-1])}
    rows = s["rows"]                                      # where the caller keeps the logits it samples from
    rows[0] = first[0]
    for i, t in enumerate(s["rest"]):
        rows[1 + i] = st.forward_token(t)
    return rows


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    if kind == "layered":
        cfg = LAYERED[case["model"]]
        n, steps, D, V = case["tokens"], case["steps"], cfg["width"], cfg["vocab"]
        every = active = pairs = 0
        for name, shape in synth.stack_shapes(cfg).items():
            if len(shape) == 2 and name not in ("embed", "head") and ".conv" not in name:
                size = shape[0] * shape[1]
                share = 1.0
                if ".e" in name:
                    r = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
                    share = r["top"] / r["experts"]
                every, active = every + size, active + size * share
        for L in cfg["layers"]:
            m = L["mixer"]
            seen = min(n, m["mask"]["size"]) / 2 if "mask" in m else 2 * m["dim"]
            pairs += m["heads"] * n * seen * 2 * (m["dim"] + m["vdim"] + m.get("rot_dim", 0))
        return {"bytes": 2.0 * (every + steps * active + (1 + steps) * V * D) + 4.0 * (n + steps) * D, "flops": 2.0 * (n + steps) * active + 2.0 * (1 + steps) * V * D + pairs}
    c = _config(case)
    per = {"f16": 2.0, "q8_0": 34.0 / 32.0}[c.weight_format]
    P, head = c.frozen_params, c.V * c.D

    def attention(rows, length):                          # scores and weighted values, causal
        return rows * length * c.Hq * c.hd * 2.0 * c.NL
    if kind == "train":
        return {"bytes": 2 * per * P + 8.0 * c.BN * c.V + 24.0 * c.NL * c.lora_layer_size, "flops": 4.0 * c.BN * P + 3 * attention(c.BN, c.seq)}
    if kind == "policy":
        return {"bytes": 22.0 * P, "flops": 6.0 * c.BN * P + 3 * attention(c.BN, c.seq)}
    if kind == "batch":
        n = case["steps"]
        return {"bytes": n * per * P + 4.0 * n * case["batch"] * c.V, "flops": 2.0 * n * case["batch"] * P + attention(n * case["batch"], n)}
    n, steps = case["tokens"], case.get("steps", 0)
    return {"bytes": (1 + steps) * per * P + 8.0 * n * c.NL * c.Hkv * c.hd, "flops": 2.0 * (n + steps) * (P - head) + 2.0 * (1 + steps) * head + attention(n + steps, n + steps)}


def tolerance(case):
    """About four times what the present code is off the 64-bit results; where a sampled id is returned, room for one tie."""
    kind = case["kind"]
    if kind == "train":                                   # F16 operands: logits 3e-3 off at 36 layers; AdamW's first step turns on the sign of small gradients
        return {"rel": 1.2e-2, "max": 0.2}
    if kind == "policy":                                  # weights rounded to F16: 2e-4
        return {"rel": 1e-3, "max": 0.05}
    if kind == "layered":                                 # F16 operands: 4e-4; a router near a tie may choose the other expert
        return {"rel": 1e-2, "max": 0.3}
    return {"rel": 6e-5, "max": 1e-3, "differ": 0.01}     # F16 or Q8_0 weights, everything else in 32 bits: 7e-6 at 500 tokens


# ---------------------------------------------------------------- the same in 64 bits

def _rms(x, g, eps=1e-6):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * g


def _gelu(x):
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _rope(x, theta):
    """[B, N, heads, hd], entry i turned together with entry i + hd / 2."""
    N, hd = x.shape[1], x.shape[3]
    f = theta ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=x.device) / hd)
    a = torch.arange(N, dtype=torch.float64, device=x.device)[:, None] * f
    cos, sin = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)


def _attend(q, k, v, scale, mask):
    """[B, N, heads, hd] each, as many key heads as query heads; mask [N, N] of what a query sees."""
    s = torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1).contiguous()) * scale
    return torch.matmul(s.masked_fill(~mask, -math.inf).softmax(-1), v.transpose(1, 2).contiguous()).transpose(1, 2)


def _decoder64(c, w, tok, lora=None, params=None, rows=None, keep=None):
    """Logits [B, N, V] (or those at the places `keep`) of tokens [B, N]; lora: flat adapters; params: weights in place of
    the pool's; rows [B, N]: False where a row is all zeros instead of a token's."""
    gemma = c.model_type == configs.GEMMA3
    get = (lambda L, k: params[f"{k}{L}"]) if params else (lambda L, k: w.matrix(w.pool, L, k).double())
    B, N = tok.shape
    x = w.embedding(w.pool)[tok].double() * (float(np.float32(math.sqrt(c.D))) if gemma else 1.0)
    if rows is not None:
        x = x * rows[..., None]
    at = 0
    mask = torch.ones(N, N, dtype=torch.bool, device=x.device).tril()
    for L, theta in enumerate(c.rope_thetas()):
        g = {k: v[L].double() for k, v in w.gammas.items()}
        h = _rms(x, g["g_in"])
        q, k, v = (h @ get(L, m).T for m in ("wq", "wk", "wv"))
        if lora is not None:
            part = []
            for r, n in ((c.R, c.D), (c.Hq * c.hd, c.R), (c.R, c.D), (c.Hkv * c.hd, c.R)):
                part.append(lora[at:at + r * n].view(r, n))
                at += r * n
            q = q + c.lora_scaling * (h @ part[0].T) @ part[1].T
            v = v + c.lora_scaling * (h @ part[2].T) @ part[3].T
        q = _rope(_rms(q.view(B, N, c.Hq, c.hd), g["g_q"]), theta)
        k = _rope(_rms(k.view(B, N, c.Hkv, c.hd), g["g_k"]), theta)
        n = c.Hq // c.Hkv
        o = _attend(q, k.repeat_interleave(n, 2), v.view(B, N, c.Hkv, c.hd).repeat_interleave(n, 2), c.hd ** -0.5, mask)
        o = o.reshape(B, N, -1) @ get(L, "wo").T
        x = x + (_rms(o, g["g_post_attn"]) if gemma else o)
        h = _rms(x, g["g_pre_ff"] if gemma else g["g_post_attn"])
        a = h @ get(L, "wg").T
        a = (_gelu(a) if gemma else a * torch.sigmoid(a)) * (h @ get(L, "wu").T)
        a = a @ get(L, "wd").T
        x = x + (_rms(a, g["g_post_ff"]) if gemma else a)
    x = _rms(x if keep is None else x[:, keep], w.g_final.double())
    return x @ (params["head"] if params else w.head(w.pool).double()).T


def _nevurax64(cfg, W, tok, keep):
    eps = cfg["norm"]["eps"]

    def layer_norm(x, g):
        d = x - x.mean(-1, keepdim=True)
        return d * torch.rsqrt((d * d).mean(-1, keepdim=True) + eps) * g
    x = W["embed"][tok] * cfg["embedding"]["scale"]
    T, dev = len(tok), x.device
    at = torch.arange(T, device=dev)
    for i, L in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", L["mixer"]
        h = layer_norm(x, W[f"l{i}.norm1"])
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        if L["type"] == "latent_attention":
            r, R = m["rot_dim"], m["kv_rank"]
            dims = m["rot"]["dims"]
            f = m["rot"]["base"] ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=dev) / dims)
            cos, sin = (at[:, None] * f).cos()[:, None], (at[:, None] * f).sin()[:, None]

            def turn(y):                                  # neighbours (2i, 2i + 1) together
                u, v = y[..., 0:dims:2], y[..., 1:dims:2]
                return torch.cat([torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2), y[..., dims:]], -1)
            q = (h @ W[p + "q"].T).view(T, H, d + r)
            low = h @ W[p + "dkv"].T
            c = _rms(low[:, :R], W[p + "dkv.norm"], eps)
            kr = turn(low[:, None, R:]).expand(T, H, r)
            k = torch.cat([(c @ W[p + "uk"].T).view(T, H, d), kr], -1)
            v = (c @ W[p + "uv"].T).view(T, H, dv)
            q = torch.cat([q[..., :d], turn(q[..., d:])], -1)
            seen = (at[None, :] <= at[:, None]) & (at[:, None] - at[None, :] < m["mask"]["size"])
            o = _attend(q[None], k[None], v[None], m["scale"], seen)[0].reshape(T, -1)
        else:
            KV, n = m["kv_heads"], m["conv"]

            def conv(key):
                y = torch.cat([x.new_zeros(n - 1, W[p + key].shape[0]), h @ W[p + key].T])
                y = sum(y[j:j + T] * W[p + key + ".conv"][:, j] for j in range(n))
                return y * torch.sigmoid(y)

            def unit(y):
                return y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6)
            q = (unit(conv("q").view(T, KV, d)) / math.sqrt(d)).repeat_interleave(H // KV, 1)
            k = unit(conv("k").view(T, KV, d)).repeat_interleave(H // KV, 1)
            v, beta = conv("v").view(T, H, dv), torch.sigmoid(h @ W[p + "b"].T)
            rate = W[p + "A_log"].exp()
            if L["type"] == "channel_delta":
                a = torch.nn.functional.softplus(h @ W[p + "a1"].T @ W[p + "a2"].T + W[p + "dt_bias"], threshold=1e9).view(T, H, d)
                g = torch.exp(-rate[:, None] * a)[..., None]
                gate = torch.sigmoid(h @ W[p + "g1"].T @ W[p + "g2"].T)
            else:
                a = torch.nn.functional.softplus(h @ W[p + "a"].T + W[p + "dt_bias"], threshold=1e9)
                g = torch.exp(-rate * a)[..., None, None]
                gate = h @ W[p + "g"].T
                gate = gate * torch.sigmoid(gate)
            S, o = x.new_zeros(H, d, dv), x.new_zeros(T, H, dv)
            for t in range(T):
                S = S * g[t]
                u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
                S = S + k[t][:, :, None] * u[:, None, :]
                o[t] = (S * q[t][:, :, None]).sum(1)
            o = _rms(o, W[p + "norm"], eps).reshape(T, -1) * gate
        y = o @ W[p + "o"].T
        if L.get("mlp"):
            p, m = f"l{i}.mlp.", L["mlp"]
            best, who = (h @ W[p + "router"].T).softmax(-1).topk(m["router"]["top"], -1)
            for e in range(m["router"]["experts"]):
                row, place = (who == e).nonzero(as_tuple=True)
                if len(row):
                    a = (h[row] @ W[f"{p}e{e}.up"].T).clamp_min(0)
                    y = y.index_add(0, row, (a * a) @ W[f"{p}e{e}.down"].T * best[row, place][:, None])
            if m.get("shared"):
                a = (h @ W[p + "shared.up"].T).clamp_min(0)
                y = y + (a * a) @ W[p + "shared.down"].T
        x = x + y
    return layer_norm(x[keep], W["final.norm"]) @ W["head"].T


def _paposun64(cfg, W, tok, keep):
    eps, mult = cfg["norm"]["eps"], cfg["residual_mult"]
    x = W["embed"][tok]
    T, dev, caches = len(tok), x.device, {}
    at = torch.arange(T, device=dev)

    def linear(name, h):
        return h @ W[name].T + W[name + ".b"]
    for i, L in enumerate(cfg["layers"]):
        p, m = f"l{i}.mix.", L["mixer"]
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        h = _rms(x, W[f"l{i}.norm1"], eps)
        if L["type"] == "attention":
            rot, G = m["rot"], m["kv_heads"]
            f = rot["base"] ** (-torch.arange(0, rot["dims"], 2, dtype=torch.float64, device=dev) / rot["dims"])
            sc = rot.get("scaling")
            if sc:                                        # long wavelengths stretched, short ones kept, a mix in between
                mix = ((sc["original"] * f / (2 * math.pi) - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
                f = f * (mix + (1 - mix) / sc["factor"])
            cos, sin = (at[:, None] * f).cos()[:, None], (at[:, None] * f).sin()[:, None]

            def turn(y):
                n = rot["dims"] // 2
                u, v = y[..., :n], y[..., n:2 * n]
                return torch.cat([u * cos - v * sin, v * cos + u * sin, y[..., 2 * n:]], -1)
            q = turn(linear(p + "q", h).view(T, H, d))
            if m.get("kv_from") is None:
                caches[i] = turn(linear(p + "k", h).view(T, G, d)), linear(p + "v", h).view(T, G, dv)
            k, v = (y.repeat_interleave(H // G, 1) for y in caches[i if m.get("kv_from") is None else m["kv_from"]])
            size = m["mask"]["size"]
            seen = (at[None, :] <= at[:, None]) & (at[None, :] // size == at[:, None] // size)
            o = _attend(q[None], k[None], v[None], m["scale"], seen)[0].reshape(T, -1)
            y = linear(p + "o", o * torch.sigmoid(h @ W[p + "g"].T))
        else:
            cap = m["gate_cap"]
            q = (h @ W[p + "q"].T).view(T, H, d) * d ** -0.5
            k, v = (h @ W[p + "k"].T).view(T, H, d), (h @ W[p + "v"].T).view(T, H, dv)
            gi = cap * torch.tanh(linear(p + "i", h) / cap)
            gf = -torch.nn.functional.softplus(-cap * torch.tanh(linear(p + "f", h) / cap), threshold=1e9)
            S, n, top, o = x.new_zeros(H, d, dv), x.new_zeros(H, d), x.new_zeros(H), x.new_zeros(T, H, dv)
            for t in range(T):
                new = torch.maximum(gf[t] + top, gi[t])
                keep_, put = torch.exp(gf[t] + top - new), torch.exp(gi[t] - new)
                S = keep_[:, None, None] * S + (put[:, None] * k[t])[:, :, None] * v[t][:, None, :]
                n, top = keep_[:, None] * n + put[:, None] * k[t], new
                o[t] = (S * q[t][:, :, None]).sum(1) / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6)[:, None]
            o = _rms(o, 1.0, eps).reshape(T, -1) * W[p + "norm"] * torch.sigmoid(h @ W[p + "g"].T)
            y = o @ W[p + "o"].T
        x = x + mult * _rms(y, W[f"l{i}.norm1b"], eps)
        if L.get("mlp"):
            y = _gelu(_rms(x, W[f"l{i}.norm2"], eps) @ W[f"l{i}.mlp.up"].T) @ W[f"l{i}.mlp.down"].T
            x = x + mult * _rms(y, W[f"l{i}.norm2b"], eps)
    return _rms(x[keep], W["final.norm"], eps) @ W["embed"].T * cfg["logit_scale"]


def exact(case, seed):
    kind = case["kind"]
    t = torch.from_numpy(_tokens(case, seed)).cuda()
    if kind == "layered":
        cfg = LAYERED[case["model"]]
        W = {k: v.double() for k, v in _layered_weights(case, seed).items()}
        n = case["tokens"]
        with torch.no_grad():
            rows = (_paposun64 if cfg["architecture"] == "Paposun" else _nevurax64)(cfg, W, t, slice(n - 1, None))
        return rows
    c = _config(case)
    w = _Weights(c, seed)
    if kind == "train":
        adapters = w.lora.double().requires_grad_(True)
        logits = _decoder64(c, w, t, lora=adapters).view(c.BN, c.V)
        losses = torch.nn.functional.cross_entropy(logits, t.roll(-1, 1).reshape(-1), reduction="none")
        losses.mean().backward()
        with torch.no_grad():                             # clipped to a norm of 1, then AdamW's first step
            g = adapters.grad / max(1.0, float(adapters.grad.norm()))
            new = adapters - LR * (g / (g.abs() + 1e-8) + 0.01 * adapters)
        return {"losses": losses.detach(), "logits": logits.detach(), "adapters": new}
    if kind == "policy":
        _, _, adv, action, valid, old = _group(case, seed, w)
        params = {f"{k}{L}": w.matrix(w.pool, L, k).double().requires_grad_(True) for L in range(c.NL) for k in synth.MATS}
        params["head"] = w.head(w.pool).double().requires_grad_(True)
        logits = _decoder64(c, w, t, params=params, rows=torch.from_numpy(valid).cuda())
        lp = logits.gather(-1, torch.from_numpy(action).cuda()[..., None])[..., 0] - logits.logsumexp(-1)
        inside = torch.from_numpy(valid & (np.arange(c.seq)[None, :] >= case["prompt"])).cuda()
        a = torch.from_numpy(adv).cuda().double()[:, None].expand_as(lp)
        ratio = torch.exp(lp.detach() - torch.from_numpy(old).cuda().double())
        clipped = ratio.clamp(1 - 0.2, 1 + 0.2)
        active = torch.where(a >= 0, ratio <= clipped, ratio >= clipped) & inside
        # the reference's rule: the row gradient is w r (softmax - onehot) with w = -advantage, over the group's size
        (lp * (a * ratio * active / case["group"])).sum().backward()
        out = {"logprobs": lp.detach(), "weights": {}}
        for k, v in params.items():
            out["weights"][k] = v.detach() - POLICY_LR * v.grad
        return out
    with torch.no_grad():
        if kind == "batch":
            logits = _decoder64(c, w, t)
            return [logits[:, i].contiguous() for i in range(case["steps"])]
        n = case["tokens"]
        rows = _decoder64(c, w, t[None], keep=slice(n - 1, None))[0]
    if kind == "prompt":
        return rows[:1]
    if case["greedy"]:
        return {"first": rows[:1], "ids": rows[1:-1].argmax(-1), "last": rows[-1]}
    return rows
