"""The work that programs give this framework, for timing: requests against quantized Llama / Qwen2 models (powerserve_amd.hip.Model) and against layer-list models
(powerserve_amd.seqmodel.SeqModel), each through the calls a serving loop makes.

A quantized model keeps a KV cache of 4096 slots and prefills in chunks of 128, four per launch sequence; a layer-list model serves in portions of 512.  Prompts
are random token ids; the weights are random numbers of the models' own shapes, drawn once per configuration, and belong to the handle a program keeps.  A layer-list
model's are drawn as a trained one behaves: the head points from every token to one that follows it, and a token has two experts of its own."""
import atexit
import json
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

from powerserve_amd import gguf, hip, seqmodel, synth

N_CTX, CHUNK, WIDE, PORTION = 4096, 128, 512, 512
WTYPES = {"Q4_0": gguf.Q4_0, "Q8_0": gguf.Q8_0, "Q4_K": gguf.Q4_K, "Q4_K_M": synth.Q4_K_M}
VOCAB, BUCKETS, TAPS, DECAY_RANK, EXPERTS, TOP = 4096, 4093, 4, 8, 8, 2


def listed():
    return [
        # the smallest model of the reference's table at its layer shape, a short chat: launches and latency
        {"name": "qwen-q8_0-decode", "family": "quant", "preset": "qwen2-0.5b-dims-2l", "wtype": "Q8_0", "what": "decode", "context": 100, "n": 32},
        # the reference's second configuration: a prompt of 512 on the 1B layer shape
        {"name": "1b-q4_0-prompt", "family": "quant", "preset": "llama-1b-dims-2l", "wtype": "Q4_0", "what": "prompt", "context": 0, "n": 512},
        # the headline at the 8B layer shape: greedy tokens behind a prompt of 2048, and that prompt
        {"name": "8b-q4_k-decode", "family": "quant", "preset": "llama-8b-dims-4l", "wtype": "Q4_K", "what": "decode", "context": 2047, "n": 32},
        {"name": "8b-q4_k-prompt", "family": "quant", "preset": "llama-8b-dims-4l", "wtype": "Q4_K", "what": "prompt", "context": 0, "n": 2048},
        # a speculative step's verification: a tree of 12 drafted tokens, the mix of weight types that files come in
        {"name": "8b-q4_k_m-tree", "family": "quant", "preset": "llama-8b-dims-4l", "wtype": "Q4_K_M", "what": "tree", "context": 700, "n": 12},
        # layer-list models: a long prompt, an ordinary ragged one, replies
        {"name": "ranutar-prompt", "family": "Ranutar", "width": 2048, "layers": 6, "dtype": "bfloat16", "what": "prompt", "context": 0, "n": 2047},
        {"name": "ranutar-prompt-ragged", "family": "Ranutar", "width": 4096, "layers": 3, "dtype": "bfloat16", "what": "prompt", "context": 0, "n": 203},
        {"name": "ranutar-decode", "family": "Ranutar", "width": 4096, "layers": 3, "dtype": "bfloat16", "what": "decode", "context": 100, "n": 32},
        # the float32 mode, which is served for those who check numbers
        {"name": "ranutar-f32-prompt", "family": "Ranutar", "width": 2048, "layers": 3, "dtype": "float32", "what": "prompt", "context": 0, "n": 300},
        {"name": "pupidra-prompt", "family": "Pupidra", "width": 2048, "layers": 6, "dtype": "bfloat16", "what": "prompt", "context": 0, "n": 1500},
        {"name": "pupidra-decode", "family": "Pupidra", "width": 2048, "layers": 6, "dtype": "bfloat16", "what": "decode", "context": 100, "n": 32},
        # a reply whose tokens a sampler on the host picks: every step's logits come back
        {"name": "pupidra-sampled", "family": "Pupidra", "width": 4096, "layers": 3, "dtype": "bfloat16", "what": "sampled", "context": 30, "n": 12},
    ]


def draw(rng):
    def spread(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    if rng.random() < 0.4:
        preset = rng.choice(["qwen2-0.5b-dims-2l", "llama-1b-dims-2l", "llama-8b-dims-4l"])
        wtype = rng.choice(["Q8_0", "Q4_0"] if preset.startswith("qwen") else ["Q8_0", "Q4_0", "Q4_K", "Q4_K_M"])
        what = rng.choice(["prompt", "decode", "tree"])
        n = spread(9, 2048) if what == "prompt" else spread(8, 64) if what == "decode" else rng.randint(2, 32)
        return {"family": "quant", "preset": preset, "wtype": wtype, "what": what, "context": 0 if what == "prompt" else spread(8, 2047), "n": n}
    width = rng.choice([2048, 4096])
    c = {"family": rng.choice(["Ranutar", "Pupidra"]), "width": width, "layers": rng.randint(1, 6 if width == 2048 else 3),
         "dtype": "float32" if rng.random() < 0.15 else "bfloat16", "what": rng.choice(["prompt", "prompt", "decode", "sampled"]), "context": 0}
    if c["what"] == "prompt":
        c["n"] = spread(5, 2047 if width == 2048 else 1000) if c["dtype"] == "bfloat16" else spread(5, 200)
    else:
        c["context"], c["n"] = spread(2, 500), spread(4, 32)
    return c


# ---------------------------------------------------------------------------------------------------------------------------- models
_CTX, _DIRS, _MODEL = [], {}, {}


def _ctx():
    if not _CTX:
        _CTX.append(hip.Ctx(0))
    return _CTX[0]


def _dir(key, write):
    if key not in _DIRS:
        d = tempfile.mkdtemp(prefix="perf_model_")
        atexit.register(shutil.rmtree, d, True)
        write(d)
        _DIRS[key] = d
    return _DIRS[key]


def _quant_dir(c):
    return _dir((c["preset"], c["wtype"]), lambda d: synth.write_model_dir(d, c["preset"], WTYPES[c["wtype"]], n_ctx=N_CTX, seed=1234))


class _Model(hip.Model):
    """A quantized model that gives its memory back with its last user."""

    def __del__(self):
        self.close()


class _View:
    """A device buffer of a model as torch.as_tensor takes it; tensors over it hold the view, and the view holds the model."""

    def __init__(self, model, ptr, shape):
        self.model = model
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (int(ptr), False), "version": 3}


class _Quant:
    """A quantized model of its own (weights and KV cache) and a request against it."""

    def __init__(self, c, seed):
        rng = np.random.default_rng(seed)
        self.c, self.m = c, _Model(_ctx(), _quant_dir(c), max_batch=WIDE, n_ctx=N_CTX)
        self.tokens, self.extra, self.tree, self.depth = _request(c, rng)
        f, L = self.m.cfg, _ctx().L
        self.kv = [(torch.as_tensor(_View(self.m, L.ps_hip_model_k_cache(self.m.h, i), (f.seq_len, f.kv_dim)), device="cuda"),
                    torch.as_tensor(_View(self.m, L.ps_hip_model_v_cache(self.m.h, i), (f.kv_dim, f.seq_len)), device="cuda")) for i in range(f.n_layers)]
        if c["context"]:
            self.m.prefill(self.tokens, CHUNK)


def _request(c, rng):
    """(the prompt, further tokens, and for a tree of them: who sees whom, how deep each is)"""
    V = synth.PRESETS[c["preset"]][7] if c["family"] == "quant" else VOCAB
    tokens = rng.integers(0, V, c["n"] if c["what"] == "prompt" else c["context"]).astype(np.int32)
    extra = rng.integers(0, V, max(1, c["n"])).astype(np.int32)
    if c["what"] != "tree":
        return tokens, extra, None, None
    n = c["n"]
    see, depth = np.eye(n, dtype=np.uint8), np.zeros(n, dtype=np.int32)
    for i in range(1, n):
        p = int(rng.integers(max(0, i - 4), i))
        see[i] |= see[p]
        depth[i] = depth[p] + 1
    return tokens, extra, see, depth


def _layer_list_config(c):
    wide = c["width"] == 4096
    W, H, ff = c["width"], 32 if wide else 16, 14336 if wide else 8192
    if c["family"] == "Ranutar":
        kinds = {"delta": dict(heads=H, kv_heads=H // 2, dim=128, vdim=128, conv=4), "wkv": dict(heads=H, dim=128),
                 "latent_attention": dict(heads=H, dim=128, vdim=128, q_rank=1536 if wide else 768, kv_rank=512, rot_dim=64, rot={"base": 1e6, "dims": 64}, mask={"size": 1024},
                                          scale=192 ** -0.5)}
        order = ["delta", "latent_attention", "wkv"]
        return synth.seq_config(W, VOCAB, [synth.seq_layer(order[i % 3], ff, **kinds[order[i % 3]]) for i in range(c["layers"])], taps=TAPS)
    order, layers = ("mal" if wide else "mmalsl")[:c["layers"]], []
    for i, k in enumerate(order):
        own = max([j for j in range(i) if order[j] == "a"], default=None)
        mixer = {"m": ("mamba2", synth.pupidra_mamba2(2 * W // 64, 64, 128, 8, 4, 8)), "l": ("latent_attention", synth.pupidra_latent(H, 128, 64, 128, 512, 192 ** -0.5, 5e5))}.get(k) \
            or ("attention", synth.pupidra_attention(H, H // 4, 128, 128, 1.0, 1024, 64, own if k == "s" else None))
        layers.append(synth.pupidra_layer(*mixer, moe=(EXPERTS, TOP, ff * 3 // 8, 2.0), shared=ff * 3 // 4))
    return synth.pupidra_config(W, VOCAB, layers, bigram=(BUCKETS, 43, 19), softcap=30.0)


def _shapes(cfg):
    """name -> (shape, how it is drawn): ("lin", gain) rows over the root of their length, ("vec", spread, mean), or a word."""
    W, s = cfg["width"], {}
    lin, vec = (lambda n, k, g=1.0: ((n, k), ("lin", g))), (lambda n, sd=0.1, mean=0.0: ((n,) if isinstance(n, int) else n, ("vec", sd, mean)))
    s["embed"] = (VOCAB, W), "embed"
    ranutar = cfg["architecture"] == "Ranutar"
    if not ranutar:
        s["bigram"] = (BUCKETS + 1, W), ("vec", 1.0, 0.0)
    for i, lc in enumerate(cfg["layers"]):
        p, m, mc, mlp = f"l{i}.", f"l{i}.mix.", lc["mixer"], lc["mlp"]
        H, kind = mc["heads"], lc["type"]
        dv = mc.get("vdim", mc.get("dim"))
        if ranutar:
            for n in ("norm1", "norm1b", "norm2", "norm2b"):
                s[p + n] = vec(W)
            for n in ("canon1", "canon2"):
                s[p + n] = vec((W, TAPS), 0.3)
            s[p + "mlp.up"], s[p + "mlp.down"], s[p + "mlp.act"] = lin(mlp["ff"], W), lin(W, mlp["ff"]), vec(2, 0.7)
        else:
            for n in "12":
                s[p + "norm" + n], s[p + "ls" + n] = vec(W, 0.2, 1.0), vec(W, 0.3, 0.8)
            ff, sf = mlp["expert"]["ff"], mlp["shared"]["ff"]
            for e in range(EXPERTS):
                s[f"{p}mlp.e{e}.up"], s[f"{p}mlp.e{e}.down"] = lin(ff, W, 1.5), lin(W, ff)
            s[p + "mlp.router"] = (EXPERTS, W), "router"
            s[p + "mlp.shared.up"], s[p + "mlp.shared.down"] = lin(sf, W, 1.5), lin(W, sf)
        if kind == "wkv":
            Hd = H * mc["dim"]
            for n in "rkvgw":
                s[m + "mu." + n] = vec(W, 0.2, 0.5)
            for n in "rkvg":
                s[m + n] = lin(Hd, W)
            s[m + "w1"], s[m + "w2"], s[m + "w0"], s[m + "u"], s[m + "norm"] = lin(DECAY_RANK, W), lin(Hd, DECAY_RANK), vec(Hd, 0.8, -0.5), vec((H, mc["dim"]), 0.5), vec(Hd, 0.2, 1.0)
        elif kind == "delta":
            KHd, Hv = mc["kv_heads"] * mc["dim"], H * dv
            for n, rows in (("q", KHd), ("k", KHd), ("v", Hv)):
                s[m + n], s[m + n + ".conv"] = lin(rows, W), vec((rows, mc["conv"]), 0.6)
            s[m + "b"], s[m + "a"], s[m + "g"] = lin(H, W), lin(H, W), lin(Hv, W)
            s[m + "A_log"], s[m + "dt_bias"], s[m + "norm"] = vec(H, 0.6, 0.7), vec(H, 0.5), vec(dv, 0.2, 1.0)
        elif kind == "mamba2":
            inner = H * dv
            chan = inner + 2 * mc["groups"] * mc["state"]
            s[m + "in"], s[m + "conv"], s[m + "conv.b"] = lin(inner + chan + H, W), vec((chan, mc["conv"]), 0.6), vec(chan, 0.3)
            s[m + "dt_bias"], s[m + "A_log"], s[m + "D"], s[m + "norm"] = vec(H, 0.7, -1.5), vec(H, 0.6, 0.2), vec(H, 0.5, 1.0), vec(inner, 0.2, 1.0)
        elif kind == "attention":
            d, G = mc["dim"], mc["kv_heads"]
            for n, r in {"q": H * d, "k": G * d, "v": G * dv}.items():
                if n == "q" or mc.get("kv_from") is None:
                    s[m + n], s[m + n + ".b"] = lin(r, W), vec(r, 0.3)
            s[m + "o.b"] = vec(W, 0.3)
        else:
            d, R, dr = mc["dim"], mc["kv_rank"], mc["rot_dim"]
            if ranutar:
                s[m + "dq"], s[m + "dq.norm"], s[m + "uq"] = lin(mc["q_rank"], W), vec(mc["q_rank"], 0.2), lin(H * (d + dr), mc["q_rank"])
                s[m + "dkv.norm"] = vec(R, 0.2, 1.0)
            else:
                s[m + "q"], s[m + "g"], s[m + "dkv.norm"] = lin(H * (d + dr), W, 1.5), lin(H, W, 2.0), vec(R, 0.3, 1.0)
            s[m + "dkv"], s[m + "uk"], s[m + "uv"] = lin(R + dr, W), lin(H * d, R), lin(H * dv, R)
        s[m + "o"] = lin(W, H * dv)
    s["final.norm"], s["head"] = vec(W, 0.1, 0.0 if ranutar else 1.0), ((VOCAB, W), "head")
    if ranutar:  # (norms over a latent: a plain weight)
        for n in [n for n in s if n.endswith("dq.norm")]:
            s[n] = vec(s[n][0][0], 0.2, 1.0)
    return s


def _weights(cfg):
    """bfloat16 tensors on the GPU.  embed: a random row plus its two experts' directions; head: row follow(t) is token t's embedding."""
    g = torch.Generator(device="cuda").manual_seed(7)

    def normal(shape):
        return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)

    W, t = cfg["width"], {}
    ways = torch.linalg.qr(normal((W, EXPERTS)))[0].t().contiguous()
    first, second = _experts()
    for n, (shape, how) in _shapes(cfg).items():
        if how == "embed":
            a = normal(shape) + 24.0 * ways[first] + 16.0 * ways[second]
        elif how == "router":
            a = 0.15 * ways + normal(shape) * (0.1 / math.sqrt(W))
        elif how == "head":
            a = normal(shape) * (0.3 / math.sqrt(W))
            a[_follow().cuda()] += t["embed"].float() * (1.5 / math.sqrt(W))
        elif how[0] == "lin":
            a = normal(shape) * (how[1] / math.sqrt(shape[1]))
        else:
            a = normal(shape) * how[1] + how[2]
        t[n] = a.to(torch.bfloat16)
    return t


def _experts():
    first = torch.arange(VOCAB) % EXPERTS
    return first, (first + 1 + (torch.arange(VOCAB) // EXPERTS) % (EXPERTS - 1)) % EXPERTS


def _follow():
    return torch.from_numpy(np.random.default_rng(3).permutation(VOCAB))


def _write_layer_list(d, cfg):
    t, meta, off = _weights(cfg), {}, 0
    for n, a in t.items():
        meta[n] = {"dtype": "BF16", "shape": list(a.shape), "data_offsets": [off, off + 2 * a.numel()]}
        off += 2 * a.numel()
    head = json.dumps(meta).encode()
    head += b" " * (-len(head) % 8)
    with open(os.path.join(d, "config.json"), "w") as f:
        json.dump(cfg, f)
    with open(os.path.join(d, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(head)) + head)
        for n in list(t):
            t.pop(n).view(torch.int16).cpu().numpy().tofile(f)


def _layer_list_model(c):
    """The model that a program loads once and serves every request from (one at a time is kept here)."""
    key = (c["family"], c["width"], c["layers"], c["dtype"])
    if key not in _MODEL:
        for m in _MODEL.values():
            m.close()
        _MODEL.clear()
        cfg = _layer_list_config(c)
        d = _dir(key[:3], lambda d: _write_layer_list(d, cfg))
        torch.cuda.empty_cache()
        _MODEL[key] = seqmodel.SeqModel(_ctx(), d, dtype=c["dtype"], max_batch=PORTION, n_slots=2, max_context=N_CTX)
    return _MODEL[key]


class _LayerList:
    """A request against a layer-list model; the slot that holds its state is taken and given back within the pass."""

    def __init__(self, c, seed):
        self.c, self.m = c, _layer_list_model(c)
        self.tokens, self.extra, _, _ = _request(c, np.random.default_rng(seed))
        self.want = _want(c["n"])


def _want(n):
    """Which of a prompt's tokens a scoring pass asks the logits of."""
    return np.unique(np.linspace(0, n - 1, 64).astype(np.int32))


def prepare(case, seed):
    return (_Quant if case["family"] == "quant" else _LayerList)(case, seed)


def run(s):
    m, what, n = s.m, s.c["what"], s.c["n"]
    if isinstance(s, _LayerList):
        slot = m.acquire()
        if what == "prompt":
            out = m.forward(slot, s.tokens, want=s.want)
        else:
            if s.tokens.size > 1:
                m.forward(slot, s.tokens[:-1])
            if what == "decode":
                ids = m.decode_greedy(slot, int(s.tokens[-1]), n)
                out = {"ids": ids, "logits": m.forward(slot, ids[-1:], want=[0])}
            else:
                out = [m.forward(slot, [t], want=[0]) for t in (s.tokens[-1], *s.extra[1:])]
        m.release(slot)
        return out
    if what == "prompt":  # everything in front of the last token without logits, that one with them
        m.reset()
        m.prefill(s.tokens[:-1], CHUNK)
        logits, ids = m.forward(s.tokens[-1:], [n - 1])
        return {"ids": ids, "logits": logits, "kv": [(k[:n], v[:, :n]) for k, v in s.kv]}
    if what == "decode":
        ids = m.decode_greedy(int(s.extra[0]), n)
        out = {"ids": ids, "logits": m.logits(1)}
        m.kv_rollback(n)
        return out
    p = m.position
    logits, ids = m.forward_tree(s.extra, p + s.depth, s.tree, want_logits=True)
    return {"ids": ids, "logits": logits, "kv": [(k[p:p + n], v[:, p:p + n]) for k, v in s.kv]}


# ---------------------------------------------------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    c, n, ctx = case, case["n"], case["context"]
    many = c["what"] in ("prompt", "tree")  # tokens that share one pass over the weights
    if c["family"] == "quant":
        arch, dim, hidden, L, H, G, hs, V, _, _, tied, _ = synth.PRESETS[c["preset"]]
        cfg = synth.llm_config(c["preset"], N_CTX)
        plan = synth.tensor_plan(cfg, arch, WTYPES[c["wtype"]], tied)
        size = {name: (ne[0] * ne[1], ne[1] * gguf.row_size(t, ne[0])) for name, t, ne in plan if len(ne) == 2}
        layers = [v for k, v in size.items() if k.startswith("blk.")]
        head = size["token_embd.weight" if tied else "output.weight"]
        params, bytes_ = (sum(v[i] for v in layers) for i in (0, 1))
        heads = 1 if c["what"] == "prompt" else n
        seen = n * (n + 1) / 2 if c["what"] == "prompt" else n * ctx + n * (n + 1) / 2
        flops = 2.0 * params * n + 2.0 * head[0] * heads + 4.0 * seen * L * H * hs
        kv = 8.0 * G * hs * L
        read = (ctx if many else n * ctx) * kv
        return {"bytes": (bytes_ + head[1]) * (1 if many else n) + read + n * kv + heads * V * 4.0, "flops": flops}
    cfg = _layer_list_config(c)
    e = 4 if c["dtype"] == "float32" else 2
    shapes = {k: v[0][0] * v[0][1] for k, v in _shapes(cfg).items() if len(v[0]) == 2 and isinstance(v[1], tuple) and v[1][0] == "lin"}
    expert = sum(v for k, v in shapes.items() if ".mlp.e" in k) / EXPERTS
    rest = sum(v for k, v in shapes.items() if ".mlp.e" not in k)
    head = VOCAB * cfg["width"]
    front = n if many else max(0, ctx - 1)  # tokens of the prompt, in one pass
    steps = 0 if many else n + (c["what"] == "decode")
    wanted = len(_want(n)) if many else (1 if c["what"] == "decode" else n)
    flops = 2.0 * (rest + TOP * expert) * (front + steps) + 2.0 * head * (wanted if many else steps)
    for lc in cfg["layers"]:
        mc = lc["mixer"]
        total = front + steps
        size = (mc.get("mask") or {}).get("size", N_CTX)
        if "attention" in lc["type"]:
            flops += 2.0 * mc["heads"] * (mc["dim"] + mc.get("rot_dim", 0) + mc["vdim"]) * sum(min(i + 1, size) for i in range(total))
        else:
            flops += 6.0 * mc["heads"] * mc.get("vdim", mc.get("dim")) * mc.get("state", mc.get("dim")) * total
    once = (rest + min(EXPERTS, max(TOP, front * TOP)) * expert) * e if front else 0
    return {"bytes": once + steps * ((rest + TOP * expert + head) * e) + (head * e if many else 0) + wanted * VOCAB * 4.0, "flops": flops}


def tolerance(case):
    if case["family"] == "quant":
        return "exact"  # the quantized path is the reference's arithmetic bit for bit
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3}  # measured against exact(): 1.4e-6
    # bfloat16 operands, rounded in every product; measured against exact(): 0.0033 and 0.0095 (rows whose routing turns on a near tie may differ by more than the rest)
    return {"rel": 0.013, "max": 0.5} if case["family"] == "Ranutar" else {"rel": 0.03, "max": 0.99}


# ---------------------------------------------------------------------------------------------------------------------------- the same in 64 bits, plainly
def _rms(a, eps):
    return a / torch.sqrt((a * a).mean(-1, keepdim=True) + eps)


def _silu(a):
    return a * torch.sigmoid(a)


def _rotate(a, pos, base, dims, pairs):
    """The first `dims` numbers of a [T, heads, d] turn: neighbours, or halves."""
    f = torch.tensor(float(base), dtype=torch.float64, device=a.device) ** (-torch.arange(0, dims, 2, device=a.device, dtype=torch.float64) / dims)
    ang = pos.to(a.device).double()[:, None, None] * f
    c, s = torch.cos(ang), torch.sin(ang)
    out = a.clone()
    i, j = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    out[..., i], out[..., j] = a[..., i] * c - a[..., j] * s, a[..., j] * c + a[..., i] * s
    return out


def _attend(q, k, v, mask, scale, minus=None):
    """q [T, H, d], k / v [S, G, .], mask [T, S] -> [T, H * dv]"""
    out = []
    r = q.shape[1] // k.shape[1]
    for h in range(q.shape[1]):
        z = q[:, h] @ k[:, h // r].t() * scale
        z = z if minus is None else z - minus[h]
        out.append(torch.softmax(z.masked_fill(~mask, -math.inf), -1) @ v[:, h // r])
    return torch.stack(out, 1).reshape(q.shape[0], -1)


def _dequantized(raw, t, n, k):
    """Rows of GGUF blocks as float64 [n, k]."""
    b = torch.from_numpy(np.array(raw)).cuda().reshape(-1, gguf.BLOCK[t][1])
    f16 = lambda lo: b[:, lo:lo + 2].contiguous().view(torch.float16).double()  # noqa: E731
    i8 = lambda lo, hi: b[:, lo:hi].contiguous().view(torch.int8).double()  # noqa: E731
    if t == gguf.Q8_0:
        w = f16(0) * i8(2, 34)
    elif t == gguf.Q4_0:
        w = f16(0) * (torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).double() - 8)
    elif t == gguf.Q4_K:
        s, q = b[:, 4:16], b[:, 16:].reshape(-1, 4, 32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = (f16(0) * sc)[:, :, None] * q - (f16(2) * mn)[:, :, None]
    else:  # Q6_K: two halves of 128; ql [64], qh [32], a scale per 16
        ql, qh, sc = b[:, 0:128].reshape(-1, 2, 64), b[:, 128:192].reshape(-1, 2, 32), i8(192, 208)
        q = torch.stack([(ql[..., :32] & 15) | ((qh & 3) << 4), (ql[..., 32:] & 15) | (((qh >> 2) & 3) << 4), (ql[..., :32] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 32:] >> 4) | ((qh >> 6) << 4)], 2)
        w = (f16(208) * sc)[:, :, None] * (q.reshape(-1, 16, 16).double() - 32)
    return w.reshape(n, k)


def _quantized(a, wide):
    """The activation operand: 8 bits per number, a scale per 256 (K-quants) or per 32, which is kept in 16 bits."""
    b = a.reshape(*a.shape[:-1], -1, 256 if wide else 32)
    amax = b.abs().amax(-1, keepdim=True).clamp_min(1e-30)
    q = torch.round(b * 127 / amax)
    d = amax / 127
    return (q * (d if wide else d.to(torch.float16).double())).reshape(a.shape)


def _exact_quant(c, seed):
    tokens, extra, tree, depth = _request(c, np.random.default_rng(seed))
    rd = gguf.GGUFReader(os.path.join(_quant_dir(c), "ggml", "weights.gguf"))
    arch, dim, hidden, L, H, G, hs, V, base, rtype, tied, eps = synth.PRESETS[c["preset"]]
    n, ctx = c["n"], c["context"]

    def vec(name):
        return torch.from_numpy(np.array(rd.data(name))).cuda().double()

    def mul(a, name, rows=None):
        ti = rd.tensors[name]
        return _quantized(a, ti.type not in (gguf.Q8_0, gguf.Q4_0)) @ _dequantized(rd.data(name), ti.type, ti.ne[1], ti.ne[0]).t()

    ids = torch.from_numpy(np.concatenate([tokens, extra]) if tree is not None else tokens).long()
    T = len(ids)
    pos = torch.arange(T)
    mask = torch.ones(T, T, dtype=torch.bool).tril()
    if tree is not None:
        pos[ctx:] = ctx + torch.from_numpy(depth).long()
        mask[ctx:, ctx:] = torch.from_numpy(tree).bool()
    mask = mask.cuda()
    ti = rd.tensors["token_embd.weight"]
    x = _dequantized(rd.data("token_embd.weight"), ti.type, ti.ne[1], ti.ne[0])[ids.cuda()]
    kv = []
    for i in range(L):
        p = f"blk.{i}."
        h = _rms(x, eps) * vec(p + "attn_norm.weight")
        q, k, v = (mul(h, p + f"attn_{s}.weight") + (vec(p + f"attn_{s}.bias") if arch == "qwen2" else 0.0) for s in "qkv")
        q, k = (_rotate(a.reshape(T, -1, hs), pos, base, hs, rtype == 0) for a in (q, k))
        kv.append((k.reshape(T, -1)[ctx:], v[ctx:].t()))
        x = x + mul(_attend(q, k, v.reshape(T, G, hs), mask, hs ** -0.5), p + "attn_output.weight")
        h = _rms(x, eps) * vec(p + "ffn_norm.weight")
        x = x + mul(_silu(mul(h, p + "ffn_gate.weight")) * mul(h, p + "ffn_up.weight"), p + "ffn_down.weight")
    h = _rms(x[-1:] if tree is None else x[ctx:], eps) * vec("output_norm.weight")
    return {"ids": None, "logits": mul(h, "token_embd.weight" if tied else "output.weight"), "kv": kv}


def _time_filter(a, w):
    """Per channel, causal: w [C, taps], the last tap is the present."""
    taps = w.shape[1]
    pad = torch.cat([a.new_zeros(taps - 1, a.shape[1]), a])
    return sum(pad[j:j + a.shape[0]] * w[:, j] for j in range(taps))


def _wkv(W, h, mc, eps):
    T, H, d = h.shape[0], mc["heads"], mc["dim"]
    prev = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
    mix = {n: h + (prev - h) * W("mu." + n) for n in "rkvgw"}
    r, k, v = ((mix[n] @ W(n).t()).reshape(T, H, d) for n in "rkv")
    decay = torch.exp(-torch.exp(torch.tanh(mix["w"] @ W("w1").t()) @ W("w2").t() + W("w0"))).reshape(T, H, d)
    S, out, u = h.new_zeros(H, d, d), [], W("u")[:, :, None]
    for t in range(T):
        kv = k[t][:, :, None] * v[t][:, None, :]
        out.append((r[t][:, None, :] @ (S + u * kv))[:, 0])
        S = decay[t][:, :, None] * S + kv
    return (_rms(torch.stack(out), eps).reshape(T, H * d) * W("norm") * _silu(mix["g"] @ W("g").t())) @ W("o").t()


def _delta(W, h, mc, eps):
    T, H, KH, d, dv = h.shape[0], mc["heads"], mc["kv_heads"], mc["dim"], mc["vdim"]
    q, k, v = (_silu(_time_filter(h @ W(n).t(), W(n + ".conv"))) for n in "qkv")
    q, k, v = q.reshape(T, KH, d), k.reshape(T, KH, d), v.reshape(T, H, dv)
    q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) / math.sqrt(d)).repeat_interleave(H // KH, 1)
    k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // KH, 1)
    beta = torch.sigmoid(h @ W("b").t())[:, :, None]
    keep = torch.exp(-torch.exp(W("A_log")) * torch.nn.functional.softplus(h @ W("a").t() + W("dt_bias")))[:, :, None, None]
    S, out = h.new_zeros(H, d, dv), []
    for t in range(T):
        S = S * keep[t]
        write = beta[t] * (v[t] - (k[t][:, None, :] @ S)[:, 0])
        S = S + k[t][:, :, None] * write[:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
    return ((_rms(torch.stack(out), eps) * W("norm")).reshape(T, H * dv) * _silu(h @ W("g").t())) @ W("o").t()


def _latent(W, h, mc, eps, ranutar):
    T, H, d, dr, dv, R = h.shape[0], mc["heads"], mc["dim"], mc["rot_dim"], mc["vdim"], mc["kv_rank"]
    i = torch.arange(T, device=h.device)
    rot = lambda a: _rotate(a, i, mc["rot"]["base"], mc["rot"]["dims"], not ranutar)  # noqa: E731
    down = h @ W("dkv").t()
    c, shared = _rms(down[:, :R], eps) * W("dkv.norm"), rot(down[:, None, R:])
    q = (((_rms(h @ W("dq").t(), eps) * W("dq.norm")) @ W("uq").t()) if ranutar else h @ W("q").t()).reshape(T, H, d + dr)
    q = torch.cat([q[..., :d], rot(q[..., d:])], -1)
    k = torch.cat([(c @ W("uk").t()).reshape(T, H, d), shared.expand(T, H, dr)], -1)
    gap = i[:, None] - i[None, :]
    o = _attend(q, k, (c @ W("uv").t()).reshape(T, H, dv), (gap >= 0) & (gap < (mc.get("mask") or {}).get("size", T)), mc["scale"])
    if not ranutar:
        o = (o.reshape(T, H, dv) * torch.sigmoid(h @ W("g").t())[:, :, None]).reshape(T, H * dv)
    return o @ W("o").t()


def _kept_window(W, h, mc, eps, source):
    T, H, G, d, dv = h.shape[0], mc["heads"], mc["kv_heads"], mc["dim"], mc["vdim"]
    proj = lambda n: h @ W(n).t() + W(n + ".b")  # noqa: E731
    q = _rms(proj("q").reshape(T, H, d), eps)
    k, v = source or (_rms(proj("k").reshape(T, G, d), eps), proj("v").reshape(T, G, dv))
    i = torch.arange(T, device=h.device)
    gap = i[:, None] - i[None, :]
    mask = (gap >= 0) & ((gap < mc["mask"]["size"]) | (i[None, :] < mc["mask"]["keep_first"]))
    minus = [2.0 ** (-8.0 * (x + 1.0) / H) * gap for x in range(H)]
    return _attend(q, k, v, mask, mc["scale"], minus) @ W("o").t() + W("o.b"), (k, v)


def _mamba2(W, h, mc, eps):
    T, H, P, N, G = h.shape[0], mc["heads"], mc["vdim"], mc["state"], mc["groups"]
    inner = H * P
    u = h @ W("in").t()
    xbc = _silu(_time_filter(u[:, inner:2 * inner + 2 * G * N], W("conv")) + W("conv.b"))
    x, B, C = xbc[:, :inner].reshape(T, H, P), *(xbc[:, inner + j * G * N:inner + (j + 1) * G * N].reshape(T, G, N).repeat_interleave(H // G, 1) for j in (0, 1))
    dt = torch.nn.functional.softplus(u[:, 2 * inner + 2 * G * N:] + W("dt_bias"))
    keep = torch.exp(-torch.exp(W("A_log")) * dt)[:, :, None, None]
    S, y = h.new_zeros(H, N, P), []
    for t in range(T):
        S = keep[t] * S + (dt[t][:, None] * B[t])[:, :, None] * x[t][:, None, :]
        y.append((C[t][:, None, :] @ S)[:, 0])
    y = (torch.stack(y) + W("D")[:, None] * x).reshape(T, inner) * _silu(u[:, :inner])
    return (_rms(y.reshape(T, mc["norm_groups"], -1), eps).reshape(T, inner) * W("norm")) @ W("o").t()


def _scaled_experts(W, h, mlp):
    s = torch.softmax(h @ W("router").t(), -1)
    w, e = s.topk(TOP, -1)
    one = lambda a, n: torch.relu(a @ W(n + ".up").t()) ** 2 @ W(n + ".down").t()  # noqa: E731
    out = one(h, "shared")
    for j in range(EXPERTS):
        at, slot = (e == j).nonzero(as_tuple=True)
        if len(at):
            out.index_add_(0, at, w[at, slot][:, None] * mlp["router"]["scale"] * one(h[at], f"e{j}"))
    return out


def _exact_stream(cfg, tensors, tokens):
    """What the final norm makes of the residual stream, [T, width]."""
    eps, ranutar = cfg["norm"]["eps"], cfg["architecture"] == "Ranutar"
    ids = torch.from_numpy(tokens).long().cuda()
    of = lambda p: (lambda n: tensors[p + n].double())  # noqa: E731
    top = of("")
    x = tensors["embed"][ids].double()
    if not ranutar:
        big = cfg["embedding"]["bigram"]
        rows = torch.cat([ids.new_full((1,), big["buckets"]), (ids[:-1] * big["mul_prev"] + ids[1:] * big["mul_cur"]) % big["buckets"]])
        x = x + tensors["bigram"][rows].double()
    kv = {}
    for i, lc in enumerate(cfg["layers"]):
        L, M, F, mc, kind = of(f"l{i}."), of(f"l{i}.mix."), of(f"l{i}.mlp."), lc["mixer"], lc["type"]
        h = x
        if ranutar:
            h = _rms(x, eps) * (1 + L("norm1"))
            h = h + _time_filter(h, L("canon1"))
        if kind == "attention":
            y, kv[i] = _kept_window(M, h, mc, eps, kv.get(mc.get("kv_from")))
        elif kind == "latent_attention":
            y = _latent(M, h, mc, eps, ranutar)
        else:
            y = {"wkv": _wkv, "delta": _delta, "mamba2": _mamba2}[kind](M, h, mc, eps)
        if ranutar:
            x = x + _rms(y, eps) * (1 + L("norm1b"))
            h = _rms(x, eps) * (1 + L("norm2"))
            z = (h + _time_filter(h, L("canon2"))) @ F("up").t()
            p, q = torch.nn.functional.softplus(F("act"))
            z = torch.where(z > 0, p * z * z + 0.5 * z, (0.5 + q) * (torch.expm1(z.clamp_max(0)) - z) + 0.5 * z)
            x = x + _rms(z @ F("down").t(), eps) * (1 + L("norm2b"))
        else:
            x = x + _rms(y, eps) * L("norm1") * L("ls1")
            x = x + _rms(_scaled_experts(F, x, lc["mlp"]), eps) * L("norm2") * L("ls2")
    return _rms(x, eps) * (top("final.norm") + (1 if ranutar else 0))


def _exact_layer_list(c, seed):
    tokens, extra, _, _ = _request(c, np.random.default_rng(seed))
    cfg = _layer_list_config(c)
    t = _weights(cfg)
    head = t["head"].double()
    cap = cfg.get("logit_softcap")
    logits = lambda rows: (cap * torch.tanh(rows @ head.t() / cap)) if cap else rows @ head.t()  # noqa: E731
    if c["what"] == "prompt":
        return logits(_exact_stream(cfg, t, tokens)[torch.from_numpy(_want(c["n"])).long().cuda()])
    if c["what"] == "sampled":
        rows = logits(_exact_stream(cfg, t, np.concatenate([tokens, extra[1:]]))[len(tokens) - 1:])
        return [r[None] for r in rows]
    seq, follow = list(tokens), _follow()
    for _ in range(c["n"]):
        seq.append(int(follow[seq[-1]]))
    for _ in range(4):  # the continuation that the head points to, mended where another token wins
        z = logits(_exact_stream(cfg, t, np.asarray(seq, dtype=np.int32))[len(tokens) - 1:])
        ids = z[:-1].argmax(-1).tolist()
        if ids == seq[len(tokens):]:
            return {"ids": None, "logits": z[-1:]}
        at = next(i for i, (a, b) in enumerate(zip(ids, seq[len(tokens):])) if a != b)
        seq[len(tokens) + at] = ids[at]
        for j in range(len(tokens) + at + 1, len(seq)):
            seq[j] = int(follow[seq[j - 1]])
    return None


def exact(case, seed):
    with torch.no_grad():
        if case["family"] != "quant":
            return _exact_layer_list(case, seed)
        # (a prompt: one activation that rounds the other way on its way to 8 bits changes every row behind it by about the rounding's own size, 1e-2)
        # a greedy continuation of random weights turns on ties: its ids, and what is computed from them, have no value of their own
        return None if case["what"] == "decode" else _exact_quant(case, seed)
