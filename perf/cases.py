"""What the framework is timed on: whole passes of its models through the host library's sequences, as a program that serves them makes them -- a prompt in one
portion (or behind an earlier one), then single-token steps.  Tokens behind the prompt are fed, not sampled, so that a pass computes the same whatever the last bits
of a logit are.  Weights are random, of the sizes that synth.py and bench.py use; a model is opened once per process and keeps its weights, every pass is a new
sequence with tokens of its own.

A case: design, format (BitNet) or size (the others), layers, `earlier` and `prompt` tokens (two portions), `steps`.  A pass leaves the logits behind the last token;
one that ends with its prompt leaves that token's residual stream, too."""
import importlib
import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

bitnet = importlib.import_module("bitnet-rs_amd")
synth = importlib.import_module("bitnet-rs_amd.synth")

CAPACITY = 8192  # positions of a sequence


def bitnet_case(name, weights, prompt, steps, cache="f32"):
    return {"name": name, "design": "BitNet", "weights": weights, "cache": cache, "layers": 30, "earlier": 0, "prompt": prompt, "steps": steps}


def stack_case(name, design, size, prompt, steps, earlier=0):
    return {"name": name, "design": design, "size": size, "layers": 4, "earlier": earlier, "prompt": prompt, "steps": steps}


def listed():
    return [
        # bitnet-b1.58-2B-4T, all 30 layers: a chat's short question and its answer, the decode step above all
        bitnet_case("bitnet i2s answer", "i2s", 128, 64),
        # a long document, then an answer from its far end, on the halved cache
        bitnet_case("bitnet qk256 long answer", "qk256", 4000, 48, "f16"),
        # time to the first token: of a document, of a page whose length is nothing round, of a line
        bitnet_case("bitnet qk256 document", "qk256", 4096, 0),
        bitnet_case("bitnet i2s page", "i2s", 777, 0),
        bitnet_case("bitnet qk256 line", "qk256", 19, 0),
        # the layer-stack designs: documents of whole and of odd lengths, and answers to short prompts
        stack_case("lasapel document", "Lasapel", "3b", 4096, 0),
        stack_case("lasapel answer", "Lasapel", "2b", 61, 48),
        stack_case("mimolix page", "Mimolix", "1b", 1531, 0),
        stack_case("mimolix answer", "Mimolix", "3b", 200, 32),
        stack_case("lurepel document", "Lurepel", "3b", 3000, 0),
        # the next turn of a talk: a question behind what was said, and its answer
        stack_case("lurepel turn", "Lurepel", "1b", 90, 40, earlier=2000),
        stack_case("sipelorn document and answer", "Sipelorn", "1b", 2048, 24),
    ]


def draw(rng):
    design = rng.choice(["BitNet", "BitNet", "Lasapel", "Mimolix", "Lurepel", "Sipelorn"])
    prompt = int(round(math.exp(rng.uniform(math.log(2.0), math.log(4000.0)))))
    steps = rng.choice([0, 0, rng.randint(1, 48)])
    if design == "BitNet":
        c = bitnet_case("", rng.choice(["i2s", "qk256"]), prompt, steps, rng.choice(["f32", "f16"]))
    else:
        earlier = rng.choice([0, 0, int(round(math.exp(rng.uniform(math.log(16.0), math.log(2000.0)))))])
        c = stack_case("", design, rng.choice(["1b", "3b"]), min(prompt, 4000 - earlier), steps, earlier)
    del c["name"]
    return c


# ---- models ----------------------------------------------------------------------------------------------------------
def config_of(case):
    make = {"Lasapel": synth.lasapel_config, "Mimolix": synth.mimolix_config, "Lurepel": synth.lurepel_config, "Sipelorn": synth.sipelorn_config}
    return make[case["design"]](case["size"], case["layers"])


def write_model(case, folder):
    write = {"Lasapel": synth.write_lasapel, "Mimolix": synth.write_mimolix, "Lurepel": synth.write_lurepel, "Sipelorn": synth.write_sipelorn}
    config = config_of(case)
    write[case["design"]](folder, config)
    if case["design"] != "Lasapel":
        settle_routers(folder, config)
    return folder


def mapped_tensors(folder, mode):
    """name -> its bf16 bits in the file"""
    path = os.path.join(folder, "model.safetensors")
    with open(path, "rb") as f:
        n, = struct.unpack("<Q", f.read(8))
        head = json.loads(f.read(n))
    raw = np.memmap(path, np.uint8, mode, offset=8 + n)
    return {name: raw[slice(*t["data_offsets"])].view(np.uint16).reshape(t["shape"]) for name, t in head.items()}


def settle_routers(folder, config):
    """A choice of experts must not hang on the last bit of the router's input.  The first columns of an embedding row say which experts its token takes, evenly spread and
    well apart from the others; nothing is added to these columns behind the embedding, and they are all that a router reads."""
    router = next(layer["mlp"]["router"] for layer in config["layers"] if layer["mlp"]["kind"] == "moe")
    n, top, groups = router["experts"] + router.get("identity", 0), router["top"], router.get("groups")
    g, V, W = np.random.default_rng(7), config["vocab"], config["width"]
    if groups:  # as many from each of the groups that are kept
        size, take = n // groups["count"], top // groups["keep"]
        group = np.argsort(g.random((V, groups["count"])), 1)[:, :groups["keep"], None] * size
        chosen = (group + np.argsort(g.random((V, groups["keep"], size)), 2)[:, :, :take]).reshape(V, top)
    else:
        chosen = np.argsort(g.random((V, n)), 1)[:, :top]
    code = -0.5 - g.random((V, n), dtype=np.float32)
    np.put_along_axis(code, chosen, (2.0 - 0.1 * np.arange(top, dtype=np.float32))[None], 1)
    if "scale" in config.get("embedding", {}):
        code /= np.float32(config["embedding"]["scale"])

    def bits(a):
        return (np.asarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)

    for name, t in mapped_tensors(folder, "r+").items():
        last = name.rsplit(".", 1)[-1]
        if name == "embed":
            t[:, :n] = bits(code)
        elif name == "bigram":
            t[:, :n] = 0
        elif last in ("o", "down", "proj"):
            t[:n] = 0
        elif last == "router":
            t[:] = bits(np.eye(n, W))
        elif name == "loop.in":
            t[:n] = bits(np.eye(n, 2 * W, W))
        elif name == "embed.norm" or last in ("norm1", "norm2"):
            t[:n] = bits(1.0)
        elif name.endswith(("norm1.b", "norm2.b")):
            t[:n] = 0


class BitNetWeights:
    """Random weights by synth.py's recipe (uniform QK256 codes; ternary codes, half of them zero, with f16 block scales), made on the GPU layer by layer."""

    VALUES = {"qk256": (-2.0, -1.0, 1.0, 2.0), "i2s": (0.0, 1.0, 0.0, -1.0)}

    def __init__(self, case):
        self.cfg = synth.ModelConfig(n_layers=case["layers"], max_pos=CAPACITY)
        self.format = case["weights"]

    def generator(self, *ids):
        return torch.Generator(device="cuda").manual_seed(42 + sum((i + 1) * 1009 ** k for k, i in enumerate(ids)))

    def codes(self, rows, cols, g):
        n = rows * cols // 4
        a = torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g)
        if self.format == "qk256":
            return a
        b = torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g)
        return (a & 0x55) | (((a & b) & 0x55) << 1)

    def scales(self, rows, cols):
        return (2.0 / ((torch.arange(rows * cols // 32, device="cuda") % 100) + 1)).half().float()

    def layer(self, i):
        g = self.generator(i)
        gain = 1.0 / (synth.W_RMS[self.format] * math.sqrt(self.cfg.hidden))
        w = {n: (torch.rand(self.cfg.hidden, device="cuda", generator=g) + 0.5) * gain for n in ("attn_norm", "ffn_norm")}
        for name, (rows, cols) in self.cfg.shapes().items():
            w[name] = self.codes(rows, cols, g)
            if self.format == "i2s":
                w[name + "_scales"] = self.scales(rows, cols)
        return w

    def globals(self):
        g = self.generator(1 << 20)
        embed = torch.randn(self.cfg.vocab, self.cfg.hidden, device="cuda", generator=g).half()
        return embed, torch.rand(self.cfg.hidden, device="cuda", generator=g) + 0.5

    def open(self, case):
        d = bitnet.HostDecoder(self.cfg)
        for i in range(self.cfg.n_layers):
            w = {k: v.cpu().numpy() for k, v in self.layer(i).items()}
            d.set_layer_qk256(i, w) if self.format == "qk256" else d.set_layer_i2s(i, w, 32)
        embed, norm = self.globals()
        d.set_globals({"embed_f16": embed.view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1), "final_norm": norm.cpu().numpy()})
        d.set_kv_f16(case["cache"] == "f16")
        return d


MODELS = {}


def model_of(case):
    key = (case["design"], case.get("weights"), case.get("cache"), case.get("size"), case["layers"])
    if key not in MODELS:
        if case["design"] == "BitNet":
            MODELS[key] = BitNetWeights(case).open(case)
        else:
            with tempfile.TemporaryDirectory() as folder:
                MODELS[key] = bitnet.open_model(write_model(case, folder), max_pos=CAPACITY)
    return MODELS[key]


def tokens_of(case, seed, vocab):
    return np.random.default_rng(seed).integers(0, vocab, case["earlier"] + case["prompt"] + case["steps"]).astype(np.int32)


def prepare(case, seed):
    m = model_of(case)
    return {"model": m, "tokens": tokens_of(case, seed, m.vocab), "earlier": case["earlier"], "prompt": case["prompt"], "steps": case["steps"]}


def run(state):
    m = state["model"]
    m.reset()
    m.feed(state["tokens"])
    if state["earlier"]:
        m.prefill(state["earlier"], with_logits=False, digits=2)
    m.prefill(state["prompt"], with_logits=True, digits=2)
    if state["steps"]:
        m.run(state["steps"])
    return {"logits": m.last_logits()} if state["steps"] else {"logits": m.last_logits(), "hidden": m.last_hidden()}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def stack_sizes(case):
    """(weights every token meets, weights of the routed experts it meets, weights of all routed experts, columns of heads that attend over all keys,
    bytes of the cache per position) of a pass over the layers, looped layers counted as often as they run"""
    c = config_of(case)
    W, always, chosen, every, attend, cache = c["width"], 0, 0, 0, 0, 0
    loop = c.get("loop") or {"start": 0, "stop": 0, "times": 1}
    for i, layer in enumerate(c["layers"]):
        times = loop["times"] if loop["start"] <= i < loop["stop"] else 1
        m, f = layer["mixer"], layer.get("mlp")
        H, D, V = m["heads"], m["dim"], m["vdim"]
        a = W * H * V
        if layer["type"] == "latent_attention":
            Q = H * (D + m["rot_dim"])
            a += (W * m["q_rank"] + m["q_rank"] * Q if m.get("q_rank") else W * Q) + (H * D + H * V) * m["kv_rank"]
            if "kv_from" not in m:
                a += W * (m["kv_rank"] + m["rot_dim"])
            attend += times * H * (D + m["rot_dim"] + V)
            cache += times * 2 * (m["kv_rank"] + m["rot_dim"])
        elif layer["type"] == "lightning":
            a += W * H * (2 * D + 2 * V)
        elif layer["type"] == "delta":
            a += W * (2 * m["kv_heads"] * D + 2 * H * V + 2 * H)
        else:
            maps, own = 2 if "diff" in m else 1, "kv_from" not in m
            a += W * (H * maps * D + (m["kv_heads"] * (maps * D + V) if own and c["architecture"] != "Lurepel" else m["kv_heads"] * D if own else 0))
            a += W * {"Lurepel": H, "Sipelorn": H * V}.get(c["architecture"], 0)
            attend += times * H * maps * (D + V)
            cache += times * 2 * m["kv_heads"] * (maps * D + V)
        if c["architecture"] == "Sipelorn":
            a += 2 * W * W + 2 * W * c["token_side"]["dim"]
        if f:
            gated = 3 if c["architecture"] == "Lurepel" or f["kind"] == "moe" and c["architecture"] == "Sipelorn" else 2
            if f["kind"] == "dense":
                a += gated * W * f["ff"]
            else:
                a += W * f["router"]["experts"] + (gated * W * f["shared"]["ff"] if f.get("shared") else 0)
                chosen += times * f["router"]["top"] * gated * W * f["expert"]["ff"]
                every += times * f["router"]["experts"] * gated * W * f["expert"]["ff"]
        always += times * a
    if c.get("loop"):
        always += loop["times"] * 2 * W * W
    return always, chosen, every, attend, cache, c["vocab"] * W


def work(case):
    """Every portion and every step reads the weights it uses once (they follow from one another, and no cache holds a model), and the keys and values behind it."""
    if case["design"] == "BitNet":
        cfg = synth.ModelConfig(n_layers=case["layers"])
        always, chosen, every = cfg.n_layers * sum(r * c for r, c in cfg.shapes().values()), 0, 0
        attend, cache, head = cfg.n_layers * 2 * cfg.n_heads * cfg.head_dim, cfg.n_layers * 2 * cfg.n_kv_heads * cfg.head_dim * (2 if case["cache"] == "f16" else 4), cfg.vocab * cfg.hidden
        each = 0.25 if case["weights"] == "qk256" else 0.3125
    else:
        always, chosen, every, attend, cache, head = stack_sizes(case)
        each = 2.0
    nbytes, flops, at = 0.0, 0.0, 0
    for n, logits in [(case["earlier"], 0), (case["prompt"], 1)] + [(1, 1)] * case["steps"]:
        if not n:
            continue
        nbytes += each * (always + min(every, n * chosen)) + logits * 2 * head + (at + n) * cache
        flops += 2.0 * n * (always + chosen) + logits * 2 * head + 2.0 * attend * (n * at + n * (n + 1) / 2)
        at += n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # four times what the passes are off their 64-bit values by: 0.0015 to 0.003 (BitNet: activations of 15 bits per group in a step, f16 rows in a prompt), 0.0005 to
    # 0.006 (bf16 rows and cache); the largest error of one logit is about five times the root mean square
    return {"rel": 0.012, "max": 0.1} if case["design"] == "BitNet" else {"rel": 0.02, "max": 0.2}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------
def read_tensors(folder):
    tensors = mapped_tensors(folder, "r")
    return lambda name: torch.from_numpy(np.array(tensors[name]).view(np.int16)).cuda().view(torch.bfloat16).double()


def rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def centred(x, w, b, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b


def silu(z):
    return z * torch.sigmoid(z)


def gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def turn(v, freq, mult=1.0, neighbours=False):
    """v [tokens, heads, dims]: the first 2 len(freq) elements, those half a part apart or neighbours"""
    n = len(freq)
    angle = torch.arange(v.shape[0], dtype=torch.float64, device=v.device)[:, None, None] * freq
    c, s = torch.cos(angle) * mult, torch.sin(angle) * mult
    out = v.clone()
    one, two = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if neighbours else (slice(0, n), slice(n, 2 * n))
    out[..., one], out[..., two] = v[..., one] * c - v[..., two] * s, v[..., two] * c + v[..., one] * s
    return out


def yarn(rot):
    dims, base, s = rot["dims"], float(rot["base"]), rot["scaling"]
    i = torch.arange(dims // 2, dtype=torch.float64, device="cuda")
    f = base ** (-2.0 * i / dims)

    def dim_of(turns):
        return dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

    lo, hi = max(math.floor(dim_of(s["fast"])), 0), min(math.ceil(dim_of(s["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0


def banded(rot):
    s = rot["scaling"]
    f = float(rot["base"]) ** (-2.0 * torch.arange(rot["dims"] // 2, dtype=torch.float64, device="cuda") / rot["dims"])
    keep = ((s["original"] * f / (2.0 * math.pi) - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
    return (1.0 - keep) * f / s["factor"] + keep * f


def attend(q, k, v, scale=1.0, sink=None, first=None, penalty=None):
    """q [n, heads, dim], k [n, kv heads, dim], v [n, kv heads, vdim]; sink [heads]: a score without a value; first [n]: the first key a token sees"""
    n, H, _ = q.shape
    at = torch.arange(n, device=q.device)
    hidden = at[None, :] > at[:, None]
    if first is not None:
        hidden = hidden | (at[None, :] < first[:, None])
    out = torch.empty(n, H, v.shape[2], dtype=q.dtype, device=q.device)
    for h in range(H):
        g = h // (H // k.shape[1])
        s = q[:, h] @ k[:, g].T * scale
        if penalty is not None:
            s = s - penalty[0][h] * torch.log1p(penalty[1][h] * (at[:, None] - at[None, :]).clamp(min=0))
        s = s.masked_fill(hidden, -math.inf)
        top = s.amax(1, keepdim=True) if sink is None else torch.maximum(s.amax(1, keepdim=True), sink[h])
        e = torch.exp(s - top)
        total = e.sum(1, keepdim=True) + (0.0 if sink is None else torch.exp(sink[h] - top))
        out[:, h] = e / total @ v[:, g]
    return out


def convolve(x, w):
    taps, out = w.shape[1], torch.zeros_like(x)
    for j in range(min(taps, len(x))):
        out[j:] += w[:, taps - 1 - j] * x[:len(x) - j]
    return out


def experts(h, get, p, ids, w, ffn):
    out = torch.zeros_like(h)
    for e in ids.unique().tolist():
        t, c = (ids == e).nonzero(as_tuple=True)
        out[t] += w[t, c][:, None] * ffn(h[t], f"{p}e{e}.")
    return out


def exact_lasapel(c, get, tokens):
    eps, x, latents = c["norm"]["eps"], get("embed")[tokens], {}
    for i, layer in enumerate(c["layers"]):
        p, m, n = f"l{i}.", layer["mixer"], len(tokens)
        q, H, D, V = p + "mix.", m["heads"], m["dim"], m["vdim"]
        h = rms(x, eps) * (1.0 + get(p + "norm1"))
        if layer["type"] == "latent_attention":
            f, mult = yarn(m["rot"])
            if "kv_from" not in m:
                z = h @ get(q + "dkv").T
                latents[i] = rms(z[:, :m["kv_rank"]], eps) * get(q + "dkv.norm"), turn(z[:, None, m["kv_rank"]:], f, mult)
            lat, kr = latents[m.get("kv_from", i)]
            qq = (rms(h @ get(q + "dq").T, eps) * get(q + "dq.norm") @ get(q + "uq").T).reshape(n, H, -1)
            qq = torch.cat([qq[..., :D], turn(qq[..., D:], f, mult)], 2)
            k = torch.cat([(lat @ get(q + "uk").T).reshape(n, H, D), kr.expand(n, H, kr.shape[2])], 2)
            y = attend(qq, k, (lat @ get(q + "uv").T).reshape(n, H, V), m["scale"], get(q + "sink")).reshape(n, H * V) @ get(q + "o").T
        else:
            a, b, v = (silu(h @ get(q + s).T).reshape(n, H, -1) for s in "qkv")
            apart = torch.arange(n, device="cuda", dtype=torch.float64)
            apart = apart[:, None] - apart[None, :]
            o = torch.stack([(a[:, j] @ b[:, j].T * torch.where(apart < 0, 0.0, m["decay"][j] ** apart.clamp(min=0))) @ v[:, j] for j in range(H)], 1)
            y = (rms(o.reshape(n, H * V), eps) * get(q + "norm") * torch.sigmoid(h @ get(q + "g").T)) @ get(q + "o").T
        x = x + rms(y, eps) * (1.0 + get(p + "norm1b")) * get(p + "ls1")
        h = rms(x, eps) * (1.0 + get(p + "norm2"))
        y = torch.relu(h @ get(p + "mlp.up").T + get(p + "mlp.up.b")) ** 2 @ get(p + "mlp.down").T + get(p + "mlp.down.b")
        x = x + rms(y, eps) * (1.0 + get(p + "norm2b")) * get(p + "ls2")
    return rms(x[-1], eps) * (1.0 + get("final.norm")) @ get("head").T, x[-1]


def exact_mimolix(c, get, tokens):
    eps, n, loop = c["norm"]["eps"], len(tokens), c["loop"]
    x = first = get("embed")[tokens] * c["embedding"]["scale"]
    order = list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], len(c["layers"])))
    for i in order:
        p, layer = f"l{i}.", c["layers"][i]
        q, m, f = p + "mix.", layer["mixer"], layer["mlp"]
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        if i == loop["start"]:
            x = torch.cat([x, first], 1) @ get("loop.in").T
        h = centred(x, get(p + "norm1"), get(p + "norm1.b"), eps)
        if layer["type"] == "attention":
            qq = rms((h @ get(q + "q").T).reshape(n, H, 2, D), eps) * get(q + "q.norm")
            k = rms((h @ get(q + "k").T).reshape(n, G, 2, D), eps) * get(q + "k.norm")
            v = (h @ get(q + "v").T).reshape(n, G, V)
            at = torch.arange(n, device="cuda", dtype=torch.float64)
            qq = qq * (m["scale"] * (1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((at + 1) / m["q_temp"]["every"]) + 1.0)))[:, None, None, None]
            lam = torch.exp(get(q + "lq1") @ get(q + "lk1")) - torch.exp(get(q + "lq2") @ get(q + "lk2")) + m["diff"]
            y = rms(attend(qq[:, :, 0], k[:, :, 0], v) - lam * attend(qq[:, :, 1], k[:, :, 1], v), eps) * (1.0 - m["diff"])
            y = y.reshape(n, H * V)
        else:
            a, b, v = (silu(convolve(h @ get(q + s).T, get(q + s + ".conv"))) for s in "qkv")
            a, b = (z.reshape(n, G, D) for z in (a, b))
            a, b = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (a, b))
            a, b, v = (a * D ** -0.5).repeat_interleave(H // G, 1), b.repeat_interleave(H // G, 1), v.reshape(n, H, V)
            step = torch.sigmoid(h @ get(q + "b").T)
            keep = torch.exp(-torch.exp(get(q + "A_log")) * torch.nn.functional.softplus(h @ get(q + "a").T + get(q + "dt_bias")))
            S, o = torch.zeros(H, V, D, dtype=torch.float64, device="cuda"), torch.empty_like(v)
            for t in range(n):
                S = S * keep[t, :, None, None]
                new = step[t, :, None] * (v[t] - (S * b[t, :, None]).sum(2))
                S = S + new[:, :, None] * b[t, :, None]
                o[t] = (S * a[t, :, None]).sum(2)
            y = (rms(o, eps) * get(q + "norm")).reshape(n, H * V) * silu(h @ get(q + "g").T)
        y = y @ get(q + "o").T

        def ffn(z, e):
            return torch.relu(z @ get(e + "up").T) ** 2 @ get(e + "down").T

        w, ids = torch.softmax(h @ get(p + "mlp.router").T, 1).topk(f["router"]["top"], 1)
        y = y + ffn(h, p + "mlp.shared.") + experts(h, get, p + "mlp.", ids, w / (w.sum(1, keepdim=True) + 1e-20) * f["router"]["scale"], ffn)
        x = x + c["residual_mult"] * y
    return centred(x[-1], get("final.norm"), get("final.norm.b"), eps) @ get("head").T, x[-1]


def exact_lurepel(c, get, tokens):
    eps, n = c["norm"]["eps"], len(tokens)
    x = rms(get("embed")[tokens], eps) * get("embed.norm")
    at = torch.arange(n, device="cuda")

    def gated(z, e, act):
        return (act(z @ get(e + "gate").T) * (z @ get(e + "up").T)) @ get(e + "down").T

    for i, layer in enumerate(c["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        q, H, G, D, chunk = p + "mix.", m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"]
        a, k = (x @ get(q + "q").T).reshape(n, H, D), (x @ get(q + "k").T).reshape(n, G, D)
        freq = banded(m["rot"])
        o = attend(rms(turn(a, freq, neighbours=True), eps), rms(turn(k, freq, neighbours=True), eps), k, m["scale"], torch.zeros(H, dtype=torch.float64, device="cuda"), at // chunk * chunk)
        y = (o * torch.sigmoid(x @ get(q + "g").T)[:, :, None]).reshape(n, H * D) @ get(q + "o").T
        x = x + rms(y, eps) * get(p + "norm1")
        if f["kind"] == "dense":
            y = gated(x, p + "mlp.", gelu_tanh)
        else:
            s = torch.softmax(x @ get(p + "mlp.router").T, 1)
            ids = (s + get(p + "mlp.correction")).topk(f["router"]["top"], 1)[1]
            y = experts(x, get, p + "mlp.", ids, s.gather(1, ids), lambda z, e: gated(z, e, silu) if int(e.rsplit("e", 1)[1][:-1]) < f["router"]["experts"] else z)
        x = x + rms(y, eps) * get(p + "norm2")
    return rms(x[-1], eps) * get("final.norm") @ get("head").T, x[-1]


def exact_sipelorn(c, get, tokens):
    eps, n, side, b = c["norm"]["eps"], len(tokens), c["token_side"]["dim"], c["embedding"]["bigram"]
    pair = (torch.cat([tokens[:1] * 0, tokens[:-1]]) * b["mul_prev"] + tokens * b["mul_cur"]) % b["buckets"]
    pair[0] = b["buckets"]
    x = get("embed")[tokens] * c["embedding"]["scale"] + get("bigram")[pair]
    brought, at, shared = get("side.embed")[tokens], torch.arange(n, device="cuda"), {}

    def gated(z, e):
        return (silu(z @ get(e + "gate").T) * (z @ get(e + "up").T)) @ get(e + "down").T

    for i, layer in enumerate(c["layers"]):
        p, m, f = f"l{i}.", layer["mixer"], layer["mlp"]
        q, H, D, V = p + "mix.", m["heads"], m["dim"], m["vdim"]
        h = centred(x, get(p + "norm1"), get(p + "norm1.b"), eps)
        if layer["type"] == "attention":
            def rows(s, heads):
                return convolve(h @ get(q + s).T + get(q + s + ".b"), get(q + s + ".conv")).reshape(n, heads, -1)

            if "kv_from" not in m:
                shared[i] = rows("k", m["kv_heads"]), rows("v", m["kv_heads"])
            k, v = shared[m.get("kv_from", i)]
            o = attend(rows("q", H), k, v, m["scale"], None, at - m["mask"]["size"] + 1, (get(q + "r1"), get(q + "r2")))
            y = o.reshape(n, H * V) * torch.sigmoid(h @ get(q + "g").T) @ get(q + "o").T
        else:
            freq, mult = yarn(m["rot"])
            z = h @ get(q + "dkv").T
            lat, kr = rms(z[:, :m["kv_rank"]], eps) * get(q + "dkv.norm"), turn(z[:, None, m["kv_rank"]:], freq, mult, True)
            a = (h @ get(q + "q").T).reshape(n, H, -1)
            a = torch.cat([a[..., :D], turn(a[..., D:], freq, mult, True)], 2)
            k = torch.cat([(lat @ get(q + "uk").T).reshape(n, H, D), kr.expand(n, H, kr.shape[2])], 2)
            y = attend(a, k, (lat @ get(q + "uv").T).reshape(n, H, V), m["scale"]).reshape(n, H * V) @ get(q + "o").T
        x = x + y * torch.sigmoid(h @ get(p + "rg1").T + get(p + "rg1.b"))
        h = centred(x, get(p + "norm2"), get(p + "norm2.b"), eps)
        if f["kind"] == "dense":
            u, (up, down) = h @ get(p + "mlp.up").T, torch.nn.functional.softplus(get(p + "mlp.act"))
            u = torch.where(u > 0, up * u * u + 0.5 * u, (0.5 + down) * (torch.expm1(u.clamp(max=0.0)) - u) + 0.5 * u)
            y = u @ get(p + "mlp.down").T
        else:
            r = f["router"]
            s = torch.sigmoid(h @ get(p + "mlp.router").T)
            choice = (s + get(p + "mlp.correction")).reshape(n, r["groups"]["count"], -1)
            best = choice.topk(2, 2)[0].sum(2).topk(r["groups"]["keep"], 1)[1]
            kept = torch.zeros(n, r["groups"]["count"], dtype=torch.bool, device="cuda").scatter_(1, best, True)
            ids = choice.masked_fill(~kept[:, :, None], -math.inf).reshape(n, -1).topk(r["top"], 1)[1]
            y = experts(h, get, p + "mlp.", ids, s.gather(1, ids), gated) + gated(h, p + "mlp.shared.") * torch.sigmoid(h @ get(p + "mlp.shared.sg").T)
        x = x + y * torch.sigmoid(h @ get(p + "rg2").T + get(p + "rg2.b"))
        g = gelu_tanh(x @ get(p + "side.gate").T) * brought[:, i * side:(i + 1) * side]
        x = x + rms(g @ get(p + "side.proj").T, eps) * get(p + "side.norm")
    return centred(x[-1], get("final.norm"), get("final.norm.b"), eps) @ get("head").T, x[-1]


def exact_bitnet(case, tokens):
    made = BitNetWeights(case)
    cfg, n = made.cfg, len(tokens)
    table = torch.tensor(made.VALUES[made.format], dtype=torch.float64, device="cuda")
    embed, final = made.globals()
    x = embed[tokens].double()
    D, H, G, zero = cfg.head_dim, cfg.n_heads, cfg.n_kv_heads, torch.zeros((), dtype=torch.float64, device="cuda")
    freq = cfg.rope_theta ** (-2.0 * torch.arange(D // 2, dtype=torch.float64, device="cuda") / D)
    for i in range(cfg.n_layers):
        w = made.layer(i)

        def product(z, name):
            rows, cols = cfg.shapes()[name]
            codes = w[name].reshape(rows, cols // 4, 1) >> torch.tensor([0, 2, 4, 6], dtype=torch.uint8, device="cuda") & 3
            m = table[codes.reshape(rows, cols).long()]
            if made.format == "i2s":
                m = m * w[name + "_scales"].double().reshape(rows, cols // 32).repeat_interleave(32, 1)
            return z @ m.T

        h = centred(x, w["attn_norm"].double(), zero, cfg.eps)
        q, k, v = (product(h, s).reshape(n, -1, D) for s in "qkv")
        x = x + product(attend(turn(q, freq), turn(k, freq), v, D ** -0.5).reshape(n, H * D), "o")
        h = centred(x, w["ffn_norm"].double(), zero, cfg.eps)
        x = x + product(silu(product(h, "gate")) * product(h, "up"), "down")
    return centred(x[-1], final.double(), zero, cfg.eps) @ embed.double().T, x[-1]


def exact(case, seed):
    if case["design"] == "BitNet":
        logits, hidden = exact_bitnet(case, torch.from_numpy(tokens_of(case, seed, synth.ModelConfig().vocab)).long().cuda())
    else:
        c = config_of(case)
        with tempfile.TemporaryDirectory() as folder:
            get = read_tensors(write_model(case, folder))
            forward = {"Lasapel": exact_lasapel, "Mimolix": exact_mimolix, "Lurepel": exact_lurepel, "Sipelorn": exact_sipelorn}[case["design"]]
            logits, hidden = forward(c, get, torch.from_numpy(tokens_of(case, seed, c["vocab"])).long().cuda())
    return {"logits": logits.cpu().numpy(), "hidden": None if case["steps"] else hidden.cpu().numpy()}
