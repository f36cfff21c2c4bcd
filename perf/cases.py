"""The work this framework is timed at: decoding, prompts and lockstep batches of the sparse LLaMA / Falcon engine, and
requests to the models described layer by layer, all through powerinfer_amd.model.

Weights are random at the scale of the repository's benchmark (0.02).  What a model decides - which neurons fire, which experts a token
goes to - is made to keep a margin, so that two correct implementations agree on it: a few channels of the residual stream mark the
token's class (nothing writes to them), and predictors and routers read the class from there.  Neuron j fires for a class with its own
Zipf(1.2) rate, one draw per class, so counts, their spread over the neurons and the growth of a batch's union are those of independent
draws.
"""
import math

import numpy as np
import torch

from powerinfer_amd import fikevik, lerasun, lib, pibalorn, pufivik, synth
from powerinfer_amd.model import LayerModel, Model

F64 = torch.float64
CLASSES = 16                    # token classes of the sparse models (token id modulo CLASSES), one marked channel each
MARKED = 32                     # channels kept free for them: one Q4_0 block
EMBED = 0.25                    # spread of embeddings
SPARSE = {"tiny": ("llama-tiny", 8), "7b": ("llama-7b", 8), "13b": ("llama-13b", 6), "falcon40b": ("falcon-40b", 4)}
DESIGNS = ("lerasun", "pibalorn", "fikevik", "pufivik")


# ---- the cases ----------------------------------------------------------------------------------------------------------------------
def sparse(name, kind, model, wtype="f16", past=0, steps=1, prompt=0, n_seq=1, hot=1.0, layers=None):
    return dict(name=name, kind=kind, model=model, wtype=wtype, past=past, steps=steps, prompt=prompt, n_seq=n_seq, hot=hot, layers=layers or SPARSE[model][1])


def request(name, model, width, prompt, steps, n_seq=1):
    return dict(name=name, kind="request", model=model, width=width, prompt=prompt, steps=steps, n_seq=n_seq)


def listed():
    return [
        # a small model answering a few tokens: launches and hand-overs, hardly any bytes
        sparse("tiny-f16-decode", "decode", "tiny", past=20, steps=16, layers=3),
        # chat at batch 1, the headline: a 7B-shaped FP16 model behind a 64-token prompt, the caller sampling from the logits
        sparse("7b-f16-decode", "decode", "7b", past=64, steps=8),
        # the same model quantised, deep in a long conversation
        sparse("7b-q4-decode-long", "decode", "7b", "q4_0", past=3001, steps=8),
        # the quantised model with a VRAM budget: the hottest 60 % of neurons on the GPU, the others on host threads
        sparse("7b-q4-split-decode", "decode", "7b", "q4_0", past=128, steps=8, hot=0.6, layers=4),
        # the largest shape, behind a 1024-token prompt
        sparse("falcon40b-f16-decode", "decode", "falcon40b", past=1024, steps=8),
        # sixteen sequences in lockstep behind a shared 512-token prompt
        sparse("13b-f16-lockstep", "lockstep", "13b", past=512, steps=4, n_seq=16),
        # a document to read before the first token
        sparse("7b-f16-prompt", "prompt", "7b", prompt=2047),
        # a question to a quantised model: a short prompt of odd length
        sparse("7b-q4-prompt", "prompt", "7b", "q4_0", prompt=131),
        # latent attention and routed experts: a long prompt
        request("lerasun-prompt", "lerasun", 4096, prompt=2048, steps=0),
        # grouped-query and linear attention, experts beside a shared one: a server's sixteen requests, ragged prompts, then steps together
        request("pibalorn-serve", "pibalorn", 2048, prompt=48, steps=12, n_seq=16),
        # gated linear attention, windows and a matrix memory: four ragged prompts read together
        request("fikevik-prompts", "fikevik", 4096, prompt=700, steps=0, n_seq=4),
        # mixed and soft-capped heads, experts: one conversation's turn, prompt and answer
        request("pufivik-chat", "pufivik", 4096, prompt=333, steps=16),
    ]


def spread(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "lockstep", "prompt", "request", "request"])
    if kind == "request":
        n_seq = rng.choice([1, 1, rng.randint(2, 16)])
        steps = rng.choice([0, rng.randint(1, 16)])
        c = request("", rng.choice(DESIGNS), rng.choice([2048, 4096]), spread(rng, 3, 1500 // n_seq), steps, n_seq)
    elif kind == "lockstep":
        model, wtype = rng.choice([("13b", "f16"), ("7b", "f16"), ("7b", "q4_0"), ("tiny", "f16")])
        c = sparse("", kind, model, wtype, past=spread(rng, 5, 450), steps=rng.randint(1, 4), n_seq=rng.randint(2, 16), layers=rng.randint(2, 4))
    elif kind == "prompt":
        model, wtype = rng.choice([("7b", "f16"), ("7b", "f16"), ("7b", "q4_0"), ("13b", "f16"), ("falcon40b", "f16"), ("tiny", "f16")])
        c = sparse("", kind, model, wtype, prompt=spread(rng, 3, 450 if model == "tiny" else 1900), layers=rng.randint(2, 4))
    else:
        model, wtype, hot = rng.choice([("tiny", "f16", 1.0), ("7b", "f16", 1.0), ("7b", "q4_0", 1.0), ("7b", "q4_0", round(rng.uniform(0.3, 0.8), 2)),
                                        ("13b", "f16", 1.0), ("falcon40b", "f16", 1.0)])
        c = sparse("", kind, model, wtype, past=spread(rng, 3, 400 if model == "tiny" else 3000), steps=rng.randint(2, 12), hot=hot,
                   layers=rng.randint(2, 4))
    del c["name"]
    return c


# ---- random tensors -----------------------------------------------------------------------------------------------------------------
class Source:
    """Tensors by name, made on the GPU from the seed alone."""

    def __init__(self, seed):
        self.seed = seed

    def generator(self, *name):
        h = self.seed & 0x7FFFFFFF
        for ch in "/".join(map(str, name)):
            h = (h * 1000003 + ord(ch)) & 0x7FFFFFFFFFFFFFFF
        return torch.Generator("cuda").manual_seed(h)

    def normal(self, name, rows, cols, std, dtype):
        x = torch.empty(rows, cols, dtype=dtype, device="cuda")
        return x.normal_(0.0, std, generator=self.generator(*name))

    def host(self, *name):
        return np.random.default_rng([self.seed, len(name)] + [ord(ch) for ch in "/".join(map(str, name))])


def q4_0_blocks(x):
    """Q4_0 blocks of fp16 rows: bytes [rows, cols / 32 * 18], and the values they hold."""
    b = x.float().reshape(-1, 32)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    d = top / -8
    q = (b * torch.where(d != 0, 1 / d, torch.zeros_like(d)) + 8.5).floor_().clamp_(0, 15).to(torch.uint8)
    out = torch.empty(b.shape[0], 18, dtype=torch.uint8, device=x.device)
    out[:, :2] = d.half().view(torch.uint8).reshape(-1, 2)
    out[:, 2:] = q[:, :16] | (q[:, 16:] << 4)
    return out.reshape(x.shape[0], -1)


def q4_0_values(blocks):
    b = blocks.reshape(-1, 18)
    d = b[:, :2].contiguous().view(torch.float16).to(F64)
    q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(F64) - 8
    return (q * d).reshape(blocks.shape[0], -1)


def cut(total, n_seq):
    """Lengths of n_seq ragged prompts around `total`."""
    return [max(1, total - (total * ((7 * s) % 16)) // 24) for s in range(n_seq)]


# ---- sparse models ------------------------------------------------------------------------------------------------------------------
def shape_of(case):
    name, _ = SPARSE[case["model"]]
    ctx = case["past"] + case["prompt"] + case["steps"] + 8
    return synth.hparams(name, n_layer=case["layers"], n_ctx=ctx, wtype=lib.Q4_0 if case["wtype"] == "q4_0" else lib.F16, hot_frac=case["hot"])


class SparseTensors:
    def __init__(self, hp, seed):
        self.hp, self.src = hp, Source(seed)

    def matrix(self, layer, kind):
        """The stored tensor: fp16, or Q4_0 blocks."""
        hp, d, f16 = self.hp, self.hp.n_embd, torch.float16
        gqa = d // hp.n_head * hp.n_head_kv
        rows, cols = {"tok_embd": (hp.n_vocab, d), "output": (hp.n_vocab, d), "wqkv": (d + 2 * gqa, d), "wo": (d, d), "ffn_gate": (hp.n_ff, d), "ffn_up": (hp.n_ff, d),
                      "ffn_down_t": (hp.n_ff, d), "fc1": (hp.n_rank, d)}[kind]
        w = self.src.normal((layer, kind), rows, cols, EMBED if kind == "tok_embd" else 0.02, f16)
        first = d - MARKED                                                   # the marked channels
        if kind == "tok_embd":
            w[:, first:] = 0
            ids = torch.arange(rows, device=w.device)
            w[ids, first + ids % CLASSES] = 4.0
        elif kind == "wo":
            w[first:] = 0
        elif kind == "ffn_down_t":
            w[:, first:] = 0
        elif kind == "fc1":                                                  # the last CLASSES hidden units see the token's class
            w[rows - CLASSES:] = 0
            for c in range(CLASSES):
                w[rows - CLASSES + c, first + c] = 8.0
        return q4_0_blocks(w) if hp.wtype == lib.Q4_0 and kind != "fc1" else w

    def rates(self, layer):
        return synth.zipf_rates(self.hp.n_ff, self.hp.mean_rate, self.src.host(layer, "rates"))[0]

    def fc2(self, layer):
        """[n_ff, rank] fp16: the class units decide with a margin, the others vary the scores."""
        hp = self.hp
        w = self.src.normal((layer, "fc2"), hp.n_ff, hp.n_rank, 0.01, torch.float16)
        fires = self.src.host(layer, "fires").random((hp.n_ff, CLASSES)) < self.rates(layer)[:, None]
        w[:, hp.n_rank - CLASSES:] = torch.from_numpy(np.where(fires, 1.0, -1.0).astype(np.float16)).to(w.device)
        return w


def sparse_tokens(case, hp, seed):
    """(prompt or shared past, [steps, n_seq] tokens behind it)"""
    rng = np.random.default_rng([seed, 77])
    first = rng.integers(0, hp.n_vocab, case["prompt"] or case["past"]).astype(np.int32)
    return first, rng.integers(0, hp.n_vocab, (case["steps"], case["n_seq"])).astype(np.int32)


def prepare_sparse(case, seed):
    hp = shape_of(case)
    src, m, held, q4 = SparseTensors(hp, seed), Model(hp), [], hp.wtype == lib.Q4_0

    def put(layer, kind, w, to_host=False):
        if to_host:
            return m.set_tensor(layer, kind, w.cpu().numpy())
        held.append(w)
        t = lib.Q4_0 if w.dtype == torch.uint8 else lib.F16
        m.set_tensor_device(layer, kind, w.data_ptr(), t, w.shape[1] // 18 * 32 if t == lib.Q4_0 else w.shape[1], w.shape[0])

    falcon, ones, zeros = hp.arch == "falcon", np.ones(hp.n_embd, np.float32), np.zeros(hp.n_embd, np.float32)
    put(-1, "tok_embd", src.matrix(-1, "tok_embd"))
    put(-1, "output", src.matrix(-1, "output"))
    m.set_tensor(-1, "output_norm", ones)
    if falcon:
        m.set_tensor(-1, "output_norm_b", zeros)
    for i in range(hp.n_layer):
        for kind in ("attn_norm", "attn_norm_2") if falcon else ("attn_norm", "ffn_norm"):
            m.set_tensor(i, kind, ones)
            if falcon:
                m.set_tensor(i, kind + "_b", zeros)
        put(i, "wqkv", src.matrix(i, "wqkv"))
        put(i, "wo", src.matrix(i, "wo"))
        for kind in ("ffn_up", "ffn_down_t") if falcon else ("ffn_gate", "ffn_up", "ffn_down_t"):
            put(i, kind, src.matrix(i, kind), to_host=hp.hot_frac < 1)
        put(i, "fc1", src.matrix(i, "fc1"))
        put(i, "fc2", src.fc2(i))
        p = src.rates(i)
        m.set_tensor(i, "neuron_rate", p.astype(np.float32))
        if hp.hot_frac < 1:
            on_gpu, bucket = synth.gpu_split(p, hp.hot_frac)
            m.set_tensor(i, "gpu_idx", on_gpu)
            m.set_tensor(i, "gpu_bucket", bucket)
    torch.cuda.synchronize()
    m.finalize()
    first, then = sparse_tokens(case, hp, seed)
    if case["kind"] == "lockstep":
        m.batch_init(case["n_seq"])
        for k, t in enumerate(first):
            m.batch_decode(np.full(case["n_seq"], t), np.full(case["n_seq"], k), want_logits=False)
    elif case["past"]:
        m.decode(first, 0, want_logits=False)
    return dict(case=case, model=m, held=held, first=first, then=then)


def run_sparse(state):
    case, m = state["case"], state["model"]
    if case["kind"] == "prompt":
        return m.decode(state["first"], 0)[1]
    past, out = case["past"], []
    for k, toks in enumerate(state["then"]):
        if case["kind"] == "lockstep":
            out.append(m.batch_decode(toks, np.full(case["n_seq"], past + k, np.int32))[1])
        else:
            out.append(m.decode(toks, past + k)[1])
    return out


def rotated(x, pos, dims, freq, pairs, length=1.0):
    """x [n, heads, dim] with its first `dims` rotated: neighbours (pairs) or halves."""
    a = pos.to(F64)[:, None] * freq[None, :]
    c, s = length * torch.cos(a)[:, None], length * torch.sin(a)[:, None]
    y = x.clone()
    u, v = (slice(0, dims, 2), slice(1, dims, 2)) if pairs else (slice(0, dims // 2), slice(dims // 2, dims))
    y[..., u], y[..., v] = x[..., u] * c - x[..., v] * s, x[..., v] * c + x[..., u] * s
    return y


def frequencies(dims, base):
    return float(base) ** (-2.0 * torch.arange(dims // 2, dtype=F64, device="cuda") / dims)


def rms(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def layer_norm(x, eps):
    return rms(x - x.mean(-1, keepdim=True), eps)


def exact_sparse(case, seed):
    hp = shape_of(case)
    src = SparseTensors(hp, seed)
    first, then = sparse_tokens(case, hp, seed)
    if case["kind"] == "prompt":
        tokens, pos, wanted = first, np.arange(len(first)), [len(first) - 1]
        owner = np.zeros(len(first), int)
    else:                                        # the past, then every sequence's own tokens: owner -1 is everybody's
        steps, n_seq = then.shape
        tokens = np.concatenate([first, then.reshape(-1)])
        pos = np.concatenate([np.arange(len(first)), np.repeat(len(first) + np.arange(steps), n_seq)])
        owner = np.concatenate([np.full(len(first), -1), np.tile(np.arange(n_seq), steps)])
        wanted = list(range(len(first), len(tokens)))
    tok, p, own = (torch.as_tensor(np.asarray(a), device="cuda").long() for a in (tokens, pos, owner))
    seen = (p[None] <= p[:, None]) & ((own[None] == own[:, None]) | (own[None] == -1))
    val = (lambda w: q4_0_values(w) if w.dtype == torch.uint8 else w.to(F64))  # noqa: E731
    falcon, H, G, D = hp.arch == "falcon", hp.n_head, hp.n_head_kv, hp.n_embd // hp.n_head
    norm = (lambda v: layer_norm(v, hp.norm_eps)) if falcon else (lambda v: rms(v, hp.norm_eps))
    freq = frequencies(D, hp.rope_freq_base)
    x = val(src.matrix(-1, "tok_embd")[tok])
    for i in range(hp.n_layer):
        h = norm(x)
        q, k, v = (h @ val(src.matrix(i, "wqkv")).T).split([H * D, G * D, G * D], 1)
        q, k = (rotated(t.reshape(len(tok), -1, D), p, D, freq, not falcon) for t in (q, k))
        v, o = v.reshape(len(tok), G, D), torch.empty(len(tok), H, D, dtype=F64, device="cuda")
        for a in range(H):
            s = (q[:, a] @ k[:, a * G // H].T / math.sqrt(D)).masked_fill(~seen, -math.inf)
            o[:, a] = torch.softmax(s, 1) @ v[:, a * G // H]
        y = o.reshape(len(tok), -1) @ val(src.matrix(i, "wo")).T
        if not falcon:
            x = x + y
            h = norm(x)
        on = torch.relu(h @ src.matrix(i, "fc1").to(F64).T) @ src.fc2(i).to(F64).T >= hp.sparse_threshold
        u = h @ val(src.matrix(i, "ffn_up")).T
        u = torch.relu(u) if falcon else torch.relu(h @ val(src.matrix(i, "ffn_gate")).T) * u
        x = x + (u * on) @ val(src.matrix(i, "ffn_down_t")) + (y if falcon else 0)
    logits = (norm(x[wanted]) @ val(src.matrix(-1, "output")).T).cpu().numpy()
    if case["kind"] == "prompt":
        return logits[0]
    logits = logits.reshape(then.shape + (-1,))
    return list(logits) if case["kind"] == "lockstep" else [r[0] for r in logits]


def work_sparse(case):
    hp = shape_of(case)
    d, ff, r = hp.n_embd, hp.n_ff, hp.n_rank
    gqa = d // hp.n_head * hp.n_head_kv
    s = 2.0 if hp.wtype == lib.F16 else 18 / 32
    mats = 2 if hp.arch == "falcon" else 3
    fires = np.minimum(1, synth.zipf_rates(ff, hp.mean_rate, np.random.default_rng(0))[0])
    prompt = case["kind"] == "prompt"
    tokens = case["prompt"] if prompt else case["n_seq"]                       # of one step
    union = float((1 - (1 - fires) ** min(tokens, CLASSES)).sum())
    past = 0 if prompt else case["past"]
    dense = (2 * d * d + 2 * d * gqa) + 0.0
    seqs_kv = 1 if prompt else case["n_seq"]
    layer = dense * s + (d * r + r * ff) * 2 + union * mats * d * s + seqs_kv * (past + 1) * 2 * gqa * 2 + (tokens * 2 * gqa * 2 if prompt else 0)
    wanted = 1 if prompt else tokens
    head = hp.n_vocab * d * s + wanted * hp.n_vocab * 4
    cells = (tokens + 1) / 2 if prompt else past + 1
    flops = hp.n_layer * tokens * 2 * (dense + d * r + r * ff + ff * hp.mean_rate * mats * d + 2 * cells * d) + wanted * 2 * hp.n_vocab * d
    n = 1 if prompt else case["steps"]
    return {"bytes": n * (hp.n_layer * layer + head), "flops": n * flops}


# ---- models described layer by layer ------------------------------------------------------------------------------------------------
VOCAB, TOP = 32000, 6
ROUTES = 64                     # token classes of a router, one marked channel each
BF16 = torch.bfloat16


def config_of(case):
    """Layers at a width, with the sizes of the repository's benchmark."""
    width, name = case["width"], case["model"]
    H, dim, experts, ff, dense_ff = width // 128, 128, 64, 1408, {2048: 5632, 4096: 11008}[width]
    kv = H // 4
    if name == "lerasun":
        lat = {"heads": H, "dim": dim, "rot_dim": 64, "vdim": dim, "kv_rank": 512, "scale": (dim + 64) ** -0.5, "rot": {"base": 10000.0}}
        moe = {"kind": "moe", "router": {"experts": experts, "top": TOP, "groups": {"count": 8, "keep": 4}}, "expert": {"ff": ff}}
        return {"width": width, "vocab": VOCAB, "norm": {"eps": 1e-6}, "logit_scale": 1.0,
                "layers": [{"type": "latent_attention", "mixer": dict(lat, kv_from=i - 1 if i % 2 else None), "mlp": moe} for i in range(4)]}
    if name == "pibalorn":
        dense = {"kind": "dense", "ff": dense_ff, "limit": 7.0}
        moe = {"kind": "moe", "router": {"experts": experts, "top": TOP}, "expert": {"ff": ff, "limit": 7.0}, "shared": {"ff": 2816, "limit": 7.0}}
        att = {"type": "attention", "mixer": {"heads": H, "kv_heads": kv, "dim": dim, "vdim": dim, "rot": {"dims": dim, "base": 10000.0}, "scale": dim ** -0.5}}
        lin = {"type": "lightning", "mixer": {"heads": H, "dim": dim, "vdim": dim, "decay": np.exp(-2.0 ** -np.linspace(0, 8, H)).tolist()}}
        return {"width": width, "vocab": VOCAB, "norm": {"eps": 1e-6}, "embedding": {"scale": 1.0, "bigram": {"buckets": 9973, "mul_prev": 29, "mul_cur": 13}},
                "loop": {"start": 2, "stop": 4, "times": 2}, "layers": [dict(att, mlp=dense), dict(lin, mlp=moe), dict(att, mlp=moe), dict(lin, mlp=moe)]}
    if name == "fikevik":
        mlp = {"kind": "dense", "ff": dense_ff}
        lin = {"type": "gla", "mixer": {"heads": H, "dim": dim, "vdim": dim, "tau": 16.0}, "mlp": mlp}
        par = {"type": "parallel", "mlp": mlp, "mixer": {
            "left": {"heads": H, "kv_heads": kv, "dim": dim, "vdim": dim, "rot": {"dims": dim, "base": 10000.0}, "scale": dim ** -0.5, "mask": {"size": 1024}},
            "right": {"heads": H, "dim": dim, "vdim": dim, "gate_cap": 15.0}, "left_scale": 0.7, "right_scale": 0.7}}
        return {"width": width, "vocab": VOCAB, "norm": {"eps": 1e-6}, "embedding": {"scale": 1.0}, "postln_alpha": 2.0,
                "layers": [lin, par, dict(lin, weights_of=0), dict(par, weights_of=1)]}
    mix = {"heads": H, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "v_mix": True}
    mlp = {"kind": "moe", "router": {"experts": experts, "top": TOP}, "expert": {"ff": ff}}
    waves = {"type": "attention", "mlp": mlp, "mixer": dict(mix, rot={"dims": 64, "base": 500000.0, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})}
    soft = {"type": "attention_2", "mlp": mlp, "mixer": dict(mix, softcap=50.0, rot={"dims": 64, "base": 10000.0, "scaling": {"factor": 4.0, "slow": 1.0, "fast": 32.0, "original": 4096}})}
    return {"width": width, "vocab": VOCAB, "norm": {"eps": 1e-6, "groups": 8}, "embedding": {"scale": 1.0}, "residual_mult": 0.5, "canon": {"taps": 4},
            "layers": [waves, soft, waves, soft]}


RANK = 16                       # of the key decays' projection


def descs_of(case, cfg):
    if case["model"] == "fikevik":
        return fikevik.layer_descs(cfg, {f"l{i}.mix.a1": np.empty((RANK, case["width"]), np.float32) for i in range(len(cfg["layers"]))})
    return {"lerasun": lerasun, "pibalorn": pibalorn, "pufivik": pufivik}[case["model"]].layer_descs(cfg)


class DesignTensors:
    """bf16 matrices by layer and role, made when asked for; `shapes` lists the roles of a layer."""

    def __init__(self, case, seed):
        self.case, self.cfg, self.src = case, config_of(case), Source(seed)
        self.descs = descs_of(case, self.cfg)

    def shapes(self, i):
        d, w = self.descs[i], self.case["width"]
        if d.get("weights_of"):
            return {}
        s, H = {}, d["n_head"]
        hd, hv = H * d["dim"], H * d["vdim"]
        if d["mixer"] == lib.MIXER_LATENT:
            s["mix_q"] = (H * (d["dim"] + d["rot_dim"]), w)
            if d["kv_from"] < 0:
                s["mix_dkv"] = (d["kv_rank"] + d["rot_dim"], w)
            s["mix_uk"], s["mix_uv"] = (hd, d["kv_rank"]), (hv, d["kv_rank"])
        elif d["mixer"] == lib.MIXER_GROUPED:
            G = d["n_kv_head"]
            s["mix_q"], s["mix_k"] = (hd, w), (G * d["dim"], w)
            if self.case["model"] != "pibalorn":                    # Pibalorn's values are its keys
                s["mix_v"] = (G * d["vdim"], w)
            if d.get("head_mix"):
                s["mix_head_gate"] = (H, w)
            if d.get("mem_heads"):
                M = d["mem_heads"]
                for k in ("mem_q", "mem_k"):
                    s[k] = (M * d["mem_dim"], w)
                for k in ("mem_v", "mem_g"):
                    s[k] = (M * d["mem_vdim"], w)
                s["mem_i"] = s["mem_f"] = (M, w)
                s["mem_o"] = (w, M * d["mem_vdim"])
        else:
            s["mix_q"] = s["mix_k"] = (hd, w)
            s["mix_v"] = s["mix_g"] = (hv, w)
            if d["mixer"] == lib.MIXER_KEYED:
                s["mix_a1"], s["mix_a2"] = (RANK, w), (hd, RANK)
        s["wo"] = (w, hv)
        if d.get("gated_residual"):
            s["res_gate"] = s["res_gate_ffn"] = (w, w)
        if d.get("glu_ff"):
            s["glu_gate"] = s["glu_up"] = (d["glu_ff"], w)
            s["glu_down"] = (w, d["glu_ff"])
        if d.get("n_expert"):
            E, f = d["n_expert"], d["expert_ff"]
            s["router"] = (E, w)
            if d["ffn"] == lib.FFN_GLU_MOE:
                s["expert_gate"] = (E * f, w)
            s["expert_up"], s["expert_down"] = (E * f, w), (E * w, f)
            if d.get("glu_ff"):
                s["shared_score"] = (1, w)
        return s

    def matrix(self, i, role, shape):
        w = self.case["width"]
        x = self.src.normal((i, role), *shape, {"tok_embd": EMBED, "bigram": EMBED / 4, "router": 0.003}.get(role, 0.02), BF16)
        if self.case["model"] == "fikevik":                          # nothing is routed
            return x
        first = w - ROUTES
        if role in ("tok_embd", "bigram"):
            x[:, first:] = 0
            if role == "tok_embd":
                ids = torch.arange(shape[0], device=x.device)
                x[ids, first + ids % ROUTES] = 2.0
        elif role in ("wo", "glu_down"):
            x[first:] = 0
        elif role == "expert_down":
            x.view(-1, w, shape[1])[:, first:] = 0
        elif role == "router":
            rng = self.src.host(i, "routes")
            for c in range(ROUTES):
                x[torch.from_numpy(self.experts(rng, shape[0])).to(x.device), first + c] = {"lerasun": 1.0, "pibalorn": 10.0, "pufivik": 3.0}[self.case["model"]]
        return x

    def experts(self, rng, n):
        """A class's experts: with eight groups of experts, two in each of two groups and one in each of two."""
        if self.case["model"] != "lerasun":
            return rng.permutation(n)[:TOP]
        size, out = n // 8, []
        for g, k in zip(rng.permutation(8)[:4], (2, 2, 1, 1)):
            out += (g * size + rng.permutation(size)[:k]).tolist()
        return np.asarray(out)

    def vectors(self, i):
        """float32 vectors of a layer by role."""
        d, w, name = self.descs[i], self.case["width"], self.case["model"]
        if d.get("weights_of"):
            return {}
        one, f32, rng, H = np.ones(w, np.float32), np.float32, self.src.host(i, "vectors"), d["n_head"]
        if name == "lerasun":
            v = {"attn_norm": 0 * one, "ffn_norm": 0 * one, "mix_sink": rng.standard_normal(H).astype(f32), "router_bias": np.zeros(d["n_expert"], f32)}
            if d["kv_from"] < 0:
                v["mix_dkv_norm"] = np.ones(d["kv_rank"], f32)
            return v
        if name == "pibalorn":
            v = {"attn_norm": one}
            if d["mixer"] == lib.MIXER_LINEAR:
                v["mix_norm"], v["mix_decay"] = np.ones(H * d["vdim"], f32), np.asarray(self.cfg["layers"][i]["mixer"]["decay"], f32)
            return v
        if name == "fikevik":
            v = {"attn_norm": one, "ffn_norm": one, "res_gate_b": 0 * one, "res_gate_ffn_b": 0 * one}
            if d["mixer"] == lib.MIXER_KEYED:
                v["mix_a2_b"], v["mix_norm"] = rng.standard_normal(H * d["dim"]).astype(f32), np.ones(H * d["vdim"], f32)
            else:
                M = d["mem_heads"]
                v.update(mix_q_norm=np.ones(d["dim"], f32), mix_k_norm=np.ones(d["dim"], f32), mix_temp=np.ones(H, f32), mem_norm=np.ones(M * d["mem_vdim"], f32),
                         mem_i_b=np.zeros(M, f32), mem_f_b=np.full(M, 4, f32))
            return v
        v = {k: one for k in ("attn_norm", "attn_norm_after", "ffn_norm", "ffn_norm_after")}
        v["mix_conv"] = (0.2 * rng.standard_normal((self.cfg["canon"]["taps"], w))).astype(f32)
        if i:
            v["mix_value"] = np.full(1, 0.4, f32)
        if d.get("head_mix"):
            v["mix_sink"] = rng.standard_normal(H).astype(f32)
            v["mix_talk"] = (np.eye(H) + 0.1 * rng.standard_normal((H, H)) / H ** 0.5).astype(f32)
        return v


def requests_of(case, seed):
    """Token lists of the prompts, and [steps, n_seq] tokens behind them."""
    rng = np.random.default_rng([seed, 99])
    prompts = [rng.integers(0, VOCAB, n).astype(np.int32) for n in cut(case["prompt"], case["n_seq"])]
    return prompts, rng.integers(0, VOCAB, (case["steps"], case["n_seq"])).astype(np.int32)


def prepare_request(case, seed):
    t, w, name, held = DesignTensors(case, seed), case["width"], case["model"], []
    prompts, then = requests_of(case, seed)
    cells = (sum(map(len, prompts)) + then.size + 32) // 32 * 32
    opts = {"lerasun": lambda: dict(norm_offset=lerasun.NORM_OFFSET), "pibalorn": lambda: pibalorn.model_opts(t.cfg), "fikevik": lambda: fikevik.model_opts(t.cfg),
            "pufivik": lambda: pufivik.model_opts(t.cfg)}[name]()
    m = LayerModel(name, t.descs, n_embd=w, n_vocab=VOCAB, n_ctx=cells, norm_eps=t.cfg["norm"]["eps"], **opts)

    def put(layer, role, shape):
        x = t.matrix(layer, role, shape)
        held.append(x)
        m.set_tensor_device(layer, role, x.data_ptr(), lib.BF16, shape[1], shape[0])

    for role, shape in whole_shapes(case).items():
        put(-1, role, shape)
    if name == "pufivik":                                            # its output matrix is its embedding
        m.set_tensor_device(-1, "output", held[0].data_ptr(), lib.BF16, w, VOCAB)
    m.set_tensor(-1, "output_norm", np.full(w, 0 if name == "lerasun" else 1, np.float32))
    if name == "lerasun":
        m.set_tensor(-1, "embd_norm", np.zeros(w, np.float32))
    if name == "pibalorn":
        m.set_tensor(-1, "loop_step", np.zeros((t.cfg["loop"]["times"], w), np.float32))
    for i in range(len(t.descs)):
        for role, v in t.vectors(i).items():
            m.set_tensor(i, role, v)
        for role, shape in t.shapes(i).items():
            put(i, role, shape)
    torch.cuda.synchronize()
    m.finalize()
    if case["n_seq"] > 1:
        m.kv_cells_init(cells)
    return dict(case=case, model=m, held=held, prompts=prompts, then=then)


def whole_shapes(case):
    s = {"tok_embd": (VOCAB, case["width"])}
    if case["model"] != "pufivik":
        s["output"] = (VOCAB, case["width"])
    if case["model"] == "pibalorn":
        s["bigram"] = (9974, case["width"])
    return s


def run_request(state):
    """The prompts, read together, and a token of every request per step: the logits behind the prompts, then those of every step."""
    m, prompts, then = state["model"], state["prompts"], state["then"]
    n = len(prompts)
    if n == 1:
        m.kv_clear()
        past = len(prompts[0])
        return [m.decode(prompts[0], 0)[1]] + [m.decode(toks, past + k)[1] for k, toks in enumerate(then)]
    m.kv_cells_clear()
    at = np.array([len(p) for p in prompts])
    tokens, masks = np.concatenate(prompts), np.repeat(np.uint32(1) << np.arange(n, dtype=np.uint32), at)
    out = [m.kv_cells_step(tokens, np.concatenate([np.arange(k) for k in at]), masks, np.cumsum(at) - 1, want_next=False)[1]]
    for k, toks in enumerate(then):
        out.append(m.kv_cells_step(toks, at + k, np.uint32(1) << np.arange(n, dtype=np.uint32), np.arange(n), want_next=False)[1])
    return out


def silu(z):
    return z * torch.sigmoid(z)


class ExactDesign:
    """The four designs in 64 bits: all tokens of all requests at once, mixers request by request."""

    def __init__(self, case, seed):
        self.case, self.t = case, DesignTensors(case, seed)
        self.cfg, self.w = self.t.cfg, case["width"]
        prompts, then = requests_of(case, seed)
        seqs = [np.concatenate([p, then[:, s]]) for s, p in enumerate(prompts)]
        self.lens, ends = [len(s) for s in seqs], np.cumsum([0] + [len(s) for s in seqs])
        self.parts = [slice(a, b) for a, b in zip(ends[:-1], ends[1:])]
        self.tokens = torch.as_tensor(np.concatenate(seqs), device="cuda").long()
        self.pos = [torch.arange(n, device="cuda") for n in self.lens]
        self.wanted = [[ends[s] + len(p) - 1 + k for s, p in enumerate(prompts)] for k in range(case["steps"] + 1)]

    def g(self, i, role):
        """A layer's tensor in 64 bits (a layer without weights of its own has its owner's)."""
        i = self.owner(i)
        v = self.t.vectors(i) if i >= 0 else {}
        if role in v:
            return torch.as_tensor(v[role], device="cuda").to(F64)
        return self.t.matrix(i, role, (self.t.shapes(i) if i >= 0 else whole_shapes(self.case))[role]).to(F64)

    def owner(self, i):
        return self.t.descs[i]["weights_of"] - 1 if i >= 0 and self.t.descs[i].get("weights_of") else i

    def project(self, i, h, role, heads=None):
        y = h @ self.g(i, role).T
        return y if heads is None else y.reshape(len(h), heads, -1)

    def attend(self, q, k, v, pos, scale, weights):
        """weights(scores [n, n] masked, head): what multiplies the values; [n, H, vdim]."""
        n, H = q.shape[:2]
        per, later = H // k.shape[1], pos[None] > pos[:, None]
        return torch.stack([weights((q[:, a] @ k[:, a // per].T * scale), later, a) @ v[:, a // per] for a in range(H)], 1)

    def mixture(self, i, h, ids, wts, expert):
        out, f = torch.zeros(len(h), self.w, dtype=F64, device="cuda"), self.t.descs[i]["expert_ff"]
        mats = {r: self.t.matrix(i, r, s) for r, s in self.t.shapes(i).items() if r.startswith("expert_")}
        for e in range(self.t.descs[i]["n_expert"]):
            at, slot = (ids == e).nonzero(as_tuple=True)
            if len(at):
                part = {r[7:]: m[e * (self.w if r == "expert_down" else f):(e + 1) * (self.w if r == "expert_down" else f)].to(F64) for r, m in mats.items()}
                out.index_add_(0, at, expert(h[at], wts[at, slot][:, None], part))
        return out

    # Lerasun
    def latent(self, i, h):
        d, H, eps = self.t.descs[i], self.t.descs[i]["n_head"], 1e-6
        D, R, freq, outs = d["dim"], d["rot_dim"], frequencies(d["rot_dim"], d["rot_base"]), []
        q = self.project(i, h, "mix_q", H)
        if d["kv_from"] < 0:
            z = self.project(i, h, "mix_dkv")
            self.lat, self.shared = rms(z[:, :d["kv_rank"]], eps), z[:, d["kv_rank"]:]
        k, v, sink = self.project(i, self.lat, "mix_uk", H), self.project(i, self.lat, "mix_uv", H), self.g(i, "mix_sink")

        def weights(s, later, a):
            s = s.masked_fill(later, -math.inf)
            top = s.max(1, keepdim=True)[0].clamp(min=float(sink[a]))
            e = torch.exp(s - top)
            return e / (e.sum(1, keepdim=True) + torch.exp(sink[a] - top))

        for part, pos in zip(self.parts, self.pos):
            qr, kr = rotated(q[part, :, D:], pos, R, freq, True), rotated(self.shared[part][:, None], pos, R, freq, True)
            outs.append(self.attend(torch.cat([q[part, :, :D], qr], 2), torch.cat([k[part], kr.expand(-1, H, -1)], 2), v[part], pos, d["scale"], weights))
        return torch.cat(outs).reshape(len(h), -1) @ self.g(i, "wo").T

    def lerasun(self, x):
        x = rms(x, 1e-6)
        for i, d in enumerate(self.t.descs):
            h = rms(x, 1e-6)
            s = torch.sigmoid(h @ self.g(i, "router").T)
            groups = s.reshape(len(s), d["n_group"], -1)
            kept = groups.topk(2, 2)[0].sum(2).topk(d["n_group_keep"], 1)[1]
            open_ = torch.zeros_like(groups, dtype=torch.bool).scatter_(1, kept[..., None].expand(-1, -1, groups.shape[2]), True).reshape(s.shape)
            ids = s.masked_fill(~open_, -1).topk(d["n_top"], 1)[1]
            wts = s.gather(1, ids)
            x = x + self.latent(i, h) + self.mixture(i, h, ids, wts / (wts.sum(1, keepdim=True) + 1e-20), lambda v, f, m: f * (torch.relu(v @ m["up"].T).square() @ m["down"].T))
        return rms(x, 1e-6)

    # Pibalorn
    def lightning(self, i, h):
        d, H = self.t.descs[i], self.t.descs[i]["n_head"]
        q, k, v = (silu(self.project(i, h, r, H)) for r in ("mix_q", "mix_k", "mix_v"))
        decay, out = self.g(i, "mix_decay")[:, None, None], torch.empty_like(v)
        for part in self.parts:
            state = torch.zeros(H, d["dim"], d["vdim"], dtype=F64, device="cuda")
            for t in range(part.start, part.stop):
                state = decay * state + k[t][:, :, None] * v[t][:, None]
                out[t] = (q[t][:, None] @ state)[:, 0]
        return rms(out.reshape(len(h), -1), 1e-6) * self.g(i, "mix_norm") * torch.sigmoid(self.project(i, h, "mix_g"))

    def unit_attention(self, i, h):
        d, freq, outs = self.t.descs[i], frequencies(self.t.descs[i]["rot_dim"], self.t.descs[i]["rot_base"]), []
        q, v = self.project(i, h, "mix_q", d["n_head"]), self.project(i, h, "mix_k", d["n_kv_head"])

        def weights(s, later, a):
            s = s.masked_fill(later, -math.inf)
            top = s.max(1, keepdim=True)[0].clamp(min=0)
            e = torch.exp(s - top)
            return e / (e.sum(1, keepdim=True) + torch.exp(-top))

        for part, pos in zip(self.parts, self.pos):
            turn = lambda y: rms(rotated(y[part], pos, d["rot_dim"], freq, False), 1e-6)  # noqa: E731, B023
            outs.append(self.attend(turn(q), turn(v), v[part], pos, d["scale"], weights))
        return torch.cat(outs).reshape(len(h), -1)

    def clamped(self, h, gate, up, down, limit=7.0):
        g, u = (h @ gate.T).clamp(max=limit), (h @ up.T).clamp(-limit, limit)
        return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ down.T

    def pibalorn(self, x):
        b, cfg = self.cfg["embedding"]["bigram"], self.cfg
        rows = torch.full_like(self.tokens, b["buckets"])
        for part in self.parts:
            t = self.tokens[part]
            rows[part.start + 1:part.stop] = (t[:-1] * b["mul_prev"] + t[1:] * b["mul_cur"]) % b["buckets"]
        x0 = x = x + self.g(-1, "bigram")[rows]
        lo, order = cfg["loop"], []
        for p in range(lo["times"]):
            order += [(i, p if i == lo["start"] else 0) for i in range(lo["start"], lo["stop"])]
        order = [(i, 0) for i in range(lo["start"])] + order + [(i, 0) for i in range(lo["stop"], len(cfg["layers"]))]
        for i, again in order:
            if again:
                x = x + x0
            h = layer_norm(x, 1e-6)
            y = (self.lightning if self.t.descs[i]["mixer"] == lib.MIXER_LINEAR else self.unit_attention)(i, h) @ self.g(i, "wo").T
            glu = self.clamped(h, *(self.g(i, r) for r in ("glu_gate", "glu_up", "glu_down")))
            if "router" in self.t.shapes(i):
                z, ids = (h @ self.g(i, "router").T).topk(TOP, 1)
                glu = torch.sigmoid(h @ self.g(i, "shared_score").T) * glu
                glu = glu + self.mixture(i, h, ids, torch.softmax(z, 1), lambda v, f, m: f * self.clamped(v, m["gate"], m["up"], m["down"]))
            x = x + y + glu
        return layer_norm(x, 1e-6)

    # Fikevik
    def gla(self, i, h):
        d, H = self.t.descs[i], self.t.descs[i]["n_head"]
        q, k, v = (self.project(i, h, r, H) for r in ("mix_q", "mix_k", "mix_v"))
        z = self.project(i, h, "mix_a1") @ self.g(i, "mix_a2").T + self.g(i, "mix_a2_b")
        decay, out = torch.exp(torch.nn.functional.logsigmoid(z) / d["decay_tau"]).reshape(len(h), H, -1), torch.empty_like(v)
        for part in self.parts:
            state = torch.zeros(H, d["dim"], d["vdim"], dtype=F64, device="cuda")
            for t in range(part.start, part.stop):
                state = decay[t][:, :, None] * state + k[t][:, :, None] * v[t][:, None]
                out[t] = (q[t][:, None] * d["dim"] ** -0.5 @ state)[:, 0]
        return (rms(out, 1e-6).reshape(len(h), -1) * self.g(i, "mix_norm") * silu(self.project(i, h, "mix_g"))) @ self.g(i, "wo").T

    def window_and_memory(self, i, h):
        d, freq, outs = self.t.descs[i], frequencies(self.t.descs[i]["rot_dim"], self.t.descs[i]["rot_base"]), []
        q, k, v = self.project(i, h, "mix_q", d["n_head"]), self.project(i, h, "mix_k", d["n_kv_head"]), rms(self.project(i, h, "mix_v", d["n_kv_head"]), 1e-6)
        for part, pos in zip(self.parts, self.pos):
            old = pos[:, None] - pos[None] >= d["window"]
            turn = lambda y: rotated(rms(y[part], 1e-6), pos, d["rot_dim"], freq, True)  # noqa: E731, B023
            outs.append(self.attend(turn(q), turn(k), v[part], pos, d["scale"], lambda s, later, a: torch.softmax(s.masked_fill(later | old, -math.inf), 1)))  # noqa: B023
        left = torch.cat(outs).reshape(len(h), -1) @ self.g(i, "wo").T
        M, cap = d["mem_heads"], d["mem_cap"]
        q, k, v = (self.project(i, h, r, M) for r in ("mem_q", "mem_k", "mem_v"))
        q, soft, out = q * d["mem_dim"] ** -0.5, lambda z: cap * torch.tanh(z / cap), torch.empty_like(v)
        gi = soft(self.project(i, h, "mem_i") + self.g(i, "mem_i_b"))
        gf = torch.nn.functional.logsigmoid(soft(self.project(i, h, "mem_f") + self.g(i, "mem_f_b")))
        for part in self.parts:
            s, z, m = torch.zeros(M, d["mem_dim"], d["mem_vdim"], dtype=F64, device="cuda"), torch.zeros(M, d["mem_dim"], dtype=F64, device="cuda"), torch.zeros(M, dtype=F64, device="cuda")
            for t in range(part.start, part.stop):
                top = torch.maximum(gf[t] + m, gi[t])
                keep, add, m = torch.exp(gf[t] + m - top), torch.exp(gi[t] - top), top
                s = keep[:, None, None] * s + (add[:, None] * k[t])[:, :, None] * v[t][:, None]
                z = keep[:, None] * z + add[:, None] * k[t]
                den = torch.maximum((z * q[t]).sum(1).abs(), torch.exp(-m)) + 1e-6
                out[t] = (q[t][:, None] @ s)[:, 0] / den[:, None]
        right = (rms(out, 1e-6).reshape(len(h), -1) * self.g(i, "mem_norm") * torch.sigmoid(self.project(i, h, "mem_g"))) @ self.g(i, "mem_o").T
        return d["out_scale"] * left + d["mem_scale"] * right

    def fikevik(self, x):
        alpha = self.cfg["postln_alpha"]
        for i, d in enumerate(self.t.descs):
            y = (self.gla if d["mixer"] == lib.MIXER_KEYED else self.window_and_memory)(i, x)
            x = rms(alpha * x + y * torch.sigmoid(x @ self.g(i, "res_gate").T), 1e-6)
            y = (silu(x @ self.g(i, "glu_gate").T) * (x @ self.g(i, "glu_up").T)) @ self.g(i, "glu_down").T
            x = rms(alpha * x + y * torch.sigmoid(x @ self.g(i, "res_gate_ffn").T), 1e-6)
        return rms(x, 1e-6)

    # Pufivik
    def scaled_frequencies(self, rot, kind):
        f, s, dims = frequencies(rot["dims"], rot["base"]), rot["scaling"], rot["dims"]
        if kind == "attention":
            turns = s["original"] * f / (2 * math.pi)
            a = ((turns - s["low"]) / (s["high"] - s["low"])).clamp(0, 1)
            return (1 - a) * f / s["factor"] + a * f, 1.0
        at = lambda turns: dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))  # noqa: E731
        lo, hi = max(math.floor(at(s["fast"])), 0), min(math.ceil(at(s["slow"])), dims - 1)
        ramp = ((torch.arange(dims // 2, device="cuda", dtype=F64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        return f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1

    def mixed_attention(self, i, h):
        d, ly = self.t.descs[i], self.cfg["layers"][i]
        m, kind, n_head = ly["mixer"], ly["type"], d["n_head"]
        q, k, v = self.project(i, h, "mix_q", n_head), self.project(i, h, "mix_k", d["n_kv_head"]), self.project(i, h, "mix_v", d["n_kv_head"])
        if i == 0:
            self.first_values = v
        else:
            lam = self.g(i, "mix_value")
            v = (1 - lam) * v + lam * self.first_values
        freq, length = self.scaled_frequencies(m["rot"], kind)
        outs = []
        for part, pos in zip(self.parts, self.pos):
            qp, kp = (rotated(y[part], pos, m["rot"]["dims"], freq, kind != "attention", length) for y in (q, k))
            if kind == "attention_2":
                outs.append(self.attend(qp, kp, v[part], pos, m["scale"], lambda s, later, a: torch.softmax((m["softcap"] * torch.tanh(s / m["softcap"])).masked_fill(later, -math.inf), 1)))
                continue
            later, per = pos[None] > pos[:, None], n_head // d["n_kv_head"]
            sink, talk = self.g(i, "mix_sink"), self.g(i, "mix_talk")
            s = torch.stack([qp[:, a] @ kp[:, a // per].T for a in range(n_head)]) * m["scale"]
            s = s.masked_fill(later, -math.inf)
            top = torch.maximum(s.max(2, keepdim=True)[0], sink[:, None, None])
            e = torch.exp(s - top)
            wts = e / (e.sum(2, keepdim=True) + torch.exp(sink[:, None, None] - top))
            wts = (talk @ wts.reshape(n_head, -1)).reshape(wts.shape)
            o = torch.stack([wts[a] @ v[part][:, a // per] for a in range(n_head)], 1)
            outs.append(o * torch.sigmoid(h[part] @ self.g(i, "mix_head_gate").T)[:, :, None])
        return torch.cat(outs).reshape(len(h), -1) @ self.g(i, "wo").T

    def pufivik(self, x):
        groups, mult = self.cfg["norm"]["groups"], self.cfg["residual_mult"]
        norm = lambda y: rms(y.reshape(len(y), groups, -1), 1e-6).reshape(y.shape)  # noqa: E731
        for i in range(len(self.t.descs)):
            h, taps = norm(x), self.g(i, "mix_conv")
            c = h.clone()
            for part in self.parts:
                rows = torch.cat([torch.zeros(len(taps) - 1, self.w, dtype=F64, device="cuda"), h[part]])
                c[part] += sum(taps[j] * rows[j:j + part.stop - part.start] for j in range(len(taps)))
            x = x + mult * norm(self.mixed_attention(i, c))
            h = norm(x)
            s, ids = torch.sigmoid(h @ self.g(i, "router").T).topk(TOP, 1)
            x = x + mult * norm(self.mixture(i, h, ids, s, lambda v, f, m: (silu(f * v @ m["gate"].T) * (f * v @ m["up"].T)) @ m["down"].T))
        return norm(x)

    def logits(self):
        x = getattr(self, self.case["model"])(self.g(-1, "tok_embd")[self.tokens])
        head = self.g(-1, "tok_embd" if self.case["model"] == "pufivik" else "output").T
        got = [(x[rows] @ head).cpu().numpy() for rows in self.wanted]
        return [g[0] for g in got] if self.case["n_seq"] == 1 else got


def work_request(case):
    t = DesignTensors(case, 0)
    tokens, steps, n_seq = sum(cut(case["prompt"], case["n_seq"])), case["steps"], case["n_seq"]
    runs = list(range(len(t.descs)))
    if case["model"] == "pibalorn":
        lo = t.cfg["loop"]
        runs += list(range(lo["start"], lo["stop"])) * (lo["times"] - 1)
    total = {"bytes": 0.0, "flops": 0.0}
    for n, times, past in ((tokens, 1, 0), (n_seq, steps, case["prompt"])):              # the step of prompts, those of single tokens
        head = VOCAB * case["width"]
        b, f = head * 2.0 + n_seq * VOCAB * 4, n_seq * 2.0 * head
        for i in runs:
            d = t.descs[i]
            own = d["weights_of"] - 1 if d.get("weights_of") else i
            for role, (r, c) in t.shapes(own).items():
                used = 1.0
                if role.startswith("expert_"):
                    used = 1 - (1 - TOP / d["n_expert"]) ** n
                    f += n * 2.0 * r * c * TOP / d["n_expert"]
                elif role not in ("mix_uk", "mix_uv"):
                    f += n * 2.0 * r * c
                b += 2.0 * r * c * used
            if d["mixer"] in (lib.MIXER_GROUPED, lib.MIXER_LATENT):
                cells = past + 1 if past else case["prompt"] / 2
                cells = min(cells, d.get("window") or cells)
                f += n * cells * d["n_head"] * 2.0 * (d["dim"] + d["rot_dim"] * (d["mixer"] == lib.MIXER_LATENT) + d["vdim"])
                cell = d["kv_rank"] + d["rot_dim"] if d["mixer"] == lib.MIXER_LATENT else d["n_kv_head"] * (d["dim"] + d["vdim"])
                b += 2.0 * cell * (n + (n_seq * cells if past else 0))
            heads, size = (d.get("mem_heads") or 0, d.get("mem_dim", 0) * d.get("mem_vdim", 0)) if d["mixer"] == lib.MIXER_GROUPED else (d["n_head"], d["dim"] * d["vdim"])
            if d["mixer"] != lib.MIXER_LATENT and heads:
                f += n * heads * size * 4.0
                b += n_seq * heads * size * 4.0 * (2 if past else 1)
        total["bytes"] += times * b
        total["flops"] += times * f
    return total


# ---- the entry points ---------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    return (prepare_request if case["kind"] == "request" else prepare_sparse)(case, seed)


def run(state):
    return (run_request if state["case"]["kind"] == "request" else run_sparse)(state)


def exact(case, seed):
    return ExactDesign(case, seed).logits() if case["kind"] == "request" else exact_sparse(case, seed)


def work(case):
    return (work_request if case["kind"] == "request" else work_sparse)(case)


def tolerance(case):
    """About four times what the paths differ by from 64 bits: fp16 0.0003 to 0.0025; bf16 0.003 to 0.02 (mixed heads); Q4_0 0.017 to 0.028,
    whose activations are rounded to eight bits between the matrices."""
    if case["kind"] == "request":
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 0.03, "max": 0.4} if case["wtype"] == "q4_0" else {"rel": 0.008, "max": 0.06}
