"""What the framework is measured on: passes through its public entry points over the range that it serves.

Four kinds of programs use it, and each gives cases:

  decode         one token for each of `batch` sequences of a W4A8KV4 Llama (runtime.DecodeRunner.step, a captured step).
  prefill        the context stage of the same model over `batch` prompts of `prompt` tokens (runtime.DecodeRunner.prefill).
  lserve_decode  four tokens of a W8A8 LServe Llama over a long context, one selection of pages among them
                 (lserve_runtime.LServeDecodeRunner.step).
  lserve_prefill its context stage, half of the kv heads streaming (LServeDecodeRunner.prefill).
  engine         a trace on the serving engine (engine.Engine.open / run / close): `seqs` prompts in one step, then `steps` single tokens
                 of every sequence, the logits of each step's last tokens.

Layer sizes are the ones of bench.py and engine/benchmark.py; models have a few layers and, of the vocabulary, about the same share."""
import math

import torch

from omniserve_amd.ckpt import load_into_runner
from omniserve_amd.engine import Engine, SequenceInput
from omniserve_amd.lserve_runtime import LServeDecodeRunner
from omniserve_amd.models.bagedra import Bagedra
from omniserve_amd.models.bobavik import Bobavik
from omniserve_amd.runtime import DecodeRunner, LlamaConfig

DEV = "cuda"

LLAMA = {
    "8b": dict(hidden=4096, inter=14336, heads=32, kv_heads=8, vocab=32000, rope_theta=500000.0),
    "70b": dict(hidden=8192, inter=28672, heads=64, kv_heads=8, vocab=16000, rope_theta=10000.0),
}
# (experts, top, ff, shared, window: Bobavik; kv_heads of the delta rule, latent, its turned part, ff: Bagedra)
BOBAVIK = {
    "4096": dict(width=4096, heads=32, kv_heads=8, experts=32, top=6, ff=1792, shared=3584, window=4096, vocab=32000),
    "2048": dict(width=2048, heads=16, kv_heads=4, experts=64, top=8, ff=640, shared=1024, window=1024, vocab=32000),
}
BAGEDRA = {
    "4096": dict(width=4096, heads=32, kv_heads=16, kv_rank=512, rot_dim=64, rank=16, ff=14336, vocab=32000),
    "2048": dict(width=2048, heads=16, kv_heads=8, kv_rank=256, rot_dim=64, rank=16, ff=6144, vocab=32000),
}
BOBAVIK_LAYERS = ("attention", "lightning", "lightning", "attention", "lightning", "attention")
BAGEDRA_LAYERS = ("gla", "delta", "latent_attention", "gla", "delta", "latent_attention")
HEAD = 128
# what a sublayer adds, of the residual it adds to: trained models' layers change little of it, random ones of unit gain would all of it, and
# would turn every rounding of a code into another model
UPDATE = 0.04
SINK, LOCAL, CTX_SINK, CTX_LOCAL, BUDGET = 128, 256, 128, 8192, 4096      # LServe's published settings


def listed():
    return [
        # one user's chat: a single short sequence, where a step is a chain of short launches
        dict(name="decode 1 sequence", kind="decode", size="8b", group=-1, batch=1, context=300),
        # the framework's headline: 16 sequences of 1024 tokens
        dict(name="decode 16 sequences", kind="decode", size="8b", group=-1, batch=16, context=1024),
        # a server at ordinary load, weights with groups of 128, lengths and batch as they come
        dict(name="decode 61 sequences g128", kind="decode", size="8b", group=128, batch=61, context=1100),
        # the large model at high load
        dict(name="decode 120 sequences 70b", kind="decode", size="70b", group=-1, batch=120, context=900),
        # one prompt of ordinary length
        dict(name="prefill 1 x 1501", kind="prefill", size="8b", group=-1, batch=1, prompt=1501),
        # several short prompts at once, weights with groups
        dict(name="prefill 7 x 333 g128", kind="prefill", size="8b", group=128, batch=7, prompt=333),
        # long-context serving: the context stage and a token behind 100 000
        dict(name="LServe prefill 1 x 12001", kind="lserve_prefill", kv="kv8", batch=1, prompt=12001),
        dict(name="LServe decode 100000", kind="lserve_decode", kv="kv8", batch=1, context=100000),
        # chat turns on the engine: prompts of some hundred tokens and answers behind them
        dict(name="Bobavik turn 16 x 500", kind="engine", arch="Bobavik", size="2048", seqs=16, prompt=500, steps=24),
        dict(name="Bagedra turn 48 x 150", kind="engine", arch="Bagedra", size="4096", seqs=48, prompt=150, steps=24),
        # a long document read in one step
        dict(name="Bobavik prompt 1 x 7999", kind="engine", arch="Bobavik", size="4096", seqs=1, prompt=7999, steps=0),
        dict(name="Bagedra prompts 2 x 8000", kind="engine", arch="Bagedra", size="2048", seqs=2, prompt=8000, steps=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "lserve_prefill", "lserve_decode", "engine", "engine", "engine", "engine"))
    if kind == "decode":
        size = rng.choice(("8b", "8b", "70b"))
        batch = _log(rng, 1, 200 if size == "8b" else 120)
        return dict(kind=kind, size=size, group=rng.choice((-1, 128)), batch=batch, context=_log(rng, 100, min(6000, 160000 // batch)))
    if kind == "prefill":
        prompt = _log(rng, 17, 4000)
        return dict(kind=kind, size="8b", group=rng.choice((-1, 128)), batch=_log(rng, 1, max(1, min(16, 6000 // prompt))), prompt=prompt)
    if kind == "lserve_prefill":
        return dict(kind=kind, kv=rng.choice(("kv8", "kv4")), batch=1, prompt=_log(rng, 2500, 12001))
    if kind == "lserve_decode":
        return dict(kind=kind, kv=rng.choice(("kv8", "kv4")), batch=1, context=_log(rng, 8000, 128000))
    arch, size = rng.choice(("Bobavik", "Bagedra")), rng.choice(("2048", "4096"))
    if rng.random() < 0.6:
        seqs = _log(rng, 1, 60)
        return dict(kind=kind, arch=arch, size=size, seqs=seqs, prompt=_log(rng, 20, min(1500, 6000 // seqs)), steps=rng.randint(12, 24))
    prompt = _log(rng, 100, 7000)
    return dict(kind=kind, arch=arch, size=size, seqs=_log(rng, 1, max(1, min(16, 7000 // prompt))), prompt=prompt, steps=0)


# ---------------------------------------------------------------------------------------------------------------------
# inputs: plain tensors, drawn from the seed alone
# ---------------------------------------------------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * seed + 17)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _ids(g, vocab, n):
    return torch.randint(0, vocab, (n,), generator=g, device=DEV)


def _w4(g, n, k, group, gain=1.0):
    """Packed 4-bit weights: codes of a bell curve around the zero point, as a quantiser leaves them."""
    code = lambda: (7.5 + 2.6 * torch.randn((n, k // 2), generator=g, device=DEV, dtype=torch.float16)).round_().clamp_(0, 15).to(torch.uint8)      # noqa: E731
    w = {"qweight": (code() | (code() << 4)).view(torch.int8)}
    spread = gain * (0.8 + 0.4 * torch.rand((n,), generator=g, device=DEV)) / (2.6 * k ** 0.5)
    if group == -1:
        w["s1_scales"] = spread.half()
        w["s1_szeros"] = (torch.randint(7, 9, (n,), generator=g, device=DEV).half() * w["s1_scales"]).half()
        return w
    s2 = torch.randint(6, 14, (k // group, n), generator=g, device=DEV)
    w["s1_scales"] = (spread / 9.5).half()
    w["s2_scales"] = s2.to(torch.int8)
    w["s2_zeros"] = (-(torch.randint(7, 9, (k // group, n), generator=g, device=DEV) * s2)).to(torch.int8)
    return w


def _llama_state(case, g):
    """A checkpoint in the QServe layout"""
    m, G = LLAMA[case["size"]], case["group"]
    H, kv = m["hidden"], m["kv_heads"] * HEAD
    s = {"model.embed_tokens.weight": _randn(g, m["vocab"], H).half(), "lm_head.weight": (H ** -0.5 * _randn(g, m["vocab"], H)).half(),
         "model.norm.weight": (1 + 0.1 * _randn(g, H)).half()}
    for i in range(_layers(case)):
        p = "model.layers.%d." % i
        for n in ("input_layernorm", "post_attention_layernorm"):
            s[p + n + ".weight"] = (1 + 0.1 * _randn(g, H)).half()
        for name, n, k in (("self_attn.q_proj", H, H), ("self_attn.k_proj", kv, H), ("self_attn.v_proj", kv, H), ("self_attn.o_proj", H, H),
                           ("mlp.gate_proj", m["inter"], H), ("mlp.up_proj", m["inter"], H), ("mlp.down_proj", H, m["inter"])):
            s.update({p + name + "." + part: t for part, t in _w4(g, n, k, G, UPDATE if n == H and "q_" not in name else 1.0).items()})
    return s


def _lserve_state(g):
    m = LLAMA["8b"]
    H, qkv = m["hidden"], (m["heads"] + 2 * m["kv_heads"]) * HEAD
    layers = []
    for _ in range(4):
        L = {n: (1 + 0.1 * _randn(g, H)).half() for n in ("ln1", "ln2")}
        for name, n, k in (("qkv", qkv, H), ("o", H, H), ("gate_up", 2 * m["inter"], H), ("down", H, m["inter"])):
            w = (32 * torch.randn((n, k), generator=g, device=DEV, dtype=torch.float16)).round_().clamp_(-127, 127).to(torch.int8)
            gain = (UPDATE if name in ("o", "down") else 1.0) / (32 * k ** 0.5)
            L[name] = (w, (gain * (0.8 + 0.4 * torch.rand((n,), generator=g, device=DEV))).half())
        layers.append(L)
    return {"layers": layers, "embed": _randn(g, m["vocab"], H).half(), "head": (H ** -0.5 * _randn(g, m["vocab"], H)).half(),
            "norm": (1 + 0.1 * _randn(g, H)).half()}


def _pages(g, m, batch, pages):
    """One layer's cache: codes [2, batch * pages, kv heads, 64, 64 bytes], scales (zero points are 7.5), places of the pages"""
    n, hk = batch * pages, m["kv_heads"]
    return (torch.randint(0, 256, (2, n, hk, 64, HEAD // 2), dtype=torch.uint8, generator=g, device=DEV),
            (0.25 + 0.25 * torch.rand((2, n, hk, 64), generator=g, device=DEV)).half(),
            [torch.randperm(n, generator=g, device=DEV).view(batch, pages) for _ in range(2)])


def _config(case):
    """A configuration of the engine's design, as its config.json holds it"""
    if case["arch"] == "Bobavik":
        s = BOBAVIK[case["size"]]
        mlp = {"kind": "moe", "expert": {"ff": s["ff"]}, "router": {"experts": s["experts"], "top": s["top"]}, "shared": {"ff": s["shared"]}}
        soft = {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": HEAD, "vdim": HEAD, "scale": HEAD ** -0.5, "v_mix": True,
                "mask": {"size": s["window"]}, "rot": {"dims": HEAD, "base": 500000.0}}
        lin = {"heads": s["heads"], "dim": HEAD, "vdim": HEAD, "decay": [0.9 + 0.099 * i / s["heads"] for i in range(s["heads"])]}
        return {"architecture": "Bobavik", "vocab": s["vocab"], "width": s["width"], "norm": {"eps": 1e-5}, "logit_scale": 1.0,
                "layers": [{"type": t, "mixer": soft if t == "attention" else lin, "mlp": mlp} for t in BOBAVIK_LAYERS]}
    s = BAGEDRA[case["size"]]
    mixers = {"latent_attention": {"heads": s["heads"], "dim": HEAD, "vdim": HEAD, "kv_rank": s["kv_rank"], "rot_dim": s["rot_dim"],
                                   "rot": {"dims": s["rot_dim"], "base": 500000.0}, "scale": (HEAD + s["rot_dim"]) ** -0.5},
              "gla": {"heads": s["heads"], "dim": HEAD, "vdim": HEAD, "tau": 16.0},
              "delta": {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": HEAD, "vdim": HEAD, "conv": 4}}
    return {"architecture": "Bagedra", "vocab": s["vocab"], "width": s["width"], "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
            "layers": [{"type": t, "mixer": mixers[t], "mlp": {"kind": "dense", "ff": s["ff"]}} for t in BAGEDRA_LAYERS]}


def _engine_state(case, g):
    """bf16 weights of unit gain; decays, step sizes and convolutions as such layers are initialised"""
    c = _config(case)
    W, bob, st = c["width"], c["architecture"] == "Bobavik", {}

    def mat(name, n, k, gain=1.0):
        st[name] = torch.randn((n, k), generator=g, device=DEV, dtype=torch.bfloat16).mul_(gain * k ** -0.5)

    def vec(name, n, spread=0.1, mean=1.0):
        st[name] = (mean + spread * _randn(g, n)).bfloat16()

    def norm(name):
        vec(name, W)
        if bob:
            vec(name + ".b", W, 0.05, 0.0)

    st["embed"] = _randn(g, c["vocab"], W).bfloat16()
    mat("head", c["vocab"], W)
    norm("final.norm")
    for i, l in enumerate(c["layers"]):
        p, m, x = "l%d." % i, l["mixer"], "l%d.mix." % i
        for n in ("norm1", "norm1b", "norm2", "norm2b") if bob else ("norm1", "norm2"):
            norm(p + n)
            if n.endswith("b") or not bob:               # behind a sublayer
                st[p + n] *= 5 * UPDATE
        H, D, E = m["heads"], m["dim"], m["vdim"]
        if l["type"] == "latent_attention":
            mat(x + "q", H * (D + m["rot_dim"]), W), mat(x + "dkv", m["kv_rank"] + m["rot_dim"], W), vec(x + "dkv.norm", m["kv_rank"])
            mat(x + "uk", H * D, m["kv_rank"]), mat(x + "uv", H * E, m["kv_rank"])
        else:
            qk = m["kv_heads"] if l["type"] == "delta" else H
            mat(x + "q", qk * D, W)
            mat(x + "k", (m["kv_heads"] if "kv_heads" in m else H) * D, W)
            mat(x + "v", (m["kv_heads"] if l["type"] == "attention" else H) * E, W)
        mat(x + "g", H * E, W), mat(x + "o", W, H * E)
        if l["type"] == "attention":
            st[x + "vmix"] = torch.tensor(0.4, device=DEV)
        if l["type"] == "lightning":
            vec(x + "norm", H * E)
        if l["type"] in ("gla", "delta"):
            vec(x + "norm", E)
        if l["type"] == "gla":
            r = BAGEDRA[case["size"]]["rank"]
            mat(x + "a1", r, W), mat(x + "a2", H * D, r), vec(x + "a2.b", H * D, 1.0, 2.0)
        if l["type"] == "delta":
            mat(x + "a", H, W), mat(x + "b", H, W)
            for n, h, size in (("q", m["kv_heads"], D), ("k", m["kv_heads"], D), ("v", H, E)):
                mat(x + n + ".conv", h * size, m["conv"])
            st[x + "A_log"] = torch.log(1 + 15 * torch.rand((H,), generator=g, device=DEV))
            dt = torch.exp(math.log(1e-3) + math.log(1e2) * torch.rand((H,), generator=g, device=DEV))
            st[x + "dt_bias"] = dt + torch.log(-torch.expm1(-dt))
        f, q = l["mlp"], p + "mlp."
        if bob:
            mat(q + "router", f["router"]["experts"], W), vec(q + "router.b", f["router"]["experts"], 0.1, 0.0)
            for n, ff in [("e%d." % e, f["expert"]["ff"]) for e in range(f["router"]["experts"])] + [("shared.", f["shared"]["ff"])]:
                mat(q + n + "gate", ff, W), mat(q + n + "up", ff, W), mat(q + n + "down", W, ff)
        else:
            for n, a, b in (("gate", f["ff"], W), ("up", f["ff"], W), ("down", W, f["ff"])):
                mat(q + n, a, b), vec(q + n + ".b", a, 0.02, 0.0)
    return c, st


def _lengths(case):
    """Prompts of a trace differ in length: `prompt` tokens and less."""
    n = case["prompt"]
    return [n - (37 * i) % (n // 3 + 1) for i in range(case["seqs"])]


def _trace(case, g, vocab):
    """Token ids of every sequence, its prompt and the tokens behind it"""
    return [_ids(g, vocab, n + case["steps"]) for n in _lengths(case)]


def _layers(case):
    return 8 if case["kind"] == "decode" and case["size"] == "8b" else 4


def _llama_config(size, layers, group=-1):
    return LlamaConfig(**{**LLAMA[size], "layers": layers}, head_dim=HEAD, group_size=group)


# ---------------------------------------------------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    g, kind = _generator(seed), case["kind"]
    if kind in ("decode", "prefill"):
        m, B = LLAMA[case["size"]], case["batch"]
        length = case["context"] if kind == "decode" else case["prompt"]
        runner = DecodeRunner(_llama_config(case["size"], _layers(case), case["group"]), B, length, 8, DEV)
        load_into_runner(runner, _llama_state(case, g), load_norm_weights=True)
        pages, size = -(-runner.max_context // 64), 64 * m["kv_heads"] * HEAD // 2
        for pools, table in zip(runner.pools, runner.block_tables):
            codes, scales, places = _pages(g, m, B, pages)
            for kv, pool in enumerate(pools):
                pool[:, :size] = codes[kv].flatten(1)
                tail = pool[:, size:].view(torch.float16).view(-1, 2, 64 * m["kv_heads"])
                tail[:, 0], tail[:, 1] = scales[kv].flatten(1), 7.5
                table[:, kv] = pool.data_ptr() + places[kv] * pool.shape[1]
        s = {"kind": kind, "runner": runner, "split": size, "length": length}
        if kind == "decode":
            s["tokens"] = _ids(g, m["vocab"], B)
            run(s)                                       # a server has its step captured
        else:
            s["tokens"] = _ids(g, m["vocab"], B * length)
        return s
    if kind in ("lserve_decode", "lserve_prefill"):
        m = LLAMA["8b"]
        length = case["context"] if kind == "lserve_decode" else case["prompt"]
        runner = LServeDecodeRunner(_llama_config("8b", _layers(case)), case["batch"], length, 64, DEV, seed=seed, kv_format=case["kv"],
                                    sink=SINK, local=LOCAL, ctx_sink=CTX_SINK, ctx_local=CTX_LOCAL, budget_tokens=BUDGET)
        w = _lserve_state(g)
        for L, new in zip(runner.layers, w["layers"]):
            L["ln1"].copy_(new["ln1"]), L["ln2"].copy_(new["ln2"])
            for n in ("qkv", "o", "gate_up", "down"):
                L[n].weight.copy_(new[n][0]), L[n].dequant_scale.copy_(new[n][1])
        runner.embed.copy_(w["embed"]), runner.lm_head.copy_(w["head"]), runner.final_norm.copy_(w["norm"])
        s = {"kind": kind, "runner": runner, "length": length}
        if kind == "lserve_decode":
            s["tokens"] = _ids(g, m["vocab"], 4 * case["batch"]).view(4, case["batch"])
            run(s)
        else:
            s["tokens"] = _ids(g, m["vocab"], case["batch"] * length)
        return s
    config, state = _engine_state(case, g)
    model = (Bobavik if case["arch"] == "Bobavik" else Bagedra).from_state(config, state, torch.bfloat16, DEV)
    del state
    trace = [t.tolist() for t in _trace(case, g, config["vocab"])]
    n = _lengths(case)
    engine = Engine(model, max_tokens=sum(64 + a + case["steps"] for a in n) + 64, max_seqs=case["seqs"])
    s = {"kind": kind, "engine": engine, "prompts": [t[:a] for t, a in zip(trace, n)], "tokens": [t[a:] for t, a in zip(trace, n)],
         "steps": case["steps"]}
    if case["steps"]:
        run(s)                                           # a server has its single-token steps captured
    return s


def run(state):
    kind = state["kind"]
    if kind == "decode":
        r = state["runner"]
        r.lengths.fill_(state["length"])                 # the pass decodes the same place again
        r.tokens.copy_(state["tokens"])
        r.step()
        return _runner_outputs(state)
    if kind == "prefill":
        state["runner"].prefill(state["length"], tokens=state["tokens"])
        return _runner_outputs(state)
    if kind == "lserve_prefill":
        hidden = state["runner"].prefill(tokens=state["tokens"], seq_len=state["length"])
        return {"hidden": hidden, "tokens": state["runner"].tokens, "last": state["runner"].normed}
    if kind == "lserve_decode":
        r, out = state["runner"], []
        r.lengths.fill_(state["length"])
        r.steps_done = 0
        for tokens in state["tokens"]:
            r.tokens.copy_(tokens)
            r.step()
            out.append((r.normed.clone(), r.tokens.clone()))
        return out
    engine = state["engine"]
    seqs = [engine.open() for _ in state["prompts"]]
    out = [engine.run([SequenceInput(q, p, [len(p) - 1]) for q, p in zip(seqs, state["prompts"])])]
    for i in range(state["steps"]):
        out.append(engine.run([SequenceInput(q, [t[i]], [0]) for q, t in zip(seqs, state["tokens"])]).clone())
    for q in seqs:
        engine.close(q)
    return out


def _runner_outputs(state):
    """Next tokens, the hidden state that the head reads, the residual, and every layer's pages: codes, scales and zero points."""
    r, split = state["runner"], state["split"]
    pages = [(p[:, :split], p[:, split:].view(torch.float16)) for pools in r.pools for p in pools]
    return {"tokens": r.tokens, "normed": r.normed, "residual": r.x, "pages": pages}


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------------------
def _causal(n, window=1 << 40):
    """Visible (query, key) pairs of a prompt of n tokens"""
    w = min(n, window)
    return w * (w + 1) // 2 + (n - w) * w


def work(case):
    kind = case["kind"]
    if kind != "engine":
        m = LLAMA[case.get("size", "8b")]
        w8 = kind.startswith("lserve")
        layers = _layers(case)
        H, I, B = m["hidden"], m["inter"], case["batch"]
        values = H * H * 2 + 2 * H * m["kv_heads"] * HEAD + 3 * H * I
        weights = values if w8 else values / 2 * (1 + (4 / 128 if case["group"] != -1 else 0))
        head = 2 * m["vocab"] * H
        row = m["kv_heads"] * (2 * HEAD + 8 if case.get("kv") == "kv8" else HEAD + 8)      # keys and values of a token and layer
        if kind in ("decode", "lserve_decode"):
            steps, keys = (4, BUDGET // 2 + (SINK + LOCAL) // 2) if w8 else (1, case["context"])
            choose = case["context"] / 16 * m["kv_heads"] // 2 * HEAD * 4 / 4 if w8 else 0      # statistics, read in one step of four
            return {"bytes": steps * (layers * (weights + B * (keys * row + choose)) + head + 4 * B * H),
                    "flops": steps * B * (layers * (2 * values + 4 * m["heads"] * HEAD * keys) + head)}
        n = case["prompt"]
        pairs = (_causal(n) + _causal(n, CTX_LOCAL + CTX_SINK)) / 2 if w8 else _causal(n)
        return {"bytes": layers * (weights + B * n * row) + head + B * n * H * (4 if w8 else 2),
                "flops": B * (layers * (2 * values * n + 4 * m["heads"] * HEAD * pairs) + head)}
    c, n, steps = _config(case), _lengths(case), case["steps"]
    W, seqs = c["width"], case["seqs"]
    tokens, flops, bytes_ = sum(n), 0, 0
    for l in c["layers"]:
        m, f = l["mixer"], l["mlp"]
        H, state, row = m["heads"], 0, 0
        if l["type"] == "attention":
            values, row = W * HEAD * (3 * H + 2 * m["kv_heads"]), 4 * HEAD * m["kv_heads"]
            pairs, per = lambda a: _causal(a, m["mask"]["size"]), 4 * H * HEAD
        elif l["type"] == "latent_attention":
            R, T = m["kv_rank"], m["rot_dim"]
            values, row = W * (H * (3 * HEAD + T) + R + T) + 2 * R * H * HEAD, 2 * (R + T)
            pairs, per = _causal, 2 * H * (2 * HEAD + T)
        else:
            heads = 4 * H if l["type"] != "delta" else 2 * H + 2 * m["kv_heads"]
            values, state = W * HEAD * (heads + H), 4 * H * HEAD * HEAD
            pairs, per = lambda a: a, 4 * H * HEAD * HEAD
        if f["kind"] == "moe":
            e, k = f["router"]["experts"], f["router"]["top"]
            used = lambda t: e * (1 - (1 - k / e) ** t)      # noqa: E731  experts that t tokens choose
            values += 3 * W * f["shared"]["ff"] + W * e
            expert = 3 * W * f["expert"]["ff"]
        else:
            used, k, expert = (lambda t: 0), 0, 0
            values += 3 * W * f["ff"]
        flops += (tokens + seqs * steps) * 2 * (values + k * expert) + sum(per * pairs(a) for a in n)
        flops += sum(per * (pairs(a + steps) - pairs(a)) for a in n)
        bytes_ += 2 * (values + used(tokens) * expert) + steps * 2 * (values + used(seqs) * expert)
        bytes_ += seqs * state + row * tokens + steps * (2 * seqs * state + row * tokens)
    head, rows = c["vocab"] * W, (1 + steps)
    return {"bytes": bytes_ + rows * (2 * head + 4 * seqs * c["vocab"]), "flops": flops + rows * seqs * 2 * head}


def tolerance(case):
    """Against 64 bits: the W4A8 models 0.01 - 0.03 (a code of the activations that rounds the other way moves a row by a part in 127, and the
    zero points' sum by more), the engine's bf16 0.003 - 0.005, and up to 0.02 in a row whose last expert is another one."""
    return {"rel": 0.02 if case.get("arch") == "Bagedra" else 0.03, "max": 0.5, "differ": 0.01}


# ---------------------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------------------------------
def _attend(q, k, v, scale, window=None, sink=0, first=0):
    """q [T, H, D] of positions first .., k, v [S, G, .]: softmax over j <= i, i - j < window or j < sink"""
    T, H, _ = q.shape
    out = q.new_empty((T, H, v.shape[2]))
    j = torch.arange(k.shape[0], device=DEV)
    for h in range(H):
        kh, vh = k[:, h * k.shape[1] // H], v[:, h * v.shape[1] // H]
        for a in range(0, T, 4096):
            i = first + torch.arange(a, min(T, a + 4096), device=DEV)[:, None]
            s = q[a:a + 4096, h] @ kh.T * scale
            unseen = j[None] > i
            if window is not None:
                unseen |= (i - j[None] >= window) & (j[None] >= sink)
            out[a:a + 4096, h] = s.masked_fill_(unseen, -math.inf).softmax(dim=1) @ vh
    return out


def _turn(x, pos, base, halves, dims=None):
    """x [T, H, D]: pairs (i, i + dims / 2), or (2 i, 2 i + 1), turned by pos * base ** (-2 i / dims)"""
    n = dims or x.shape[2]
    a = pos.double()[:, None, None] * base ** (-torch.arange(0, n, 2, device=DEV, dtype=torch.float64) / n)
    c, s, y = a.cos(), a.sin(), x.clone()
    one, two = (slice(0, n // 2), slice(n // 2, n)) if halves else (slice(0, n, 2), slice(1, n, 2))
    u, v = x[..., one], x[..., two]
    y[..., one], y[..., two] = u * c - v * s, v * c + u * s
    return y


def _codes(w, k):
    """The 4-bit weights behind QServe's order of 32 x 32 tiles, [n, k]"""
    b = w["qweight"].view(torch.uint8)
    n = b.shape[0]
    b = b.view(n // 32, k // 32, 8, 4, 2, 2, 4)
    return torch.stack((b & 15, b >> 4), dim=-1).permute(0, 7, 5, 2, 1, 4, 3, 6).reshape(n, k)


def _quantised(x):
    """int8 codes of every row, their scale, the row's sum"""
    top = x.abs().amax(dim=1, keepdim=True)
    return (x * (127 / top)).round_(), top / 127, x.sum(dim=1, keepdim=True)


def _w4_product(x, w, group):
    q, scale, total = _quantised(x)
    u = _codes(w, x.shape[1])
    if group == -1:
        return q @ u.double().T * scale * w["s1_scales"].double() - total * w["s1_szeros"].double()
    n, k = u.shape
    own = lambda t: t.view(torch.uint8).view(-1, n // 32, 8, 4).transpose(2, 3).reshape(-1, n).T.to(torch.int32)      # noqa: E731  [n, groups]
    v = (u.view(n, -1, group).int() * own(w["s2_scales"])[..., None] + own(w["s2_zeros"])[..., None]) % 256
    v = torch.where(v > 127, v - 256, v).reshape(n, k).double()
    return q @ v.T * (scale * w["s1_scales"].double())


def _w8_product(x, w):
    q, scale, _ = _quantised(x)
    return q @ w[0].double().T * scale * w[1].double()


def _norm_centred(x, g):
    """The reference's norm in front of a quantiser: the mean leaves the row, but not its mean square."""
    return (x - x.mean(dim=1, keepdim=True)) * torch.rsqrt(x.square().mean(dim=1, keepdim=True) + 1e-5) * g.double()


def _rms(x, g, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + eps) * g.double()


def _llama_layer(x, ln1, ln2, product, attention, m):
    """product(name, rows); attention(q, k, v) -> rows"""
    y = product("qkv", _norm_centred(x, ln1))
    q, k, v = y.view(y.shape[0], -1, HEAD).split((m["heads"], m["kv_heads"], m["kv_heads"]), dim=1)
    x = x + product("o", attention(q, k, v).flatten(1))
    gate, up = product("gate_up", _norm_centred(x, ln2)).chunk(2, dim=1)
    return x + product("down", torch.nn.functional.silu(gate) * up)


def _exact_llama(case, g):
    m, B, group = LLAMA[case["size"]], case["batch"], case["group"]
    st = _llama_state(case, g)
    decode = case["kind"] == "decode"
    n = case["context"] if decode else case["prompt"]
    caches = [_pages(g, m, B, -(-(n + 9) // 64)) for _ in range(_layers(case))]
    tokens = _ids(g, m["vocab"], B if decode else B * n)
    x = st["model.embed_tokens.weight"][tokens].double()
    names = {"qkv": ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj"), "o": ("self_attn.o_proj",),
             "gate_up": ("mlp.gate_proj", "mlp.up_proj"), "down": ("mlp.down_proj",)}
    scale = HEAD ** -0.5

    for i in range(_layers(case)):
        p = "model.layers.%d." % i

        def product(name, rows):
            parts = [{k: st[p + f + "." + k] for k in ("qweight", "s1_scales", "s1_szeros", "s2_scales", "s2_zeros") if p + f + "." + k in st}
                     for f in names[name]]
            return torch.cat([_w4_product(rows, w, group) for w in parts], dim=1)

        def decode_attention(q, k, v):
            pos = torch.full((B,), n, device=DEV)
            q, k = _turn(q, pos, m["rope_theta"], True), _turn(k, pos, m["rope_theta"], True)
            codes, scales, places = caches[i]
            out = []
            for b in range(B):
                old = []
                for kv in range(2):
                    c = codes[kv][places[kv][b]]
                    c = torch.stack((c & 15, c >> 4), dim=-1).flatten(-2).double() - 7.5
                    old.append((c * scales[kv][places[kv][b]].double()[..., None]).transpose(1, 2).flatten(0, 1)[:n])
                out.append(_attend(q[b:b + 1], torch.cat((old[0], k[b:b + 1])), torch.cat((old[1], v[b:b + 1])), scale, first=n))
            return torch.cat(out)

        def prompt_attention(q, k, v):
            pos = torch.arange(n, device=DEV)
            out = []
            for b in range(B):
                at = slice(b * n, b * n + n)
                out.append(_attend(_turn(q[at], pos, m["rope_theta"], True), _turn(k[at], pos, m["rope_theta"], True), v[at], scale))
            return torch.cat(out)

        x = _llama_layer(x, st[p + "input_layernorm.weight"], st[p + "post_attention_layernorm.weight"], product,
                         decode_attention if decode else prompt_attention, m)
    x = x if decode else x.view(B, n, -1)[:, -1]
    normed = _rms(x, st["model.norm.weight"])
    tokens = (normed @ st["lm_head.weight"].double().T).argmax(dim=1)
    return {"tokens": tokens, "normed": normed, "residual": x, "pages": None}


def _exact_lserve_prefill(case, g):
    m, n, B = LLAMA["8b"], case["prompt"], case["batch"]
    w = _lserve_state(g)
    x = w["embed"][_ids(g, m["vocab"], B * n)].double()
    pos = torch.arange(n, device=DEV)
    full = torch.arange(m["kv_heads"], device=DEV) % 2 == 0              # every second kv head sees all keys, the others stream
    own = full.repeat_interleave(m["heads"] // m["kv_heads"])

    def attention(q, k, v):
        out = torch.empty_like(q)
        for b in range(B):
            at = slice(b * n, b * n + n)
            qt, kt = _turn(q[at], pos, m["rope_theta"], True), _turn(k[at], pos, m["rope_theta"], True)
            out[at, own] = _attend(qt[:, own], kt[:, full], v[at][:, full], HEAD ** -0.5)
            out[at, ~own] = _attend(qt[:, ~own], kt[:, ~full], v[at][:, ~full], HEAD ** -0.5, CTX_LOCAL, CTX_SINK)
        return out

    for L in w["layers"]:
        x = _llama_layer(x, L["ln1"], L["ln2"], lambda name, rows, L=L: _w8_product(rows, L[name]), attention, m)
    last = _rms(x.view(B, n, -1)[:, -1], w["norm"])
    return {"hidden": x, "tokens": (last @ w["head"].double().T).argmax(dim=1), "last": last}


def _linear(h, w):
    return h @ w.double().T


def _each(parts, f):
    return torch.cat([f(a) for a in parts])


def _layer_norm(x, st, name):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], st[name].double(), st[name + ".b"].double(), 1e-5)


def _decayed(q, k, v, decay):
    """S <- decay S + k v^T, o = S^T q over one sequence, [T, H, .], in chunks"""
    T, H, D = q.shape
    S, out, lam = q.new_zeros((H, D, v.shape[2])), torch.empty_like(v), torch.tensor(decay, dtype=torch.float64, device=DEV)
    for a in range(0, T, 128):
        qc, kc, vc = (t[a:a + 128].transpose(0, 1) for t in (q, k, v))
        i = torch.arange(qc.shape[1], device=DEV, dtype=torch.float64)
        d = i[:, None] - i[None]
        mask = torch.where(d >= 0, lam[:, None, None] ** d.clamp(min=0), 0.0)
        out[a:a + 128] = ((qc @ kc.transpose(1, 2) * mask) @ vc + lam[:, None, None] ** (i[:, None] + 1) * (qc @ S)).transpose(0, 1)
        S = lam[:, None, None] ** float(len(i)) * S + (kc * lam[:, None, None] ** (len(i) - 1 - i)[:, None]).transpose(1, 2) @ vc
    return out


def _recurrence(parts, q, k, v, log_decay, beta=None):
    """Token by token, all sequences side by side.  log_decay [T, H, D] or [T, H, 1]; beta [T, H]: the delta rule."""
    n = [len(a) for a in parts]
    N = max(n)
    lay = lambda t: torch.stack([torch.nn.functional.pad(t[a], (0, 0) * (t.dim() - 1) + (0, N - len(a))) for a in parts], dim=1)      # noqa: E731
    q, k, v, d = lay(q), lay(k), lay(v), lay(log_decay).exp()
    S, out = q.new_zeros((*q.shape[1:], v.shape[3])), torch.empty_like(v)
    beta = None if beta is None else lay(beta)
    for t in range(N):
        S *= d[t][..., None]
        u = v[t] if beta is None else beta[t][..., None] * (v[t] - (k[t].unsqueeze(2) @ S).squeeze(2))
        S += k[t][..., None] * u.unsqueeze(2)
        out[t] = (q[t].unsqueeze(2) @ S).squeeze(2)
    return torch.cat([out[:m, i] for i, m in enumerate(n)])


def _mixture(h, st, p, f):
    z = _linear(h, st[p + "router"]) + st[p + "router.b"].double()
    top, ids = z.topk(f["router"]["top"], dim=1)
    wt = top.softmax(dim=1)
    glu = lambda x, n: _linear(torch.nn.functional.silu(_linear(x, st[p + n + "gate"])) * _linear(x, st[p + n + "up"]), st[p + n + "down"])      # noqa: E731
    y = glu(h, "shared.")
    for e in range(f["router"]["experts"]):
        t, c = torch.nonzero(ids == e, as_tuple=True)
        if len(t):
            y.index_add_(0, t, wt[t, c, None] * glu(h[t], "e%d." % e))
    return y


def _exact_engine(case, g):
    c, st = _engine_state(case, g)
    trace, n = _trace(case, g, c["vocab"]), _lengths(case)
    total = [len(t) for t in trace]
    ends = [sum(total[:i + 1]) for i in range(len(total))]
    parts = [torch.arange(e - t, e, device=DEV) for e, t in zip(ends, total)]
    pos = torch.cat([torch.arange(t, device=DEV) for t in total])
    bob = c["architecture"] == "Bobavik"
    x, first, silu = st["embed"][torch.cat(trace)].double(), None, torch.nn.functional.silu
    for i, l in enumerate(c["layers"]):
        p, m = "l%d.mix." % i, l["mixer"]
        h = _layer_norm(x, st, "l%d.norm1" % i) if bob else x
        lin = lambda name: _linear(h, st[p + name])      # noqa: E731
        H, T = m["heads"], len(x)
        if l["type"] == "attention":
            q, k = (_turn(lin(a).view(T, -1, HEAD), pos, m["rot"]["base"], False) for a in "qk")
            v = lin("v").view(T, -1, HEAD)
            raw, v = v, v if first is None else (1 - 0.4) * v + 0.4 * first
            first = raw if first is None else first
            o = _each(parts, lambda a: _attend(q[a], k[a], v[a], m["scale"], m["mask"]["size"])).flatten(1) * torch.sigmoid(lin("g"))
        elif l["type"] == "latent_attention":
            R, rot = m["kv_rank"], m["rot_dim"]
            d = lin("dkv")
            lat = _rms(d[:, :R], st[p + "dkv.norm"])
            shared = _turn(d[:, None, R:], pos, m["rot"]["base"], True).expand(T, H, rot)
            q = lin("q").view(T, H, HEAD + rot)
            q = torch.cat((q[..., :HEAD], _turn(q[..., HEAD:], pos, m["rot"]["base"], True)), dim=-1)
            k = torch.cat((_linear(lat, st[p + "uk"]).view(T, H, HEAD), shared), dim=-1)
            v = _linear(lat, st[p + "uv"]).view(T, H, HEAD)
            o = _each(parts, lambda a: _attend(q[a], k[a], v[a], m["scale"])).flatten(1) * torch.sigmoid(lin("g"))
        elif l["type"] == "lightning":
            q, k, v = (silu(lin(a)).view(T, H, HEAD) for a in "qkv")
            o = _each(parts, lambda a: _decayed(q[a], k[a], v[a], m["decay"])).flatten(1)
            o = _rms(o, st[p + "norm"]) * torch.sigmoid(lin("g"))
        else:
            if l["type"] == "gla":
                q, k, v = (lin(a).view(T, H, HEAD) for a in "qkv")
                z = _linear(lin("a1"), st[p + "a2"]) + st[p + "a2.b"].double()
                o = _recurrence(parts, q * HEAD ** -0.5, k, v, (torch.nn.functional.logsigmoid(z) / m["tau"]).view(T, H, HEAD))
            else:
                G, taps = m["kv_heads"], m["conv"]

                def convolved(name, heads):
                    y, w = lin(name), st[p + name + ".conv"].double()
                    one = lambda a: sum(torch.nn.functional.pad(y[a], (0, 0, taps - 1, 0))[j:j + len(a)] * w[:, j] for j in range(taps))      # noqa: E731
                    return silu(_each(parts, one)).view(T, heads, HEAD)

                unit = lambda t: (t * torch.rsqrt(t.square().sum(dim=-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, dim=1)      # noqa: E731
                q, k, v = unit(convolved("q", G)) * HEAD ** -0.5, unit(convolved("k", G)), convolved("v", H)
                rate = -st[p + "A_log"].double().exp() * torch.nn.functional.softplus(lin("a") + st[p + "dt_bias"].double())
                o = _recurrence(parts, q, k, v, rate[..., None], torch.sigmoid(lin("b")))
            o = _rms(o, st[p + "norm"]).flatten(1) * silu(lin("g"))
        y = _linear(o, st[p + "o"])
        x = x + (_layer_norm(y, st, "l%d.norm1b" % i) if bob else _rms(y, st["l%d.norm1" % i]))
        p = "l%d.mlp." % i
        if bob:
            y = _mixture(_layer_norm(x, st, "l%d.norm2" % i), st, p, l["mlp"])
            x = x + _layer_norm(y, st, "l%d.norm2b" % i)
        else:
            act = torch.nn.functional.gelu(_linear(x, st[p + "gate"]) + st[p + "gate.b"].double(), approximate="tanh")
            y = _linear(act * (_linear(x, st[p + "up"]) + st[p + "up.b"].double()), st[p + "down"]) + st[p + "down.b"].double()
            x = x + _rms(y, st["l%d.norm2" % i])
    starts = [e - t for e, t in zip(ends, total)]
    out = []
    for step in range(case["steps"] + 1):
        h = x[torch.tensor([s + a - 1 + step for s, a in zip(starts, n)], device=DEV)]
        h = _layer_norm(h, st, "final.norm") if bob else _rms(h, st["final.norm"])
        out.append(_linear(h, st["head"]))
    return out


def exact(case, seed):
    g = _generator(seed)
    if case["kind"] in ("decode", "prefill"):
        return _exact_llama(case, g)
    if case["kind"] == "lserve_prefill":
        return _exact_lserve_prefill(case, g)
    if case["kind"] == "engine":
        return _exact_engine(case, g)
    return None      # (the cached pages are the runner's own)
