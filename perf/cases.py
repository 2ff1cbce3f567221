"""The steps this framework is measured on: what a server does all day, one model step at a time.

A case is one step of a model: a *prompt* step (whole prompts of new requests, packed) or a *decode* step (one token of
each running request, as a captured graph, the way the engine replays it). The models are the ones of the benchmark with
their layer sizes (bench.py, bench/*_bench.py):

  llama    Llama-3-8B shapes, 8 of the 32 layers and the whole vocabulary;
  dofivik  latent attention in a window and a generalized delta rule in turn;
  loluzen  grouped attention behind short convolutions, and head-mixing attention beside a gated linear recurrence;
  vizonex  chunked attention with a sink and state-space layers in turn, dense feed-forwards.

"1b" is width 2048 with 8 layers, "8b" width 4096 with 4 layers. `experts` is the routed feed-forward of a Vizonex layer
(router, selection, experts, shared expert) on its own: behind a router a close call between two experts turns a rounding
error into another token's answer, so routed layers are compared by themselves, on given inputs.

Serving runs in bfloat16, with fp32 residuals, norms, softmax and recurrent states; so do all cases. A decode step starts
from pages and states of requests in full swing, a prompt step from nothing. Weights are random with the spread that keeps
a trained model's activations near 1.
"""
import math

import torch
import torch.nn.functional as F

BLOCK = 16          # cache page, tokens (the engine's default)
EPS = 1e-5
SINK_ALPHA = 1.702  # slope of the sigmoid in the experts' clamped gate
UNIT_KEY_EPS = 1e-6

SIZES = {
    "1b": dict(width=2048, layers=8, ff=8192, vocab=32000,
               dofivik=dict(heads=32, dim=64, rot=32, vdim=64, R=256, Rq=768, window=1024, d_heads=32, d_dim=64),
               loluzen=dict(heads=32, kv=8, dim=64, rot=32, l_heads=16, l_kv=2, r_heads=16, r_dim=64, r_vdim=128),
               vizonex=dict(heads=32, kv=8, dim=64, chunk=1024, s_heads=64, s_vdim=64, s_state=128, s_groups=8),
               experts=dict(ff=2048)),
    "8b": dict(width=4096, layers=4, ff=14336, vocab=32000,
               dofivik=dict(heads=32, dim=128, rot=64, vdim=128, R=512, Rq=1536, window=4096, d_heads=64, d_dim=64),
               loluzen=dict(heads=32, kv=8, dim=128, rot=64, l_heads=16, l_kv=2, r_heads=32, r_dim=64, r_vdim=128),
               vizonex=dict(heads=32, kv=8, dim=128, chunk=4096, s_heads=128, s_vdim=64, s_state=128, s_groups=8),
               experts=dict(ff=3584)),
}
LLAMA = dict(width=4096, layers=8, heads=32, kv=8, dim=128, ff=14336, vocab=128256, theta=500000.0)
EXPERTS = dict(experts=8, top=2, groups=4, keep=2, scale=2.5, limit=7.0)
ROT_SCALING = {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}
LENGTHS = 5         # a prompt step holds up to this many prompts


def _case(name, model, size, kind, **kw):
    return dict(name=name, model=model, size=size, kind=kind, **kw)


def _prompts(*lengths):
    """The lengths of a prompt step's prompts as plain values (0: no such prompt)."""
    return {f"len{i}": (lengths[i] if i < len(lengths) else 0) for i in range(LENGTHS)}


def listed():
    return [
        # one user chatting with an otherwise idle server: latency and launches
        _case("llama decode 1", "llama", "8b", "decode", rows=1, low=640, high=640),
        # the headline load: 64 requests of 512 prompt tokens somewhere in their 256 output tokens
        _case("llama decode 64", "llama", "8b", "decode", rows=64, low=512, high=767),
        # the prompt of one new request: its time to the first token
        _case("llama prompt 512", "llama", "8b", "prompt", **_prompts(512)),
        # a full batch of long prompts, the largest step
        _case("llama prompts 4x2048", "llama", "8b", "prompt", **_prompts(2048, 2048, 2048, 2048)),
        # a full decode batch at the benchmark's context
        _case("dofivik decode 64", "dofivik", "1b", "decode", rows=64, low=1024, high=1024),
        # the benchmark's prompt step
        _case("dofivik prompts 4x2048", "dofivik", "1b", "prompt", **_prompts(2048, 2048, 2048, 2048)),
        # a single request of the wide model, contexts and all states its own
        _case("vizonex decode 1", "vizonex", "8b", "decode", rows=1, low=1531, high=1531),
        # prompts as they arrive: of very different lengths, none a round number
        _case("vizonex prompts ragged", "vizonex", "1b", "prompt", **_prompts(1531, 700, 257, 33)),
        # a half full server, requests of different ages
        _case("loluzen decode 17", "loluzen", "8b", "decode", rows=17, low=300, high=1500),
        # one long prompt by itself: few sequences, many tokens
        _case("loluzen prompt 4001", "loluzen", "1b", "prompt", **_prompts(4001)),
        # the routed feed-forward in a full decode batch, and in the benchmark's prompt step
        _case("experts 64", "experts", "8b", "tokens", tokens=64),
        _case("experts 8192", "experts", "8b", "tokens", tokens=8192),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    model = rng.choice(["llama", "dofivik", "loluzen", "vizonex", "experts"])
    size = "8b" if model == "llama" else rng.choice(["1b", "8b"])
    c = dict(model=model, size=size)
    if model == "experts":
        return dict(c, kind="tokens", tokens=_log_uniform(rng, 1, 8192))
    if rng.random() < 0.5:
        low = _log_uniform(rng, 64, 2048)
        return dict(c, kind="decode", rows=_log_uniform(rng, 1, 64), low=low, high=low + rng.randrange(0, 512))
    n = rng.randrange(1, LENGTHS)
    total = _log_uniform(rng, 64 * n, 4096)
    cuts = sorted(rng.uniform(0.2, 1.0) for _ in range(n))
    return dict(c, kind="prompt", **_prompts(*[max(1, int(total * x / sum(cuts))) for x in cuts]))


# ------------------------------------------------------------------------------------------------ the step's sequences
def _sequences(case):
    """[(new tokens, tokens before them)] of the step."""
    if case["kind"] == "decode":
        n, lo, hi = case["rows"], case["low"], case["high"]
        return [(1, lo + (i * 37) % (hi - lo + 1)) for i in range(n)]
    return [(case[f"len{i}"], 0) for i in range(LENGTHS) if case[f"len{i}"]]


class _Step:
    """Tokens, positions, pages and slots of the step, on the GPU. Pages are handed out in a random order."""

    def __init__(self, case, vocab, gen):
        dev = gen.device
        self.seqs = _sequences(case)
        self.S, self.T = len(self.seqs), sum(q for q, _ in self.seqs)
        self.max_q, self.max_len = max(q for q, _ in self.seqs), max(q + c for q, c in self.seqs)
        pages = [-(-(q + c) // BLOCK) for q, c in self.seqs]
        self.num_blocks, width = sum(pages) + 1, max(pages)
        order = torch.randperm(self.num_blocks, generator=gen, device=dev).to(torch.int32)
        self.tables = torch.zeros(self.S, width, dtype=torch.int32, device=dev)
        first, at = [0], 0
        for i, n in enumerate(pages):
            self.tables[i, :n] = order[at:at + n]
            at += n
            first.append(first[-1] + self.seqs[i][0])
        self.first = first
        i32 = dict(dtype=torch.int32, device=dev)
        self.qsl = torch.tensor(first, **i32)
        self.lens = torch.tensor([q + c for q, c in self.seqs], **i32)
        self.slots = torch.arange(self.S, **i32)
        self.token_seq = torch.repeat_interleave(self.slots, torch.tensor([q for q, _ in self.seqs], device=dev))
        self.pos = torch.cat([torch.arange(c, c + q, **i32) for q, c in self.seqs])
        page = self.tables[self.token_seq.long(), (self.pos // BLOCK).long()]
        self.rows = page * BLOCK + self.pos % BLOCK                      # cache row of every token
        self.ids = torch.randint(0, vocab, (self.T,), generator=gen, device=dev).to(torch.int32)
        self.last = (self.qsl[1:] - 1).long()

    def held(self, s, before=True):
        """Cache rows of the tokens that sequence s holds before the step (or of those it adds)."""
        q, c = self.seqs[s]
        p = torch.arange(0, c, device=self.tables.device) if before else torch.arange(c, c + q, device=self.tables.device)
        return (self.tables[s, (p // BLOCK)].long() * BLOCK + p % BLOCK)


# ------------------------------------------------------------------------------------------------ weights and contexts
def _layer_kinds(case):
    m, n = case["model"], (LLAMA if case["model"] == "llama" else SIZES[case["size"]])["layers"]
    pair = {"llama": ("attention",) * 2, "dofivik": ("latent_attention", "general_delta"),
            "loluzen": ("attention", "parallel"), "vizonex": ("attention", "mamba2")}[m]
    return [pair[i % 2] for i in range(n)]


def _tables(case):
    """name -> (shape, spread, mean, fp32?) of every weight, under the model's parameter names."""
    t = {}

    def mat(name, rows, cols, gain=1.0):
        t[name] = ((rows, cols), gain / math.sqrt(cols), 0.0, False)

    def vec(name, shape, spread, mean=0.0, wide=True):
        t[name] = (shape if isinstance(shape, tuple) else (shape,), spread, mean, wide)
    model = case["model"]
    if model == "llama":
        z = LLAMA
        W, V, ff, D = z["width"], z["vocab"], z["ff"], z["dim"]
        t["embed"] = ((V, W), 1.0, 0.0, False)
        mat("lm_head", V, W)
        for i in range(z["layers"]):
            b = f"layers.{i}."
            mat(b + "qkv", (z["heads"] + 2 * z["kv"]) * D, W)
            mat(b + "o", W, z["heads"] * D)
            mat(b + "gate", ff, W)
            mat(b + "up", ff, W)
            mat(b + "down", W, ff)
        return t
    z = SIZES[case["size"]]
    W = z["width"]
    if model == "experts":
        E, ff = EXPERTS["experts"], z["experts"]["ff"]
        t["router"] = ((E, W), 2.0 / math.sqrt(W), 0.0, True)
        vec("correction", E, 0.2)
        t["w13"] = ((E, 2 * ff, W), 1.0 / math.sqrt(W), 0.0, False)
        t["w2"] = ((E, W, ff), 1.0 / math.sqrt(ff), 0.0, False)
        mat("shared.gate_up", 2 * ff, W)
        mat("shared.down", W, ff)
        return t
    s, V, ff = z[model], z["vocab"], z["ff"]
    t["embed"] = ((V, W), W ** -0.5 if model == "loluzen" else 1.0, 0.0, False)   # loluzen scales its rows by sqrt(W)
    mat("head", V, W)
    vec("final_norm", W, 0.1, 1.0 if model == "vizonex" else 0.0)
    if model == "vizonex":
        t["pos"] = ((_max_position(case), W), 0.3, 0.0, False)
    for i, kind in enumerate(_layer_kinds(case)):
        b = f"layers.{i}."
        x = b + "mix."
        vec(b + "norm1", W, 0.1, 1.0 if model == "vizonex" else 0.0)
        if model == "dofivik":
            vec(b + "canon1", (W, 4), 0.3)
            vec(b + "canon2", (W, 4), 0.3)
            vec(b + "norm2", W, 0.1)
            if kind == "latent_attention":
                H = s["heads"]
                mat(x + "in_proj", s["Rq"] + s["R"] + s["rot"] + H, W)
                vec(x + "q_norm", s["Rq"], 0.1, 1.0)
                vec(x + "kv_norm", s["R"], 0.1, 1.0)
                mat(x + "uq", H * (s["dim"] + s["rot"]), s["Rq"])
                mat(x + "uk", H * s["dim"], s["R"])
                mat(x + "uv", H * s["vdim"], s["R"])
                mat(x + "o", W, H * s["vdim"])
            else:
                n = s["d_heads"] * s["d_dim"]
                mat(x + "in_proj", 5 * n + 32, W)
                mat(x + "w2", n, 32)
                vec(x + "w0", n, 1.0)
                vec(x + "a_bias", n, 0.5)
                vec(x + "norm", n, 0.1, 1.0)
                mat(x + "o", W, n)
            mat(b + "mlp.up", ff, W)
            mat(b + "mlp.down", W, ff)
            vec(b + "mlp.up_b", ff, 0.1)
            vec(b + "mlp.down_b", W, 0.1)
            vec(b + "mlp.act", 2, 0.5)
        elif model == "loluzen":
            for n in ("norm1b", "norm2", "norm2b"):
                vec(b + n, W, 0.1)
            if kind == "attention":
                ch = (s["heads"] + 2 * s["kv"]) * s["dim"]
                mat(x + "in_proj", ch + s["heads"], W)
                vec(x + "conv_w", (ch, 4), 0.4, 0.25)
                vec(x + "q_norm", s["dim"], 0.1, 1.0)
                vec(x + "k_norm", s["dim"], 0.1, 1.0)
                mat(x + "o", W, s["heads"] * s["dim"])
            else:
                H, left, n = s["l_heads"], (s["l_heads"] + 2 * s["l_kv"]) * s["dim"], s["r_heads"] * s["r_dim"]
                mat(x + "in_proj", left + H + 2 * n + s["r_heads"] * s["r_vdim"], W)
                vec(x + "in_bias", left + H + 2 * n + s["r_heads"] * s["r_vdim"], 0.1, 0.0, False)
                vec(x + "left.r1", H, 0.5, 0.75)
                vec(x + "left.r2", H, 0.4, 1.0)
                vec(x + "left.talk", (H, H), 0.3)
                mat(x + "left.o", W, H * s["dim"])
                vec(x + "left.out_norm", W, 0.1, 1.0)
                vec(x + "right.lower", n, 0.2, 0.45)
                vec(x + "right.norm", s["r_vdim"], 0.1, 1.0)
                mat(x + "right.o", W, s["r_heads"] * s["r_vdim"])
                vec(x + "right.out_norm", W, 0.1, 1.0)
            mat(b + "mlp.up", ff, W)
            mat(b + "mlp.down", W, ff)
            vec(b + "mlp.up_b", ff, 0.1)
            vec(b + "mlp.down_b", W, 0.1)
        else:
            vec(b + "ls1", W, 0.1, 0.5)
            vec(b + "ls2", W, 0.1, 0.5)
            vec(b + "canon1", (W, 4), 0.3)
            if kind == "attention":
                nq, nk = s["heads"] * s["dim"], s["kv"] * s["dim"]
                mat(x + "qkv", nq + 2 * nk, W)
                vec(x + "q_norm", nq, 0.1, 1.0)
                vec(x + "k_norm", nk, 0.1, 1.0)
                vec(x + "temp", s["heads"], 0.1, 1.0)
                vec(x + "sink", s["heads"], 0.5)
                mat(x + "o", W, nq)
            else:
                H, inner, gn = s["s_heads"], s["s_heads"] * s["s_vdim"], s["s_groups"] * s["s_state"]
                mat(x + "in_proj", 2 * inner + 2 * gn + H, W)
                vec(x + "conv_w", (inner + 2 * gn, 4), 0.4)
                vec(x + "conv_b", inner + 2 * gn, 0.1)
                vec(x + "dt_bias", H, 0.5, -1.0)
                vec(x + "A_log", H, 0.5, -0.5)
                vec(x + "D", H, 0.3, 1.0)
                vec(x + "norm", inner, 0.1, 1.0)
                mat(x + "o", W, inner)
            mat(b + "mlp.gate_up", 2 * ff, W)
            mat(b + "mlp.down", W, ff)
    return t


def _max_position(case):
    return 4096 if case["kind"] == "prompt" else 4096 * (-(-case["high"] // 4096))


def _weights(case, gen):
    out = {}
    for name, (shape, spread, mean, wide) in _tables(case).items():
        w = torch.empty(shape, dtype=torch.float32 if wide else torch.bfloat16, device=gen.device)
        out[name] = w.normal_(mean, spread, generator=gen)
    for name, w in out.items():
        if name.endswith("left.talk"):
            w += torch.eye(w.shape[0], device=w.device)
        elif name.endswith("in_proj") and name[:-len("in_proj")] + "a_bias" in out:
            # a delta layer's r leans towards k: with r and k at right angles a sequence's first read, v (k . r), would
            # be rounding noise that the norm behind it blows up
            n = out[name[:-len("in_proj")] + "a_bias"].shape[0]
            w[:n] = 0.8 * w[:n] + 0.6 * w[n:2 * n]
        elif name.endswith("left.r2"):
            w.clamp_(min=0.05)
        elif name.endswith("right.lower"):
            w.clamp_(0.0, 0.9)
        elif name.endswith("in_bias"):   # the left branch's gate and the recurrence's q and v have none
            s = SIZES[case["size"]]["loluzen"]
            left, n = (s["l_heads"] + 2 * s["l_kv"]) * s["dim"], s["r_heads"] * s["r_dim"]
            w[left:left + s["l_heads"] + n] = 0
            w[left + s["l_heads"] + 2 * n:] = 0
    return out


def _contexts(case, step, gen):
    """Per layer what the sequences hold before the step: pages ("k" / "v" / "latent", [cache rows, ...]) and states (one
    row per sequence). Nothing for prompts."""
    if case["kind"] == "prompt":
        return None
    rows, S = step.num_blocks * BLOCK, step.S

    def page(*n):
        return torch.empty(rows, *n, dtype=torch.bfloat16, device=gen.device).normal_(generator=gen)

    def state(*n):
        return torch.empty(S, *n, dtype=torch.float32, device=gen.device).normal_(0.0, 0.5, generator=gen)
    if case["model"] == "llama":
        return [dict(k=page(LLAMA["kv"], LLAMA["dim"]), v=page(LLAMA["kv"], LLAMA["dim"])) for _ in range(LLAMA["layers"])]
    z = SIZES[case["size"]]
    s, W, out = z[case["model"]], z["width"], []
    for kind in _layer_kinds(case):
        if case["model"] == "dofivik":
            c = dict(conv1=state(3, W), conv2=state(3, W))
            if kind == "latent_attention":
                c["latent"] = page(s["R"] + s["rot"])
            else:
                c["delta"] = state(s["d_heads"], s["d_dim"], s["d_dim"])
        elif case["model"] == "loluzen":
            if kind == "attention":
                c = dict(k=page(s["kv"] * s["dim"]), v=page(s["kv"] * s["dim"]),
                         mix_conv=state(3, (s["heads"] + 2 * s["kv"]) * s["dim"]))
            else:
                c = dict(k=page(s["l_kv"] * s["dim"]), v=page(s["l_kv"] * s["dim"]),
                         gla=state(s["r_heads"], s["r_dim"], s["r_vdim"]))
        else:
            c = dict(conv1=state(3, W))
            if kind == "attention":
                c.update(k=page(s["kv"] * s["dim"]), v=page(s["kv"] * s["dim"]))
            else:
                ch = s["s_heads"] * s["s_vdim"] + 2 * s["s_groups"] * s["s_state"]
                c.update(mix_conv=state(3, ch), ssm=state(s["s_heads"], s["s_state"], s["s_vdim"]))
        out.append(c)
    return out


STATES = ("conv1", "conv2", "mix_conv", "delta", "ssm", "gla")


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    if case["model"] == "experts":
        w = _weights(case, gen)
        return w, torch.empty(case["tokens"], SIZES[case["size"]]["width"], device="cuda").normal_(generator=gen), None
    step = _Step(case, (LLAMA if case["model"] == "llama" else SIZES[case["size"]])["vocab"], gen)
    return _weights(case, gen), step, _contexts(case, step, gen)


# ------------------------------------------------------------------------------------------------ the framework's side
def _config(case, step):
    from xgserve.models.config import ModelConfig, dofivik_config, loluzen_config, vizonex_config
    name, top = "-".join((case["model"], case["size"])), 16384
    if case["model"] == "llama":
        z = LLAMA
        return ModelConfig(name, "llama", z["width"], z["layers"], z["heads"], z["kv"], z["dim"], z["ff"], z["vocab"], top,
                           z["theta"], norm_eps=EPS)
    z = SIZES[case["size"]]
    s, layers = z[case["model"]], []
    for kind in _layer_kinds(case):
        mlp = {"kind": "dense", "ff": z["ff"]}
        if kind == "latent_attention":
            m = {"heads": s["heads"], "dim": s["dim"], "rot_dim": s["rot"], "vdim": s["vdim"], "kv_rank": s["R"],
                 "q_rank": s["Rq"], "scale": (s["dim"] + s["rot"]) ** -0.5, "mask": {"size": s["window"]},
                 "rot": {"base": 5e5, "dims": s["rot"]}}
        elif kind == "general_delta":
            m = {"heads": s["d_heads"], "dim": s["d_dim"]}
        elif kind == "mamba2":
            m = {"heads": s["s_heads"], "vdim": s["s_vdim"], "state": s["s_state"], "groups": s["s_groups"],
                 "norm_groups": s["s_groups"], "conv": 4}
        elif kind == "parallel":
            m = {"left": {"heads": s["l_heads"], "kv_heads": s["l_kv"], "dim": s["dim"], "vdim": s["dim"],
                          "scale": s["dim"] ** -0.5},
                 "right": {"heads": s["r_heads"], "dim": s["r_dim"], "vdim": s["r_vdim"]}}
        else:
            m = {"heads": s["heads"], "kv_heads": s["kv"], "dim": s["dim"], "vdim": s["dim"], "scale": s["dim"] ** -0.5}
            if case["model"] == "vizonex":
                m["mask"] = {"size": s["chunk"]}
            else:
                m.update(conv=4, rot={"base": 5e5, "dims": s["rot"], "scaling": dict(ROT_SCALING)})
        layers.append({"type": kind, "mixer": m, "mlp": mlp})
    if case["model"] == "dofivik":
        return dofivik_config(name, z["width"], z["vocab"], layers, postln_alpha=2.0, taps=4, eps=EPS, max_position=top)
    if case["model"] == "loluzen":
        return loluzen_config(name, z["width"], z["vocab"], layers, embed_scale=z["width"] ** 0.5, residual_mult=0.5,
                              eps=EPS, max_position=top)
    return vizonex_config(name, z["width"], z["vocab"], layers, taps=4, eps=EPS, max_position=_max_position(case))


def _fill(model, weights):
    from xgserve.ops.linear import interleave_gate_up
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("gate_up") and name not in weights:
                b = name[:-len("gate_up")]
                p.copy_(interleave_gate_up(weights[b + "gate"], weights[b + "up"]))
            elif name in weights:
                p.copy_(weights[name])
            else:
                p.fill_(1.0)   # Llama's norms


def _experts_module(case, weights):
    from xgserve.models.vizonex import GroupedRouterMoE
    z, e = SIZES[case["size"]], EXPERTS
    ff = z["experts"]["ff"]
    m = GroupedRouterMoE(z["width"], {
        "expert": {"ff": ff, "limit": e["limit"]}, "shared": {"ff": ff, "limit": e["limit"]},
        "router": {"experts": e["experts"], "top": e["top"], "scale": e["scale"],
                   "groups": {"count": e["groups"], "keep": e["keep"]}}}, torch.device("cuda", 0), torch.bfloat16)
    _fill(m, weights)
    return m


@torch.no_grad()
def prepare(case, seed):
    from xgserve import ops
    from xgserve.models import AttnMeta, DofivikForCausalLM, LlamaForCausalLM, LoluzenForCausalLM, VizonexForCausalLM
    from xgserve.ops.attention import DecodeWorkspace
    from xgserve.ops.seqmix import SeqMeta
    from xgserve.tuning import enable_gemm_table
    dev = torch.device("cuda", 0)
    enable_gemm_table(dev)
    weights, step, ctx = _inputs(case, seed)
    if case["model"] == "experts":
        return dict(experts=_experts_module(case, weights), rows=step, act=step.to(torch.bfloat16))
    cls = {"llama": LlamaForCausalLM, "dofivik": DofivikForCausalLM, "loluzen": LoluzenForCausalLM,
           "vizonex": VizonexForCausalLM}[case["model"]]
    model = cls(_config(case, step), device=dev, dtype=torch.bfloat16)
    _fill(model, weights)
    decode = case["kind"] == "decode"
    meta = AttnMeta(num_tokens=step.T, num_decodes=step.S if decode else 0, positions=step.pos, slot_mapping=step.rows)
    if decode:
        meta.dec_block_tables, meta.dec_seq_lens = step.tables, step.lens
    else:
        meta.pre_block_tables, meta.pre_qsl, meta.pre_seq_lens = step.tables, step.qsl, step.lens
        meta.pre_max_q = step.max_q
    if case["model"] == "llama":
        model.fold_norms()
        z = LLAMA
        kv = torch.zeros(z["layers"], 2, step.num_blocks, z["kv"], BLOCK, z["dim"], dtype=torch.bfloat16, device=dev)
        cache = [(kv[i, 0], kv[i, 1]) for i in range(z["layers"])]
        for c, (k, v) in zip(ctx or (), cache):
            for pages, t in ((c["k"], k), (c["v"], v)):
                t.copy_(pages.view(step.num_blocks, BLOCK, z["kv"], z["dim"]).transpose(1, 2))
        wgs = max(1, step.S * z["kv"])   # the engine's rule: two workgroups per compute unit
        meta.num_splits = 1 if 4 * wgs >= 3 * 512 else min(16, -(-512 // wgs))
        meta.workspace = DecodeWorkspace(step.S, z["heads"], z["dim"], 16, dev)
        states = []
    else:
        if case["model"] == "dofivik":
            model.finalize_weights()
        if hasattr(model, "set_max_positions"):
            model.set_max_positions(step.max_len + 1)
        meta.seq = SeqMeta(num_seqs=step.S, max_q=step.max_q, qsl=step.qsl, seq_lens=step.lens, slots=step.slots,
                           block_tables=step.tables, token_seq=step.token_seq, positions=step.pos, slot_mapping=step.rows)
        cache = model.alloc_cache(step.num_blocks, BLOCK, step.S)
        for c, lc in zip(ctx or (), cache.layers):
            for name, t in c.items():
                getattr(lc, name).copy_(t.view_as(getattr(lc, name)))
        states = [getattr(lc, n) for lc in cache.layers for n in STATES if getattr(lc, n) is not None]

    def body():
        h = model(step.ids, meta, cache)
        last = h if decode else h.index_select(0, step.last)
        logits = model.compute_logits(last)
        return dict(hidden=h, logits=logits, logprob=ops.argmax_logprob(logits)[1], states=states)
    state = dict(body=body, graph=None)
    if decode:   # a decode step is a graph replay; warm up on the buffers, then put the contexts back
        keep = [t.clone() for t in states]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            body()
            body()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["out"] = body()
        for t, k in zip(states, keep):
            t.copy_(k)
    return state


@torch.no_grad()
def run(state):
    if "experts" in state:
        return state["experts"](state["rows"], state["act"])
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return state["body"]()


# ------------------------------------------------------------------------------------------------ what a step needs
def work(case):
    if case["model"] == "experts":
        z, e, n = SIZES[case["size"]], EXPERTS, case["tokens"]
        W, ff, E, top = z["width"], z["experts"]["ff"], e["experts"], e["top"]
        seen = E * (1 - (1 - top / E) ** n)
        return {"bytes": 2 * 3 * W * ff * (seen + 1) + 4 * E * W + n * W * (4 + 2 + 2 + 4),
                "flops": 2.0 * n * (3 * W * ff * (top + 1) + E * W)}
    seqs = _sequences(case)
    S, T = len(seqs), sum(q for q, _ in seqs)
    z = LLAMA if case["model"] == "llama" else SIZES[case["size"]]
    s = z if case["model"] == "llama" else z[case["model"]]
    W, V = z["width"], z["vocab"]
    # weights: all but the tables that are looked up; the output matrix works on the last tokens alone
    bytes_, flops = T * W * 2, 0.0
    for name, (shape, _, _, wide) in _tables(case).items():
        if name in ("embed", "pos"):
            continue
        bytes_ += math.prod(shape) * (4 if wide else 2)
        if len(shape) == 2 and min(shape) > 4:
            flops += 2.0 * math.prod(shape) * (S if name in ("head", "lm_head") else T)
    bytes_ += T * W * 2 + S * V * 2
    for kind in _layer_kinds(case):
        if kind in ("general_delta", "mamba2", "parallel"):
            d = {"general_delta": lambda: (s["d_heads"], s["d_dim"], s["d_dim"], 8),
                 "mamba2": lambda: (s["s_heads"], s["s_state"], s["s_vdim"], 5),
                 "parallel": lambda: (s["r_heads"], s["r_dim"], s["r_vdim"], 5)}[kind]()
            flops += d[3] * T * d[0] * d[1] * d[2]
            bytes_ += 4 * S * d[0] * d[1] * d[2] * (2 if case["kind"] == "decode" else 1)
        if kind in ("attention", "parallel", "latent_attention"):
            H = s["l_heads"] if kind == "parallel" else s["heads"]
            if kind == "latent_attention":
                row, pair, size = s["R"] + s["rot"], 2 * (s["dim"] + s["rot"] + s["vdim"]), s["window"]
            else:
                row, pair = 2 * (s["l_kv"] if kind == "parallel" else s["kv"]) * s["dim"], 4 * s["dim"]
                size = s.get("chunk", 1 << 30)
            for q, c in seqs:
                if "chunk" in s:
                    pairs = sum(p % size + 1 for p in range(c, c + q))
                    rows = (c % size + 1) if q == 1 else q
                else:
                    pairs = sum(min(p + 1, size) for p in range(c, c + q))
                    rows = min(c + q, size + q)
                flops += float(pair) * H * pairs
                bytes_ += 2 * row * rows
    return {"bytes": float(bytes_), "flops": float(flops)}


def tolerance(case):
    # bf16 activations and products between fp32 norms, softmax and states. Measured against 64 bits: 0.003 for the experts
    # alone, up to 0.011 after 8 to 16 sublayers
    if case["model"] == "experts":
        return {"rel": 0.012, "max": 0.2}
    return {"rel": 0.03, "max": 0.5}


# ------------------------------------------------------------------------------------------------ in 64 bits
def _lin(x, w):
    return x @ w.double().t()


def _unit(v, eps=EPS):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)


def _conv(x, w, hist):
    """Causal convolution per channel behind the rows `hist` [taps - 1, C]; and the rows it leaves behind."""
    ext = torch.cat([hist, x])
    n, w = x.shape[0], w.double()
    return sum(w[:, j] * ext[j:j + n] for j in range(w.shape[1])), ext[ext.shape[0] - (w.shape[1] - 1):]


def _turn(v, pos, freqs, dims, halves):
    """Rotation of the first `dims` entries by pos * freqs: pairs (i, i + dims / 2) or (2 i, 2 i + 1)."""
    a = pos.double()[:, None, None] * freqs
    c, s = a.cos(), a.sin()
    i, j = (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
    out = v.clone()
    out[..., i] = v[..., i] * c - v[..., j] * s
    out[..., j] = v[..., j] * c + v[..., i] * s
    return out


def _frequencies(dims, base, scaling, dev):
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=dev) / dims)
    if scaling:
        wave, o = 2 * math.pi / f, scaling["original"]
        s = (o / wave - scaling["low"]) / (scaling["high"] - scaling["low"])
        mid = (1 - s) * f / scaling["factor"] + s * f
        f = torch.where(wave < o / scaling["high"], f, torch.where(wave > o / scaling["low"], f / scaling["factor"], mid))
    return f


def _attend(q, k, v, ctx, scale, window=None, chunk=None, sink=None, temp=None, dist=None, talk=None):
    """q [n, H, dk] at positions ctx .., k / v [ctx + n, G, d] -> [n, H, dv]."""
    n, H, _ = q.shape
    G, L = k.shape[1], k.shape[0]
    i = torch.arange(ctx, ctx + n, device=q.device)[:, None]
    j = torch.arange(L, device=q.device)[None, :]
    seen = j <= i
    if window is not None:
        seen &= i - j < window
    if chunk is not None:
        seen &= i // chunk == j // chunk
    out, maps = [], []
    for h in range(H):
        s = q[:, h] @ k[:, h // (H // G)].t() * scale
        if temp is not None:
            s = s * temp[h]
        if dist is not None:
            s = s - dist[0][h] * torch.log1p(dist[1][h] * (i - j).clamp(min=0).double())
        s = s.masked_fill(~seen, -math.inf)
        top = s.amax(-1, keepdim=True) if sink is None else torch.maximum(s.amax(-1, keepdim=True), sink[h])
        e = torch.exp(s - top)
        p = e / (e.sum(-1, keepdim=True) + (0 if sink is None else torch.exp(sink[h] - top)))
        if talk is not None:
            maps.append(p)
        else:
            out.append(p @ v[:, h // (H // G)])
    for h in range(H if talk is not None else 0):
        p = sum(talk[h, g] * maps[g] for g in range(H))
        out.append(p @ v[:, h // (H // G)])
    return torch.stack(out, 1)


class _Exact:
    """One step of one model in 64 bits, the tokens of all sequences packed as the framework packs them."""

    def __init__(self, case, weights, step, ctx):
        self.case, self.w, self.st, self.ctx = case, weights, step, ctx
        self.z = LLAMA if case["model"] == "llama" else SIZES[case["size"]]
        self.s = self.z if case["model"] == "llama" else self.z[case["model"]]
        self.states = []

    def before(self, layer, name, s, shape):
        if self.ctx is None:
            return torch.zeros(shape, dtype=torch.float64, device="cuda")
        return self.ctx[layer][name][s].double()

    def pages(self, layer, name, s, new):
        """The rows a sequence attends to: its pages and the new tokens'."""
        if self.ctx is None:
            return new
        return torch.cat([self.ctx[layer][name][self.st.held(s)].double().view(-1, *new.shape[1:]), new])

    def each(self, f):
        """f(sequence, its rows) for every sequence, packed again."""
        return torch.cat([f(s, slice(self.st.first[s], self.st.first[s + 1])) for s in range(self.st.S)])

    def conv(self, x, w, layer, name):
        kept, out = [], []
        for s in range(self.st.S):
            y, left = _conv(x[self.st.first[s]:self.st.first[s + 1]], w, self.before(layer, name, s, (w.shape[1] - 1, x.shape[1])))
            out.append(y)
            kept.append(left)
        self.put(name, torch.stack(kept))
        return torch.cat(out)

    def put(self, name, t):
        self.layer_states[name] = t

    def recur(self, layer, name, shape, step_of):
        """step_of(token, S) -> (S, out) along every sequence, for all heads at once."""
        kept, out = [], []
        for s in range(self.st.S):
            S = self.before(layer, name, s, shape)
            for t in range(self.st.first[s], self.st.first[s + 1]):
                S, o = step_of(t, S)
                out.append(o)
            kept.append(S)
        self.put(name, torch.stack(kept))
        return torch.stack(out)

    # ---- mixers
    def llama_attention(self, i, h):
        z, st, b = self.s, self.st, f"layers.{i}."
        H, G, D = z["heads"], z["kv"], z["dim"]
        f = _frequencies(D, z["theta"], None, "cuda")
        q, k, v = _lin(h, self.w[b + "qkv"]).split([H * D, G * D, G * D], 1)
        q = _turn(q.reshape(-1, H, D), st.pos, f, D, True)
        k, v = _turn(k.reshape(-1, G, D), st.pos, f, D, True), v.reshape(-1, G, D)
        o = self.each(lambda s, r: _attend(q[r], self.pages(i, "k", s, k[r]), self.pages(i, "v", s, v[r]), st.seqs[s][1],
                                           D ** -0.5))
        return _lin(o.flatten(1), self.w[b + "o"])

    def latent(self, i, h):
        z, st, w = self.s, self.st, lambda n: self.w[f"layers.{i}.mix.{n}"]
        H, dn, rd, dv, R, Rq = z["heads"], z["dim"], z["rot"], z["vdim"], z["R"], z["Rq"]
        f = _frequencies(rd, 5e5, None, "cuda")
        cq, lat, key, gate = _lin(h, w("in_proj")).split([Rq, R, rd, H], 1)
        q = _lin(_unit(cq) * w("q_norm").double(), w("uq")).view(-1, H, dn + rd)
        q = torch.cat([q[..., :dn], _turn(q[..., dn:], st.pos, f, rd, False)], -1)
        row = torch.cat([_unit(lat) * w("kv_norm").double(), _turn(key[:, None], st.pos, f, rd, False)[:, 0]], 1)

        def one(s, r):
            rows = self.pages(i, "latent", s, row[r])
            k = torch.cat([_lin(rows[:, :R], w("uk")).view(-1, H, dn), rows[:, None, R:].expand(-1, H, -1)], -1)
            v = _lin(rows[:, :R], w("uv")).view(-1, H, dv)
            return _attend(q[r], k, v, st.seqs[s][1], (dn + rd) ** -0.5, window=z["window"])
        o = self.each(one) * torch.sigmoid(gate)[..., None]
        return _lin(o.flatten(1), w("o"))

    def delta(self, i, h):
        z, w = self.s, lambda n: self.w[f"layers.{i}.mix.{n}"]
        H, D = z["d_heads"], z["d_dim"]
        n = H * D
        r, k, v, g, a, low = _lin(h, w("in_proj")).split([n, n, n, n, n, 32], 1)
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(_lin(torch.tanh(low), w("w2")) + w("w0"))).view(-1, H, D, 1)
        r, k, v = r.reshape(-1, 1, H, D).transpose(1, 2), k.reshape(-1, H, D), v.reshape(-1, H, 1, D)
        u = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + UNIT_KEY_EPS))
        au = (torch.sigmoid(a + w("a_bias")).view(-1, H, D) * u)[..., None]
        u, k = u[:, :, None], k[..., None]

        def one(t, S):
            S = decay[t] * S - au[t] * (u[t] @ S) + k[t] * v[t]
            return S, r[t] @ S
        o = self.recur(i, "delta", (H, D, D), one).view(-1, H, D)
        return _lin(_unit(o).flatten(1) * w("norm") * torch.sigmoid(g), w("o"))

    def conv_attention(self, i, h):
        z, st, w = self.s, self.st, lambda n: self.w[f"layers.{i}.mix.{n}"]
        H, G, D = z["heads"], z["kv"], z["dim"]
        f = _frequencies(z["rot"], 5e5, ROT_SCALING, "cuda")
        p, gate = _lin(h, w("in_proj")).split([(H + 2 * G) * D, H], 1)
        q, k, v = self.conv(p, w("conv_w"), i, "mix_conv").split([H * D, G * D, G * D], 1)
        q = _turn(_unit(q.reshape(-1, H, D)) * w("q_norm"), st.pos, f, z["rot"], False)
        k = _turn(_unit(k.reshape(-1, G, D)) * w("k_norm"), st.pos, f, z["rot"], False)
        v = v.reshape(-1, G, D)
        o = self.each(lambda s, r: _attend(q[r], self.pages(i, "k", s, k[r]), self.pages(i, "v", s, v[r]), st.seqs[s][1],
                                           D ** -0.5))
        return _lin((o * torch.sigmoid(gate)[..., None]).flatten(1), w("o"))

    def two_branches(self, i, h):
        z, st, w = self.s, self.st, lambda n: self.w[f"layers.{i}.mix.{n}"]
        H, G, D, rh, dk, dv = z["l_heads"], z["l_kv"], z["dim"], z["r_heads"], z["r_dim"], z["r_vdim"]
        p = _lin(h, w("in_proj")) + w("in_bias").double()
        q, k, v, gate, rq, rf, rv = p.split([H * D, G * D, G * D, H, rh * dk, rh * dk, rh * dv], 1)
        q, k, v = q.reshape(-1, H, D), k.reshape(-1, G, D), v.reshape(-1, G, D)
        o = self.each(lambda s, r: _attend(q[r], self.pages(i, "k", s, k[r]), self.pages(i, "v", s, v[r]), st.seqs[s][1],
                                           D ** -0.5, dist=(w("left.r1").double(), w("left.r2").double()),
                                           talk=w("left.talk").double()))
        left = _lin((o * torch.sigmoid(gate)[..., None]).flatten(1), w("left.o"))
        low = w("right.lower").double()
        f = (low + (1 - low) * torch.sigmoid(rf)).view(-1, rh, dk, 1)
        rq, rv = F.silu(rq).view(-1, rh, 1, dk), rv.reshape(-1, rh, 1, dv)

        def one(t, S):
            S = f[t] * S + (1 - f[t]) * rv[t]
            return S, rq[t] @ S
        o = self.recur(i, "gla", (rh, dk, dv), one).view(-1, rh, dv)
        right = _lin((_unit(o) * w("right.norm")).flatten(1), w("right.o"))
        return 0.5 * (_unit(left) * w("left.out_norm") + _unit(right) * w("right.out_norm"))

    def chunk_attention(self, i, h):
        z, st, w = self.s, self.st, lambda n: self.w[f"layers.{i}.mix.{n}"]
        H, G, D = z["heads"], z["kv"], z["dim"]
        q, k, v = _lin(h, w("qkv")).split([H * D, G * D, G * D], 1)
        q, k = (_unit(q) * w("q_norm")).view(-1, H, D), (_unit(k) * w("k_norm")).view(-1, G, D)
        v = v.reshape(-1, G, D)
        o = self.each(lambda s, r: _attend(q[r], self.pages(i, "k", s, k[r]), self.pages(i, "v", s, v[r]), st.seqs[s][1],
                                           D ** -0.5, chunk=z["chunk"], sink=w("sink").double(), temp=w("temp").double()))
        return _lin(o.flatten(1), w("o"))

    def state_space(self, i, h):
        z, w = self.s, lambda n: self.w[f"layers.{i}.mix.{n}"]
        H, P, N, G = z["s_heads"], z["s_vdim"], z["s_state"], z["s_groups"]
        inner = H * P
        gate, xbc, dt = _lin(h, w("in_proj")).split([inner, inner + 2 * G * N, H], 1)
        xbc = F.silu(self.conv(xbc, w("conv_w"), i, "mix_conv") + w("conv_b"))
        x, B, C = xbc.split([inner, G * N, G * N], 1)
        x = x.reshape(-1, H, 1, P)
        B, C = (t.reshape(-1, G, N).repeat_interleave(H // G, 1) for t in (B, C))
        dt = F.softplus(dt + w("dt_bias"))[..., None, None]
        decay = torch.exp(-torch.exp(w("A_log").double())[:, None, None] * dt)
        B, C = dt * B[..., None], C[:, :, None]
        D = w("D").double()[:, None, None]

        def one(t, S):
            S = decay[t] * S + B[t] * x[t]
            return S, C[t] @ S + D * x[t]
        y = self.recur(i, "ssm", (H, N, P), one).reshape(-1, inner) * F.silu(gate)
        y = _unit(y.view(-1, G, inner // G)).reshape(-1, inner) * w("norm")
        return _lin(y, w("o"))

    # ---- models
    def forward(self):
        w, st, z, model = self.w, self.st, self.z, self.case["model"]
        x = w["embed"][st.ids.long()].double()
        if model == "loluzen":
            x = x * z["width"] ** 0.5
        elif model == "vizonex":
            x = x + w["pos"][st.pos.long()].double()
        mixers = {("llama", "attention"): self.llama_attention, ("dofivik", "latent_attention"): self.latent,
                  ("dofivik", "general_delta"): self.delta, ("loluzen", "attention"): self.conv_attention,
                  ("loluzen", "parallel"): self.two_branches, ("vizonex", "attention"): self.chunk_attention,
                  ("vizonex", "mamba2"): self.state_space}
        for i, kind in enumerate(_layer_kinds(self.case)):
            self.layer_states = {}
            g = lambda n: w[f"layers.{i}.{n}"]  # noqa: E731
            mix = mixers[model, kind]
            if model == "llama":
                x = x + mix(i, _unit(x))
                h = _unit(x)
                x = x + _lin(F.silu(_lin(h, g("gate"))) * _lin(h, g("up")), g("down"))
            elif model == "dofivik":
                h = x + self.conv(x, g("canon1"), i, "conv1")
                x = _unit(2.0 * x + mix(i, h)) * (1 + g("norm1"))
                h = x + self.conv(x, g("canon2"), i, "conv2")
                v = _lin(h, g("mlp.up")) + g("mlp.up_b")
                sp, cn = F.softplus(g("mlp.act").double())
                v = torch.where(v > 0, sp * v * v, (0.5 + cn) * (torch.expm1(v.clamp(max=0)) - v)) + 0.5 * v
                x = _unit(2.0 * x + _lin(v, g("mlp.down")) + g("mlp.down_b")) * (1 + g("norm2"))
            elif model == "loluzen":
                x = x + 0.5 * _unit(mix(i, _unit(x) * (1 + g("norm1")))) * (1 + g("norm1b"))
                v = F.relu(_lin(_unit(x) * (1 + g("norm2")), g("mlp.up")) + g("mlp.up_b")) ** 2
                x = x + 0.5 * _unit(_lin(v, g("mlp.down")) + g("mlp.down_b")) * (1 + g("norm2b"))
            else:
                n = _unit(x) * g("norm1")
                y = mix(i, n + self.conv(n, g("canon1"), i, "conv1"))
                gate, up = _lin(n, g("mlp.gate_up")).chunk(2, 1)
                x = x + y * g("ls1") + _lin(F.gelu(gate, approximate="tanh") * up, g("mlp.down")) * g("ls2")
            self.states += [self.layer_states[n] for n in STATES if n in self.layer_states]
        h = _unit(x)
        if model != "llama":
            h = h * (w["final_norm"].double() + (0.0 if model == "vizonex" else 1.0))
        logits = _lin(h[st.last], w["lm_head" if model == "llama" else "head"])
        return dict(hidden=h, logits=logits, logprob=torch.log_softmax(logits, -1).amax(-1), states=self.states)


@torch.no_grad()
def exact(case, seed):
    weights, step, ctx = _inputs(case, seed)
    if case["model"] != "experts":
        return _Exact(case, weights, step, ctx).forward()
    e = EXPERTS
    n32 = step.double()
    x = step.to(torch.bfloat16).double()   # the experts read the rounded rows, the router the fp32 ones

    def gated(h, w13, w2):
        g, u = _lin(h, w13).chunk(2, 1)
        g, u = g.clamp(max=e["limit"]), u.clamp(-e["limit"], e["limit"])
        return _lin(g * torch.sigmoid(SINK_ALPHA * g) * (u + 1.0), w2)
    score = torch.sigmoid(_lin(n32, weights["router"]))
    pick = score + weights["correction"].double()
    parts = pick.view(-1, e["groups"], e["experts"] // e["groups"])
    kept = torch.zeros_like(parts[..., 0]).scatter_(1, parts.topk(2, -1).values.sum(-1).topk(e["keep"], -1).indices, 1.0)
    pick = pick.masked_fill(kept.repeat_interleave(parts.shape[2], 1) == 0, -math.inf)
    ids = pick.topk(e["top"], -1).indices
    share = torch.zeros_like(score).scatter_(1, ids, score.gather(1, ids) * e["scale"])
    routed = torch.zeros_like(n32)
    for k in range(e["experts"]):
        at = share[:, k].nonzero()[:, 0]
        routed[at] += share[at, k, None] * gated(x[at], weights["w13"][k], weights["w2"][k])
    return gated(x, weights["shared.gate_up"], weights["shared.down"]), routed
