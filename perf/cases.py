"""The work this framework is used for, as cases that can be timed and checked.

Three kinds of programs use it: a chat node whose engine answers prompts with a Llama or Mixtral
model (``engine.Engine``), a server or a trace runner on a hybrid model (``engine.hybrid``), and a
model author who builds layers from the registered parts (``models.hybrid``).  A case is one step
of such a program: a batch of prompts run to their logits (prefill), one decode step of running
sequences, or one mixture-of-experts layer.  Engines and weights are kept between steps, as a
server keeps them; prompts, pages and state slots belong to a request.

``exact`` is the same mathematics in 64 bits, written token by token where a mechanism is defined
that way, on plain tensors.
"""
from __future__ import annotations

import math
import random

import torch

DEV = "cuda"
WEIGHT_SEED = 20        # the served models' weights; a case's seed draws its inputs

LLAMA = {"llama3.1-8b": dict(hidden=4096, heads=32, kv=8, ffn=14336, vocab=128256, theta=500000.0,
                             scaling=(8.0, 1.0, 4.0, 8192), experts=0),
         "mixtral-8x7b": dict(hidden=4096, heads=32, kv=8, ffn=14336, vocab=32000, theta=1e6,
                              scaling=None, experts=8)}
HEAD, TOP = 128, 2      # head size and experts per token of those models
VOCAB = 32000           # hybrid models


def listed() -> list:
    # the dense model runs with a quarter of its layers: through all of them bf16 rounding alone moves
    # the logits by 4 %, more than a comparison can tell from a mistake
    return [
        # a suggested reply being written: one token after a chat prompt of median length
        dict(name="reply decode", family="llama", model="llama3.1-8b", layers=8, phase="decode",
             seqs=1, tokens=107),
        # the time to the first token of that reply
        dict(name="reply prefill", family="llama", model="llama3.1-8b", layers=8, phase="prefill",
             seqs=1, tokens=44),
        # many peers being answered at once, each at another length
        dict(name="peers decode", family="llama", model="llama3.1-8b", layers=8, phase="decode",
             seqs=19, tokens=900),
        # a long thread and shorter ones arriving together
        dict(name="threads prefill", family="llama", model="llama3.1-8b", layers=8, phase="prefill",
             seqs=3, tokens=1111),
        # a prompt on the sparse model (two of its layers: all of them do not fit three times over)
        dict(name="sparse prefill", family="llama", model="mixtral-8x7b", layers=2, phase="prefill",
             seqs=1, tokens=700),
        # the hybrid benchmark's prompt and its decode step, at its larger width
        dict(name="regesun prefill", family="hybrid", model="regesun", width=2048, blocks=2, phase="prefill",
             seqs=1, tokens=2048, dtype="bf16"),
        dict(name="regesun decode", family="hybrid", model="regesun", width=2048, blocks=2, phase="decode",
             seqs=8, tokens=512, dtype="bf16"),
        # prompts of several lengths in one step
        dict(name="rasepel prefill", family="hybrid", model="rasepel", width=2048, blocks=2, phase="prefill",
             seqs=3, tokens=1201, dtype="bf16"),
        # a single user on a small model: launches and latency
        dict(name="rasepel decode", family="hybrid", model="rasepel", width=1024, blocks=2, phase="decode",
             seqs=1, tokens=333, dtype="bf16"),
        # attention only, every key in sight
        dict(name="tarunex prefill", family="hybrid", model="tarunex", width=2048, blocks=1, phase="prefill",
             seqs=1, tokens=2048, dtype="bf16"),
        # the exact number format (traces replayed for comparison), routed experts, ragged
        dict(name="tarunex fp32 prefill", family="hybrid", model="tarunex", width=1024, blocks=1,
             phase="prefill", seqs=2, tokens=389, dtype="fp32"),
        # the routed experts of the hybrid models by themselves
        dict(name="experts", family="experts", width=2048, ff=1024, experts=8, top=2, rows=2048, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(("llama", "llama", "llama", "sparse", "regesun", "regesun", "rasepel", "rasepel",
                       "tarunex", "tarunex", "tarunex fp32", "experts"))
    if kind in ("llama", "sparse"):
        c = dict(family="llama", model="llama3.1-8b", layers=8, phase=rng.choice(("decode", "prefill")))
        if kind == "sparse":
            c.update(model="mixtral-8x7b", layers=2, phase="prefill")
        c["seqs"] = _log_int(rng, 1, 32) if c["phase"] == "decode" else rng.randint(1, 3)
        c["tokens"] = _log_int(rng, 24, 1000)
        return c
    if kind == "experts":
        w = rng.choice((1024, 2048))
        return dict(family="experts", width=w, ff=w // 2, experts=8, top=2, rows=_log_int(rng, 1, 2048),
                    dtype=rng.choice(("bf16", "bf16", "bf16", "fp32")))
    c = dict(family="hybrid", model=kind.split()[0], width=rng.choice((1024, 2048)), blocks=2,
             phase=rng.choice(("decode", "prefill", "prefill")), dtype="bf16")
    if kind.startswith("tarunex"):
        c["blocks"] = 1
    if kind == "tarunex fp32":
        c.update(width=1024, dtype="fp32", seqs=rng.randint(1, 2), tokens=_log_int(rng, 16, 512))
        return c
    c["seqs"] = _log_int(rng, 1, 16) if c["phase"] == "decode" else rng.randint(1, 3)
    c["tokens"] = _log_int(rng, 16, 640 if c["phase"] == "decode" else 1024 if c["seqs"] > 1 else 2048)
    return c


def lengths(case) -> list:
    """Tokens that each sequence has: the first the case's number, the others fewer."""
    n = case["tokens"]
    return [n] + [max(1, n * ((5 * i + 2) % 9 + 1) // 10 + i % 3) for i in range(1, case["seqs"])]


def prompts_of(case, seed) -> list:
    """Token ids per sequence; a decode step's last one is the token it runs."""
    vocab = LLAMA[case["model"]]["vocab"] if case["family"] == "llama" else VOCAB
    g = torch.Generator().manual_seed(int(seed) * 7919 + 13)
    extra = 1 if case["phase"] == "decode" else 0
    return [torch.randint(3, vocab, (n + extra,), generator=g).tolist() for n in lengths(case)]


# ----------------------------------------------------------------------- models
def _llama_tensors(case) -> dict:
    """A random checkpoint by its published names (projections N(0, 0.02), gains near 1)."""
    m = LLAMA[case["model"]]
    g = torch.Generator(device=DEV).manual_seed(WEIGHT_SEED)

    def rnd(*shape, std=0.02):
        return torch.empty(*shape, device=DEV, dtype=torch.bfloat16).normal_(0.0, std, generator=g)

    def gain(n):
        return (1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)).bfloat16()

    h, f = m["hidden"], m["ffn"]
    t = {"model.embed_tokens.weight": rnd(m["vocab"], h, std=1.0), "model.norm.weight": gain(h),
         "lm_head.weight": rnd(m["vocab"], h)}
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        t[p + "input_layernorm.weight"], t[p + "post_attention_layernorm.weight"] = gain(h), gain(h)
        t[p + "self_attn.q_proj.weight"] = rnd(m["heads"] * HEAD, h)
        t[p + "self_attn.k_proj.weight"] = rnd(m["kv"] * HEAD, h)
        t[p + "self_attn.v_proj.weight"] = rnd(m["kv"] * HEAD, h)
        t[p + "self_attn.o_proj.weight"] = rnd(h, m["heads"] * HEAD)
        if not m["experts"]:
            t[p + "mlp.gate_proj.weight"], t[p + "mlp.up_proj.weight"] = rnd(f, h), rnd(f, h)
            t[p + "mlp.down_proj.weight"] = rnd(h, f)
            continue
        p += "block_sparse_moe."
        t[p + "gate.weight"] = rnd(m["experts"], h, std=0.5)
        for e in range(m["experts"]):
            q = p + "experts.%d." % e
            t[q + "w1.weight"], t[q + "w3.weight"], t[q + "w2.weight"] = rnd(f, h), rnd(f, h), rnd(h, f)
    return t


def _hybrid_config(case) -> dict:
    """The hybrid benchmark's stacks, cut to ``blocks`` of their blocks.  In bf16 the attention-only
    one takes dense feed-forwards (rounding alone decides close calls of a router)."""
    w, nh = case["width"], case["width"] // 128
    clamped = {"kind": "dense", "ff": 4 * w, "limit": 7.0}
    c = {"width": w, "vocab": VOCAB, "norm": {"eps": 1e-5}}
    if case["model"] == "regesun":
        gd = {"type": "general_delta", "mixer": {"heads": w // 64, "dim": 64}, "mlp": None}
        mb = {"type": "mamba2", "mixer": {"heads": w // 32, "vdim": 64, "state": 128, "groups": 8, "conv": 4,
                                          "norm_groups": 8}, "mlp": None}
        la = {"type": "latent_attention", "mixer": {"heads": nh, "dim": 128, "vdim": 128, "kv_rank": w // 4,
                                                    "mask": {"size": 1024}, "scale": 128 ** -0.5}, "mlp": clamped}
        return dict(c, architecture="Regesun", max_positions=8192, layers=[gd, mb, mb, la] * case["blocks"])
    if case["model"] == "rasepel":
        mb = {"type": "mamba1", "mixer": {"inner": 2 * w, "state": 16, "dt_rank": w // 16, "conv": 4}, "mlp": None}
        lg = {"type": "lightning", "mixer": {"heads": nh, "dim": 128, "vdim": 128,
                                             "decay": [1.0 - 2.0 ** (-1.0 - 8.0 * i / nh) for i in range(nh)]},
              "mlp": None}
        at = {"type": "attention", "mixer": {"heads": nh, "kv_heads": max(1, nh // 4), "dim": 128, "vdim": 128,
                                             "conv": 4, "mask": {"size": 1024, "pool": 16},
                                             "rot": {"base": 500000.0, "dims": 64}, "scale": 128 ** -0.5},
              "mlp": clamped}
        return dict(c, architecture="Rasepel", embedding={"scale": 1.0}, layers=[mb, lg, mb, at] * case["blocks"])
    ff = {"kind": "dense", "ff": 2 * w} if case["dtype"] == "bf16" else \
        {"kind": "moe", "expert": {"ff": w // 2}, "shared": {"ff": w // 2}, "router": {"experts": 8, "top": 2}}
    ba = {"type": "attention", "mixer": {"heads": nh, "kv_heads": max(1, nh // 4), "dim": 128, "vdim": 128,
                                         "scale": 128 ** -0.5, "softcap": 50.0,
                                         "q_temp": {"coef": 0.1, "every": 512}}, "mlp": ff}
    la = {"type": "latent_attention", "mixer": {"heads": nh, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 448,
                                                "q_rank": w // 2, "rot": {"base": 10000.0, "dims": 64},
                                                "scale": 192 ** -0.5}, "mlp": ff}
    return dict(c, architecture="Tarunex", embedding={"scale": w ** 0.5}, logit_scale=0.5, logit_softcap=50.0,
                loop={"start": 1, "stop": 3, "times": 2}, layers=[ba, la, ba, la] * case["blocks"])


def _part_shapes(kind, m, w) -> dict:
    """Tensor shapes of one mixer."""
    if kind == "general_delta":
        n = m["heads"] * m["dim"]
        return dict({k: (n, w) for k in "rkvga"}, **{"a.b": (n,), "w1": (32, w), "w2": (n, 32), "w0": (n,),
                                                     "norm": (n,), "o": (w, n)})
    if kind == "mamba2":
        inner, gn = m["heads"] * m["vdim"], m["groups"] * m["state"]
        return {"in": (2 * inner + 2 * gn + m["heads"], w), "conv": (inner + 2 * gn, m["conv"]),
                "conv.b": (inner + 2 * gn,), "dt_bias": (m["heads"],), "A_log": (m["heads"],), "D": (m["heads"],),
                "norm": (inner,), "o": (w, inner)}
    if kind == "mamba1":
        i, n, r = m["inner"], m["state"], m["dt_rank"]
        return {"in": (2 * i, w), "conv": (i, m["conv"]), "conv.b": (i,), "x": (r + 2 * n, i), "dt": (i, r),
                "dt.b": (i,), "A_log": (i, n), "D": (i,), "o": (w, i)}
    h, d, v = m["heads"], m["dim"], m["vdim"]
    if kind == "lightning":
        return {"q": (h * d, w), "k": (h * d, w), "v": (h * v, w), "g": (h * v, w), "norm": (h * v,), "o": (w, h * v)}
    if kind == "latent_attention":
        r = m["kv_rank"]
        s = {"dkv.norm": (r,), "uk": (h * d, r), "uv": (h * v, r), "o": (w, h * v)}
        if "q_rank" in m:
            return dict(s, **{"dq": (m["q_rank"], w), "dq.norm": (m["q_rank"],), "g": (h, w),
                              "uq": (h * (d + m["rot_dim"]), m["q_rank"]), "dkv": (r + m["rot_dim"], w)})
        return dict(s, q=(h * d, w), dkv=(r, w), sink=(h,), g=(h * v, w))
    g = m["kv_heads"]
    s = {"q": (h * d, w), "q.b": (h * d,), "k": (g * d, w), "k.b": (g * d,), "v": (g * v, w), "v.b": (g * v,),
         "o": (w, h * v)}
    if "pool" in m.get("mask", {}):
        return dict(s, **{"q.conv": (h * d, m["conv"]), "k.conv": (g * d, m["conv"]), "v.conv": (g * v, m["conv"]),
                          "temp": (h,), "g": (h * v, w), "o.b": (w,)})
    return dict(s, r1=(h,), r2=(h,), g=(h, w))


def _ff_shapes(m, w) -> dict:
    def unit(p, f):
        return {p + "gate": (f, w), p + "up": (f, w), p + "down": (w, f)}

    if m["kind"] == "dense":
        return unit("", m["ff"])
    s = {"router": (m["router"]["experts"], w), "router.b": (m["router"]["experts"],)}
    for e in range(m["router"]["experts"]):
        s.update(unit("e%d." % e, m["expert"]["ff"]))
    if m.get("shared"):
        s.update(unit("shared.", m["shared"]["ff"]))
    return s


def _draw_tensor(name, shape, offset, g):
    """Projections ~ N(0, 1/inputs), gains near 1, decays and steps where the recurrences hold."""
    t = torch.randn(shape or (1,), generator=g, device=DEV)
    u = torch.rand(shape or (1,), generator=g, device=DEV)
    leaf = name.split(".", 1)[1] if name[0] == "l" and "." in name and name != "loop.step" else name
    if leaf.endswith("A_log"):
        t = u * 1.5 - 1.0
    elif leaf.endswith("conv") or leaf in ("loop.step",):
        t = t * 0.5
    elif leaf in ("embed", "pos"):
        pass
    elif len(shape) == 2:
        t = t / shape[1] ** 0.5
    elif leaf in ("norm1", "norm2", "norm1b", "norm2b", "final.norm"):
        t = 1.0 - offset + 0.1 * t
    elif leaf.endswith("norm"):
        t = 1.0 + 0.1 * t
    elif leaf in ("ls1", "ls2"):
        t = 0.5 + 0.1 * t
    elif leaf.endswith("mix.r1"):
        t = u * 2.0
    elif leaf.endswith("mix.r2"):
        t = u * 0.3
    elif leaf.endswith("mix.dt.b"):
        t = t - 2.0
    elif leaf.endswith("mix.temp"):
        t = 1.0 + 0.2 * t
    else:
        t = t * 0.5
    return t.bfloat16().reshape(shape)


def _hybrid_tensors(case) -> dict:
    c, w = _hybrid_config(case), case["width"]
    kind = c["architecture"]
    shapes = {"embed": (VOCAB, w), "final.norm": () if kind == "Tarunex" else (w,)}
    if kind != "Rasepel":
        shapes["head"] = (VOCAB, w)
    if kind == "Regesun":
        shapes["pos"] = (c["max_positions"], w)
    if "loop" in c:
        shapes["loop.step"] = (c["loop"]["times"], w)
    for i, layer in enumerate(c["layers"]):
        p = "l%d." % i
        for q in (1, 2) if layer["mlp"] else (1,):
            shapes[p + "norm%d" % q] = () if kind == "Tarunex" else (w,)
            if kind == "Regesun":
                shapes[p + "norm%db" % q] = shapes[p + "ls%d" % q] = (w,)
        shapes.update({p + "mix." + k: s for k, s in _part_shapes(layer["type"], layer["mixer"], w).items()})
        if layer["mlp"]:
            shapes.update({p + "mlp." + k: s for k, s in _ff_shapes(layer["mlp"], w).items()})
    g = torch.Generator(device=DEV).manual_seed(WEIGHT_SEED)
    offset = 1.0 if kind == "Rasepel" else 0.0
    return {k: _draw_tensor(k, s, offset, g) for k, s in shapes.items()}


def _experts_config(case) -> dict:
    return {"kind": "moe", "expert": {"ff": case["ff"]}, "router": {"experts": case["experts"], "top": case["top"]}}


def _experts_tensors(case) -> dict:
    g = torch.Generator(device=DEV).manual_seed(WEIGHT_SEED)
    return {k: _draw_tensor("l0.mlp." + k, s, 0.0, g)
            for k, s in _ff_shapes(_experts_config(case), case["width"]).items()}


_SERVED = {}    # the engine (or layer) of the model that is being served


def _served(case):
    key = tuple(case.get(k) for k in ("family", "model", "layers", "width", "blocks", "dtype", "ff", "experts"))
    if key not in _SERVED:
        _SERVED.clear()
        torch.cuda.empty_cache()
        _SERVED[key] = _load(case)
    return _SERVED[key]


def _dtype(case):
    return torch.float32 if case.get("dtype") == "fp32" else torch.bfloat16


def _load(case):
    if case["family"] == "llama":
        from p2p_llm_chat_go_amd.engine import Engine
        from p2p_llm_chat_go_amd.models.config import get_config
        from p2p_llm_chat_go_amd.models.weights import EngineWeights

        cfg = get_config(case["model"]).replace(n_layers=case["layers"])
        eng = Engine(cfg, weights=EngineWeights.from_state_dict(_llama_tensors(case), cfg, DEV), device=DEV,
                     kv_pages=2048, max_batch=64)
        eng.autotune((1, 2, 4, 8, 16, 32, 48, 64))
        return eng
    if case["family"] == "hybrid":
        from p2p_llm_chat_go_amd.models.hybrid import HybridConfig, HybridWeights
        from p2p_llm_chat_go_amd.models.registry import make_engine

        cfg = HybridConfig.from_dict(_hybrid_config(case), name=case["model"])
        t = {k: v.cpu() for k, v in _hybrid_tensors(case).items()}   # as a file's tensors arrive
        return make_engine(cfg, HybridWeights(cfg, t, DEV, _dtype(case)), DEV, kv_pages=1536, max_batch=16,
                           num_slots=96, max_prefill_tokens=4096)
    from p2p_llm_chat_go_amd.models.hybrid import FEEDFORWARDS

    ff = FEEDFORWARDS["moe_top"](_experts_config(case), case["width"])
    t = _experts_tensors(case)
    ff.load(lambda k: t[k], _dtype(case), DEV)
    return ff


# ----------------------------------------------------------------------- requests
class LlamaRequests:
    """Prompts and the pages they hold; a decode step's prompts are in the cache already."""

    def __init__(self, eng, case, seed):
        from p2p_llm_chat_go_amd.engine.kv_cache import pages_for
        from p2p_llm_chat_go_amd.engine.sampling import SamplingParams

        self.eng, self.prompts = eng, prompts_of(case, seed)
        self.pages = [eng.kv.allocator.alloc(pages_for(len(p))) for p in self.prompts]
        # replies are sampled with the usual options, so a step's logits are there to be read
        self.params = [SamplingParams(temperature=0.8, top_k=40, top_p=0.9, seed=seed + b)
                       for b in range(len(self.prompts))]
        self.rows, self.ctx = sum(len(p) for p in self.prompts), max(len(p) for p in self.prompts)
        self.decode = case["phase"] == "decode"
        self.captured = not eng.cfg.is_moe and self.rows <= eng.max_prefill_tokens
        if self.decode:
            eng.prefill([p[:-1] for p in self.prompts], self.pages, graph=False)
            eng.decode_graph(len(self.prompts), self.ctx, greedy=False)
            self.last, self.at = [p[-1] for p in self.prompts], [len(p) - 1 for p in self.prompts]
        elif self.captured:
            eng.prefill_graph(self.rows, len(self.prompts), self.ctx, greedy=False)

    def __del__(self):
        for p in getattr(self, "pages", ()):
            self.eng.kv.allocator.free(p)

    def run(self):
        eng, n = self.eng, len(self.prompts)
        if self.decode:
            eng.decode_steps(self.last, self.at, self.pages, self.ctx, 1, params=self.params)
            return eng.decode_graph(n, self.ctx, greedy=False).state.ws.logits[:n]
        if self.captured:
            eng.prefill(self.prompts, self.pages, sampling=self.params)
            return eng.prefill_graph(self.rows, n, self.ctx, greedy=False).ws.logits[:n]
        return eng.prefill(self.prompts, self.pages, return_logits=True)[1]


class HybridRequests:
    """Prompts and the sequences they are; a decode step's sequences are open already."""
    MOST = 60   # recurrent states that are looked at

    def __init__(self, eng, case, seed):
        self.eng, self.prompts = eng, prompts_of(case, seed)
        self.keys = [(id(self), b) for b in range(len(self.prompts))]
        self.decode = case["phase"] == "decode"
        if self.decode:
            for k, p in zip(self.keys, self.prompts):
                eng.step([(k, p[:-1], [])])
            seqs = [eng.cache.get(k) for k in self.keys]
            for s in seqs:
                eng.cache.reserve(s, s.length + 1)
            self.rows = [(s.slot, s.pages, s.length, p[-1]) for s, p in zip(seqs, self.prompts)]
            self.graph = eng.decode_graph(len(self.rows), max(len(s.pages) for s in seqs))

    def close(self):
        for k in getattr(self, "keys", ()):
            if k in self.eng.cache:
                self.eng.release(k)

    def __del__(self):
        self.close()

    def states(self):
        """Recurrent states after the step, the first sequences' first."""
        st = self.eng.cache.state
        every = [st[i]["S"][self.eng.cache.get(k).slot] for k in self.keys for i in sorted(st) if "S" in st[i]]
        return every[:self.MOST]

    def run(self):
        if self.decode:
            self.graph.step(self.rows)
            logits = self.graph.logits[:len(self.rows)]
        else:
            self.close()   # the prompts come anew
            logits = self.eng.step([(k, p, [len(p) - 1]) for k, p in zip(self.keys, self.prompts)])
        return {"logits": logits, "states": self.states()}


def prepare(case, seed):
    served = _served(case)
    if case["family"] == "llama":
        return LlamaRequests(served, case, seed)
    if case["family"] == "hybrid":
        return HybridRequests(served, case, seed)
    return served, _experts_input(case, seed).to(_dtype(case))


def _experts_input(case, seed):
    """Normed rows."""
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 13)
    return torch.randn(case["rows"], case["width"], generator=g, device=DEV).bfloat16()


def run(state):
    if isinstance(state, tuple):
        return state[0].forward(state[1])
    return state.run()


# ----------------------------------------------------------------------- work
def _numbers(shapes) -> int:
    return sum(math.prod(s) for s in shapes)


def work(case) -> dict:
    size = 4 if case.get("dtype") == "fp32" else 2
    if case["family"] == "experts":
        n, w, f = case["rows"], case["width"], case["ff"]
        hit = min(case["experts"], n * case["top"])
        return {"bytes": size * (hit * 3 * w * f + 2 * n * w) + 4 * case["experts"] * w,
                "flops": 6.0 * n * case["top"] * w * f + 2.0 * n * case["experts"] * w}
    lens, decode = lengths(case), case["phase"] == "decode"
    rows = len(lens) if decode else sum(lens)
    # (query, key) pairs of an attention over a window; keys that a step reads
    pairs = lambda win: sum(min(n + 1, win) if decode else sum(min(i + 1, win) for i in range(n)) for n in lens)
    read = lambda win: sum(min(n, win) for n in lens) if decode else 0
    if case["family"] == "llama":
        m = LLAMA[case["model"]]
        h, f, kv = m["hidden"], m["ffn"], m["kv"] * HEAD
        attn = h * (m["heads"] * HEAD + 2 * kv) + m["heads"] * HEAD * h
        used = min(m["experts"], rows * TOP) if m["experts"] else 1
        each = TOP if m["experts"] else 1
        head = h * m["vocab"]
        return {"bytes": 2.0 * (case["layers"] * (attn + 3 * h * f * used + 2 * kv * (rows + read(1 << 30))) + head
                                + rows * h) + 4.0 * len(lens) * m["vocab"],
                "flops": 2.0 * case["layers"] * (rows * (attn + 3 * h * f * each)
                                                 + 2 * pairs(1 << 30) * m["heads"] * HEAD) + 2.0 * len(lens) * head}
    c, w = _hybrid_config(case), case["width"]
    nbytes = size * (VOCAB * w + rows * w) + 4.0 * len(lens) * VOCAB
    flops = 2.0 * len(lens) * VOCAB * w
    runs = [i for i, _t, _f in _runs(c)]
    for i, layer in enumerate(c["layers"]):
        times, m = runs.count(i), layer["mixer"]
        shapes = _part_shapes(layer["type"], m, w)
        nbytes += size * _numbers(shapes.values())
        flops += 2.0 * times * rows * _numbers(s for k, s in shapes.items() if len(s) == 2 and "conv" not in k
                                               and "A_log" not in k)
        if layer["mlp"]:
            ff = layer["mlp"]
            if ff["kind"] == "dense":
                nbytes += size * 3 * w * ff["ff"]
                flops += 6.0 * times * rows * w * ff["ff"]
            else:
                e, top, f = ff["router"]["experts"], ff["router"]["top"], ff["expert"]["ff"]
                nbytes += size * (3 * w * f * min(e, rows * top) + 3 * w * ff["shared"]["ff"])
                flops += 6.0 * times * rows * w * (top * f + ff["shared"]["ff"])
        if layer["type"] in ("general_delta", "mamba2", "mamba1", "lightning"):
            state = m["inner"] * m["state"] if layer["type"] == "mamba1" else \
                m["heads"] * m["dim" if "dim" in m else "state"] * m.get("vdim", m.get("dim"))
            nbytes += 4.0 * state * len(lens) * (2 if decode else 1)
            flops += (8.0 if layer["type"] == "general_delta" else 6.0) * rows * state
            continue
        win = m.get("mask", {}).get("size", 1 << 30)
        if layer["type"] == "latent_attention":
            kept, per = m["kv_rank"] + m.get("rot_dim", 0), 2 * m["dim"] + m.get("rot_dim", 0)
        else:
            kept, per = m["kv_heads"] * 2 * m["dim"], 2 * m["dim"]
        nbytes += size * times * kept * (rows + read(win))
        flops += 2.0 * times * pairs(win) * m["heads"] * per
    return {"bytes": nbytes, "flops": flops}


def tolerance(case) -> dict:
    # about four times what the outputs are off exact(): whole models in bf16 round every layer's
    # activations, the Llama family's residual stream too
    if case.get("dtype") == "fp32":
        return {"rel": 2e-5}
    return {"rel": {"experts": 0.012, "hybrid": 0.03, "llama": 0.03}[case["family"]]}


# ----------------------------------------------------------------------- 64 bits
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _rotate(x, angles, halves):
    """x [T, heads, n]: channel pairs (i, i + n/2), or (2i, 2i + 1), turned by ``angles`` [T, n/2]."""
    c, s = torch.cos(angles)[:, None], torch.sin(angles)[:, None]
    if halves:
        a, b = x.chunk(2, -1)
        return torch.cat([a * c - b * s, b * c + a * s], -1)
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2)


def _angles(T, dims, base, scaling=None):
    f = base ** (-torch.arange(0, dims, 2, device=DEV, dtype=torch.float64) / dims)
    if scaling:
        factor, low, high, original = scaling
        wave = 2 * math.pi / f
        smooth = ((original / wave - low) / (high - low)).clamp(0.0, 1.0)
        f = (1 - smooth) * f / factor + smooth * f
    return torch.arange(T, device=DEV, dtype=torch.float64)[:, None] * f


def _causal(T, window=1 << 30):
    d = torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)[None]
    return (d >= 0) & (d < window)


def _exact_llama(case, t, ids):
    """Logits of the last position."""
    m, T = LLAMA[case["model"]], len(ids)
    w = lambda name: t[name].double()
    x = t["model.embed_tokens.weight"][torch.tensor(ids, device=DEV)].double()
    ang, group = _angles(T, HEAD, m["theta"], m["scaling"]), m["heads"] // m["kv"]
    keep = _causal(T)
    for i in range(case["layers"]):
        p = "model.layers.%d." % i
        h = _rms(x, 1e-5) * w(p + "input_layernorm.weight")
        q, k, v = ((h @ w(p + "self_attn.%s_proj.weight" % n).T).view(T, -1, HEAD) for n in "qkv")
        q, k = _rotate(q, ang, True), _rotate(k, ang, True)
        o = torch.empty_like(q)
        for g in range(m["kv"]):
            s = torch.einsum("tgd,sd->gts", q[:, g * group:(g + 1) * group], k[:, g]) / HEAD ** 0.5
            a = torch.softmax(s.masked_fill(~keep, -math.inf), -1)
            o[:, g * group:(g + 1) * group] = (a @ v[:, g]).transpose(0, 1)
        x = x + o.reshape(T, -1) @ w(p + "self_attn.o_proj.weight").T
        h = _rms(x, 1e-5) * w(p + "post_attention_layernorm.weight")
        if not m["experts"]:
            x = x + (_silu(h @ w(p + "mlp.gate_proj.weight").T) * (h @ w(p + "mlp.up_proj.weight").T)) \
                @ w(p + "mlp.down_proj.weight").T
            continue
        p += "block_sparse_moe."
        weight, idx = torch.softmax(h @ w(p + "gate.weight").T, -1).topk(TOP, -1)
        weight = weight / weight.sum(-1, keepdim=True)
        for e in range(m["experts"]):
            q = p + "experts.%d." % e
            rows, slot = (idx == e).nonzero(as_tuple=True)
            y = (_silu(h[rows] @ w(q + "w1.weight").T) * (h[rows] @ w(q + "w3.weight").T)) @ w(q + "w2.weight").T
            x.index_add_(0, rows, y * weight[rows, slot][:, None])
    return (_rms(x[-1], 1e-5) * w("model.norm.weight")) @ w("lm_head.weight").T


def _short_conv(u, w):
    """y_t = sum_j w[:, j] u_(t - taps + 1 + j), nothing before token 0."""
    T, taps = u.shape[0], w.shape[1]
    pad = torch.cat([u.new_zeros(taps - 1, u.shape[1]), u])
    return sum(pad[j:j + T] * w[:, j] for j in range(taps))


def _general_delta(h, t, m, eps, states):
    H, D, T = m["heads"], m["dim"], h.shape[0]
    r, k, v = ((h @ t[n].T).view(T, H, D) for n in "rkv")
    w = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(h @ t["w1"].T) @ t["w2"].T + t["w0"])).view(T, H, D)
    a = torch.sigmoid(h @ t["a"].T + t["a.b"]).view(T, H, D)
    u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    au, S, out = a * u, h.new_zeros(H, D, D), torch.empty_like(r)
    for i in range(T):
        S = w[i, :, :, None] * S - au[i, :, :, None] * (u[i, :, None] @ S) + k[i, :, :, None] * v[i, :, None]
        out[i] = (r[i, :, None] @ S)[:, 0]
    states.append(S)
    return (_rms(out, eps).reshape(T, H * D) * t["norm"] * torch.sigmoid(h @ t["g"].T)) @ t["o"].T


def _mamba2(h, t, m, eps, states):
    H, P, N, G, T = m["heads"], m["vdim"], m["state"], m["groups"], h.shape[0]
    inner = H * P
    z, xbc, dt = (h @ t["in"].T).split([inner, inner + 2 * G * N, H], -1)
    x, B, C = _silu(_short_conv(xbc, t["conv"]) + t["conv.b"]).split([inner, G * N, G * N], -1)
    x = x.reshape(T, H, P)
    B, C = (q.reshape(T, G, N).repeat_interleave(H // G, 1) for q in (B, C))
    dt = torch.nn.functional.softplus(dt + t["dt_bias"], threshold=1e9)
    decay, dx, S, y = torch.exp(-torch.exp(t["A_log"]) * dt), dt[..., None] * x, h.new_zeros(H, N, P), torch.empty_like(x)
    for i in range(T):
        S = decay[i, :, None, None] * S + B[i, :, :, None] * dx[i, :, None]
        y[i] = (C[i, :, None] @ S)[:, 0]
    states.append(S)
    y = (y + t["D"][:, None] * x).reshape(T, inner) * _silu(z)
    return (_rms(y.view(T, m["norm_groups"], -1), eps).reshape(T, inner) * t["norm"]) @ t["o"].T


def _mamba1(h, t, m, eps, states):
    n, r, T = m["state"], m["dt_rank"], h.shape[0]
    x, z = (h @ t["in"].T).chunk(2, -1)
    x = _silu(_short_conv(x, t["conv"]) + t["conv.b"])
    low, B, C = (x @ t["x"].T).split([r, n, n], -1)
    dt = torch.nn.functional.softplus(low @ t["dt"].T + t["dt.b"], threshold=1e9)
    A, dx, S, y = -torch.exp(t["A_log"]).T, dt * x, h.new_zeros(n, m["inner"]), torch.empty_like(x)
    for i in range(T):
        S = torch.exp(dt[i] * A) * S + B[i, :, None] * dx[i]
        y[i] = C[i] @ S
    states.append(S)
    return ((y + t["D"] * x) * _silu(z)) @ t["o"].T


def _lightning(h, t, m, eps, states):
    H, D, T = m["heads"], m["dim"], h.shape[0]
    q, k, v = (_silu(h @ t[n].T).view(T, H, -1) for n in "qkv")
    decay = torch.tensor(m["decay"], device=DEV, dtype=torch.float64)[:, None, None]
    S, o = h.new_zeros(H, D, m["vdim"]), torch.empty_like(v)
    for i in range(T):
        S = decay * S + k[i, :, :, None] * v[i, :, None]
        o[i] = (q[i, :, None] @ S)[:, 0]
    states.append(S)
    return (_rms(o.reshape(T, -1), eps) * t["norm"] * torch.sigmoid(h @ t["g"].T)) @ t["o"].T


def _latent_attention(h, t, m, eps, states):
    H, D, V, T = m["heads"], m["dim"], m["vdim"], h.shape[0]
    rank, rd = m["kv_rank"], m.get("rot_dim", 0)
    q = h if not rd else _rms(h @ t["dq"].T, eps) * t["dq.norm"]
    q = (q @ t["uq" if rd else "q"].T).view(T, H, D + rd)
    c, kr = (h @ t["dkv"].T).split([rank, rd], -1)
    c = _rms(c, eps) * t["dkv.norm"]
    k, v = (c @ t["uk"].T).view(T, H, D), (c @ t["uv"].T).view(T, H, V)
    s = torch.einsum("thd,shd->hts", q[..., :D], k)
    if rd:
        ang = _angles(T, rd, m["rot"]["base"])
        s = s + torch.einsum("thd,sd->hts", _rotate(q[..., D:], ang, False), _rotate(kr[:, None], ang, False)[:, 0])
    s = (s * m["scale"]).masked_fill(~_causal(T, m.get("mask", {}).get("size", 1 << 30)), -math.inf)
    if not rd:   # one more key with a score of its own and no value
        s = torch.cat([t["sink"][:, None, None].expand(H, T, 1), s], -1)
    a = torch.softmax(s, -1)[..., 0 if rd else 1:]
    gate = torch.sigmoid(h @ t["g"].T).view(T, H, -1)
    return ((torch.einsum("hts,shd->thd", a, v)) * gate).reshape(T, H * V) @ t["o"].T


def _attention(h, t, m, eps, states):
    H, G, D, V, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], h.shape[0]
    q, k, v = (h @ t[n].T + t[n + ".b"] for n in "qkv")
    pool = m.get("mask", {}).get("pool")
    if pool:     # behind short convolutions; blocks of older tokens by their mean
        q, k, v = (_short_conv(z, t[n + ".conv"]) for z, n in ((q, "q"), (k, "k"), (v, "v")))
    q, k, v = q.view(T, H, D), k.view(T, G, D), v.view(T, G, V)
    at = torch.arange(T, device=DEV)
    if pool:
        d, size = m["rot"]["dims"], m["mask"]["size"]
        ang = _angles(T, d, m["rot"]["base"])
        q, k = (_rms(torch.cat([_rotate(z[..., :d], ang, True), z[..., d:]], -1), eps) for z in (q, k))
        q = q * t["temp"][:, None]
        nb = T // pool
        k, v = (torch.cat([z, z[:nb * pool].view(nb, pool, G, -1).mean(1)]) for z in (k, v))
        ends = torch.arange(nb, device=DEV) * pool + pool - 1
        keep = torch.cat([_causal(T, size), ends[None] <= at[:, None] - size], 1)
    else:
        every, coef = m["q_temp"]["every"], m["q_temp"]["coef"]
        q = q * (1.0 + coef * torch.log(torch.floor((at.double() + 1) / every) + 1))[:, None, None]
        keep = _causal(T)
    k, v = (z.repeat_interleave(H // G, 1) for z in (k, v))
    s = torch.einsum("thd,shd->hts", q, k) * m["scale"]
    if pool:
        o = torch.einsum("hts,shd->thd", torch.softmax(s.masked_fill(~keep, -math.inf), -1), v)
        return (o.reshape(T, H * V) * torch.sigmoid(h @ t["g"].T)) @ t["o"].T + t["o.b"]
    dist = (at[:, None] - at[None]).clamp(min=0).double()
    s = m["softcap"] * torch.tanh(s / m["softcap"]) - t["r1"][:, None, None] * torch.log(1 + t["r2"][:, None, None] * dist)
    s = torch.cat([s.new_zeros(H, T, 1), s.masked_fill(~keep, -math.inf)], -1)   # one more key: score 0, no value
    o = torch.einsum("hts,shd->thd", torch.softmax(s, -1)[..., 1:], v) * torch.sigmoid(h @ t["g"].T)[..., None]
    return o.reshape(T, H * V) @ t["o"].T


_MIXERS = {"general_delta": _general_delta, "mamba2": _mamba2, "mamba1": _mamba1, "lightning": _lightning,
           "latent_attention": _latent_attention, "attention": _attention}


def _unit(h, t, p, limit=None):
    g, u = h @ t[p + "gate"].T, h @ t[p + "up"].T
    if limit is None:
        return (_silu(g) * u) @ t[p + "down"].T
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ t[p + "down"].T


def _feed_forward(h, t, m):
    if m["kind"] == "dense":
        return _unit(h, t, "", m.get("limit"))
    z, idx = (h @ t["router"].T + t["router.b"]).topk(m["router"]["top"], -1)
    weight = torch.softmax(z, -1)
    out = _unit(h, t, "shared.") if m.get("shared") else torch.zeros_like(h)
    for e in range(m["router"]["experts"]):
        rows, slot = (idx == e).nonzero(as_tuple=True)
        out.index_add_(0, rows, _unit(h[rows], t, "e%d." % e) * weight[rows, slot][:, None])
    return out


def _runs(c) -> list:
    """(layer, pass, first of its pass) in the order they run."""
    n = len(c["layers"])
    if "loop" not in c:
        return [(i, None, False) for i in range(n)]
    a, b = c["loop"]["start"], c["loop"]["stop"]
    again = [(i, p, i == a) for p in range(c["loop"]["times"]) for i in range(a, b)]
    return [(i, None, False) for i in range(a)] + again + [(i, None, False) for i in range(b, n)]


def _exact_hybrid(c, t, ids):
    """Logits of the last position and the recurrent states after it."""
    eps, kind, states = c["norm"]["eps"], c["architecture"], []
    x0 = t["embed"][torch.tensor(ids, device=DEV)] * c.get("embedding", {}).get("scale", 1.0)
    x = x0 + t["pos"][:len(ids)] if kind == "Regesun" else x0
    for i, turn, first in _runs(c):
        layer = c["layers"][i]
        sub = lambda p: {k[len(p):]: v for k, v in t.items() if k.startswith(p)}
        p = "l%d." % i
        mix = lambda h: _MIXERS[layer["type"]](h, sub(p + "mix."), layer["mixer"], eps, states)
        ff = lambda h: _feed_forward(h, sub(p + "mlp."), layer["mlp"])
        if kind == "Tarunex":
            if first:
                x = x + t["loop.step"][turn] + (x0 if turn else 0.0)
            u = _rms(x, eps)
            x = x + mix(u * t[p + "norm1"]) + ff(u * t[p + "norm2"])
        elif kind == "Rasepel":
            x = x + _rms(mix(x), eps) * (1 + t[p + "norm1"])
            if layer["mlp"]:
                x = x + _rms(ff(x), eps) * (1 + t[p + "norm2"])
        else:
            x = x + _rms(mix(_rms(x, eps) * t[p + "norm1"]), eps) * t[p + "norm1b"] * t[p + "ls1"]
            if layer["mlp"]:
                x = x + _rms(ff(_rms(x, eps) * t[p + "norm2"]), eps) * t[p + "norm2b"] * t[p + "ls2"]
    z = _rms(x[-1], eps) * (t["final.norm"] + (1.0 if kind == "Rasepel" else 0.0))
    z = (z @ t["embed" if kind == "Rasepel" else "head"].T) * c.get("logit_scale", 1.0)
    cap = c.get("logit_softcap")
    return (cap * torch.tanh(z / cap) if cap else z), states


@torch.no_grad()
def exact(case, seed):
    if case["family"] == "experts":
        t = {k: v.double() for k, v in _experts_tensors(case).items()}
        return _feed_forward(_experts_input(case, seed).double(), t, _experts_config(case))
    prompts = prompts_of(case, seed)
    if case["family"] == "llama":
        t = _llama_tensors(case)
        return torch.stack([_exact_llama(case, t, p) for p in prompts])
    t = {k: v.double() for k, v in _hybrid_tensors(case).items()}
    got = [_exact_hybrid(_hybrid_config(case), t, p) for p in prompts]
    return {"logits": torch.stack([z for z, _s in got]),
            "states": [s for _z, states in got for s in states][:HybridRequests.MOST]}


if __name__ == "__main__":
    for one in listed() + [draw(random.Random(0))]:
        print(one, work(one))
