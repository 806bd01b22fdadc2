"""Token sampling: greedy (fused into the LM head kernel, see ops.lm_head_argmax)
and Ollama-style temperature / top-k / top-p sampling for requests that ask for
it (``options`` of ``/api/generate``; Ollama's defaults are temperature 0.8,
top_k 40, top_p 0.9).

The stochastic path is ``ops.sample`` (csrc/kernels/sampling.hip), captured in
the decode graph right after the LM head: top-k first (k <= 128, radix select,
so the full-vocab softmax is never materialised), then top-p over the k
survivors, then an exponential-race draw (argmax of p / Exp(1)), equivalent to
multinomial sampling.  The random stream is keyed by (request seed, position,
token id), so replays draw fresh numbers with no host state and a given seed
reproduces a reply.  Rows with temperature <= 0 are greedy.
"""
from __future__ import annotations

import dataclasses
import random

import torch


@dataclasses.dataclass
class SamplingParams:
    temperature: float = 0.0   # 0 = greedy (engine default: deterministic)
    top_k: int = 40
    top_p: float = 0.9
    seed: int | None = None
    max_tokens: int = 128
    stop_on_eos: bool = True

    @property
    def greedy(self) -> bool:
        return self.temperature <= 0.0

    def resolved_seed(self) -> int:
        """The request's random-stream key: ``seed`` if given, else drawn once per request."""
        if self.seed is None:
            self.seed = random.getrandbits(62)
        return int(self.seed) & ((1 << 63) - 1)

    @classmethod
    def from_ollama(cls, options: dict | None, default_max: int = 128) -> "SamplingParams":
        o = options or {}
        n = int(o.get("num_predict", default_max))
        if n < 0:
            n = default_max
        # ignore_eos (llama.cpp server option; benchmarks): decode exactly num_predict tokens
        return cls(temperature=float(o.get("temperature", 0.0)), top_k=int(o.get("top_k", 40)),
                   top_p=float(o.get("top_p", 0.9)), seed=o.get("seed"), max_tokens=max(1, n),
                   stop_on_eos=not bool(o.get("ignore_eos", False)))


class HostImage:
    """Page-locked host image of a device buffer that is filled anew for every step.  From pageable memory a copy
    is a staging round trip of some 35 us that the host waits for; from here it is queued like a launch.  The
    image is written again only once its last copy has been read (``fill`` waits for that)."""

    def __init__(self, dev: torch.Tensor):
        self.dev = dev
        cuda = dev.device.type == "cuda"
        self.host = torch.zeros(dev.shape, dtype=dev.dtype, pin_memory=cuda)
        self.sent = torch.cuda.Event() if cuda else None
        self.busy = False

    def fill(self):
        """The image as a numpy array, free to be written."""
        if self.busy:
            self.sent.synchronize()
            self.busy = False
        return self.host.numpy()

    def send(self, lo: int = 0, hi: int | None = None):
        """Queue the copy of words lo .. hi - 1 (None: all)."""
        self.dev[lo:hi].copy_(self.host[lo:hi], non_blocking=True)
        if self.sent is not None:
            self.sent.record(torch.cuda.current_stream(self.dev.device))
            self.busy = True


_PADDING = (0.0, 40, 0.9, 0)   # a row no sequence has: greedy, and the same in every step


class SamplerSlots:
    """Per-row sampling parameters of a decode batch as device tensors, read by the
    graph-captured ``ops.sample`` launch (so a sampled decode step replays like a
    greedy one): views of one buffer, which ``load`` fills with one copy (each time: the native loop writes them too).
    With ``image`` they are its words from ``at`` (even) on, and ``fill`` leaves the copy to the owner, who sends
    them with its own words."""

    def __init__(self, B: int, device, image: HostImage | None = None, at: int = 0):
        self.B, self.at = B, at
        self.image = HostImage(torch.zeros(self.words(B), device=device, dtype=torch.int32)) if image is None else image
        o = (3 * B + 1) // 2 * 2   # the seeds' 64-bit words after three 32-bit ones per row
        self.buf = self.image.dev[at:at + self.words(B)]
        (self.temp, self.topk, self.topp, self.seeds), self.parts = (
            (v[:B].view(torch.float32), v[B:2 * B], v[2 * B:3 * B].view(torch.float32), v[o:].view(torch.int64))
            for v in (self.buf, self.image.host[at:at + self.words(B)]))
        self.load([])

    @staticmethod
    def words(B: int) -> int:
        return (3 * B + 1) // 2 * 2 + 2 * B

    def fill(self, params: list):
        """The rows' parameters into the image, which ``image.fill`` has freed."""
        params = params[:self.B]
        rows = [(p.temperature, p.top_k, p.top_p, p.resolved_seed()) for p in params]
        rows += [_PADDING] * (self.B - len(rows))
        for view, col in zip(self.parts, zip(*rows)):
            view.numpy()[:] = col

    def load(self, params: list):
        self.image.fill()
        self.fill(params)
        self.image.send(self.at, self.at + self.words(self.B))


def sample(logits: torch.Tensor, params: list, pos) -> torch.Tensor:
    """logits [B, V] fp32 -> int32 token ids [B] (one SamplingParams per row; pos =
    the position each row's token is drawn for).  Runs ops.sample (the GPU kernel,
    or its PyTorch reference on CPU tensors)."""
    from .. import ops

    B = logits.shape[0]
    params = list(params[:B]) + [SamplingParams()] * (B - len(params))
    dev = logits.device
    temp = torch.tensor([p.temperature for p in params], dtype=torch.float32).to(dev)
    topk = torch.tensor([p.top_k for p in params], dtype=torch.int32).to(dev)
    topp = torch.tensor([p.top_p for p in params], dtype=torch.float32).to(dev)
    seeds = torch.tensor([p.resolved_seed() for p in params], dtype=torch.int64).to(dev)
    pos = torch.as_tensor(pos, dtype=torch.int32).to(dev)
    return ops.sample(logits, temp, topk, topp, seeds, pos)


def sample_tp(model, logits: torch.Tensor, params: list, pos) -> torch.Tensor:
    """Vocab-parallel ``sample`` (TP prefill): per-shard top-128 candidates, one all-gather,
    then the same draw on every rank (see DecodeState.body_sampled)."""
    from .. import ops

    B = logits.shape[0]
    params = list(params[:B]) + [SamplingParams()] * (B - len(params))
    dev = logits.device
    W = model.tp
    temp = torch.tensor([p.temperature for p in params], dtype=torch.float32).to(dev)
    topk = torch.tensor([p.top_k for p in params], dtype=torch.int32).to(dev)
    topp = torch.tensor([p.top_p for p in params], dtype=torch.float32).to(dev)
    seeds = torch.tensor([p.resolved_seed() for p in params], dtype=torch.int64).to(dev)
    posd = torch.tensor(list(pos), dtype=torch.int32).to(dev)
    cv = torch.empty(B, 128, device=dev, dtype=torch.float32)
    ci = torch.empty(B, 128, device=dev, dtype=torch.int32)
    ops.topk_candidates(logits, model.w.tp_rank * (model.cfg.vocab // W), cv, ci)
    av = torch.empty(W * B, 128, device=dev, dtype=torch.float32)
    ai = torch.empty(W * B, 128, device=dev, dtype=torch.int32)
    model.comm.all_gather_rows_into(av, cv)
    model.comm.all_gather_rows_into(ai, ci)
    out = torch.empty(B, dtype=torch.int32, device=dev)
    return ops.sample_candidates(av, ai, W, temp, topk, topp, seeds, posd, out)
