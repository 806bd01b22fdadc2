"""Attention of prompts over keys and values formed from latents (``ops.seqmix.formed_attn``) against the PyTorch rendering of the
same op, and the latent layers that take it against their form in latent space."""
import pytest
import torch

from p2p_llm_chat_go_amd.models import hybrid as hy
from p2p_llm_chat_go_amd.ops import seqmix as sm
from tests.test_attn_tile_gpu import DEV, PAGE, _close, _step

STEPS = ["portions", "prompts", "short"]


def _formed(ent, win):
    """Places of each entry's keys among the formed ones, and their number."""
    base, n = [], 0
    for _r0, rows, start, _s in ent:
        lo = max(0, start - win + 1)
        base.append(n - lo)
        n += start + rows - lo
    return torch.tensor(base, dtype=torch.int32), n


@pytest.mark.gpu
@pytest.mark.parametrize("step", STEPS)
@pytest.mark.parametrize("H,D,Rd,V", [(16, 128, 64, 128), (3, 24, 8, 40), (2, 72, 0, 128), (5, 128, 0, 64), (1, 64, 40, 8)])
@pytest.mark.parametrize("win,sunk,gated", [(1 << 30, False, "heads"), (37, True, "channels"), (64, False, None), (1, True, None)])
def test_formed_attention(step, H, D, Rd, V, win, sunk, gated):
    ent, row_ent, pos, bt, R, g = _step(step, 11)
    dt, rank = torch.bfloat16, 48
    q = torch.randn(R, H * (D + 8), generator=g).to(dt)
    qrot = torch.randn(R, H * Rd, generator=g).to(dt) if Rd else None
    pool = torch.randn((int(bt.max()) + 1) * PAGE, rank + Rd, generator=g).to(dt)
    kbase, n = _formed(ent, win)
    kv = torch.randn(n, H * (D + V), generator=g).to(dt)
    sink = torch.randn(H, generator=g) if sunk else None
    gate = torch.randn(R, H * V + 3, generator=g).to(dt)[:, 1:] if gated else None    # rows that are not aligned
    kw = dict(out_scale=0.7, gate_channels=gated == "channels")
    args = (sink, 1.3 / (D + Rd) ** 0.5, win)
    want = sm.formed_attn(q, D + 8, qrot, kv, kbase, pool, rank, bt, row_ent, pos, *args, torch.empty(R, H * V).to(dt), PAGE, H, D,
                          V, None, gate=gate, **kw)
    to = lambda t: None if t is None else t.to(DEV)
    units = sm.make_units(ent, sm.FORMED_PAIRS).to(DEV)
    out = torch.full((R, H * V + 2), 7.0, dtype=dt, device=DEV)
    sm.formed_attn(to(q), D + 8, to(qrot), to(kv), to(kbase), to(pool), rank, to(bt), to(row_ent), to(pos), to(sink), *args[1:],
                   out[:, :H * V], PAGE, H, D, V, units, gate=to(gate), **kw)
    _close(out[:, :H * V], want)
    assert bool((out[:, H * V:] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["key", "value", "rotated", "query"])
def test_a_token_that_is_not_finite_reaches_only_the_rows_that_see_it(what):
    ent, row_ent, pos, bt, R, g = _step("portions", 5)
    H, D, Rd, V, rank, win, dt = 3, 64, 16, 64, 48, 40, torch.bfloat16
    q, qrot = torch.randn(R, H * D, generator=g).to(dt), torch.randn(R, H * Rd, generator=g).to(dt)
    pool = torch.randn((int(bt.max()) + 1) * PAGE, rank + Rd, generator=g).to(dt)
    kbase, n = _formed(ent, win)
    kv = torch.randn(n, H * (D + V), generator=g).to(dt)
    bad = int(kbase[0]) + 20                                    # token 20 of the first entry
    if what == "key":
        kv[bad, D + 3] = float("nan")
    elif what == "value":
        kv[bad, H * D + 3] = float("inf")
    elif what == "rotated":
        pool[int(bt[0, 0]) * PAGE + 20, rank + 1] = float("nan")
    else:
        q[9, 3] = float("nan")
    args = (None, 0.1, win)
    want = sm.formed_attn(q, D, qrot, kv, kbase, pool, rank, bt, row_ent, pos, *args, torch.empty(R, H * V).to(dt), PAGE, H, D, V, None)
    to = lambda t: t.to(DEV)
    out = sm.formed_attn(to(q), D, to(qrot), to(kv), to(kbase), to(pool), rank, to(bt), to(row_ent), to(pos), *args,
                         torch.empty(R, H * V, dtype=dt, device=DEV), PAGE, H, D, V,
                         sm.make_units(ent, sm.FORMED_PAIRS).to(DEV)).cpu()
    lost = ~want.isfinite()
    assert lost.any() and not lost.all() and torch.equal(lost, ~out.isfinite())
    _close(out[~lost], want[~lost])


MIXERS = {"latent_attention": {"heads": 4, "dim": 64, "vdim": 64, "kv_rank": 128, "mask": {"size": 100}, "scale": 0.125},
          "rope_latent_attention": {"heads": 4, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 96, "q_rank": 64,
                                    "rot": {"base": 10000.0, "dims": 24}, "scale": 96 ** -0.5},
          "direct_latent_attention": {"heads": 3, "dim": 40, "rot_dim": 16, "vdim": 128, "kv_rank": 64,
                                      "rot": {"base": 10000.0, "dims": 16}, "scale": 56 ** -0.5}}


@pytest.mark.parametrize("dev", ["cpu", pytest.param(DEV, marks=pytest.mark.gpu)])
@pytest.mark.parametrize("kind", sorted(MIXERS))
@pytest.mark.parametrize("steps", [[(0, 130), (0, 70)], [(90, 150), (0, 33)]], ids=["whole", "portions"])
def test_layers_form_keys_as_they_attend_in_latent_space(kind, steps, dev, monkeypatch):
    W, dt = 128, torch.float32 if dev == "cpu" else torch.bfloat16
    mix = hy.MIXERS[kind](dict(MIXERS[kind]), W, 1e-5)
    g = torch.Generator().manual_seed(3)
    t = {k: torch.randn(s, generator=g) / (s[-1] ** 0.5 if len(s) == 2 else 1.0) for k, s in mix.tensor_shapes().items()}
    mix.load(lambda k: t[k], dt, dev)
    pages = [[3, 7, 1, 5], [2, 8, 6]]
    pool = torch.randn(10 * PAGE, mix.cache_spec()[1], generator=g).to(dev, dt)
    b = hy.StepBatch([(i, pages[i], s, [0] * n) for i, (s, n) in enumerate(steps)], [[0], [0]], dev)
    h = torch.randn(b.R, W, generator=g).to(dev, dt)
    cache = type("Cache", (), {"paged": {0: pool}})()
    got = []
    for formed in (False, True):
        monkeypatch.setattr(sm, "latent_forms", lambda *a, **k: formed)
        if dev == "cpu":
            monkeypatch.setattr(sm, "formed_ok", lambda *a, **k: True)
        got.append(mix.forward(h, b, cache, 0).float())
    # the same sums in another order: fp32 as such, bf16 with keys, values and products rounded at 2^-9 each
    off = ((got[1] - got[0]).norm() / got[0].norm()).item()
    assert off < (1e-5 if dev == "cpu" else 1.5e-2), off
