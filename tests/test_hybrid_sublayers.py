"""Feed-forwards and mixers of every kind in the designs whose residual passes may leave a sublayer's input to the
product that reads it (``sm.NormedRows``: steps of up to four rows): routed experts, which read their input more than
once, against the oracles, prompts and steps of few rows."""
import pytest
import torch

import rasepel_oracle
import regesun_oracle
import rotutar_oracle
import test_rasepel_model as Ra
import test_regesun_model as Re
from p2p_llm_chat_go_amd.models import hybrid as Hy

DEVICES = ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)]
MOE = {"kind": "moe", "limit": 1.2, "expert": {"ff": 48, "limit": 1.2},
       "router": {"experts": 6, "top": 2, "groups": {"count": 3, "keep": 2}}}
CUTS = [9, 1, 1, 4, 3, 2, 1, 5, 1]   # rows of the steps: a prompt, then few and more


def _few_rows_everywhere(monkeypatch):
    """Steps of few rows leave their rows unformed on the CPU too (where no kernel forms them in the product)."""
    whole = Hy.HybridModel._residual

    def residual(self, b):
        x, spare = whole(self, b)
        return x, torch.empty_like(x) if spare is None and b.R <= Hy.sm.NORMED_ROWS else spare
    monkeypatch.setattr(Hy.HybridModel, "_residual", residual)


def _build(design, monkeypatch, layers=None):
    if design == "Regesun":
        monkeypatch.setattr(regesun_oracle, "dense_ff", lambda h, t, p, ml: (
            rotutar_oracle.moe_ff if ml["kind"] == "moe" else dense_ff)(h, t, p, ml))
        return (Re, regesun_oracle) + Re.make(layers or [dict(Re.GD, mlp=MOE), dict(Re.MB, mlp=MOE), Re.LA, Re.GD,
                                                         dict(Re.MB, mlp=MOE)], seed=2)
    monkeypatch.setattr(rasepel_oracle, "clamped_unit", lambda h, t, p, limit: (
        rotutar_oracle.moe_ff(h, t, p, MOE) if p + "router" in t else clamped_unit(h, t, p, limit)))
    return (Ra, rasepel_oracle) + Ra.make(layers or [Ra.layer(Ra.LG, MOE), Ra.layer(Ra.MB, MOE), Ra.layer(Ra.AT, Ra.FF),
                                                     Ra.LG, Ra.layer(Ra.AT, MOE)], seed=2)


dense_ff, clamped_unit = regesun_oracle.dense_ff, rasepel_oracle.clamped_unit


def _run(mod, eng, t, cuts):
    at, outs = 0, []
    for n in cuts:
        outs.append(eng.step([("a", t[at:at + n], list(range(n)))]))
        at += n
    eng.release("a")
    return torch.cat(outs)


@pytest.mark.parametrize("dev", DEVICES)
@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("design", ["Regesun", "Rasepel"])
def test_routed_feed_forwards(dev, few, design, monkeypatch):
    if few:
        _few_rows_everywhere(monkeypatch)
    mod, O, c, cfg, sd = _build(design, monkeypatch)
    assert cfg.is_moe
    t = mod.toks(sum(CUTS), cfg.vocab, 3)
    ref = O.forward(c, sd, t)
    eng = mod.engine(cfg, sd, dev)
    mod.close(mod.run_whole(eng, "w", t), ref)
    mod.close(_run(mod, eng, t, CUTS), ref)


@pytest.mark.parametrize("dev", DEVICES)
@pytest.mark.parametrize("design", ["Regesun", "Rasepel"])
def test_a_feed_forward_of_an_author(dev, design, monkeypatch):
    """A registered class of its own, with no base and nothing but what the contract names."""
    class Doubled:
        w_in = w_out = None
        n_mid = 0

        def __init__(self, spec, width):
            self.width = width

        def tensor_shapes(self):
            return {"m": (self.width, self.width)}

        def load(self, get, dtype, dev):
            self.m = get("m").to(dev, dtype).contiguous()

        def forward(self, h):
            return torch.nn.functional.linear(h, self.m) + h

    monkeypatch.setitem(Hy.FEEDFORWARDS, "doubled", Doubled)
    _few_rows_everywhere(monkeypatch)
    ml = {"kind": "doubled", "limit": 1.0}
    base = [dict(Re.GD, mlp=ml), dict(Re.MB, mlp=ml)] if design == "Regesun" else [Ra.layer(Ra.LG, ml), Ra.layer(Ra.MB, ml)]
    mod, O, c, cfg, sd = _build(design, monkeypatch, base)
    monkeypatch.setattr(O, "dense_ff" if design == "Regesun" else "clamped_unit",
                        lambda h, t, p, _: h @ t[p + "m"].T + h)
    t = mod.toks(sum(CUTS), cfg.vocab, 4)
    mod.close(_run(mod, mod.engine(cfg, sd, dev), t, CUTS), O.forward(c, sd, t))


@pytest.mark.parametrize("dev", DEVICES)
@pytest.mark.parametrize("design", ["Regesun", "Rasepel"])
def test_parts_below_a_registered_one(dev, design, monkeypatch):
    """A class below a registered one whose forward() is its own reads a tensor, in steps of any number of rows; one that
    keeps the forward() it inherits, or says so itself, takes rows that are not formed."""
    seen = []

    def reading(base, **more):
        def forward(self, h, *a):
            seen.append((h.shape[0], type(h)))
            return base.forward(self, h * 1.0, *a)
        return type("Reading" + base.__name__, (base,), dict(more, forward=forward))

    first, second = (Hy.GeneralDelta, Hy.Mamba2) if design == "Regesun" else (Hy.Lightning, Hy.Mamba1)
    for base in (first, second):
        monkeypatch.setitem(Hy.MIXERS, base.kind, reading(base))
    monkeypatch.setitem(Hy.FEEDFORWARDS, "dense", reading(Hy.DenseFF))
    _few_rows_everywhere(monkeypatch)
    layers = [dict(Re.GD, mlp=Re.LA["mlp"]), Re.MB, Re.GD] if design == "Regesun" else [Ra.layer(Ra.LG, Ra.FF), Ra.MB, Ra.LG]
    mod, O, c, cfg, sd = _build(design, monkeypatch, layers)
    t = mod.toks(sum(CUTS), cfg.vocab, 5)
    mod.close(_run(mod, mod.engine(cfg, sd, dev), t, CUTS), O.forward(c, sd, t))
    assert {n for n, _ in seen} == set(CUTS) and {k for _, k in seen} == {torch.Tensor}

    part = lambda cls: Hy.takes_unformed(object.__new__(cls))
    for base in (first, second, Hy.DenseFF, Hy.LatentAttention, Hy.ConvAttention):
        assert part(base) and part(type("Kept", (base,), {})) and part(reading(base, one_input=True))
        assert not part(reading(base)) and not part(type("Below", (reading(base),), {}))
    assert part(Hy.GeluFF) and not part(Hy.WindowAttention) and not part(Hy.MoEFF) and not part(Hy.Parallel)
