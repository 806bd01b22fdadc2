"""Feed-forwards that a model author derives from the registered ones, in every design that can leave a unit's product to them."""
import pytest
import torch

from p2p_llm_chat_go_amd.models import hybrid as hy
from p2p_llm_chat_go_amd.models.config import get_config
from p2p_llm_chat_go_amd.models.registry import make_engine


def _logits(name):
    """Logits of a tiny model on the CPU, a prompt of 20 and one of three tokens."""
    cfg = get_config(name)
    eng = make_engine(cfg, hy.HybridWeights.random(cfg, "cpu", seed=3, dtype=torch.float32), "cpu", kv_pages=16, num_slots=4,
                      max_batch=4, dtype=torch.float32)
    return eng.step([("a", list(range(5, 25)), [19]), ("b", [7, 8, 9], [0, 2])])


@pytest.mark.parametrize("name", ["tiny-regesun", "tiny-tarunex", "tiny-rasepel", "tiny-nosuzen"])
@pytest.mark.parametrize("method", ["fill", "fill_routed", "forward_proj"])
def test_overridden_methods_are_given_the_product(name, method, monkeypatch):
    want = _logits(name)
    used = {hy.DESIGNS[get_config(name).design].ff_key(L.mlp.get("kind", "dense")) for L in get_config(name).layers if L.mlp}
    calls = []
    for key in used:
        base = hy.FEEDFORWARDS[key]
        if not hasattr(base, method):
            continue

        def over(self, proj, *args, _f=getattr(base, method)):
            calls.append(method)
            if getattr(self, "w_in", None) is not None:
                assert proj is not None and proj.shape[1] == self.w_in.shape[0]   # [gate | up]
            return _f(self, proj, *args)

        monkeypatch.setitem(hy.FEEDFORWARDS, key, type("Own" + base.__name__, (base,), {method: over}))
    got = _logits(name)
    # the same sums: the product and the unit apart
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5 * want.abs().max().item())
