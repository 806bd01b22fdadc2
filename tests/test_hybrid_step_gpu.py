"""A captured decode step's metadata, written in place, against ``StepBatch.build_host``."""
import random

import pytest
import torch

from p2p_llm_chat_go_amd.engine.hybrid import HybridDecodeGraph
from p2p_llm_chat_go_amd.models.config import get_config
from p2p_llm_chat_go_amd.models.hybrid import StepBatch
from p2p_llm_chat_go_amd.models.registry import make_engine
from p2p_llm_chat_go_amd.ops import PAGE
from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,maxp", [(1, 1), (4, 2), (8, 5)])
def test_metadata_in_place(rows, maxp):
    eng = make_engine(get_config("tiny-regesun"), None, "cuda:0", kv_pages=64, max_batch=8)
    g = HybridDecodeGraph(eng.model, rows, maxp)
    rng = random.Random(rows)
    for turn in range(12):      # fewer and more rows, longer and shorter tables, the same ones again
        n = rng.randint(0, rows) if turn else rows
        live = []
        for i in range(n):
            p = rng.randrange(min(maxp * PAGE, eng.cfg.max_pos))
            pages = [rng.randrange(1, 60) for _ in range(rng.randint(p // PAGE + 1, maxp))]
            live.append((i, pages, p, rng.randrange(100)))
        g._fill(live)
        padded = [(s, pg + [0] * (maxp - len(pg)), p, [t]) for s, pg, p, t in live] + [g.pad] * (rows - n)
        want, _ = StepBatch.build_host(padded, [[0]] * rows, maxp)
        assert torch.equal(g.host, want)
        sm.copy_words(g.host, g.batch.flat)
        torch.cuda.synchronize()
        assert torch.equal(g.batch.flat.cpu(), want)
    for bad in ([(0, [1] * (maxp + 1), 0, 1)], [(0, [1], maxp * PAGE, 1)], [(0, [1], 0, 1)] * (rows + 1),
                [(0, [1] * maxp, eng.cfg.max_pos, 1)]):
        with pytest.raises(ValueError):
            g._fill(bad)
    out = torch.zeros(300, dtype=torch.int32).pin_memory()
    sm.copy_words(torch.arange(300, dtype=torch.int32, device="cuda:0"), out)
    torch.cuda.synchronize()
    assert out.tolist() == list(range(300))
