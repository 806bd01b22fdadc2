"""Tables that a step's layers derive from its entries, formed on the device, against those formed on the host."""
import random

import pytest
import torch

from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("E", [1, 3, 255, 257, 600])
@pytest.mark.parametrize("size,least", [(64, 128), (64, 1), (16, 33), (1, 2), (7, 5)])
def test_tables(E, size, least):
    rng = random.Random(E * size)
    row, ents = 0, []
    for i in range(E):
        n = rng.choice((1, size, size + 1, rng.randint(1, 300 if E < 300 else 40)))
        ents.append((row, n, rng.randint(0, 5000), rng.randint(0, 99)))
        row += n
    ent = torch.tensor(ents, dtype=torch.int32, device=DEV)
    assert torch.equal(sm.device_units(ents, size, ent).cpu(), sm.make_units(ents, size))
    for got, want in zip(sm.chunk_tables(ents, size, DEV, ent), sm.scan_chunks(ents, size)):
        assert torch.equal(got.cpu(), want)
    for got, want in zip(sm.portion_tables(ents, size, least, DEV, ent), sm.portion_tables(ents, size, least, DEV)):
        assert (got is None and want is None) or torch.equal(got, want)


def test_entries_elsewhere_are_copied():
    ents = [(0, 70, 0, 1), (70, 1, 5, 2)]
    host = torch.tensor(ents, dtype=torch.int32)
    wide = torch.zeros(2, 8, dtype=torch.int32, device=DEV)[:, :4]
    for ent in (None, host, wide):
        assert torch.equal(sm.chunk_tables(ents, 64, DEV, ent)[0].cpu(), sm.scan_chunks(ents, 64)[0])
    assert torch.equal(sm.device_units(ents, 16, host), sm.make_units(ents, 16))
    long = sm.portion_tables(ents, 64, 100, DEV, host.to(DEV))   # no entry of so many rows
    assert long[0].shape[0] == 0 and long[2].shape[0] == 2
