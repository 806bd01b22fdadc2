"""Values at the ends of what the kernels take: sinks that weigh nothing or everything, tokens that are not
finite (they must not reach the tokens before them), step sizes and decays of mixed size."""
import math

import pytest
import torch

from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAGE = 64
INF, NAN = float("inf"), float("nan")


def _step(lens, starts, seed):
    ent, r0 = [], 0
    for i, (n, s) in enumerate(zip(lens, starts)):
        ent.append((r0, n, s, i))
        r0 += n
    row_ent = torch.tensor([i for i, e in enumerate(ent) for _ in range(e[1])], dtype=torch.int32)
    pos = torch.tensor([e[2] + k for e in ent for k in range(e[1])], dtype=torch.int32)
    g = torch.Generator().manual_seed(seed)
    bt = (torch.randperm(len(ent) * 4, generator=g) + 1).to(torch.int32).view(len(ent), 4)
    return ent, row_ent, pos, bt, r0, g


def _rows(dt, per_wave, tiled):
    return 4 * per_wave if tiled and dt == torch.bfloat16 else per_wave


def _tol(dt):
    # as in the tests of the same kernels on ordinary inputs: two roundings to bf16 of values up to about 4.5; fp32
    # sums of up to 512 products behind an exponential
    return dict(rtol=1e-2, atol=1.8e-2) if dt == torch.bfloat16 else dict(rtol=2e-5, atol=2e-5)


def _to(x):
    return tuple(_to(t) for t in x) if isinstance(x, tuple) else x.to(DEV) if isinstance(x, torch.Tensor) else x


# ------------------------------------------------------------------ sinks
SINKS = torch.tensor([-INF, -3.4e38, -1e30, -1e9, -1e6, -300.0, 0.5, 300.0, 3e38])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tiled", [True, False])
@pytest.mark.parametrize("max_keys", [None, 700])    # whole windows / cut into runs
@pytest.mark.parametrize("win", [1 << 30, 19])
def test_sinks_of_any_size(dt, tiled, max_keys, win):
    """A sink far below the scores changes nothing, one far above leaves nothing."""
    ent, row_ent, pos, bt, R, g = _step([129, 70], [0, 64], 1)
    H, D = len(SINKS), 64
    pool = torch.randn((int(bt.max()) + 1) * PAGE, 2 * D, generator=g).to(dt)
    q = torch.randn(R, H * D, generator=g).to(dt)
    per = sm.window_rows_per_wave(H)
    units = sm.make_units(ent, _rows(dt, per, tiled)).to(DEV)
    a = (q, pool, bt, row_ent, pos, SINKS, 0.15, win)
    want = sm.window_attn(*a, torch.empty(R, H * D, dtype=dt), PAGE, H, 1, D, D)
    got = sm.window_attn(*_to(a), torch.empty(R, H * D, dtype=dt, device=DEV), PAGE, H, 1, D, D, units=units,
                         unit_rows=_rows(dt, per, tiled), max_keys=max_keys)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))
    qa = q.view(R, H, D).transpose(0, 1).contiguous()
    cache = pool[:, :D].contiguous()
    a = (qa, cache, bt, row_ent, pos, SINKS, 0.15, win)
    want = sm.latent_attn(*a, torch.empty(H, R, D, dtype=dt), PAGE)
    got = sm.latent_attn(*_to(a), torch.empty(H, R, D, dtype=dt, device=DEV), PAGE, units=units,
                         unit_rows=_rows(dt, per, tiled), max_keys=max_keys)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(dt))
