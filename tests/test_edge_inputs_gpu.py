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


# ------------------------------------------------------------------ weights in 16 bits
@pytest.mark.parametrize("scale", [0.03, 0.1, 0.3, 1.0])    # from even weights to one key that takes all
@pytest.mark.parametrize("win", [1 << 30, 100])
@pytest.mark.parametrize("form", ["window", "latent"])
def test_shared_tiles_are_as_exact_as_a_wavefront_each(scale, win, form):
    """Against 64 bits the two kernels differ by the rounding of the weights to bf16 only: the largest one is exact in both."""
    ent, row_ent, pos, bt, R, g = _step([200, 130], [0, 0], 7)
    H, D = 8, 128
    pool = torch.randn((int(bt.max()) + 1) * PAGE, (2 if form == "window" else 1) * D, generator=g).to(torch.bfloat16)
    q = torch.randn(R, H * D, generator=g).to(torch.bfloat16)
    per, errs = sm.window_rows_per_wave(H), []
    j, i = torch.arange(200)[None], pos.long()[:, None]
    tok = bt.long()[row_ent.long()][:, :4].repeat_interleave(PAGE, 1)[:, :200] * PAGE + torch.arange(200) % PAGE   # [R, 200]
    kv = pool[tok].double()
    s = torch.matmul(q.view(R, H, D).double(), kv[..., :D].transpose(1, 2).contiguous()) * scale
    s = s.masked_fill(~((j <= i) & (j > i - win))[:, None], -INF)
    want = torch.matmul(torch.softmax(s, -1), kv[..., -D:].contiguous())                                            # [R, H, D]
    for rows in (per, 4 * per):
        kw = dict(units=sm.make_units(ent, rows).to(DEV), unit_rows=rows)
        if form == "window":
            a = (q, pool, bt, row_ent, pos, None, scale, win)
            o = sm.window_attn(*_to(a), torch.empty(R, H * D, dtype=q.dtype, device=DEV), PAGE, H, 1, D, D, **kw)
            o = o.view(R, H, D)
        else:
            a = (q.view(R, H, D).transpose(0, 1).contiguous(), pool, bt, row_ent, pos, None, scale, win)
            o = sm.latent_attn(*_to(a), torch.empty(H, R, D, dtype=q.dtype, device=DEV), PAGE, **kw).transpose(0, 1)
        errs.append(_err(o.cpu(), want))
    # both round every result once (1.66e-3); the weights' roundings are drawn anew where tiles begin elsewhere: 1 %
    assert errs[1] < 1.01 * errs[0], errs


# ------------------------------------------------------------------ tokens that are not finite
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bad", [INF, -INF, NAN])
@pytest.mark.parametrize("max_keys", [None, 700])
@pytest.mark.parametrize("form", ["window", "padded", "blocks", "kept", "maps", "latent", "latent512"])
def test_attention_keeps_values_that_are_not_finite_to_later_rows(dt, bad, max_keys, form):
    """Position 70's value is not finite: rows before it, and rows whose window has passed it, are as they were."""
    ent, row_ent, pos, bt, R, g = _step([150, 40], [0, 37], 2)
    H, D = 4, {"latent512": 512, "padded": 72}.get(form, 64)
    M = 2 if form == "maps" else 1
    win = 50 if form != "window" else 1 << 30
    latent = form.startswith("latent")
    width = D if latent else (M + 1) * D
    pool = torch.randn((int(bt.max()) + 1) * PAGE, width, generator=g).to(dt)
    q = torch.randn(R, H * M * D, generator=g).to(dt)
    kw = {"blocks": dict(every=16), "kept": dict(keep=9), "maps": dict(diff=(0.4, 1e-4))}.get(form, {})
    if form == "blocks":
        kw["blk"] = torch.randn((int(bt.max()) + 1) * sm.blocks_per_page(PAGE, 16), width, generator=g).to(dt)
        kw["blk"][int(bt[0, 1]) * 4, D + 3] = bad        # the block of tokens 64 .. 79
    if form == "kept":
        pool[int(bt[0, 0]) * PAGE + 4, D + 3] = bad      # a kept token, seen by all rows from there on
    else:
        pool[int(bt[0, 1]) * PAGE + 6, width - D + 3] = bad
    per = sm.window_rows_per_wave(H)
    units = sm.make_units(ent, _rows(dt, per, True)).to(DEV)
    more = dict(units=units, unit_rows=_rows(dt, per, True), max_keys=max_keys)
    if latent:
        a = (q.view(R, H, D).transpose(0, 1).contiguous(), pool, bt, row_ent, pos, None, 0.05, win)
        want = sm.latent_attn(*a, torch.empty(H, R, D, dtype=dt), PAGE)
        got = sm.latent_attn(*_to(a), torch.empty(H, R, D, dtype=dt, device=DEV), PAGE, **more)
        # a latent is key and value: the rows that see it are lost as a whole
        lost = ~want.isfinite()
    else:
        a = (q, pool, bt, row_ent, pos, None, 0.1, win)
        want = sm.window_attn(*a, torch.empty(R, H * D, dtype=dt), PAGE, H, 1, D, D, **kw)
        got = sm.window_attn(*_to(a), torch.empty(R, H * D, dtype=dt, device=DEV), PAGE, H, 1, D, D, **more,
                             **{k: _to(v) for k, v in kw.items()})
        lost = ~want.isfinite()
    assert lost.any() and not lost.all()
    got = got.cpu()
    assert torch.equal(lost, ~got.isfinite())
    torch.testing.assert_close(got[~lost].float(), want[~lost].float(), **_tol(dt))


@pytest.mark.parametrize("where", ["x", "B", "C", "dt", "z"])
@pytest.mark.parametrize("bad", [INF, NAN])
@pytest.mark.parametrize("P", [64, 40, 200])
def test_mamba_scan_keeps_tokens_that_are_not_finite_to_later_ones(where, bad, P):
    g = torch.Generator().manual_seed(3)
    H, N, G = 2, 32, 1
    inner, C = H * P, H * P + 2 * N
    lens, at = [130, 40], 74
    ent_h = [(0, 130, 0, 0), (130, 40, 9, 1)]
    ent = torch.tensor(ent_h, dtype=torch.int32)
    R = sum(lens)
    conv, zx = torch.randn(R, C, generator=g), torch.randn(R, 2 * inner + 2 * N + H, generator=g)
    dtb, Al, Dp = (torch.randn(H, generator=g) for _ in range(3))
    S0, T0 = torch.randn(2, H, N, P, generator=g), torch.zeros(2, 3, C)
    if where == "dt":
        zx[at, inner + C] = bad                  # head 0's step size
    elif where == "z":
        zx[at, 5] = bad
    else:
        conv[at, {"x": 5, "B": inner + 5, "C": inner + N + 5}[where]] = bad
    res = []
    for dev in ("cpu", DEV):
        S = S0.clone().to(dev)
        y = sm.mamba_scan(conv.to(dev), zx.to(dev), inner, inner + C, dtb.to(dev), Al.to(dev), Dp.to(dev), S,
                          T0.clone().to(dev), ent.to(dev), ent_h, torch.empty(R, inner, device=dev), H, P, N, G)
        res.append((y.cpu(), S.cpu()))
    (y1, s1), (y2, s2) = res
    for a, b in ((y1, y2), (s1, s2)):
        ok = a.isfinite()
        assert not ok.all() or where in ("C", "z") and a is s1
        assert torch.equal(ok, b.isfinite())
        torch.testing.assert_close(b[ok], a[ok], rtol=1e-4, atol=1e-5 * float(a[ok].abs().max()))


@pytest.mark.parametrize("where", ["r", "k", "v", "g", "a", "lo"])
@pytest.mark.parametrize("bad", [INF, NAN])
@pytest.mark.parametrize("D", [64, 40, 7])
def test_gdelta_scan_keeps_tokens_that_are_not_finite_to_later_ones(where, bad, D):
    g = torch.Generator().manual_seed(4)
    H, at = 2, 74
    n = H * D
    ent_h = [(0, 130, 0, 0), (130, 40, 9, 1)]
    ent, R = torch.tensor(ent_h, dtype=torch.int32), 170
    proj, lo = torch.randn(R, 5 * n, generator=g), torch.randn(R, n, generator=g)
    w0, ab, nw = (torch.randn(n, generator=g) for _ in range(3))
    S0 = torch.randn(2, H, D, D, generator=g)
    if where == "lo":
        lo[at, D - 1] = bad                      # in head 0, as below
    else:
        proj[at, "rkvga".index(where) * n + D - 1] = bad
    res = []
    for dev in ("cpu", DEV):
        S, p = S0.clone().to(dev), proj.to(dev)
        o = sm.gdelta_scan(*[p[:, i * n:(i + 1) * n] for i in range(5)], lo.to(dev), w0.to(dev), ab.to(dev), nw.to(dev),
                           S, ent.to(dev), ent_h, torch.empty(R, n, device=dev), H, D, 1e-5)
        res.append((o.cpu(), S.cpu()))
    (o1, s1), (o2, s2) = res
    harmless = bad == INF and where in ("g", "a", "lo")   # behind a sigmoid
    assert o1.isfinite().all() == harmless
    for a, b in ((o1, o2), (s1, s2)):
        ok = a.isfinite()
        assert torch.equal(ok, b.isfinite())
        torch.testing.assert_close(b[ok], a[ok], rtol=1e-4, atol=1e-4)   # as in the tests of ordinary inputs


# ------------------------------------------------------------------ decays
def _err(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("steps", ["even", "drawn", "large first"])
@pytest.mark.parametrize("lens", [[64], [300, 40]])
def test_mamba_scan_decays_in_64_bits(steps, lens):
    """A weight between two tokens is as exact as the decays between them, whatever decayed before (A = 16)."""
    g = torch.Generator().manual_seed(5)
    H, P, N, G = 2, 64, 128, 1
    inner, C = H * P, H * P + 2 * N
    ent_h, r0 = [], 0
    for i, n in enumerate(lens):
        ent_h.append((r0, n, 7, i))
        r0 += n
    ent, R = torch.tensor(ent_h, dtype=torch.int32), r0
    conv, zx = torch.randn(R, C, generator=g), torch.randn(R, 2 * inner + 2 * N + H, generator=g)
    raw = {"even": torch.full((R, H), math.log(math.expm1(0.05))), "drawn": torch.randn(R, H, generator=g) - 2,
           "large first": torch.where((torch.arange(R) % 64 < 32)[:, None], torch.randn(R, H, generator=g) + 4,
                                      torch.full((R, H), -7.0))}[steps]
    zx[:, inner + C:] = raw
    Al, Dp, zero = torch.full((H,), math.log(16.0)), torch.randn(H, generator=g), torch.zeros(H)
    S0 = torch.randn(len(lens), H, N, P, generator=g)
    S, T = S0.clone().to(DEV), torch.zeros(len(lens), 3, C, device=DEV)
    y = sm.mamba_scan(conv.to(DEV), zx.to(DEV), inner, inner + C, zero.to(DEV), Al.to(DEV), Dp.to(DEV), S, T,
                      ent.to(DEV), ent_h, torch.empty(R, inner, device=DEV), H, P, N, G).cpu()
    x, B, Cc = (t.double() for t in conv.split([inner, N, N], -1))
    dt, A = torch.nn.functional.softplus(raw.double(), threshold=1e9), -torch.exp(Al.double())
    z, want, ends = zx[:, :inner].double(), torch.empty(R, inner, dtype=torch.float64), []
    for row0, n, _s, slot in ent_h:
        st = S0[slot].double()
        for t in range(row0, row0 + n):
            xt = x[t].view(H, P)
            st = torch.exp(A * dt[t])[:, None, None] * st + B[t][None, :, None] * (dt[t][:, None] * xt)[:, None]
            want[t] = ((Cc[t] @ st + Dp.double()[:, None] * xt).reshape(inner)) * z[t] * torch.sigmoid(z[t])
        ends.append(st)
    # fp32 products and sums: a few roundings of 6e-8; a step of 4 at A = 16 carries its own rounding times 64
    assert _err(y, want) < 6e-7
    assert _err(S.cpu(), torch.stack(ends)) < 6e-7


@pytest.mark.parametrize("D", [64, 40])
@pytest.mark.parametrize("w0", [-3.0, 0.0, 20.0])
def test_gdelta_scan_decays_in_64_bits(D, w0):
    g = torch.Generator().manual_seed(6)
    H, R = 2, 64
    n = H * D
    proj, lo = torch.randn(R, 5 * n, generator=g), torch.randn(R, n, generator=g) + w0
    ab, nw, zero = torch.zeros(n), torch.ones(n), torch.zeros(n)
    proj[:, 3 * n:4 * n] = 40.0                      # gates of one
    S0 = torch.randn(1, H, D, D, generator=g)
    ent_h = [(0, R, 7, 0)]
    S, p = S0.clone().to(DEV), proj.to(DEV)
    o = sm.gdelta_scan(*[p[:, i * n:(i + 1) * n] for i in range(5)], lo.to(DEV), zero.to(DEV), ab.to(DEV), nw.to(DEV), S,
                       torch.tensor(ent_h, dtype=torch.int32, device=DEV), ent_h, torch.empty(R, n, device=DEV), H, D,
                       0.0).cpu()
    r, k, v, _g, a = (proj[:, i * n:(i + 1) * n].double().view(R, H, D) for i in range(5))
    w = torch.exp(-math.exp(-0.5) * torch.sigmoid(lo.double())).view(R, H, D)
    st, want = S0[0].double(), torch.empty(R, H, D, dtype=torch.float64)
    for t in range(R):
        u = k[t] / torch.sqrt((k[t] * k[t]).sum(-1, keepdim=True) + 1e-6)
        us = (u[:, None] @ st)
        st = w[t][:, :, None] * st - (torch.sigmoid(a[t]) * u)[:, :, None] * us + k[t][:, :, None] * v[t][:, None]
        q = (r[t][:, None] @ st)[:, 0]
        want[t] = q / torch.sqrt((q * q).mean(-1, keepdim=True))
    # what 64 tokens of fp32 products and sums leave: outputs 1.4 to 1.6e-7 (a walk over the tokens the same), states
    # 0.7 to 1.7e-7 (0.4 to 1.4e-7)
    assert _err(o, want.reshape(R, n)) < 2e-7
    assert _err(S[0].cpu(), st) < 2.2e-7
