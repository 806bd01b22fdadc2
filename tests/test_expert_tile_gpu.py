"""Routing of many rows and the tiled expert products against the PyTorch rendering of the same ops:
experts without slots and with one, counts off the tiles' grid, row lengths that end inside a step,
columns that end inside a tile, every tile size, the activations."""
import pytest
import torch

from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("R,W,E,top,groups,keep,kw", [
    (256, 72, 8, 2, 1, 1, dict(score="top_softmax", bias=True)),
    (301, 200, 12, 3, 4, 2, dict()),
    (1000, 64, 70, 5, 7, 3, dict(score="softmax", group_score="max", renorm=True, scale=1.5)),
    (259, 40, 3, 1, 1, 1, dict(score="softmax", corr=True)),
    # 17 to 32 experts, rows longer than the wavefronts' chunks at once; one row fewer than sixteen take
    (230, 2104, 20, 4, 5, 3, dict(bias=True)), (199, 72, 8, 2, 1, 1, dict(score="top_softmax")),
    (200, 72, 33, 2, 1, 1, dict()),
    # many experts: a row per workgroup up to R * 28 = E * W, sixteen from there on
    (300, 100, 128, 8, 8, 3, dict(renorm=True)), (365, 80, 128, 8, 8, 3, dict()), (366, 80, 128, 8, 8, 3, dict()),
    (1300, 72, 256, 8, 1, 1, dict(score="softmax")),
    # 17 to 32 experts and long rows from 400 (bf16) and 503 rows (fp32) on
    (520, 2104, 20, 4, 5, 3, dict(bias=True)), (502, 2104, 20, 4, 5, 3, dict(bias=True))])
def test_routing_of_many_rows(dt, R, W, E, top, groups, keep, kw):
    g = torch.Generator().manual_seed(2)
    h, wr = torch.randn(R, W, generator=g).to(dt), torch.randn(E, W, generator=g) / W ** 0.5
    extra = {k: torch.randn(E, generator=g) * 0.3 for k in ("bias", "corr") if kw.get(k)}
    kw = dict(kw, **extra)
    res = []
    for dev in ("cpu", DEV):
        ids, wts = torch.empty(R, top, dtype=torch.int32, device=dev), torch.empty(R, top, device=dev)
        cnt, rows = torch.empty(E, dtype=torch.int32, device=dev), torch.full((E, R * top), -1, dtype=torch.int32, device=dev)
        k2 = {k: v.to(dev) if isinstance(v, torch.Tensor) else v for k, v in kw.items()}
        sm.group_route(h.to(dev), wr.to(dev), top, groups, keep, ids, wts, cnt, rows, **k2)
        res.append([t.cpu() for t in (ids, wts, cnt, rows)])
    (i1, w1, _c1, _r1), (i2, w2, c2, r2) = res
    # two scores that differ by less than fp32 sums may come in either order
    assert (i1 != i2).float().mean() < 0.005
    same = (i1 == i2).all(1)
    torch.testing.assert_close(w2[same], w1[same], rtol=1e-5, atol=1e-6)
    # every slot is in its expert's list, once
    for e in range(E):
        assert sorted(r2[e, :int(c2[e])].tolist()) == (i2.reshape(-1) == e).nonzero()[:, 0].tolist()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("W,E,top,at", [(2048, 8, 2, (200, 260)), (1024, 20, 3, (292, 368)), (72, 5, 1, (200, 200))])
def test_routing_below_and_above_the_row_threshold(dt, W, E, top, at):
    """From a number of rows on (at: bf16, fp32) a router's logits are summed in another order: both within fp32 rounding of
    64 bits, and the same experts wherever no two scores are closer than that."""
    R = at[dt == torch.float32]
    g = torch.Generator().manual_seed(W)
    h, wr = torch.randn(R, W, generator=g).to(dt), torch.randn(E, W, generator=g) / W ** 0.5
    h[:7] = 0.0
    h[:7, :E] = 1.0
    wr[:, :E] = wr[0, :E]                                     # rows 0 .. 6: sums of E products, all experts tied
    z = h.double() @ wr.double().t()
    bound = W * 2.0 ** -24 * (h.double().abs() @ wr.double().abs().t())   # W fp32 products and sums, in any order
    score = torch.sigmoid(z)
    # the sigmoid carries a quarter of a logit's error on at most, and adds its own few roundings
    off = bound / 4 + 8 * 2.0 ** -24
    ranked, order = score.sort(1, descending=True)
    clear = ranked[:, top - 1] - ranked[:, top] > 2 * off.amax(1)
    inside = (ranked[:, :top - 1] - ranked[:, 1:top] > 2 * off.amax(1, keepdim=True)).all(1)
    assert clear[7:].float().mean() > 0.95 and not clear[:7].any()
    for rows in (R - 1, R):
        ids, wts = torch.empty(rows, top, dtype=torch.int32, device=DEV), torch.empty(rows, top, device=DEV)
        cnt, lists = torch.empty(E, dtype=torch.int32, device=DEV), torch.empty(E, rows * top, dtype=torch.int32, device=DEV)
        sm.group_route(h[:rows].to(DEV), wr.to(DEV), top, 1, 1, ids, wts, cnt, lists)
        ids, wts = ids.cpu().long(), wts.cpu().double()
        assert ((wts - score[:rows].gather(1, ids)).abs() <= off[:rows].gather(1, ids)).all()
        assert torch.equal(ids[clear[:rows]].sort(1)[0], order[:rows, :top][clear[:rows]].sort(1)[0])
        both = (clear & inside)[:rows]
        assert torch.equal(ids[both], order[:rows, :top][both])


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts,N,K", [
    ([0, 1, 130, 400, 17], 100, 40),        # 64 x 64 tiles; K ends inside a step of either type
    ([700, 129, 300], 3000, 72),            # 96 x 128 tiles (bf16)
    ([700, 129, 300], 5152, 72),            # 64 x 64 (fp32; the ones before 32 x 64)
    ([700, 129, 300], 7008, 72),
    ([3, 0, 1], 160, 200),                  # few slots
    ([0, 1, 129, 170, 100], 5152, 72),      # 128 x 128 (bf16)
    ([321, 1, 158, 0, 170], 5152, 72)])     # 160 x 128 (bf16)
@pytest.mark.parametrize("act", [None, "silu_glu", "relu2", "limit"])
def test_expert_products(dt, counts, N, K, act):
    tiles = {(548, 100): (64, 32), (1129, 3000): (96, 32), (1129, 5152): (96, 64), (1129, 7008): (96, 64), (4, 160): (0, 0),
             (400, 5152): (128, 32), (650, 5152): (160, 32)}
    assert sm.lib().p2p_sm_expert_tile(len(counts), N, K, sum(counts), dt == torch.float32) == \
        tiles[sum(counts), N][dt == torch.float32]
    if act in ("silu_glu", "limit"):
        N = N // 32 * 32
    g = torch.Generator().manual_seed(4)
    E, S = len(counts), sum(counts)
    order = torch.randperm(S, generator=g).to(torch.int32)
    rows, at = torch.zeros(E, S, dtype=torch.int32), 0
    for e, n in enumerate(counts):
        rows[e, :n] = order[at:at + n]
        at += n
    cnt = torch.tensor(counts, dtype=torch.int32)
    x = torch.randn((S + 1) // 2, K + 8, generator=g).to(dt)[:, :K]       # two slots per row, strided
    w = (torch.randn(E, N, K, generator=g) / K ** 0.5).to(dt)
    kw = {"silu_glu": dict(silu_glu=True), "relu2": dict(relu2=True), "limit": dict(act_limit=0.9), None: {}}[act]
    F = N // 2 if act in ("silu_glu", "limit") else N
    want = sm.expert_gemm(x, 2, w, cnt, rows, torch.zeros(S, F, dtype=dt), S, **kw)
    x2 = torch.empty((S + 1) // 2, K + 8, dtype=dt, device=DEV)[:, :K].copy_(x)
    out = torch.full((S, F + 8), 7.0, dtype=dt, device=DEV)
    sm.expert_gemm(x2, 2, w.to(DEV), cnt.to(DEV), rows.to(DEV), out[:, :F], S, **kw)
    # sums of K products of about 1 / sqrt(K): fp32 rounding in either order, one rounding to bf16 (of values
    # up to about 5, squared under relu2: up to 25)
    tol = dict(rtol=1e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=2e-5, atol=1e-5)
    torch.testing.assert_close(out[:, :F].cpu().float(), want.float(), **tol)
    assert bool((out[:, F:] == 7.0).all())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("counts", [[3, 0, 1], [130, 70]])    # few slots / tiles
@pytest.mark.parametrize("N,K", [(48, 8), (64, 16), (20, 24), (70, 4), (33, 12)])
def test_expert_products_of_short_rows(dt, counts, N, K):
    """Rows shorter than one step of the kernels, the last ones at the end of their tensors."""
    if dt == torch.bfloat16 and K % 8:
        K *= 2
    g = torch.Generator().manual_seed(5)
    E, S = len(counts), sum(counts)
    rows, at = torch.zeros(E, S, dtype=torch.int32), 0
    for e, n in enumerate(counts):
        rows[e, :n] = torch.arange(at, at + n)
        at += n
    cnt = torch.tensor(counts, dtype=torch.int32)
    x, w = torch.randn(S, K, generator=g).to(dt), (torch.randn(E, N, K, generator=g) / K ** 0.5).to(dt)
    want = sm.expert_gemm(x, 1, w, cnt, rows, torch.zeros(S, N, dtype=dt), S)
    out = sm.expert_gemm(x.to(DEV), 1, w.to(DEV), cnt.to(DEV), rows.to(DEV), torch.zeros(S, N, dtype=dt, device=DEV), S)
    # up to 24 products of about 1 / sqrt(K) in fp32, one rounding to bf16 of values up to about 5
    tol = dict(rtol=1e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=2e-5, atol=1e-5)
    torch.testing.assert_close(out.cpu().float(), want.float(), **tol)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("K", [640, 200, 136])    # steps of a wavefront's share off the depth of its loads
def test_small_expert_products_with_infinite_weights(dt, K):
    """An infinite weight gives an infinite result, and only in its column."""
    g = torch.Generator().manual_seed(6)
    N, S = 70, 5
    x, w = torch.randn(S, K, generator=g).abs().to(dt), torch.randn(1, N, K, generator=g).to(dt)
    for k in (40, K - 3):
        w[0, k % N, k] = float("inf")
    cnt, rows = torch.tensor([S], dtype=torch.int32), torch.arange(S, dtype=torch.int32)[None]
    want = x.double() @ w[0].double().T
    out = sm.expert_gemm(x.to(DEV), 1, w.to(DEV), cnt.to(DEV), rows.to(DEV), torch.zeros(S, N, dtype=dt, device=DEV), S).cpu()
    fin = want.isfinite()
    assert torch.equal(out[~fin].double(), want[~fin]) and (~fin).sum() == 2 * S
    torch.testing.assert_close(out[fin].double(), want[fin], rtol=1e-2 if dt == torch.bfloat16 else 1e-5, atol=1e-4)


@pytest.mark.parametrize("R", [3, 300])      # a row per workgroup / sixteen
@pytest.mark.parametrize("score,groups,keep", [("sigmoid", 1, 1), ("softmax", 4, 2), ("top_softmax", 4, 1)])
def test_routing_of_rows_that_are_not_finite(R, score, groups, keep):
    """Every slot goes to an expert that exists and is in that expert's list, whatever the scores are; the other
    rows' choices are as they were."""
    g = torch.Generator().manual_seed(3)
    W, E, top = 40, 12, 3
    h, wr = torch.randn(R, W, generator=g), torch.randn(E, W, generator=g)
    corr = torch.randn(E, generator=g)
    bad = h.clone()
    bad[1], bad[2, 7], bad[R - 1, 3] = float("nan"), float("inf"), -3e38
    low = torch.full((E,), float("-inf"))     # no expert wanted
    res = []
    for x, c in ((h, corr), (bad, corr), (h, low)):
        ids, wts = torch.full((R, top), -1, dtype=torch.int32, device=DEV), torch.empty(R, top, device=DEV)
        cnt, rows = torch.empty(E, dtype=torch.int32, device=DEV), torch.full((E, R * top), -1, dtype=torch.int32, device=DEV)
        sm.group_route(x.to(DEV), wr.to(DEV), top, groups, keep, ids, wts, cnt, rows, score=score, corr=c.to(DEV))
        ids, cnt, rows = ids.cpu(), cnt.cpu(), rows.cpu()
        assert int(ids.min()) >= 0 and int(ids.max()) < E
        assert all(len(set(r)) == top for r in ids.tolist())
        for e in range(E):
            assert sorted(rows[e, :int(cnt[e])].tolist()) == (ids.reshape(-1) == e).nonzero()[:, 0].tolist()
        res.append(ids)
    same = [r for r in range(R) if r not in (1, 2, R - 1)]
    assert torch.equal(res[0][same], res[1][same])
