"""HIP kernels of ops.seqmix against the PyTorch rendering of the same ops (CPU tensors),
in fp32 and bf16, at sizes that are not multiples of the kernels' tiles, with several
entries per step and state carried over a second step."""
import pytest
import torch

from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ents(lens, starts, slots):
    ent, r0 = [], 0
    for n, s, sl in zip(lens, starts, slots):
        ent.append((r0, n, s, sl))
        r0 += n
    row_ent = [i for i, e in enumerate(ent) for _ in range(e[1])]
    return ent, torch.tensor(ent, dtype=torch.int32), torch.tensor(row_ent, dtype=torch.int32), r0


def _tol(dt):
    return dict(rtol=2e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=2e-4, atol=2e-5)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("wide", [200, 4100])   # rows kept in registers / rows read twice
def test_embed_norms(dt, wide):
    g = torch.Generator().manual_seed(0)
    V, W, R = 50, wide, 37
    emb, ptab = torch.randn(V, W, generator=g).to(dt), torch.randn(64, W, generator=g).to(dt)
    ids = torch.randint(0, V, (R,), generator=g, dtype=torch.int32)
    pos = torch.randint(0, 64, (R,), generator=g, dtype=torch.int32)
    a = sm.embed_pos(emb, ptab, ids, pos, torch.empty(R, W))
    b = sm.embed_pos(emb.to(DEV), ptab.to(DEV), ids.to(DEV), pos.to(DEV), torch.empty(R, W, device=DEV))
    torch.testing.assert_close(b.cpu(), a, rtol=0, atol=0)
    w = torch.randn(W, generator=g)
    for parts in (1, 4) if wide % 4 == 0 else (1,):
        o1 = sm.rmsnorm(a, w, 1e-5, torch.empty(R, W, dtype=dt), parts=parts)
        o2 = sm.rmsnorm(b, w.to(DEV), 1e-5, torch.empty(R, W, dtype=dt, device=DEV), parts=parts)
        torch.testing.assert_close(o2.cpu().float(), o1.float(), **_tol(dt))
    # gather + scatter
    inr = torch.tensor([5, 0, 36], dtype=torch.int32)
    outr = torch.tensor([7, -1, 2], dtype=torch.int32)
    y = a.to(dt)
    o1 = sm.rmsnorm(y, w, 1e-5, torch.zeros(9, W, dtype=dt), in_rows=inr, out_rows=outr)
    o2 = sm.rmsnorm(y.to(DEV), w.to(DEV), 1e-5, torch.zeros(9, W, dtype=dt, device=DEV),
                    in_rows=inr.to(DEV), out_rows=outr.to(DEV))
    torch.testing.assert_close(o2.cpu().float(), o1.float(), **_tol(dt))
    ls = torch.randn(W, generator=g)
    x1 = sm.norm_scale_add(a.clone(), y, w, ls, 1e-5)
    x2 = sm.norm_scale_add(b.clone(), y.to(DEV), w.to(DEV), ls.to(DEV), 1e-5)
    torch.testing.assert_close(x2.cpu(), x1, rtol=1e-5, atol=1e-5)
    # ... and the next sublayer's normed input in the same pass
    w2 = torch.randn(W, generator=g)
    h1, h2 = torch.empty(R, W, dtype=dt), torch.empty(R, W, dtype=dt, device=DEV)
    x1 = sm.norm_scale_add(a.clone(), y, w, ls, 1e-5, next_w=w2, next_out=h1)
    x2 = sm.norm_scale_add(b.clone(), y.to(DEV), w.to(DEV), ls.to(DEV), 1e-5, next_w=w2.to(DEV), next_out=h2)
    torch.testing.assert_close(x2.cpu(), x1, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(h2.cpu().float(), h1.float(), **_tol(dt))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_pointwise(dt):
    g = torch.Generator().manual_seed(1)
    R, H, V, Fd = 9, 3, 20, 70
    x = torch.randn(R, 40, generator=g).to(dt)
    a = sm.tanh_(x[:, 10:33].clone())
    big = x.to(DEV)
    b = sm.tanh_(big[:, 10:33])
    torch.testing.assert_close(b.cpu().float(), a.float(), **_tol(dt))
    o, gt = torch.randn(H, R, V, generator=g).to(dt), torch.randn(R, H * V, generator=g).to(dt)
    a = sm.sigmoid_gate(o, gt, torch.empty(R, H * V, dtype=dt), H, V)
    b = sm.sigmoid_gate(o.to(DEV), gt.to(DEV), torch.empty(R, H * V, dtype=dt, device=DEV), H, V)
    torch.testing.assert_close(b.cpu().float(), a.float(), **_tol(dt))
    gu = (3 * torch.randn(R, 2 * Fd, generator=g)).to(dt)
    a = sm.ff_act(gu, torch.empty(R, Fd, dtype=dt), 1.75)
    b = sm.ff_act(gu.to(DEV), torch.empty(R, Fd, dtype=dt, device=DEV), 1.75)
    torch.testing.assert_close(b.cpu().float(), a.float(), **_tol(dt))


@pytest.fixture(params=[64, 8], ids=["onepass", "chunks8"])
def scan_chunk(request, monkeypatch):
    """Both forms of the recurrent scans: one pass over a portion, and chunks of 8 tokens
    side by side (used for portions of 16 tokens and more)."""
    monkeypatch.setattr(sm, "SCAN_CHUNK", request.param)
    return request.param


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D", [(2, 40), (3, 20), (1, 72), (2, 64), (1, 136), (2, 7)])
def test_gdelta(dt, H, D, scan_chunk):
    g = torch.Generator().manual_seed(2)
    n = H * D
    slots = 5
    w0, ab, nw = (torch.randn(n, generator=g) for _ in range(3))
    st_c = torch.zeros(slots, H, D, D)
    st_g = st_c.to(DEV)
    for lens, starts in (([40, 1, 7], [0, 0, 0]), ([3, 1, 35], [40, 1, 7])):
        ent_h, ent, row_ent, R = _ents(lens, starts, [3, 0, 4])
        proj = torch.randn(R, 5 * n + 3, generator=g).to(dt)
        lo = torch.randn(R, n, generator=g).to(dt)
        v5 = lambda p: [p[:, i * n:(i + 1) * n] for i in range(5)]
        a = sm.gdelta_scan(*v5(proj), lo, w0, ab, nw, st_c, ent, ent_h, torch.empty(R, n, dtype=dt), H, D, 1e-5)
        pg = proj.to(DEV)
        b = sm.gdelta_scan(*v5(pg), lo.to(DEV), w0.to(DEV), ab.to(DEV), nw.to(DEV), st_g, ent.to(DEV),
                           ent_h, torch.empty(R, n, dtype=dt, device=DEV), H, D, 1e-5)
        torch.testing.assert_close(b.cpu().float(), a.float(), **_tol(dt))
        torch.testing.assert_close(st_g.cpu()[[3, 0, 4]], st_c[[3, 0, 4]], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,P,N,G,K", [(6, 40, 24, 3, 3), (4, 24, 16, 1, 4), (2, 72, 80, 2, 2), (2, 200, 256, 1, 4), (8, 64, 128, 4, 4)])
def test_mamba(dt, H, P, N, G, K, scan_chunk):
    g = torch.Generator().manual_seed(3)
    inner, C = H * P, H * P + 2 * G * N
    slots = 4
    cw, cb = torch.randn(C, K, generator=g) * 0.5, torch.randn(C, generator=g) * 0.1
    dtb, Al, Dp = torch.randn(H, generator=g), torch.rand(H, generator=g) - 0.5, torch.randn(H, generator=g)
    S_c, T_c = torch.zeros(slots, H, N, P), torch.zeros(slots, K - 1, C)
    S_g, T_g = S_c.to(DEV), T_c.to(DEV)
    for lens, starts in (([1, 30, 2], [0, 0, 0]), ([1, 1, 33], [1, 30, 2]), ([5, 1, 1], [2, 31, 35])):
        ent_h, ent, row_ent, R = _ents(lens, starts, [2, 0, 3])
        zx = torch.randn(R, 2 * inner + 2 * G * N + H, generator=g).to(dt)
        c1 = sm.mamba_conv(zx, inner, cw, cb, T_c, ent, ent_h, row_ent, torch.empty(R, C))
        zg = zx.to(DEV)
        c2 = sm.mamba_conv(zg, inner, cw.to(DEV), cb.to(DEV), T_g, ent.to(DEV), ent_h, row_ent.to(DEV),
                           torch.empty(R, C, device=DEV))
        torch.testing.assert_close(c2.cpu(), c1, rtol=1e-4, atol=1e-5)
        y1 = sm.mamba_scan(c1, zx, inner, inner + C, dtb, Al, Dp, S_c, T_c, ent, ent_h, torch.empty(R, inner), H, P, N, G)
        y2 = sm.mamba_scan(c2, zg, inner, inner + C, dtb.to(DEV), Al.to(DEV), Dp.to(DEV), S_g, T_g, ent.to(DEV),
                           ent_h, torch.empty(R, inner, device=DEV), H, P, N, G)
        torch.testing.assert_close(y2.cpu(), y1, rtol=2e-4, atol=2e-4)
        torch.testing.assert_close(S_g.cpu()[[2, 0, 3]], S_c[[2, 0, 3]], rtol=2e-4, atol=2e-4)
        torch.testing.assert_close(T_g.cpu()[[2, 0, 3]], T_c[[2, 0, 3]], rtol=0, atol=0)


@pytest.fixture
def walks(monkeypatch):
    """SCAN_CHUNK = 0: no scan forms chunks, whatever its portions are."""
    def tables(*_a):
        raise AssertionError("a scan formed chunks")
    monkeypatch.setattr(sm, "SCAN_CHUNK", 0)
    monkeypatch.setattr(sm, "chunk_tables", tables)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D", [(2, 40), (3, 20), (1, 72), (2, 64), (1, 136), (2, 7)])
def test_gdelta_walks(dt, H, D, walks):
    test_gdelta(dt, H, D, 0)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,P,N,G,K", [(6, 40, 24, 3, 3), (2, 72, 80, 2, 2), (2, 200, 256, 1, 4), (8, 64, 128, 4, 4)])
def test_mamba_walks(dt, H, P, N, G, K, walks):
    test_mamba(dt, H, P, N, G, K, 0)


GD_FORMS = [
    # portions, heads, head size, the form that runs first, the portions that are in it
    ([38], 2, 64, "walk", [38]), ([40], 2, 64, "matrix", [40]), ([40, 5], 2, 32, "walk", [40, 5]),
    ([64] * 8, 33, 40, "matrix", [64] * 8), ([64] * 8, 40, 40, "walk", [64] * 8),
    ([100, 40, 1], 32, 64, "matrix", [100, 40, 1]), ([64, 1, 5, 1], 256, 8, "matrix", [64]),
    ([1100], 128, 8, "chunks", [1100]), ([1000, 3], 128, 8, "matrix", [1000]), ([130, 5], 2, 72, "chunks", [130, 5])]


@pytest.mark.parametrize("lens,H,D,form,first", GD_FORMS)
def test_gdelta_forms(lens, H, D, form, first, monkeypatch):
    """Both sides of the lines between the walk, walked chunks and matrix products; what is left walks."""
    ran = []
    for nm in ("p2p_sm_gdelta_scan", "p2p_sm_gdelta_scan_chunked", "p2p_sm_gdelta_chunk"):
        f = getattr(sm.lib(), nm)
        monkeypatch.setattr(sm.lib(), nm, lambda *a, f=f, nm=nm: (ran.append(nm), f(*a))[1])
    test_gdelta_long_portions(torch.float32, lens, [3 * i for i in range(len(lens))], H, D, 0.0)
    names = {"walk": "p2p_sm_gdelta_scan", "chunks": "p2p_sm_gdelta_scan_chunked", "matrix": "p2p_sm_gdelta_chunk"}
    assert ran == [names[form]] + ([names["walk"]] if first != lens else [])


@pytest.mark.parametrize("lens,H,P,N,first", [
    ([31, 1], 4, 64, 128, []), ([32], 4, 64, 128, []), ([36], 4, 64, 128, [36]), ([130, 1, 20], 4, 64, 128, [130, 20, 1]),
    ([64, 1, 5, 1], 128, 64, 128, [64]), ([1, 130, 1, 70, 31], 128, 64, 128, [130, 70, 31])])
def test_mamba_portions_in_chunks(lens, H, P, N, first, monkeypatch):
    """Decoded tokens join a prompt's chunks where that is cheap and walk where it is not."""
    cut, whole = [], sm.scan_chunks
    monkeypatch.setattr(sm, "scan_chunks", lambda e, c: (cut.extend(x[1] for x in e), whole(e, c))[1])
    test_mamba_long_portions(lens, [2 * i for i in range(len(lens))], H, P, N, 2, False)
    assert sorted(cut) == sorted(first)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,rank,win", [(6, 120, 36), (3, 40, 7), (5, 96, 200), (16, 512, 33), (20, 64, 64), (1, 8, 3)])
def test_latent_attn(dt, H, rank, win):
    g = torch.Generator().manual_seed(4)
    page, npages = 64, 12
    cache = torch.randn(npages * page, rank, generator=g).to(dt)
    bt = torch.tensor([[3, 7, 1, 9], [2, 5, 0, 0]], dtype=torch.int32)
    # entry 0: rows at positions 100..139 (crosses a page border), entry 1: single token at 70
    pos = torch.tensor(list(range(100, 140)) + [70], dtype=torch.int32)
    row_ent = torch.tensor([0] * 40 + [1], dtype=torch.int32)
    R = pos.numel()
    qa = (torch.randn(R, H, rank, generator=g) * 0.3).to(dt).transpose(0, 1)   # strided [H, R, rank]
    sink = torch.randn(H, generator=g)
    a = sm.latent_attn(qa, cache, bt, row_ent, pos, sink, 0.2, win, torch.empty(H, R, rank, dtype=dt), page)
    b = sm.latent_attn(qa.to(DEV), cache.to(DEV), bt.to(DEV), row_ent.to(DEV), pos.to(DEV), sink.to(DEV), 0.2,
                       win, torch.empty(H, R, rank, dtype=dt, device=DEV), page)
    torch.testing.assert_close(b.cpu().float(), a.float(), **_tol(dt))
    if dt == torch.bfloat16:
        # the matrix-core kernel: queries as a contiguous [H, R, rank] tensor, row groups per wave
        qc = qa.contiguous().to(DEV)
        assert sm.latent_mfma_ok(qc, cache.to(DEV))
        units = sm.make_units([(0, 40, 100, 0), (40, 1, 70, 1)], sm.latent_rows_per_wave(H)).to(DEV)
        c = sm.latent_attn(qc, cache.to(DEV), bt.to(DEV), row_ent.to(DEV), pos.to(DEV), sink.to(DEV), 0.2,
                           win, torch.empty(H, R, rank, dtype=dt, device=DEV), page, units=units)
        torch.testing.assert_close(c.cpu().float(), a.float(), **_tol(dt))
        # few rows, long windows: every window cut into runs of key tiles and merged
        d = sm.latent_attn(qc, cache.to(DEV), bt.to(DEV), row_ent.to(DEV), pos.to(DEV), sink.to(DEV), 0.2,
                           win, torch.empty(H, R, rank, dtype=dt, device=DEV), page, units=units,
                           max_keys=140)
        torch.testing.assert_close(d.cpu().float(), a.float(), **_tol(dt))


@pytest.mark.parametrize("runs", [1, 2, 3, 5])
@pytest.mark.parametrize("H,rank,win,sunk", [(3, 72, 300, True), (20, 200, 131, False), (1, 384, 65, True), (16, 512, 300, True)])
def test_latent_attn_shared_by_wavefronts(monkeypatch, H, rank, win, sunk, runs):
    """Latents over 64 numbers in a step: 64 keys of four wavefronts, runs of an odd number of 32 keys, runs that are
    empty, units of one to 16 rows, padded ranks."""
    monkeypatch.setattr(sm, "_key_runs", lambda *a: runs)
    g = torch.Generator().manual_seed(H)
    page = 48
    cache = torch.randn(page * 16, rank, generator=g).bfloat16()
    bt = torch.randperm(16, generator=g).to(torch.int32).view(2, 8)
    pos = torch.tensor(list(range(280, 299)) + [0, 63], dtype=torch.int32)
    row_ent = torch.tensor([0] * 19 + [1, 1], dtype=torch.int32)
    qa = (torch.randn(H, 21, rank, generator=g) * 0.2).bfloat16()
    sink = torch.randn(H, generator=g) if sunk else None
    want = sm.latent_attn(qa, cache, bt, row_ent, pos, sink, 0.2, win, torch.empty(H, 21, rank).bfloat16(), page)
    units = sm.make_units([(0, 19, 280, 0), (19, 1, 0, 1), (20, 1, 63, 1)], sm.latent_rows_per_wave(H)).to(DEV)
    got = sm.latent_attn(qa.to(DEV), cache.to(DEV), bt.to(DEV), row_ent.to(DEV), pos.to(DEV), None if sink is None else
                         sink.to(DEV), 0.2, win, torch.empty(H, 21, rank, device=DEV).bfloat16(), page, units=units,
                         max_keys=300)
    torch.testing.assert_close(got.cpu().float(), want.float(), **_tol(torch.bfloat16))


@pytest.mark.parametrize("lens,starts", [([130, 64, 1], [0, 7, 3]), ([65], [0]), ([33, 200], [5, 0])])
@pytest.mark.parametrize("H,P,N,G", [(4, 64, 128, 2), (2, 30, 17, 1), (1, 256, 256, 1), (3, 36, 20, 1), (2, 100, 44, 1)])
@pytest.mark.parametrize("steep", [False, True])
def test_mamba_long_portions(lens, starts, H, P, N, G, steep):
    """Chunks of 64 on the matrix instruction: remainders, single-chunk portions beside long ones, and
    decays so steep that a quotient of running products would overflow."""
    g = torch.Generator().manual_seed(6)
    inner, C = H * P, H * P + 2 * G * N
    slots = len(lens) + 1
    ent_h, ent, _row_ent, R = _ents(lens, starts, list(range(len(lens)))[::-1])
    conv = torch.randn(R, C, generator=g)
    zx = torch.randn(R, 2 * inner + 2 * G * N + H, generator=g)
    dtb, Dp = torch.randn(H, generator=g) + (3.0 if steep else 0.0), torch.randn(H, generator=g)
    Al = torch.rand(H, generator=g) + (3.0 if steep else -1.0)
    S0, T0 = torch.randn(slots, H, N, P, generator=g), torch.zeros(slots, 3, C)
    res = []
    for dev in ("cpu", DEV):
        S, T = S0.clone().to(dev), T0.clone().to(dev)
        y = sm.mamba_scan(conv.to(dev), zx.to(dev), inner, inner + C, dtb.to(dev), Al.to(dev), Dp.to(dev), S, T,
                          ent.to(dev), ent_h, torch.empty(R, inner, device=dev), H, P, N, G)
        res.append((y.cpu(), S.cpu()))
    (y1, s1), (y2, s2) = res
    # sums of up to 64 x 256 fp32 products in another order, exponents of sums of 64 steps
    for a, b in ((y1, y2), (s1, s2)):
        torch.testing.assert_close(b, a, rtol=1e-4, atol=1e-5 * float(a.abs().max()))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,P,N,G", [(8, 64, 128, 2), (6, 32, 16, 3), (4, 100, 44, 1), (2, 64, 30, 1), (2, 200, 8, 1)])
def test_mamba_groups_share_their_products(dt, H, P, N, G):
    """Heads of a group take the products of B and C from one workgroup, and z and y four numbers at a time where rows
    allow it: to the bit what every head forms by itself (a group each, with the same B and C) and what odd rows give."""
    g = torch.Generator().manual_seed(H + P + N)
    inner, lens = H * P, [150, 64, 33]
    ent_h, ent, _row_ent, R = _ents(lens, [0, 5, 0], [2, 1, 0])
    x, bc = torch.randn(R, inner, generator=g), torch.randn(2, R, G, N, generator=g)
    zx = torch.randn(R, 2 * inner + 2 * H * N + H, generator=g).to(dt).to(DEV)
    dtb, Al, Dp = (torch.randn(H, generator=g).to(DEV) for _ in range(3))
    S0 = torch.randn(4, H, N, P, generator=g)
    res = []
    for groups, pad in ((G, 0), (H, 0), (G, 1)):
        B, C = (b.repeat_interleave(groups // G, 1).reshape(R, groups * N) for b in bc)
        conv = torch.cat([x, B, C], 1).to(DEV)
        z = torch.nn.functional.pad(zx, (0, pad))
        S, T = S0.to(DEV), torch.zeros(4, 3, conv.shape[1], device=DEV)
        y = sm.mamba_scan(conv, z, inner, zx.shape[1] - H, dtb, Al, Dp, S, T, ent.to(DEV), ent_h,
                          torch.empty(R, inner, device=DEV), H, P, N, groups)
        res.append((y, S))
    for y, S in res[1:]:
        assert torch.equal(y, res[0][0]) and torch.equal(S, res[0][1])


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("lens,starts", [([130, 64, 1], [0, 7, 3]), ([65], [0]), ([33, 200], [5, 0])])
@pytest.mark.parametrize("H,D", [(4, 64), (2, 33), (1, 5)])
@pytest.mark.parametrize("decay", [-20.0, 0.0, 20.0])
def test_gdelta_long_portions(dt, lens, starts, H, D, decay):
    """Chunks of 64 on the matrix instruction: remainders, single-chunk portions beside long ones, decays of one, mixed,
    and the strongest there are."""
    g = torch.Generator().manual_seed(8)
    n, slots = H * D, len(lens) + 1
    ent_h, ent, _row_ent, R = _ents(lens, starts, list(range(len(lens)))[::-1])
    proj, lo = torch.randn(R, 5 * n + 3, generator=g).to(dt), torch.randn(R, n, generator=g).to(dt)
    w0, ab, nw = torch.randn(n, generator=g) + decay, torch.randn(n, generator=g), torch.randn(n, generator=g)
    S0 = torch.randn(slots, H, D, D, generator=g)
    res = []
    for dev in ("cpu", DEV):
        S, p = S0.clone().to(dev), proj.to(dev)
        o = sm.gdelta_scan(*[p[:, i * n:(i + 1) * n] for i in range(5)], lo.to(dev), w0.to(dev), ab.to(dev), nw.to(dev), S,
                           ent.to(dev), ent_h, torch.empty(R, n, dtype=dt, device=dev), H, D, 1e-5)
        res.append((o.cpu().float(), S.cpu()))
    (o1, s1), (o2, s2) = res
    # 200 tokens of fp32 sums in another order; without decay nothing is forgotten on the way
    torch.testing.assert_close(s2, s1, rtol=2e-4, atol=2e-5 * float(s1.abs().max()))
    torch.testing.assert_close(o2, o1, **(_tol(dt) if dt == torch.bfloat16 else dict(rtol=1e-3, atol=2e-4)))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 1030, 1024), (2, 4096, 8), (8, 2048, 1000), (9, 40, 512), (16, 10304, 1024),
                                   (8, 10304, 2048), (16, 2051, 1544)])
@pytest.mark.parametrize("form", ["plain", "norm", "tanh", "conv", "conv32"])
def test_products_form_their_rows(dt, M, N, K, form, monkeypatch):
    """A product that forms its input rows (and convolves its columns) on the way leaves the bits of the separate passes:
    rows, halves of the workgroup and widths that do not fill, strided y, one to four taps, slots at position 0."""
    if dt == torch.float32 and K > 1024:
        pytest.skip("no kernel: longer rows than registers hold")
    g = torch.Generator().manual_seed(M + N + K)
    rnd = lambda *s: torch.randn(*s, generator=g).to(DEV)
    x, spare, h = rnd(M, K), torch.empty(M, K, device=DEV), torch.empty(M, K, device=DEV, dtype=dt)
    y, w, gain, ls = rnd(M, K + 8).to(dt)[:, :K], (rnd(N, K) * K ** -0.5).to(dt), rnd(K), rnd(K)
    nw, b = (rnd(K), None) if form in ("norm", "conv32") else (None, rnd(N).to(dt))
    taps = 1 + (M + N) % 4 if form == "conv32" else 4
    c0, C = N // 3, N // 2
    cw, cb, tail = rnd(C, taps), rnd(C), rnd(M + 2, taps - 1, C)
    ent = [(r, 1, 0 if r == 1 else 5 + r, M + 1 - r) for r in range(M)]
    entd, re = torch.tensor(ent, dtype=torch.int32, device=DEV), torch.arange(M, dtype=torch.int32, device=DEV)
    co = torch.empty(M, C, device=DEV, dtype=torch.float32 if form == "conv32" else dt)
    # the passes one by one
    x1, t1, co1 = x.clone(), tail.clone(), co.clone()
    if not sm._skinny(h, w):
        pytest.skip("no kernel: the library's shape")
    h1 = torch.empty_like(h)
    sm.norm_scale_add(x1, y, gain, ls if form != "plain" else None, 1e-5, next_w=nw, next_out=h1)
    tanh = N // 2 if form == "tanh" else None
    want = sm.linear(h1, w, None if form.startswith("conv") else b, tanh_from=tanh)
    monkeypatch.setattr(sm, "NORMED_ROWS", 16)
    p = sm.NormedRows(x, spare, y, gain, ls if form != "plain" else None, 1e-5, nw, h)
    x0 = x.clone()
    if form.startswith("conv"):
        sm.mamba_conv(want, c0, cw, cb, t1, entd, ent, re, co1, roll=True)
        t2, co2 = tail.clone(), torch.empty_like(co)   # ... of rows that are there
        assert torch.equal(sm.linear_conv(h1, w, c0, cw, cb, t2, entd, ent, re, co2), want)
        assert torch.equal(t2, t1) and torch.equal(co2, co1)
        got = p.linear(w, conv=(c0, cw, cb, tail, entd, co))
        assert got is not None
        assert torch.equal(co, co1) and torch.equal(tail, t1)
    else:
        got = p.linear(w, b, tanh)
        assert got is not None
    assert torch.equal(got, want) and torch.equal(p.x, x1) and p.x is spare and torch.equal(x, x0)
    if not form.startswith("conv"):
        z = (want.float() * 0.5) if tanh is None else None
        if z is not None and b is None:
            assert torch.equal(sm.logits(h1, w, 0.0, 0.5), z)
            assert torch.equal(sm.logits(h1, w, 3.0, 0.5), sm.softcap(want, 3.0, torch.empty_like(z), scale=0.5))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 7, 16, 17])
@pytest.mark.parametrize("N,K", [(1, 8), (1024, 4), (1040, 64), (1031, 1000), (1025, 2048), (33, 4096), (16, 4104)])
@pytest.mark.parametrize("off,bias", [(0, False), (8, True), (3, True)])
def test_linear_few_rows(dt, M, N, K, off, bias):
    """Edges of the 16 columns, of the 128-byte pieces and of the eight wavefronts' turns, strided and unaligned
    rows; shapes on both sides of the rule."""
    g = torch.Generator().manual_seed(9)
    x = torch.randn(M, K + 24, generator=g).to(dt).to(DEV)[:, off:off + K]
    w, b = torch.randn(N, K, generator=g).to(dt).to(DEV), torch.randn(N, generator=g).to(dt).to(DEV) if bias else None
    y = sm.linear(x, w, b)
    ref = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    # one rounding of the result, and K products summed in fp32: eps |x| |w| sqrt(K) with room for the tail
    eps = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -23
    torch.testing.assert_close(y.double(), ref, rtol=eps, atol=8 * 2.0 ** -24 * K + 1e-6)
    assert y.dtype == dt and y.is_contiguous()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [4, 256, 260, 1023, 1024, 1028, 2048, 2052, 4096, 4100])
@pytest.mark.parametrize("off", [0, 4, 1])   # first column of the rows and vectors: aligned for one wide load, or not
def test_row_passes_by_width(dt, n, off):
    """The row passes at the edges of the widths that a form takes, and on rows that wide loads cannot take."""
    g = torch.Generator().manual_seed(10)
    R = 5
    x, big = torch.randn(R, n, generator=g), torch.randn(R, 3 * n + 12, generator=g).to(dt)
    vecs = torch.randn(4, 2 * n + 8, generator=g)
    res = []
    for dev in ("cpu", DEV):
        b, v = big.to(dev), [t.to(dev)[off:off + n] for t in vecs]
        ya, yb = b[:, off:off + n], b[:, n + 4 + off:n + 4 + off + n]
        out = [torch.zeros(R, n + 8, dtype=dt, device=dev)[:, off:off + n] for _ in range(5)]
        x1 = sm.norm_scale_add(x.clone().to(dev), ya, v[0], v[1], 1e-5, v[2], out[0])
        x2 = sm.add_norm(x.clone().to(dev), ya, yb, 1e-5, v[0], out[1])
        x3 = sm.add_norm2(x.clone().to(dev), ya, yb, vec=v[3], eps=1e-5, w1=v[0], out1=out[2], w2=v[1][:1], out2=out[3])
        parts = 2 if n % 2 == 0 else 1
        sm.rmsnorm(ya, v[1], 1e-5, out[4], parts=parts)
        res.append([t.float().cpu() for t in [x1, x2, x3] + out])
    # sums of up to 4100 fp32 squares in another order, then one rounding; the two wide inputs double the scale
    for p, q in zip(*res):
        torch.testing.assert_close(q, p, **(_tol(dt) if dt == torch.bfloat16 else dict(rtol=1e-5, atol=1e-5)))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("F,off", [(4, 0), (252, 0), (256, 0), (1020, 0), (1023, 0), (1028, 4), (1028, 1), (1, 0)])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh"])
def test_glu_act_by_width(dt, F, off, act):
    """Four channels per thread at the edges of a block, and the widths and rows that take one."""
    gu = (torch.randn(3, 2 * F + 8, generator=torch.Generator().manual_seed(11)) * 2).to(dt)
    res = [sm.glu_act(gu.to(d)[:, off:off + 2 * F], torch.zeros(3, F + 4, dtype=dt, device=d)[:, :F], act).cpu()
           for d in ("cpu", DEV)]
    torch.testing.assert_close(res[1], res[0], **_tol(dt))


@pytest.mark.parametrize("R,H,V,K,per_head", [(1, 16, 128, 512, False), (8, 3, 40, 72, False), (16, 2, 24, 448, True),
                                              (9, 1, 1, 8, True), (17, 2, 24, 64, False),
                                              (8, 32, 512, 512, False), (8, 32, 513, 512, False)])
def test_heads_gated(R, H, V, K, per_head):
    """Products of few rows per head with the gate in the epilogue: as the library's product, rounded, and the gate pass
    (one bf16 step apart where the sums round differently), also from rows with a gap and into rows with a gap."""
    g = torch.Generator().manual_seed(R + V)
    x = torch.randn(H, R, K + 8, generator=g).bfloat16().to(DEV)[:, :, :K]
    w = (torch.randn(H, V, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    gate = torch.randn(R, H * V + 3, generator=g).bfloat16().to(DEV)
    out = torch.full((R, H * V + 5), 7.0, device=DEV).bfloat16()
    wt = w.transpose(1, 2).contiguous()
    sm.heads_gated(x, w, wt, gate, out[:, :H * V], per_head=per_head)
    o = torch.stack([x[h].double() @ w[h].double().T for h in range(H)])
    z = torch.sigmoid(gate.double())
    z = z[:, :H].repeat_interleave(V, 1) if per_head else z[:, :H * V]
    want = o.permute(1, 0, 2).reshape(R, H * V) * z
    assert ((out[:, :H * V].double() - want).abs() <= 2 ** -7 * want.abs() + 1e-5 * o.abs().max()).all()
    assert (out[:, H * V:] == 7).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,part", [(1, 1, 1), (8, 17, 9), (16, 4096, 64), (5, 4112, 65), (8, 8203, 128), (16, 13000, 2),
                                      (3, 8200, 256), (2, 4120, 257), (16, 50, 511),
                                      (7, 5000, 161), (2, 2040, 192), (4, 2032, 192),
                                      (4, 4112, 57), (16, 8210, 81), (8, 4500, 225), (4, 3080, 192)])
def test_few_row_products_walk_over_columns(dt, M, N, part):
    """K of ``part`` 16-byte fragments: one to four pieces per wavefront and beyond, whole ones and rests; one to several
    tiles per workgroup, the last one cut; rows with a gap.  Against 64 bits: one rounding of the result and one of each
    of the K sums in fp32."""
    K = part * (16 // dt.itemsize)
    g = torch.Generator().manual_seed(part)
    x = torch.randn(M, K + 16, generator=g).to(dt).to(DEV)[:, :K]
    w = torch.randn(N, K, generator=g).to(dt).to(DEV)
    b = torch.randn(N, generator=g).to(dt).to(DEV)
    y = torch.full((M + 1, N), 7.0, dtype=dt, device=DEV)
    sm._chk(sm.lib().p2p_sm_skinny(x.data_ptr(), x.stride(0), w.data_ptr(), b.data_ptr(), y.data_ptr(), M, N, K, N,
                                   int(dt == torch.float32), sm._st(x)), "skinny")
    want = x.double() @ w.double().T + b.double()
    size = x.double().abs() @ w.double().abs().T + b.double().abs()
    half = 2.0 ** -24 if dt == torch.float32 else 2.0 ** -8
    assert ((y[:M].double() - want).abs() <= half * want.abs() + (K + 1) * 2.0 ** -23 * size).all()
    assert (y[M] == 7).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 8, 16, 17, 300])
def test_linear_with_tanh_columns(dt, M):
    """tanh of the columns from one on, from none on as well: bit for bit the product and then the pass over them."""
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, 1024, generator=g).to(dt).to(DEV)
    w = (torch.randn(1104, 1024, generator=g) / 32).to(dt).to(DEV)
    for at in (0, 1072, 1087, 1104):
        want = sm.linear(x, w)
        if at < 1104:
            sm.tanh_(want[:, at:])
        assert torch.equal(sm.linear(x, w, tanh_from=at), want), at


def test_mamba_tails_move_in_the_convolution():
    """A step of single tokens: outputs, states and tails are those of a convolution that leaves its tails to the scan."""
    g = torch.Generator().manual_seed(5)
    H, P, N, G, K, E = 4, 64, 32, 2, 4, 5
    inner = H * P
    C = inner + 2 * G * N
    zx = torch.randn(E, 2 * inner + 2 * G * N + H, generator=g).bfloat16().to(DEV)
    cw, cb = torch.randn(C, K, generator=g).to(DEV), torch.randn(C, generator=g).to(DEV)
    dtb, al, dp = (torch.randn(H, generator=g).to(DEV) for _ in range(3))
    ent_h, ent, row_ent, R = _ents([1] * E, [3, 0, 7, 1, 9], [4, 0, 2, 1, 3])
    got = []
    for roll in (False, True):
        S, T = torch.randn(6, H, N, P, generator=torch.Generator().manual_seed(1)).to(DEV), torch.randn(
            6, K - 1, C, generator=torch.Generator().manual_seed(2)).to(DEV)
        conv = torch.empty(R, C, device=DEV)
        sm.mamba_conv(zx, inner, cw, cb, T, ent.to(DEV), ent_h, row_ent.to(DEV), conv, roll=roll)
        y = torch.empty(R, inner, device=DEV)
        sm.mamba_scan(conv, zx, inner, inner + C, dtb, al, dp, S, T, ent.to(DEV), ent_h, y, H, P, N, G, roll=not roll)
        got.append((y, S, T))
    for a, b in zip(*got):
        assert torch.equal(a, b)
