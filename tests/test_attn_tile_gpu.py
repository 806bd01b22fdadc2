"""The attention kernels whose wavefronts share key tiles in LDS against the PyTorch rendering of the
same ops, and the fp32 kernels of the same inputs: row groups that are full, ragged and of one row, portions that begin inside a sequence,
tiles cut by the window's ends, key lists of blocks and of kept tokens, windows cut into runs."""
import pytest
import torch

from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
PAGE = 64
# portions (rows, first position): tile remainders, a long prefix, a single row among them
STEPS = {"prompts": ([129, 37, 64], [0, 0, 64]), "portions": ([70, 9, 1], [3, 180, 131]), "short": ([5], [0])}


def _step(name, seed):
    lens, starts = STEPS[name]
    ent, r0 = [], 0
    for i, (n, s) in enumerate(zip(lens, starts)):
        ent.append((r0, n, s, i))
        r0 += n
    row_ent = torch.tensor([i for i, e in enumerate(ent) for _ in range(e[1])], dtype=torch.int32)
    pos = torch.tensor([e[2] + k for e in ent for k in range(e[1])], dtype=torch.int32)
    g = torch.Generator().manual_seed(seed)
    bt = (torch.randperm(len(ent) * 3, generator=g) + 1).to(torch.int32).view(len(ent), 3)
    return ent, row_ent, pos, bt, r0, g


def _close(got, want):
    if want.dtype == torch.float32:
        # scores of size up to about 8 from sums of up to 512 products, off by a few 1e-6; weights of fp32
        # exponentials and a weighted mean of values of about one carry that on
        torch.testing.assert_close(got.cpu(), want, rtol=2e-5, atol=2e-5)
        return
    # probabilities and results are rounded to bf16 (2^-9 each) beside values of about one: a weighted
    # mean of values up to 4.5 in size is off by at most 2 * 2^-9 * 4.5 = 1.8e-2
    torch.testing.assert_close(got.cpu().float(), want.float(), rtol=1e-2, atol=1.8e-2)


@pytest.mark.parametrize("step", sorted(STEPS))
@pytest.mark.parametrize("H,G,D,V", [(8, 2, 128, 128), (3, 1, 24, 40), (4, 4, 16, 8), (34, 2, 8, 16),
                                     (4, 2, 136, 200), (16, 1, 64, 256),
                                     # windows alone with both sides of 33 to 128: two sizes, padded ones, groups of 3 and 5
                                     (6, 2, 64, 128), (6, 2, 128, 64), (8, 2, 72, 40), (10, 2, 96, 104)])
@pytest.mark.parametrize("form", ["window", "sink", "biased", "blocks", "kept", "maps"])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_window_attention_tiles(step, H, G, D, V, form, dt):
    ent, row_ent, pos, bt, R, g = _step(step, 3)
    M = 2 if form == "maps" else 1
    win = {"window": 1 << 30, "biased": 1 << 30, "sink": 33, "blocks": 50, "kept": 21, "maps": 40}[form]
    q = torch.randn(R, H * M * D, generator=g).to(dt)
    pool = torch.randn((int(bt.max()) + 1) * PAGE, G * (M * D + V), generator=g).to(dt)
    sink, kw, dev = None, dict(out_scale=0.7), {}
    if form == "sink":
        sink = torch.randn(H, generator=g)
    if form == "biased":
        sink = torch.zeros(H)
        dev.update(dist=(torch.rand(H, generator=g) * 2, torch.rand(H, generator=g) * 0.3),
                   gate=torch.randn(R, H + 3, generator=g).to(dt))
        kw.update(softcap=9.0)
    if form == "blocks":
        dev.update(blk=torch.randn((int(bt.max()) + 1) * sm.blocks_per_page(PAGE, 12), G * (D + V),
                                   generator=g).to(dt), gate=torch.randn(R, H * V, generator=g).to(dt))
        kw.update(every=12, gate_channels=True)
    if form in ("kept", "maps"):
        kw.update(keep=9)
    if form == "maps":
        kw.update(diff=(0.4, 1e-4))
    scale = 1.3 / D ** 0.5
    want = sm.window_attn(q, pool, bt, row_ent, pos, sink, scale, win, torch.empty(R, H * V).to(dt), PAGE, H, G,
                          D, V, **kw, **dev)
    to = lambda t: tuple(x.to(DEV) for x in t) if isinstance(t, tuple) else t.to(DEV) if t is not None else None
    # four wavefronts' rows for bf16, one's for fp32
    rows = (4 if dt == torch.bfloat16 else 1) * sm.window_rows_per_wave(H // G)
    units = sm.make_units(ent, rows).to(DEV)
    dev = {k: to(v) for k, v in dev.items()}
    for max_keys in (None, 700):    # whole key lists / cut into runs
        out = torch.full((R, H * V + 8), 7.0, dtype=dt, device=DEV)
        sm.window_attn(to(q), to(pool), to(bt), to(row_ent), to(pos), to(sink), scale, win, out[:, :H * V], PAGE, H, G,
                       D, V, units=units, unit_rows=rows, max_keys=max_keys, **kw, **dev)
        _close(out[:, :H * V], want)
        assert bool((out[:, H * V:] == 7.0).all())


@pytest.mark.parametrize("step", ["portions", "prompts"])
@pytest.mark.parametrize("H,G,D,V", [(4, 2, 32, 256), (4, 2, 256, 32), (4, 2, 128, 24), (2, 1, 16, 136), (8, 2, 72, 32)])
@pytest.mark.parametrize("form", ["window", "sink", "blocks", "kept", "maps"])
def test_window_attention_tiles_of_one_narrow_side(step, H, G, D, V, form):
    """Tiles of 32 keys whose key or value rows are so short that two wavefronts copy them."""
    test_window_attention_tiles(step, H, G, D, V, form, torch.bfloat16)


@pytest.mark.parametrize("step", sorted(STEPS))    # few and many workgroups: either side of the lines between the kernels
@pytest.mark.parametrize("H,G,D,V", [(8, 2, 192, 128), (8, 2, 132, 40), (16, 16, 260, 72), (16, 8, 512, 256), (16, 16, 200, 136),
                                     (8, 2, 64, 512), (16, 16, 200, 260)])
@pytest.mark.parametrize("form", ["window", "sink", "blocks"])
def test_window_attention_of_long_rows(step, H, G, D, V, form):
    """fp32 keys or values of more than 128 numbers: a wavefront per tile, or all four on it."""
    test_window_attention_tiles(step, H, G, D, V, form, torch.float32)


def test_group_size():
    one = [(i, 1, 5, i) for i in range(8)]
    assert sm.attn_unit_rows(4, one) == 4                     # decoded tokens
    assert sm.attn_unit_rows(4, [(0, 300, 0, 0)]) == 16       # a prompt
    assert sm.attn_unit_rows(4, [(0, 300, 0, 0)] + [(300 + i, 1, 9, i + 1) for i in range(8)]) == 16
    assert sm.attn_unit_rows(4, [(0, 7, 0, 0)]) == 4          # less than half of one group
    assert [sm.attn_unit_rows(1, [(0, n, 0, 0)], 128) for n in (32, 33)] == [1, 4]    # short latents
    assert [sm.attn_unit_rows(1, [(0, n, 0, 0)], 64) for n in (64, 65)] == [1, 4]
    assert sm.attn_unit_rows(1, [(0, 16, 0, 0)], 256) == 4
    # few workgroups: runs of 64 keys; more, or short windows: of 256 where wavefronts share tiles
    assert [sm._key_runs(15, 500, t) for t in (0, 1)] == [8, 8] and sm._key_runs(16, 500, 1) == 2
    assert sm._key_runs(2, 255, 1) == 1 and sm._key_runs(2, 256, 1) == 4 and sm._key_runs(40, 5000, 1) == 12
    q = torch.zeros(2, 8, dtype=torch.bfloat16, device=DEV)
    z = torch.zeros(2, dtype=torch.int32, device=DEV)
    with pytest.raises(ValueError):
        sm.window_attn(q, torch.zeros(64, 16, dtype=torch.bfloat16, device=DEV), z.view(2, 1), z, z, None, 1.0, 1, q,
                       PAGE, 1, 1, 8, 8, units=sm.make_units([(0, 2, 0, 0)], 16).to(DEV), unit_rows=5)


@pytest.mark.parametrize("step", sorted(STEPS))
@pytest.mark.parametrize("H,rank", [(16, 512), (3, 64), (1, 72), (34, 40), (8, 256), (5, 328), (16, 128)])
@pytest.mark.parametrize("win,sunk", [(1 << 30, False), (37, True), (64, False)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_latent_attention_tiles(step, H, rank, win, sunk, dt):
    ent, row_ent, pos, bt, R, g = _step(step, 7)
    qa = torch.randn(H, R, rank + 8, generator=g).to(dt)[:, :, :rank]
    cache = torch.randn((int(bt.max()) + 1) * PAGE, rank, generator=g).to(dt)
    sink = torch.randn(H, generator=g) if sunk else None
    scale = 1.3 / rank ** 0.5
    want = sm.latent_attn(qa, cache, bt, row_ent, pos, sink, scale, win, torch.empty(H, R, rank).to(dt), PAGE)
    rows = (4 if dt == torch.bfloat16 else 1) * sm.latent_rows_per_wave(H)
    units = sm.make_units(ent, rows).to(DEV)
    for max_keys in (None, 700):    # whole windows / cut into runs
        out = torch.full((H, R, rank), 7.0, dtype=dt, device=DEV)
        q2 = torch.empty(H, R, rank + 8, dtype=dt, device=DEV)[:, :, :rank].copy_(qa)
        sm.latent_attn(q2, *(t.to(DEV) for t in (cache, bt, row_ent, pos)), sink.to(DEV) if sunk else None, scale, win,
                       out, PAGE, units=units, unit_rows=rows, max_keys=max_keys)
        _close(out, want)


@pytest.mark.parametrize("step", sorted(STEPS))
@pytest.mark.parametrize("size", [4, 8, 12, 20])
def test_fp32_keys_shorter_than_a_step(step, size):
    """Nothing beside a key's own numbers is read with it: here all of that is not a number."""
    ent, row_ent, pos, bt, R, g = _step(step, 9)
    H, units = 3, None
    q = torch.randn(R, H * size, generator=g)
    top = (int(bt.max()) + 1) * PAGE
    full = torch.full((top, size), float("nan"))
    for r in range(R):      # only the rows that belong to the sequences
        for j in range(int(pos[r]) + 1):
            full[int(bt[int(row_ent[r]), j // PAGE]) * PAGE + j % PAGE] = 0.0
    keep = full[:, 0] == 0.0
    full[keep] = torch.randn(int(keep.sum()), size, generator=g)
    units = sm.make_units(ent, sm.latent_rows_per_wave(H)).to(DEV)
    qa = q.view(R, H, size).transpose(0, 1).contiguous()
    want = sm.latent_attn(qa, full, bt, row_ent, pos, None, 0.5, 40, torch.empty(H, R, size), PAGE)
    out = sm.latent_attn(*(t.to(DEV) for t in (qa, full, bt, row_ent, pos)), None, 0.5, 40,
                         torch.empty(H, R, size, device=DEV), PAGE, units=units)
    _close(out, want)
    pool = torch.cat([full, full[:, :4]], 1).contiguous()    # key of `size`, value of four numbers
    want = sm.window_attn(q, pool, bt, row_ent, pos, None, 0.5, 40, torch.empty(R, H * 4), PAGE, H, 1, size, 4)
    out = sm.window_attn(*(t.to(DEV) for t in (q, pool, bt, row_ent, pos)), None, 0.5, 40,
                         torch.empty(R, H * 4, device=DEV), PAGE, H, 1, size, 4, units=units)
    _close(out, want)


@pytest.mark.parametrize("max_keys", [None, 700])
@pytest.mark.parametrize("what", ["score", "sink"])
def test_fp32_rows_that_are_not_a_number_say_so(what, max_keys):
    """A query, or a sink, that is not a number gives a result that is not one, in its row (head) only."""
    ent, row_ent, pos, bt, R, g = _step("portions", 4)
    H, D = 3, 16
    q, pool = torch.randn(R, H * D, generator=g), torch.randn((int(bt.max()) + 1) * PAGE, 2 * D, generator=g)
    sink = torch.zeros(H)
    if what == "sink":
        sink[1] = float("nan")
    else:
        q[5, D + 2] = float("nan")
    units = sm.make_units(ent, sm.window_rows_per_wave(H)).to(DEV)
    want = sm.window_attn(q, pool, bt, row_ent, pos, sink, 0.3, 40, torch.empty(R, H * D), PAGE, H, 1, D, D)
    out = sm.window_attn(*(t.to(DEV) for t in (q, pool, bt, row_ent, pos, sink)), 0.3, 40, torch.empty(R, H * D, device=DEV),
                         PAGE, H, 1, D, D, units=units, max_keys=max_keys).cpu()
    lost = want.isnan()
    assert lost.any() and torch.equal(lost, out.isnan())
    _close(out[~lost], want[~lost])
