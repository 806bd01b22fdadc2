"""Layouts the GEMM kernels rely on (CPU): fragment-major activations (ops.gemm.pack_frag)
and weights (tile_weight) follow the v_mfma_f32_16x16x32_bf16 operand layout."""
import pytest
import torch

from p2p_llm_chat_go_amd.ops import _lib
from p2p_llm_chat_go_amd.ops import gemm as G


def test_pack_frag_layout():
    torch.manual_seed(0)
    M, K = 37, 256
    x = torch.randn(M, K).to(torch.bfloat16)
    xp = G.pack_frag(x)
    assert xp.shape == (48, K)
    flat = xp.reshape(-1, 8)  # 16-byte chunks in (m-tile, k-step, lane) order
    S = K // 32
    for mt in range(3):
        for s in (0, S - 1):
            for lane in (0, 15, 16, 63):
                row, k = 16 * mt + (lane & 15), 32 * s + 8 * (lane >> 4)
                got = flat[(mt * S + s) * 64 + lane]
                want = x[row, k:k + 8] if row < M else torch.zeros(8, dtype=x.dtype)
                assert torch.equal(got, want), (mt, s, lane)


def test_tile_weight_roundtrip():
    w = torch.randn(64, 128).to(torch.bfloat16)
    assert torch.equal(G.untile_weight(G.tile_weight(w)), w)


@pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
@pytest.mark.parametrize("epi", [G.EPI_STORE, G.EPI_RESID, G.EPI_SILU, G.EPI_F32, G.EPI_QKV_ROPE, G.EPI_ARGMAX])
def test_every_width_of_128_columns_has_a_tile(epi):
    """The heuristic gives every shape that tiles (K a multiple of 64, N of 128; SwiGLU: of 256) a tile that is built for
    its epilogue; none is left to the register-staged kernel behind it.  (128 x 192 tiles are not built for SwiGLU:
    feed-forwards of 3072 to 18432 columns whose gate and up divide by 192 were.)"""
    L = _lib.lib()
    for N in range(256 if epi == G.EPI_SILU else 128, 40960, 256 if epi == G.EPI_SILU else 128):
        for M in (1, 64, 65, 100, 128, 129, 192, 193, 200, 256, 257, 300, 384, 385, 512, 513, 640, 641, 768, 1024, 2048, 4100):
            assert L.p2p_prefill_tile(M, N, 1024, epi) > 0, (M, N)
    for ffn, M in ((3072, 1024), (4608, 640), (6144, 400), (6912, 300), (9216, 200), (12288, 200), (18432, 100)):
        assert L.p2p_prefill_tile(M, 2 * ffn, 4096, G.EPI_SILU) not in (0, 9)
    assert L.p2p_prefill_tile(700, 6144, 4096, G.EPI_QKV_ROPE) == 9   # one round of 128 x 192
    assert L.p2p_prefill_tile(700, 6144, 4096, G.EPI_SILU) == 7       # ... and of 192 x 128
    assert L.p2p_prefill_tile(2048, 3072, 1024, G.EPI_RESID) == 6     # short rows: two tiles to a CU
    # long rows: 128 x 256 in two slices of K, in four of 2048 and more, 128 x 128 where they would be shorter or eight
    for M, N, K, tile in ((1024, 4096, 14336, 2), (398, 4096, 14336, 2), (200, 4096, 14336, 3), (700, 4096, 6144, 2),
                          (398, 4096, 6144, 3), (1024, 4096, 4096, 3),
                          # 192 x 128 where 128 x 256 leaves a quarter of the CUs idle, from K = 8192 on
                          (256, 4096, 14336, 3), (257, 4096, 14336, 7), (300, 4096, 14336, 7), (350, 4096, 14336, 7),
                          (384, 4096, 14336, 7), (385, 4096, 14336, 2), (576, 4096, 14336, 2), (577, 4096, 14336, 7),
                          (700, 4096, 14336, 7), (768, 4096, 14336, 7), (769, 4096, 14336, 2), (700, 4096, 8192, 7),
                          (700, 4096, 8128, 2)):
        assert L.p2p_prefill_tile(M, N, K, G.EPI_RESID) == tile, (M, N, K)
    # SwiGLU widths: the tile whose rounds of 256 CUs are the shortest
    for M, N, tile in ((128, 28672, 3), (150, 28672, 7), (250, 28672, 2), (300, 28672, 8), (500, 28672, 1), (700, 28672, 2),
                       (1024, 28672, 1), (300, 22016, 7), (600, 22016, 2), (300, 36864, 2)):
        assert L.p2p_prefill_tile(M, N, 4096, G.EPI_SILU) == tile, (M, N)
    assert L.p2p_prefill_tile(300, 100, 1024, epi) == 0 and L.p2p_prefill_tile(300, 256, 100, epi) == 0


@pytest.mark.skipif(not _lib.available(), reason="kernel library not built")
def test_grouped_product_has_no_scales_of_its_own():
    """Normed grouped products of more than 64 rows write the rows' scales to the caller's buffer and refuse a call without
    one: a buffer inside the library was shared by every stream and device."""
    L = _lib.lib()
    at = 4096   # no launch is reached, so nothing is read
    args = [at, 0, 2, at, at, 128, 1, None, at, 64, 100, 64, 256, G.EPI_SILU, 1, at, 128, 1e-5, 0]
    assert L.p2p_grouped_gemm(*args, None, None) != 0
    args[8] = at + 2   # rows that the scales' wide loads cannot take
    assert L.p2p_grouped_gemm(*args, at, None) != 0


def test_launch_codes_of_few_rows_keep_their_own_size():
    """1, 2, 3-4, 5-8 and 9-16 rows share a 16-row tile but keep a code each; a size that was not tuned takes the
    tile's (the largest tuned in it), and sizes above 16 rows have the tile's alone."""
    w = torch.zeros(16, 8, 16, 32)
    saved = dict(G._TUNE)
    try:
        G._TUNE.clear()
        for M, code in ((1, 11), (2, 12), (16, 16), (48, 48)):
            G.set_tune(G.tune_key(w, M, G.EPI_RESID, False), code, M)
        got = {M: G._code(w, M, G.EPI_RESID, False, 0) for M in (1, 2, 3, 8, 9, 16, 17, 33, 48)}
        assert got == {1: 11, 2: 12, 3: 16, 8: 16, 9: 16, 16: 16, 17: 0, 33: 48, 48: 48}
        assert G._code(w, 1, G.EPI_RESID, False, 7) == 7 and G._code(w, 1, G.EPI_SILU, False, 0) == 0
    finally:
        G._TUNE.clear()
        G._TUNE.update(saved)


def test_a_launch_code_without_rows_holds_for_all_of_its_tile():
    """set_tune(key, code), as a program sets a code of its own, is what every size of the tile runs on, also where the
    tuner has recorded sizes before; other shapes keep theirs."""
    w, other = torch.zeros(16, 8, 16, 32), torch.zeros(8, 8, 16, 32)
    saved = dict(G._TUNE)
    try:
        G._TUNE.clear()
        for v in (w, other):
            for M in (1, 2, 4, 8, 16, 48):
                G.set_tune(G.tune_key(v, M, G.EPI_RESID, False), M, M)
        G.set_tune(G.tune_key(w, 1, G.EPI_RESID, False), 77)
        assert [G._code(w, M, G.EPI_RESID, False, 0) for M in (1, 2, 3, 8, 9, 16, 48)] == [77] * 6 + [48]
        assert [G._code(other, M, G.EPI_RESID, False, 0) for M in (1, 2, 3, 8, 9, 16)] == [1, 2, 4, 8, 16, 16]
        G.set_tune(G.tune_key(w, 2, G.EPI_RESID, False), 5, 2)
        assert [G._code(w, M, G.EPI_RESID, False, 0) for M in (1, 2, 3)] == [5, 5, 5]
    finally:
        G._TUNE.clear()
        G._TUNE.update(saved)


@pytest.mark.parametrize("nq,nkv", [(32, 32), (32, 16), (32, 8), (64, 8), (4, 1), (24, 8)])
def test_query_tiles_by_rows(nq, nkv):
    """v2 tiles of 128 query rows from 128 rows on, of 256 from 512 workgroups on (8 heads per kv head and models with a
    router: 128); other head groups 16 tokens."""
    from p2p_llm_chat_go_amd.ops import attention as A

    G = nq // nkv
    for rows in (1, 127, 128, 500, 1024, 2049, 40000):
        blocks = -(-rows // (256 // G)) * nkv
        many = blocks >= 128
        wide = blocks >= (128 if G == 8 else 512)
        want = 16 if G == 3 else 256 // G if wide else 128 // G if G < 8 and rows >= 128 else 16
        assert A.flash_tile(nq, nkv, rows) == want
        assert A.flash_tile(nq, nkv, rows, routed=True) == (256 // G if G != 3 and many else 16)


@pytest.mark.parametrize("nq,nkv,rows,dense,routed", [
    # query heads, key/value heads, rows of a chunk -> tokens per query tile, of a model without and with a router
    (32, 8, 1, 16, 16), (32, 8, 127, 16, 16), (32, 8, 128, 32, 16), (32, 8, 700, 32, 16), (32, 8, 960, 32, 16),
    (32, 8, 961, 32, 64), (32, 8, 4032, 32, 64), (32, 8, 4033, 64, 64), (32, 8, 8192, 64, 64),
    (32, 32, 127, 16, 16), (32, 32, 128, 128, 16), (32, 32, 768, 128, 16), (32, 32, 769, 128, 256), (32, 32, 3840, 128, 256),
    (32, 32, 3841, 256, 256), (32, 16, 128, 64, 16), (32, 16, 896, 64, 16), (32, 16, 897, 64, 128), (32, 16, 3969, 128, 128),
    (64, 8, 128, 16, 16), (64, 8, 480, 16, 16), (64, 8, 481, 32, 32), (64, 8, 4096, 32, 32), (4, 1, 4096, 32, 16),
    (24, 8, 100, 16, 16), (24, 8, 4096, 16, 16)])
def test_query_tiles_that_kernels_take(nq, nkv, rows, dense, routed):
    """The tile of a prompt's attention on both sides of every line, and what its kernels need: 256 rows of (token, query
    head) at most, 1, 2, 4 or 8 query heads per key/value head above 16 tokens, and room in a captured chunk."""
    from types import SimpleNamespace

    from p2p_llm_chat_go_amd import ops
    from p2p_llm_chat_go_amd.engine.graph import PrefillGraph
    from p2p_llm_chat_go_amd.ops import attention as A

    G = nq // nkv
    for want, r in ((dense, False), (routed, True)):
        tile = A.flash_tile(nq, nkv, rows, r)
        assert tile == want
        assert tile == A.QTILE or (G in (1, 2, 4, 8) and A.QTILE < tile <= ops.kernel_lib().p2p_flash_prefill_tile(nq, nkv)
                                   and tile * G <= 256)
        # a captured chunk of these rows, filled or with dummy rows behind its sequences
        model = SimpleNamespace(device=torch.device("cpu"), nq=nq, nkv=nkv, tp=1, cfg=SimpleNamespace(is_moe=r))
        pages = -(-rows // A.PAGE)
        g = PrefillGraph(model, None, rows, 3, pages, pages * A.PAGE)
        for lens in ([rows], [max(1, rows // 3), rows // 2], [1, 1, 1]):
            chunk = [(b, t, 5) for b, n in enumerate(lens) for t in range(n)][:rows]
            at, n = g.offsets["tiles"]
            tiles = g.host_meta(chunk, [list(range(1, pages + 1))] * 3, [0])[at:at + n].view(-1, 4)
            assert g.qtile == A.flash_tile(nq, nkv, rows, r, 3, pages * A.PAGE * 3 // 4)
            assert int(tiles[:, 1].max()) <= g.qtile and int(tiles[:, 1].sum()) == rows


@pytest.mark.parametrize("nq,nkv,seqs,each,past,tile", [
    # 16-token tiles: short contexts while workgroups x context is 65536 at most (here 512 x 128, 512 x 144) ..
    (32, 8, 20, 44, 0, 16), (32, 8, 8, 33, 0, 16), (32, 8, 1, 192, 0, 16), (32, 8, 1, 193, 0, 32), (32, 32, 2, 128, 0, 16),
    (32, 32, 2, 128, 16, 128), (32, 32, 8, 128, 128, 128),
    # .. and prompts of a tile from 384 workgroups on
    (32, 8, 48, 16, 4000, 16), (32, 8, 47, 16, 4000, 32), (32, 8, 48, 17, 4000, 32), (32, 8, 128, 1, 900, 16),
    # as before: many rows, 8 heads to one
    (32, 8, 256, 17, 0, 64), (64, 8, 60, 8, 0, 16), (64, 8, 61, 8, 0, 32)])
def test_query_tiles_of_short_prompts(nq, nkv, seqs, each, past, tile):
    """The tile by the sequences of a chunk and its longest context; without them as for one long sequence."""
    from p2p_llm_chat_go_amd.ops import attention as A

    assert A.flash_tile(nq, nkv, seqs * each, False, seqs, past + each) == tile
    assert A.flash_tile(nq, nkv, seqs * each, True, seqs, past + each) == A.flash_tile(nq, nkv, seqs * each, True)


@pytest.mark.parametrize("M,N,K,tile", [
    # fewer than 160 tiles of 256 x 256: pairs up to 512 of 128 x 128, 128 x 256 beyond; pairs again ..
    (1024, 8192, 1024, 6), (1536, 6144, 1024, 2), (1280, 8192, 1024, 6), (2048, 8192, 1024, 6), (4096, 6144, 2048, 6), (2560, 4096, 3072, 6),
    # .. phased where K is long enough and its last round fills five of six CUs
    (2048, 8192, 2560, 1), (2048, 8192, 2496, 6), (1500, 8192, 3072, 6), (2800, 5120, 2560, 1), (4096, 6144, 3072, 6),
    (2048, 8192, 3136, 1)])
def test_tiles_of_residual_products_with_a_short_k(M, N, K, tile):
    assert _lib.lib().p2p_prefill_tile(M, N, K, G.EPI_RESID) == tile
