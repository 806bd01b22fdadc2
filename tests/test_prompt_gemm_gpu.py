"""Products of prompts (``ops.seqmix.linear`` above 16 rows, ``linear_unit``) against 64-bit products."""
import pytest
import torch
import torch.nn.functional as F

from p2p_llm_chat_go_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TILES = 14


def _case(M, N, K, ld=None, seed=0, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed + M * 7 + N)
    x = torch.randn(M, ld or K, generator=g, device=DEV).to(dtype)[:, :K]
    return x, (torch.randn(N, K, generator=g, device=DEV) / K ** 0.5).to(dtype)


def _close(got, x, w, b):
    """got = x w^T + b as one rounding to bf16 (2^-8 of the value at most) of fp32 sums of K products and b, whose roundings are
    at most K 2^-24 of what the products' magnitudes sum to."""
    ref = x.double() @ w.double().t() + b.double()
    sums = (x.shape[1] + 1) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    assert bool(((got.double() - ref).abs() <= 2.0 ** -8 * (ref.abs() + sums) + sums).all())


def _tanh_close(got, z):
    """got = tanh of the bf16 numbers z to 2e-6 of it, rounded to bf16: to half of the last of 8 bits."""
    t = torch.tanh(z.double())
    last = torch.exp2(torch.floor(torch.log2(t.abs().clamp(min=2.0 ** -126))) - 7)
    assert bool(((got.double() - t).abs() <= last / 2 * (1 + 2.0 ** -20) + 2e-6 * t.abs()).all())


# rows and columns at the edges of every tile (32 to 256), one 64 of K, fewer stages than a tile keeps, groups of K left over
@pytest.mark.parametrize("tile", range(TILES + 1))
@pytest.mark.parametrize("M,N,K,ld", [(1, 8, 64, 64), (140, 200, 32, 40), (31, 100, 128, 136), (33, 33, 192, 192), (257, 264, 448, 456),
                                      (200, 77, 1088, 1088), (513, 520, 320, 320)])
def test_tiles(tile, M, N, K, ld):
    x, w = _case(M, N, K, ld)
    b = torch.randn(N, device=DEV).bfloat16()
    for shift in (0, 3, 4):   # 16-byte, 2-byte and 8-byte places of the rows
        whole = torch.full((M + 2, N + 16), 9.0, device=DEV, dtype=torch.bfloat16)
        out = whole[1:M + 1, shift:shift + N]
        sm._prompt_gemm(x, w, b, out, tile=tile)
        _close(out, x, w, b)
        z = out.clone()
        sm._prompt_gemm(x, w, b, out, tanh_from=N - 5, tile=tile)
        assert torch.equal(out[:, :N - 5], z[:, :N - 5])
        _tanh_close(out[:, N - 5:], z[:, N - 5:])
        out.fill_(9.0)
        assert bool((whole == 9.0).all())   # nothing beside it was written


def test_tanh_of_every_number():
    """All finite bf16 numbers as products of a row's one 1: around the switch of the two forms at 1/4, at their ends, beyond."""
    every = torch.arange(1 << 16, device=DEV, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    every = every[every.isfinite() & ((every == 0) | (every.abs() >= 2.0 ** -126))]
    n = every.numel() // 64
    z = every[:64 * n].view(64, n)
    out = sm.linear(torch.eye(64, device=DEV).bfloat16(), z.t().contiguous(), tanh_from=0)
    _tanh_close(out, z)
    odd = torch.tensor([float("inf"), float("-inf"), float("nan")], device=DEV).bfloat16().repeat_interleave(16)[:, None]
    x = torch.zeros(48, 64, device=DEV).bfloat16()
    x[:, :1] = odd
    out = sm.linear(x, torch.ones(8, 64, device=DEV).bfloat16(), tanh_from=0).float()
    assert bool((out[:16] == 1).all() and (out[16:32] == -1).all() and out[32:].isnan().all())


@pytest.mark.parametrize("tile", [0] + list(range(2, TILES - 1)))
@pytest.mark.parametrize("act,limit", [("silu", None), ("gelu_tanh", None), ("silu", 1.0)])
def test_units(tile, act, limit):
    M, n, K = 131, 330, 256
    x, w = _case(M, 2 * n, K)
    ref = x.double() @ (3 * w).double().t()
    g, u = ref[:, :n], ref[:, n:]
    if limit is not None:
        g = g.clamp(max=limit)
        want = g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1)
    else:
        want = (F.silu(g) if act == "silu" else F.gelu(g, approximate="tanh")) * u
    out = torch.empty(M, n, device=DEV, dtype=torch.bfloat16)
    sm._prompt_gemm(x, 3 * w, None, out, act=sm.GLU_ACTS[act] if limit is None else 2, limit=limit or 0.0, alpha=sm.FF_ALPHA,
                    tile=tile)
    assert ((out.double() - want).norm() / want.norm()).item() < 2.0 ** -8
    got = sm.linear_unit(x, 3 * w, torch.empty_like(out), act, limit)
    assert ((got.double() - want).norm() / want.norm()).item() < 2.0 ** -8


# fp32 sums of K products: against the library's sums of the same inputs, of which neither has another order's rounding on its
# side (a chain of K / 4 sums each: their errors are alike, and twice the library's is far outside of what orders do)
@pytest.mark.parametrize("tile", range(10))
@pytest.mark.parametrize("M,N,K,ld", [(1, 8, 32, 32), (140, 200, 16, 20), (31, 100, 64, 68), (129, 132, 224, 224), (200, 77, 1056, 1060), (300, 520, 512, 512)])
def test_float32(tile, M, N, K, ld):
    x, w = _case(M, N, K, ld, dtype=torch.float32)
    b = torch.randn(N, device=DEV)
    ref = x.double() @ w.double().t() + b.double()
    lib = ((F.linear(x, w, b).double() - ref).norm() / ref.norm()).item()
    for shift in (0, 1):
        whole = torch.full((M + 2, N + 8), 9.0, device=DEV)
        out = whole[1:M + 1, shift:shift + N]
        sm._prompt_gemm(x, w, b, out, tile=tile)
        assert ((out.double() - ref).norm() / ref.norm()).item() <= 2 * lib + 6e-8
        out.fill_(9.0)
        assert bool((whole == 9.0).all())
    if tile in (1, 7) or N % 2:
        return
    h = N // 2
    want = F.silu(ref[:, :h] - b[:h].double()) * (ref[:, h:] - b[h:].double())
    out = sm._prompt_gemm(x, w, None, torch.empty(M, h, device=DEV), act=0, tile=tile)
    assert ((out.double() - want).norm() / want.norm()).item() < 1e-6


@pytest.mark.parametrize("act,limit", [("silu", None), ("gelu_tanh", None), ("silu", 7.0)])
def test_float32_units_keep_the_bits_of_the_pass(act, limit):
    # rows of one 1: every product is a number of w itself, so what is off is the unit's.  Gates of -40 to 40, where
    # e^-g has lost all bits if its argument was rounded
    n, K, M = 512, 32, 32
    x = torch.eye(K, device=DEV)[:M]
    gate = torch.linspace(-40, 40, n * M, device=DEV).view(n, M)
    if act == "gelu_tanh":
        gate = gate / 8                                       # (z + 0.044715 z^3: beyond 5 nothing but z or 0 is left)
    up = torch.linspace(0.5, 2.0, n * M, device=DEV).view(n, M).flip(0)
    w = torch.cat([gate, up], 0).contiguous()
    g, u = gate.t().double(), up.t().double()
    if limit is not None:
        g = g.clamp(max=limit)
        want, y = g * torch.sigmoid(1.702 * g) * (u.clamp(-limit, limit) + 1), 1.702 * g
    elif act == "silu":
        want, y = g * torch.sigmoid(g) * u, torch.zeros_like(g)
    else:
        y = 2 * (2 / torch.pi) ** 0.5 * (g + 0.044715 * g ** 3)
        want = g * torch.sigmoid(y) * u
    got = sm.linear_unit(x, w, torch.empty(M, n, device=DEV), act, limit)
    # e^-y to 2^-23 of it, the sum, the division and two products each 2^-24 more; where y is formed (not for silu), its own
    # roundings, up to four of 2^-24, reach e^-y by |y|
    bound = (6 + 4 * y.abs()) * 2.0 ** -24 * want.abs() + 1e-37
    assert bool(((got.double() - want).abs() <= bound).all())


def test_rows_and_other_rows():
    x, w = _case(300, 96, 128, 160)
    rows = torch.randint(0, 300, (45,), device=DEV, dtype=torch.int32)
    assert torch.equal(sm.linear(x, w, rows=rows), sm.linear(x[rows.long()].contiguous(), w))
    y = sm.linear(x, w)
    x[7], x[299, 3] = float("inf"), float("nan")   # a row's values reach no other row
    z = sm.linear(x, w)
    keep = [i for i in range(300) if i not in (7, 299)]
    assert torch.equal(z[keep], y[keep]) and not bool(torch.isfinite(z[7]).any())


def test_other_forms_stay_with_the_library():
    x, w = _case(40, 64, 96)                                  # K not in steps of 64
    assert torch.equal(sm.linear(x, w), F.linear(x, w))
    x, w = _case(40, 64, 128, 132)                            # rows that 16-byte copies cannot read
    assert torch.equal(sm.linear(x, w), F.linear(x, w))
    x, w = _case(40, 64, 128)
    for a, b in ((x[:1].expand(40, 128), w), (x, w.t().contiguous().t()), (x.t().contiguous().t(), w), (x[None], w)):
        assert not sm._prompt_gemm_ok(a, b)
        assert torch.equal(sm.linear(a, b), F.linear(a, b))
    w.requires_grad_(True)                                    # whose gradient somebody wants
    sm.linear(x, w).sum().backward()
    assert w.grad is not None
    assert sm.linear(x[:0], w.detach()).shape == (0, 64)


@pytest.mark.parametrize("M", [3, 16, 40])
def test_biases_of_other_shapes(M):
    x, w = _case(M, 64, 128)
    for b in (torch.full((1,), 0.75, device=DEV).bfloat16(), torch.randn(1, 64, device=DEV).bfloat16()):
        assert not sm._bias_ok(b, w, x)
        assert torch.equal(sm.linear(x, w, b), F.linear(x, w, b))
    for b in (torch.randn(63, device=DEV).bfloat16(), torch.randn(65, device=DEV).bfloat16()):
        with pytest.raises(RuntimeError):
            sm.linear(x, w, b)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [3, 40])
def test_tanh_of_the_last_columns(M, dt):
    x, w = _case(M, 64, 128, dtype=dt)
    z = sm.linear(x, w)
    for n in (5, 64, 70):
        y = sm.linear(x, w, tanh_from=-n)
        assert torch.equal(y, sm.linear(x, w, tanh_from=max(0, 64 - n)))
        assert torch.equal(y[:, :max(0, 64 - n)], z[:, :max(0, 64 - n)]) and not torch.equal(y, z)


def test_transforms_and_modes_are_served_as_by_the_library():
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx

    x, w = _case(40, 64, 128, dtype=torch.float32)
    xs = torch.stack([x, 2 * x, -x])
    assert torch.equal(torch.func.vmap(lambda a: sm.linear(a, w))(xs), torch.func.vmap(lambda a: F.linear(a, w))(xs))
    t = torch.randn_like(x)
    y, dy = torch.func.jvp(lambda a: sm.linear(a, w), (x,), (t,))
    assert torch.equal(y, F.linear(x, w)) and torch.equal(dy, F.linear(t, w))
    with forward_ad.dual_level():
        y, dy = forward_ad.unpack_dual(sm.linear(forward_ad.make_dual(x, t), w))
        assert dy is not None and torch.equal(dy, F.linear(t, w))
    assert torch.equal(torch.func.grad(lambda a: sm.linear(a, w).sum())(x), torch.func.grad(lambda a: F.linear(a, w).sum())(x))
    traced = make_fx(lambda a: sm.linear(a, w))(x)            # a trace holds the product, not its result
    assert torch.equal(traced(2 * x), F.linear(2 * x, w))
    traced = torch.jit.trace(lambda a: sm.linear(a, w), (x,), check_trace=False)
    assert torch.equal(traced(2 * x), F.linear(2 * x, w))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert sm.linear(x, w).dtype == torch.bfloat16 == F.linear(x, w).dtype
    rows = torch.arange(3, 23, device=DEV, dtype=torch.int32)
    assert torch.equal(torch.func.vmap(lambda a: sm.linear(a, w, rows=rows))(xs), F.linear(xs[:, 3:23], w))
    assert sm._prompt_gemm_ok(x, w)                           # (nothing of that is left on)
