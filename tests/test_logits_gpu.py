"""Logits of untuned shapes on both sides of the wide kernel's rule, against a product in 64 bits."""
import pytest
import torch

from p2p_llm_chat_go_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("M", [1, 15, 16, 17, 48, 64, 70])
@pytest.mark.parametrize("N,K", [(32000, 256), (32128, 1280), (31984, 512), (32000, 288), (16384, 512), (16512, 4096), (20480, 256)])
@pytest.mark.parametrize("norm", [False, True])
def test_logits_by_rows(M, N, K, norm):
    g = torch.Generator(device=DEV).manual_seed(M + K)
    w = (torch.randn(N, K, generator=g, device=DEV) * 0.05).to(torch.bfloat16)
    x = torch.randn(M, K + 16, generator=g, device=DEV).to(torch.bfloat16)[:, 8:8 + K]
    y = ops.skinny_gemm(ops.tile_weight(w), x, ops.EPI_F32, norm=norm)
    xd = x.double()
    ref = xd @ w.double().t()
    if norm:
        ref = ref * torch.rsqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-5)
    # exact products of bf16 numbers, K of them summed in fp32: 2^-24 K |x| |w| at the very most
    bound = 2.0 ** -24 * K * (xd.abs() @ w.double().abs().t()).max()
    assert (y.double() - ref).abs().max() < bound
