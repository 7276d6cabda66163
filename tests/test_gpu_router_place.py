"""Which router the layer call takes above 240 tokens, and rows that the norm takes
element by element (GPU). Routing is compared bit for bit with the oracle."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from moe_cases import bf16_np, forward_args

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda:0")


# the first size of the two-phase router, with its scratch in the expert buffers; a
# reduction of forty slices; expert buffers smaller than the scratch and a hidden size
# it does not take (the all-VALU router); two halves of 128 experts, the second partial
@pytest.mark.parametrize(
    "T,D,E,K,I",
    [(241, 512, 32, 4, 128), (300, 2560, 64, 6, 64), (300, 512, 256, 1, 64), (260, 640, 32, 2, 64),
     (500, 768, 176, 8, 64)],
)  # fmt: skip
def test_layer_routing_above_the_split_router(dev, T, D, E, K, I):
    from kappa_amd.qwen3 import quantize_weight
    from kappa_amd.qwen3.ffn_moe import _moe_forward

    g = torch.Generator(device="cuda").manual_seed(T + D)
    x = torch.randn(T, D, generator=g, device=dev).to(torch.bfloat16)
    router = (torch.randn(D, E, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    ws = [quantize_weight(torch.randn(*s, generator=g, device=dev) * 0.05) for s in ((E, D, I), (E, D, I), (E, I, D))]
    _, idx, w = _moe_forward(x.reshape(1, T, D), router, *ws, num_experts=E, num_experts_per_tok=K, packed=None,
                             return_routing=True, **forward_args("gather_einsum"))  # fmt: skip
    lg = oracle.router_logits(bf16_np(x), router.float().cpu().numpy())
    oidx, ow = oracle.topk_softmax(lg, K, act_bf16=True)
    np.testing.assert_array_equal(idx.cpu().numpy(), oidx)
    assert np.all(np.abs(w.float().cpu().numpy() - ow) <= 2.0**-8 * np.abs(ow))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("which", ["x", "scale"])
def test_rms_norm_off_alignment(dev, dtype, which):
    """Rows or a scale that are not 16-byte aligned: the same values bit for bit."""
    from kappa_amd.qwen3 import rms_norm

    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(9, 2048, generator=g, device=dev).to(dtype)
    s = torch.randn(2048, generator=g, device=dev).to(dtype)
    want = rms_norm(x, s)

    def shifted(t):
        v = torch.zeros(t.numel() + 8, dtype=t.dtype, device=dev)[1 : 1 + t.numel()].view(t.shape)
        v.copy_(t)
        return v

    got = rms_norm(shifted(x) if which == "x" else x, shifted(s) if which == "scale" else s)
    assert torch.equal(got, want)
