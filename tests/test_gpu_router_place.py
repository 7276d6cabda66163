"""Routing of the layer call above 240 tokens where the choice between its two routers
changes (the choice itself is checked on the CPU, sanitize/host_checks.cpp), and rows
that the norm takes element by element (GPU). Routing is compared bit for bit with the
oracle."""

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
# it does not take (the all-VALU router); two halves of 128 experts, the second partial;
# a small router at 511 tokens and one above; the sizes that the all-VALU router keeps,
# and the first after them
@pytest.mark.parametrize(
    "T,D,E,K,I",
    [(241, 512, 32, 4, 128), (300, 2560, 64, 6, 64), (300, 512, 256, 1, 64), (260, 640, 32, 2, 64),
     (500, 768, 176, 8, 64), (511, 512, 64, 4, 64), (601, 512, 64, 4, 64), (512, 2048, 64, 4, 64),
     (513, 2048, 64, 4, 64), (256, 2304, 96, 4, 64), (257, 2304, 96, 4, 64), (1020, 2304, 48, 4, 64),
     (1021, 2304, 48, 4, 64)],
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


def _shifted(t):
    """The same values one element into a storage: not 16-byte aligned."""
    v = torch.zeros(t.numel() + 8, dtype=t.dtype, device=t.device)[1 : 1 + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def test_route_off_alignment(dev):
    """Rows that are not 16-byte aligned take the all-VALU router: the same selections."""
    from kappa_amd.qwen3 import moe_stages

    g = torch.Generator(device="cuda").manual_seed(6)
    x = torch.randn(300, 1024, generator=g, device=dev).to(torch.bfloat16)
    router = (torch.randn(1024, 64, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    want = moe_stages.route(x, router, num_experts=64, k=4, logits=False)
    got = moe_stages.route(_shifted(x), router, num_experts=64, k=4, logits=False)
    for n in ("idx", "w", "hist"):
        assert torch.equal(got[n], want[n]), n


def test_route_underflowing_norms(dev):
    """Router columns whose squares all underflow in f32, with a tie at the K-th place that
    another sum order breaks: expert 9's terms at hidden indices 32..63 are each below
    half an ulp of its running canonical sum and vanish, but summed by themselves
    they lift the logit over a value with few bits. The lower index has to win."""
    from kappa_amd.qwen3 import moe_stages

    T, D, E = 300, 512, 16
    r = np.zeros((D, E), np.float32)
    r[0, [3, 9]] = 2.0**-77 * (1 + 2.0**-7)
    r[1, [3, 9]] = -(2.0**-97)
    r[32:64, 9] = 250 / 256 * 2.0**-101
    x = np.full((T, D), 2.0**30, np.float32)
    lg = oracle.router_logits(x, r)
    assert (lg[:, 3] == lg[:, 9]).all() and (lg[:, 3] > 0).all() and (np.float32(r[0, 3]) ** 2 == 0)
    xd, rd = (torch.from_numpy(a).to(dev).to(torch.bfloat16) for a in (x, r))
    assert torch.equal(xd.float().cpu(), torch.from_numpy(x)) and torch.equal(rd.float().cpu(), torch.from_numpy(r))
    got = moe_stages.route(xd, rd, num_experts=E, k=1, logits=False)
    assert (got["idx"] == 3).all()


@pytest.mark.parametrize("short,shift", [(0, 0), (0, 4), (1, 0)])
def test_route_scratch_forms(dev, short, shift):
    """kmoe_route with its scratch, with one that is not 16-byte aligned, and with one
    that is too small for the two-phase form: the selections of a call without."""
    import ctypes

    from kappa_amd import _lib
    from kappa_amd.qwen3 import moe_stages
    from kappa_amd.qwen3.ffn_moe import _desc, _stream
    from kappa_amd.qwen3.quant import weight_struct

    T, D, E, K = 300, 1024, 64, 4
    g = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn(T, D, generator=g, device=dev).to(torch.bfloat16)
    router = (torch.randn(D, E, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    want = moe_stages.route(x, router, num_experts=E, k=K)
    desc = _desc(T, D, E, K, 1, x.dtype)
    r, keep = weight_struct(router, dev, n_out=E, n_groups=None, name="router_w")
    n = ctypes.c_size_t()
    _lib.check(_lib.lib().kmoe_route_scratch_bytes(desc, ctypes.byref(n)))
    buf = torch.zeros(n.value + 64, dtype=torch.uint8, device=dev)
    got = {k: torch.full_like(want[k], -1) for k in ("idx", "w", "hist")}
    _lib.check(_lib.lib().kmoe_route(desc, x.data_ptr(), r, None, buf.data_ptr() + shift, n.value - short,
                                     got["idx"].data_ptr(), got["w"].data_ptr(), got["hist"].data_ptr(), _stream(dev)))  # fmt: skip
    for k in got:
        assert torch.equal(got[k], want[k]), k
    assert bool(buf.any()) == (not short and not shift)


def test_workspace_off_alignment(dev):
    """A workspace that is not 16-byte aligned (layout-native f32 weights, which ask for no
    alignment of it): the output of an aligned one."""
    import ctypes

    from kappa_amd import _lib
    from kappa_amd.qwen3.ffn_moe import _desc, _stream
    from kappa_amd.qwen3.quant import weight_struct

    T, D, E, K, I = 260, 512, 32, 2, 64
    g = torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn(T, D, generator=g, device=dev).to(torch.bfloat16)
    router = (torch.randn(D, E, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    ws = [torch.randn(*s, generator=g, device=dev) * 0.05 for s in ((E, D, I), (E, D, I), (E, I, D))]
    desc = _desc(T, D, E, K, I, x.dtype)
    n = ctypes.c_size_t()
    _lib.check(_lib.lib().kmoe_workspace_bytes(desc, ctypes.byref(n)))
    buf = torch.zeros(n.value + 64, dtype=torch.uint8, device=dev)
    args = [weight_struct(w, dev, n_out=w.shape[-1], n_groups=None if w is router else E, name="w")
            for w in (router, *ws)]  # fmt: skip
    outs = []
    for shift in (0, 4):
        out = torch.empty_like(x)
        _lib.check(_lib.lib().kmoe_forward(desc, x.data_ptr(), *(a[0] for a in args), None, out.data_ptr(), None, None,
                                           buf.data_ptr() + shift, n.value, _stream(dev)))  # fmt: skip
        outs.append(out)
    assert torch.equal(*outs)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("which", ["x", "scale"])
def test_rms_norm_off_alignment(dev, dtype, which):
    """Rows or a scale that are not 16-byte aligned: the same values bit for bit."""
    from kappa_amd.qwen3 import rms_norm

    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(9, 2048, generator=g, device=dev).to(dtype)
    s = torch.randn(2048, generator=g, device=dev).to(dtype)
    want = rms_norm(x, s)
    got = rms_norm(_shifted(x) if which == "x" else x, _shifted(s) if which == "scale" else s)
    assert torch.equal(got, want)
