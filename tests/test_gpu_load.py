"""The load-time kernels (quantiser and relayout) at the edges of their tiles (GPU).
Whole results are compared bit for bit."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda:0")


def _shifted(t):
    """The same values one element into a storage: not 16-byte aligned."""
    s = torch.zeros(t.numel() + 16, dtype=t.dtype, device=t.device)
    v = s[1 : 1 + t.numel()].view(t.shape)
    v.copy_(t)
    return v


# rows: inside one sweep, either number of sweeps in registers, and beyond them
# (128 bf16 or 64 f32 rows per sweep, 8 or 16 sweeps); columns: one piece, a
# partial strip, several strips, and a width that the strips do not take
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("rows,cols", [(1, 8), (129, 72), (1024, 64), (1025, 200), (2049, 64), (700, 30)])
def test_quantiser_edges(dev, rows, cols, dtype):
    from kappa_amd.qwen3 import quantize_weight_per_channel

    rng = np.random.default_rng(rows + cols)
    w = (rng.standard_normal((2, rows, cols)) * 0.02).astype(np.float32)
    # exact ties: channels whose scale is a power of two and whose values are n + 1/2 of it
    n = rng.integers(-126, 126, (rows, 4)) + 0.5
    n[0] = 127.0
    w[0, :, :4] = n * 2.0**-9
    w[1, :, 1] = 0.0  # an all-zero channel: the smallest scale
    wt = torch.from_numpy(w).to(dev).to(dtype)
    qo, so = oracle.quantize_per_channel(wt.float().cpu().numpy())
    for t in (wt, _shifted(wt)):
        q, s = quantize_weight_per_channel(t)
        np.testing.assert_array_equal(q.cpu().numpy(), qo)
        np.testing.assert_array_equal(s.cpu().numpy(), so)


@pytest.mark.parametrize("rows", [300, 2300])
def test_quantiser_non_finite(dev, rows):
    """Infinities and NaN against the oracle: NaN does not count for a channel's scale, and
    a quotient that is NaN (which the oracle leaves to C's conversion) quantises to
    -128. Both kernels: aligned, and of any alignment."""
    from kappa_amd.qwen3 import quantize_weight_per_channel

    g = torch.Generator(device=dev)
    g.manual_seed(3)
    w = (torch.randn(1, rows, 64, generator=g, device=dev) * 0.02).to(torch.bfloat16)
    w[0, 5, 0], w[0, 7, 1], w[0, rows - 1, 2], w[0, rows - 2, 3] = float("nan"), float("inf"), float("-inf"), 3e38
    w[0, :, 4] = float("nan")
    w[0, :, 5] *= 1e-37
    wn = w.float().cpu().numpy()
    with np.errstate(invalid="ignore"):
        qo, so = oracle.quantize_per_channel(wn)
        nan = np.isnan(wn / so)
    assert nan.any() and not nan.all()
    for t in (w, _shifted(w)):
        q, s = quantize_weight_per_channel(t)
        np.testing.assert_array_equal(s.cpu().numpy().view(np.int32), so.view(np.int32))
        np.testing.assert_array_equal(q.cpu().numpy(), np.where(nan, -128, qo))


@pytest.mark.parametrize("E,D,I", [(2, 64, 64), (3, 320, 192), (1, 576, 1088)])
def test_prepack_edges(dev, E, D, I):
    """Partial column and k blocks, from sources of any alignment."""
    from kappa_amd.qwen3 import Q8Weight, prepack_moe_experts

    rng = np.random.default_rng(E + D + I)
    qs = [rng.integers(-128, 128, shp).astype(np.int8) for shp in ((E, D, I), (E, D, I), (E, I, D))]
    one = torch.tensor(0.01, device=dev)
    for place in (lambda t: t, _shifted):
        p = prepack_moe_experts(*(Q8Weight(place(torch.from_numpy(q).to(dev)), one) for q in qs))
        w13 = p.w13.cpu().numpy().reshape(E, I // 16, 2, D // 16, 16, 16)
        for which in (0, 1):
            src = qs[which].reshape(E, D // 16, 16, I // 16, 16)
            np.testing.assert_array_equal(w13[:, :, which], src.transpose(0, 3, 1, 4, 2))
        w2 = p.w2.cpu().numpy().reshape(E, D // 16, I // 16, 16, 16)
        np.testing.assert_array_equal(w2, qs[2].reshape(E, I // 16, 16, D // 16, 16).transpose(0, 3, 1, 4, 2))
