"""Plain bf16 expert weights (the unquantised checkpoint) on the MFMA kernels of
expert_bf16.hip, against the oracle (GPU).

The layer shape has widths that are multiples of 64 but not of the kernels' wider
tiles (128 gate/up columns, 256 down columns) and a reduction that the eight waves
of a decode block split unevenly. Bars as in test_gpu_parity: the routing
bit-exact, outputs within max-abs 2e-2 and mean-rel 1e-3 (f32 sums in another
order than the oracle's move a value to a neighbouring bf16 now and then).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from moe_cases import forward_args, mean_rel

pytestmark = pytest.mark.gpu

D, E, K, I = 320, 8, 3, 192


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch.device("cuda:0")


def _layer(seed: int, T: int):
    rng = np.random.default_rng(seed)
    r = lambda *s, sc=1.0: oracle.bf16_round((rng.standard_normal(s) * sc).astype(np.float32))  # noqa: E731
    return r(T, D), r(D, E, sc=0.1), r(E, D, I, sc=D**-0.5), r(E, D, I, sc=D**-0.5), r(E, I, D, sc=I**-0.5)


def _forward(dev, x, router, ws, impl, capacity=0):
    from kappa_amd.qwen3.ffn_moe import _moe_forward

    return _moe_forward(
        x.reshape(1, -1, D), router, *ws, num_experts=E, num_experts_per_tok=K, packed=None, return_routing=True,
        capacity=capacity, **forward_args(impl),
    )  # fmt: skip


def _dev_bf16(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev).to(torch.bfloat16)


# one 16-row group and its edges, the second group, the largest GEMV batch, the
# grouped GEMM with a nearly empty tile and with several row tiles per expert
@pytest.mark.parametrize("impl", ["gather_einsum", "ragged", "fixed_capacity"])
@pytest.mark.parametrize("T", [1, 15, 17, 47, 64, 65, 171, 400])
def test_bf16_weights(dev, T, impl):
    host = _layer(T, T)
    cap = max(1, T * K // (2 * E)) if impl == "fixed_capacity" else None
    x, router, *ws = (_dev_bf16(a, dev) for a in host)
    out, idx, _ = _forward(dev, x, router, ws, impl, cap or 0)
    ref = oracle.forward(*host, k=K, act_bf16=True, impl=impl, capacity=cap)
    np.testing.assert_array_equal(idx.cpu().numpy(), ref["idx"])
    got = out.reshape(T, D).float().cpu().numpy()
    print(f"max-abs {np.abs(got - ref['out']).max():.2e} mean-rel {mean_rel(got, ref['out']):.2e}")
    assert np.abs(got - ref["out"]).max() <= 2e-2
    assert mean_rel(got, ref["out"]) <= 1e-3


@pytest.mark.parametrize("T", [5, 100])
def test_bf16_weights_off_alignment(dev, T):
    """Weights and activations at addresses that are not 16-byte aligned (a view one
    element into a storage) run on the layout-native kernels, with the same result
    to rounding."""
    host = _layer(7, T)
    ref = oracle.forward(*host, k=K, act_bf16=True, impl="ragged")
    x, router, *ws = (_dev_bf16(a, dev) for a in host)

    def shifted(t):
        s = torch.zeros(t.numel() + 8, dtype=t.dtype, device=dev)
        v = s[1 : 1 + t.numel()].view(t.shape)
        v.copy_(t)
        return v

    for which in range(4):
        args = [shifted(t) if i == which else t for i, t in enumerate((x, *ws))]
        out, idx, _ = _forward(dev, args[0], router, args[1:], "ragged")
        np.testing.assert_array_equal(idx.cpu().numpy(), ref["idx"])
        got = out.reshape(T, D).float().cpu().numpy()
        assert np.abs(got - ref["out"]).max() <= 2e-2 and mean_rel(got, ref["out"]) <= 1e-3, which


@pytest.mark.parametrize("T", [5, 100])
def test_bf16_stage_writes_every_row(dev, T):
    """The stage call computes the rows past an expert's capacity too (the whole call's
    combine is what drops them)."""
    from kappa_amd.qwen3 import moe_stages

    xn, rn, *wn = _layer(T + 1, T)
    x, router, *ws = (_dev_bf16(a, dev) for a in (xn, rn, *wn))
    r = moe_stages.route(x, router, num_experts=E, k=K)
    d = moe_stages.dispatch(r["idx"], r["hist"], num_experts=E, capacity=1)
    assert bool((d["group_sizes"] > 1).any())
    _, y = moe_stages.expert_ffn(x, d, *ws, k=K, impl="fixed_capacity", capacity=1)
    _, ref = oracle.expert_ffn(xn, d["offsets"].cpu().numpy(), d["sorted_token"].cpu().numpy(), *wn, True,
                               impl="fixed_capacity")  # fmt: skip
    got = y.float().cpu().numpy()
    assert np.abs(got - ref).max() <= 2e-2 and mean_rel(got, ref) <= 1e-3


@pytest.mark.parametrize("impl", ["gather_einsum", "ragged"])
@pytest.mark.parametrize("T", [5, 100])
def test_bf16_infinite_weight(dev, T, impl):
    """An infinite down weight gives the infinities of the chain's order, not NaN where h's
    two planes differ in sign or the lower one is zero."""
    xn, rn, *wn = _layer(T + 2, T)
    wn[2][:, 5, 7] = np.inf
    wn[2][1, 6, 9] = np.nan
    ref = oracle.forward(xn, rn, *wn, k=K, act_bf16=True, impl=impl)
    x, router, *ws = (_dev_bf16(a, dev) for a in (xn, rn, *wn))
    out, _, _ = _forward(dev, x, router, ws, impl)
    got = out.reshape(T, D).float().cpu().numpy()
    fin = np.isfinite(ref["out"])
    assert np.isinf(ref["out"][:, 7]).any() and np.isnan(ref["out"][:, 9]).any()
    np.testing.assert_array_equal(got[~fin], ref["out"][~fin])
    assert np.isfinite(got[fin]).all() and mean_rel(got[fin], ref["out"][fin]) <= 1e-3
