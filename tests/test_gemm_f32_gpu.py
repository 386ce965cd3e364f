"""The float32 matrix kernels under the INT4 + LoRA linear, elementwise
against float64 with the bound of a float32 sum.

A sum of n float32 products is within n * 2^-24 * sum |a||b| of the exact one
whatever its order (first order in 2^-24; 2^-23 below leaves room for the
higher ones), and each later product adds its own term. The shapes sit around
the kernels' edges: 16 x 16 and 64 x 64 outputs, K blocks of 32 (taken in turn
by four groups of waves from K = 256 on: last rounds in which some groups have a
part of a block or none, forward and input gradient) and thin steps of 256, odd
K, group scales of 2 (one element at a time), 4 and 64.
"""

from __future__ import annotations

import pytest
import torch

from representax_amd import ops

pytestmark = pytest.mark.gpu
F64 = torch.float64
EPS = 2.0 ** -23


def _exact_weight(packed, scales, k):
    p = packed.to(torch.int32)
    q = torch.stack((p & 15, p >> 4), -1).reshape(p.shape[0], -1)[:, :k]
    q = torch.where(q < 8, q, q - 16).float()
    s = scales.view(torch.bfloat16).float().reshape(p.shape[0], -1)
    return (q * s.repeat_interleave(k // s.shape[1], 1)).to(torch.bfloat16).to(F64)


# (m, k, n, r, group)
SHAPES = [(1, 33, 5, 1, None), (63, 64, 65, 3, 2), (65, 100, 129, 16, 4), (64, 31, 64, 17, None),
          (200, 768, 192, 65, 64), (129, 1, 70, 1, None), (3000, 96, 48, 2, 32),
          (130, 300, 330, 3, 4), (70, 420, 290, 17, None), (67, 261, 259, 1, None)]


@pytest.mark.parametrize("m,k,n,r,group", SHAPES)
def test_float32_linear(m, k, n, r, group):
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n)

    def rnd(*s):
        return torch.randn(s, generator=g, device="cuda")

    packed, scales = ops.int4_pack(rnd(n, k), group)
    x, a, b, gy = rnd(m, k), rnd(r, k), rnd(n, r), rnd(m, n)
    c = 1.5
    y, h = ops.int4lora_forward(x, packed, scales, a, b, scaling=c, group_size=group)
    dx, d_a, d_b = ops.int4lora_backward(gy, x, packed, scales, a, b, h, scaling=c,
                                         group_size=group)
    w = _exact_weight(packed, scales, k)
    xd, ad, bd, gd = (t.to(F64) for t in (x, a, b, gy))
    hd = xd @ ad.t()
    want = {"h": hd, "y": xd @ w.t() + c * (hd @ bd.t()),
            "dx": gd @ w + c * (gd @ bd) @ ad, "dA": c * (gd @ bd).t() @ xd,
            "dB": c * gd.t() @ hd}
    xa, aa, ba, ga, wa = (t.abs() for t in (xd, ad, bd, gd, w))
    ha = xa @ aa.t()
    gb = ga @ ba
    bound = {"h": k * ha, "y": (k + r + 4) * (xa @ wa.t() + c * ha @ ba.t()),
             "dx": (n + r + 4) * (ga @ wa + c * gb @ aa), "dA": (m + n + 4) * c * gb.t() @ xa,
             "dB": (m + k + 4) * c * ga.t() @ ha}
    for name, got in {"h": h, "y": y, "dx": dx, "dA": d_a, "dB": d_b}.items():
        assert got.dtype == torch.float32
        assert ((got.to(F64) - want[name]).abs() <= EPS * bound[name]).all(), name


def test_float32_linear_keeps_infinities_nan_and_tiny_values():
    """Non-finite operands reach exactly the outputs their products reach, and
    products in the subnormal range are kept (no operand is split)."""

    m, k, n, r = 70, 64, 80, 2
    inf = float("inf")
    packed, scales = ops.int4_pack(torch.eye(n, k, device="cuda") * 7.0)
    x = torch.zeros((m, k), device="cuda")
    x[3, 5], x[4, 6], x[66, 63] = inf, float("nan"), 1e-38
    # the adapter passes on column 5 alone, so that its infinity stays one
    a, b = torch.zeros((r, k), device="cuda"), torch.ones((n, r), device="cuda")
    a[:, 5] = 1.0
    w = ops.int4_dequant(packed, scales, k).float()
    y, h = ops.int4lora_forward(x, packed, scales, a, b, scaling=1.0)
    # infinity times the weight's zeros is NaN; column 5 has none
    assert torch.isnan(y[4]).all() and torch.isnan(h[4]).all() and (h[3] == inf).all()
    others = [j for j in range(n) if j != 5]
    assert y[3, 5] == inf and torch.isnan(y[3, others]).all()
    rest = [i for i in range(m) if i not in (3, 4)]
    assert torch.equal(y[rest], x[rest] @ w.t())
    small, _ = ops.int4lora_forward(x[65:] * 1e-4, packed, scales, a, b, scaling=1.0)
    assert torch.equal(small[1, 63], (x[66, 63] * 1e-4) * w[63, 63]) and small[1, 63] != 0


def test_more_tiles_than_one_grid_dimension():
    """2^26 rows and three more are more thin tiles than a launch holds in one
    dimension: the rows around the limits equal a small call's, bit for bit."""

    m, k, n, r = (1 << 26) + 3, 40, 2, 1
    g = torch.Generator(device="cuda").manual_seed(3)
    base = torch.randn((1 << 12, k), generator=g, device="cuda")
    packed, scales = ops.int4_pack(torch.randn((n, k), generator=g, device="cuda"))
    a, b = (torch.randn(s, generator=g, device="cuda") for s in ((r, k), (n, r)))
    want, h_want = ops.int4lora_forward(base, packed, scales, a, b, scaling=1.5)
    x = torch.empty((m, k), device="cuda")
    x[:1 << 26].view(1 << 14, 1 << 12, k).copy_(base.expand(1 << 14, 1 << 12, k))
    x[1 << 26:] = base[:3]
    y, h = ops.int4lora_forward(x, packed, scales, a, b, scaling=1.5)
    for got, part in ((y, want), (h, h_want)):
        for at in (0, 1 << 25, (1 << 26) - (1 << 12)):  # row 0, the second grid row, the last
            assert torch.equal(got[at:at + (1 << 12)], part)
        assert torch.equal(got[1 << 26:], part[:3])
    del x, y, h, got
    torch.cuda.empty_cache()
