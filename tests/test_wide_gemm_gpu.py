"""The persistent 256-row GEMM tiles against the other tiles, bit for bit.

Both tiles are forced on shapes with ragged rows and output widths around
their 256-row, 192- and 256-column edges, with one and with more tiles than
workgroups per row, every rank block count and every epilogue. They run the
MFMA sequence of the fused GEMM's tiles, so every output must have the same
bits (the fused tiles are pinned to the oracle elsewhere).
"""

from __future__ import annotations

import pytest
import torch

from representax_amd import ops
from tests.helpers import kernel_names

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
WIDE = [18, 19]
# (m, k, n, rank, group, bias)
SHAPES = [(65, 64, 16, 16, None, True), (255, 128, 184, 16, 64, False),
          (257, 192, 200, 32, None, True), (513, 64, 584, 32, 32, True),
          (66000, 64, 256, 16, None, False)]


def _operands(m, k, n, r, group, bias):
    g = torch.Generator(device="cuda").manual_seed(m + n + r)

    def rnd(*s, scale=1.0):
        return (torch.randn(s, generator=g, device="cuda") * scale).to(BF16)

    packed, scales = ops.int4_pack(rnd(n, k, scale=0.05), group)
    return dict(x=rnd(m, k), packed=packed, scales=scales, a=rnd(r, k, scale=0.1),
                b=rnd(n, r, scale=0.3), gy=rnd(m, n), zy=rnd(m, n, scale=2.0), zx=rnd(m, k, scale=2.0),
                gx=rnd(m, k, scale=2.0),
                bias=rnd(n).view(torch.uint16) if bias else None)


@pytest.mark.parametrize("activation", ["none", "gelu", "silu_mul"])
@pytest.mark.parametrize("m,k,n,r,group,bias", SHAPES)
def test_forward(m, k, n, r, group, bias, activation):
    p = _operands(m, k, n, r, group, bias)

    def run(tile):
        with ops.tuning(int4_tile=tile):
            if activation == "none":
                return ops.int4lora_forward(p["x"], p["packed"], p["scales"], p["a"], p["b"],
                                            scaling=1.7, group_size=group, bias_bits=p["bias"])
            return ops.int4lora_forward_act(
                p["x"], p["packed"], p["scales"], p["a"], p["b"], activation=activation,
                scaling=1.7, group_size=group, bias_bits=p["bias"],
                gate=p["zy"] if activation == "silu_mul" else None)

    want = run(3)
    for tile in WIDE:
        for w, g in zip(want, run(tile)):
            assert torch.equal(w, g), tile


@pytest.mark.parametrize("activation", ["none", "gelu", "silu_mul", "add"])
@pytest.mark.parametrize("m,n,r", [(255, 128, 16), (300, 192, 32), (66000, 64, 16)])
@pytest.mark.parametrize("k", [192, 448])
def test_input_gradient(m, k, n, r, activation):
    p = _operands(m, k, n, r, 64, False)
    h = ops.int4lora_forward(p["x"], p["packed"], p["scales"], p["a"], p["b"], scaling=2.0,
                             group_size=64)[1]

    def run(tile):
        with ops.tuning(bf16_tile=tile):
            if activation == "none":
                return ops.int4lora_backward(p["gy"], p["x"], p["packed"], p["scales"], p["a"],
                                             p["b"], h, scaling=2.0, group_size=64)
            return ops.int4lora_backward_act(
                p["gy"], p["x"], p["packed"], p["scales"], p["a"], p["b"], h,
                activation=activation, z=p["zx"],
                gate=p["gx"] if activation == "silu_mul" else None, scaling=2.0, group_size=64)

    want = run(6)
    for tile in WIDE:
        for w, g in zip(want, run(tile)):
            assert w is None or torch.equal(w, g), tile


def test_without_workspace_takes_the_fused_gemm():
    """A workspace too small for the bf16 weight copy is no error: the call
    falls back to the fused GEMM, which needs none."""

    from representax_amd import _native as nat

    m, k, n, r = 512, 256, 512, 16
    p = _operands(m, k, n, r, None, False)
    want, h_want = ops.int4lora_forward(p["x"], p["packed"], p["scales"], p["a"], p["b"],
                                        scaling=2.0)
    y, h = torch.empty_like(want), torch.empty_like(h_want)
    with ops.tuning(int4_tile=18):
        assert nat.query("rpx_int4lora_forward_workspace", m, n, k, 0, r, nat.DTYPE_BF16) >= 2 * n * k
        nat.call("rpx_int4lora_forward", p["x"].data_ptr(), nat.DTYPE_BF16, m, k,
                 p["packed"].data_ptr(), p["scales"].data_ptr(), n, 0, None, p["a"].data_ptr(),
                 p["b"].data_ptr(), r, 2.0, y.data_ptr(), h.data_ptr(), None, 0,
                 torch.cuda.current_stream().cuda_stream)
    assert torch.equal(y, want) and torch.equal(h, h_want)


@pytest.mark.parametrize("r,wide", [(16, True), (32, True), (24, False)])
def test_automatic_choice(r, wide):
    """Without a forced tile: the large products of rank 16 and 32 run the wide
    kernel, forward and input gradient, and another rank runs none of it, with
    the bits of the forced small tile either way."""

    m, k, n = 16384, 768, 3072
    p = _operands(m, k, n, r, 64, True)

    def forward():
        return ops.int4lora_forward(p["x"], p["packed"], p["scales"], p["a"], p["b"], scaling=1.7,
                                    group_size=64, bias_bits=p["bias"])

    (y, h), names = kernel_names(forward)
    assert any("k_gemm_wide" in name for name in names) == wide
    with ops.tuning(int4_tile=3):
        want, _ = forward()
    assert torch.equal(y, want)

    def backward():
        return ops.int4lora_backward(p["gy"], p["x"], p["packed"], p["scales"], p["a"], p["b"], h,
                                     scaling=1.7, group_size=64)

    got, names = kernel_names(backward)
    assert any("k_gemm_wide" in name for name in names) == wide
    with ops.tuning(bf16_tile=6):
        want = backward()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


# more tiles than the 256 workgroups, so that the load pipeline runs on into a
# second tile, over reductions of two and three 64-deep slices (the stages'
# parity carries over), ragged rows and columns: (m, reduction, forward columns,
# input gradient's columns, rank)
SECOND_TILE = [(257 * 256 + 65, 128, 200, 192, 16), (257 * 256 + 65, 192, 200, 192, 32),
               (130 * 256 + 3, 192, 584, 576, 16)]


@pytest.mark.parametrize("m,k,n,columns,r", SECOND_TILE)
def test_second_tile_of_a_workgroup(m, k, n, columns, r):
    p = _operands(m, k, n, r, 64, True)
    back = _operands(m, columns, k, r, None, False)  # its input gradient reduces over k

    def forward(tile):
        with ops.tuning(int4_tile=tile):
            return ops.int4lora_forward_act(p["x"], p["packed"], p["scales"], p["a"], p["b"],
                                            activation="gelu", scaling=1.7, group_size=64,
                                            bias_bits=p["bias"])

    def backward(tile):
        with ops.tuning(bf16_tile=tile):
            return ops.int4lora_backward_act(back["gy"], back["x"], back["packed"], back["scales"],
                                             back["a"], back["b"], back["gy"][:, :r].contiguous(),
                                             activation="gelu", z=back["zx"], scaling=2.0)

    for run, small in ((forward, 3), (backward, 6)):
        want = run(small)
        for tile in WIDE:
            got, names = kernel_names(lambda: run(tile))
            assert any("k_gemm_wide" in name for name in names), (run.__name__, tile)
            for w, g in zip(want, got):
                assert w is None or torch.equal(w, g), (run.__name__, tile)
