"""Casts of several tensors in one launch: the same bits as torch's, at the
edges of a thread's eight elements and a workgroup's 2048, and the gradients
of masters that the fused calls cast themselves (GPU)."""

from __future__ import annotations

import pytest
import torch

from representax_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _values(n, seed):
    g = torch.Generator().manual_seed(seed)
    t = torch.randn(n, generator=g) * 10.0 ** torch.randint(-40, 38, (n,), generator=g).float()
    t[: n // 9] = torch.tensor([float("inf"), -0.0, float("-inf"), 1e-45]).repeat(n)[: n // 9]
    return t.to(DEV)


@pytest.mark.parametrize("counts", [(1, 7), (8, 9, 2047), (2048, 2049, 1, 4099), (5,) * 16,
                                    (3,) * 17, (4096,)])
def test_same_bits_as_torch(counts):
    f32 = [_values(n, i) for i, n in enumerate(counts)]
    bf16 = ops.cast_many(f32, torch.bfloat16)
    for t, got in zip(f32, bf16):
        assert torch.equal(got.view(torch.int16), t.to(torch.bfloat16).view(torch.int16))
    nan = ops.cast_many([torch.full((8,), float("nan"), device=DEV)] * 2, torch.bfloat16)
    assert all(t.isnan().all() for t in nan)


def test_views_that_are_not_dense_or_aligned():
    base = _values(4000, 3)
    odd = [base[1:1001], base[::2], base[:64].reshape(8, 8).t(), base[:0]]
    for t, got in zip(odd, ops.cast_many(odd, torch.bfloat16)):
        assert torch.equal(got, t.to(torch.bfloat16))


@pytest.mark.parametrize("m,k,n,rank", [(70, 96, 80, 16), (5, 40, 24, 3), (300, 768, 768, 32)])
def test_master_gradients_are_those_of_the_cast(m, k, n, rank):
    """A float32 master given to the fused call gets what autograd returns
    through an explicit bf16 view of it, bit for bit: also in shapes outside
    the MFMA kernels."""

    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, k, generator=g).to(DEV, torch.bfloat16).requires_grad_(True)
    gy = torch.randn(m, n, generator=g).to(DEV, torch.bfloat16)
    packed, scales = ops.int4_pack(torch.randn(n, k, generator=g).to(DEV))
    a = torch.randn(rank, k, generator=g).to(DEV).requires_grad_(True)
    b = torch.randn(n, rank, generator=g).to(DEV).requires_grad_(True)
    outs = []
    for pair in ((a, b), (a.to(torch.bfloat16), b.to(torch.bfloat16))):
        y = ops.Int4LoRALinearFn.apply(x, *pair, packed, scales, None, 2.0, None)
        outs.append((y.detach(), *torch.autograd.grad(y, [x, a, b], gy)))
    assert outs[0][2].dtype == torch.float32
    assert all(torch.equal(p, q) for p, q in zip(*outs))
