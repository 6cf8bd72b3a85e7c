"""GPU: the LayerNorm backward at the widths and row counts where its team
split changes, against fp64; the forward's row mean bit for bit in the order
its wave adds.

dx rounds once to 16 bits (2^-9 of a bf16 value; with the residual gradient
the sum of two rounded values rounds again, so twice that of each); its fp32
arithmetic and the fp32 column sums over `rows` rows add at most rows * 2^-23
of the summed magnitudes."""

import numpy as np
import pytest
import torch

from eth_amd import kernels as K
from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 383, 384, 700])
@pytest.mark.parametrize("cols", [2048, 2056, 2560, 3072, 3080, 4096, 4104, 5120, 6144, 6152, 8192])
def test_backward_widths(cuda, rows, cols):
    announce(f"layer norm backward {rows}x{cols}")
    gen = torch.Generator(device=cuda).manual_seed(rows * 31 + cols)
    x, dy, dres = (torch.randn(rows, cols, device=cuda, generator=gen).bfloat16() for _ in range(3))
    gamma = (torch.randn(cols, device=cuda, generator=gen) * 0.1 + 1).bfloat16()
    beta = torch.zeros(cols, device=cuda).bfloat16()
    _y, mean, rstd = K.layer_norm_fwd(x, gamma, beta)
    xd, gd = x.double().requires_grad_(True), gamma.double().requires_grad_(True)
    bd = beta.double().requires_grad_(True)
    torch.nn.functional.layer_norm(xd, (cols,), gd, bd, 1e-5).backward(dy.double())
    for residual in (False, True):
        dg, db = torch.empty(cols, device=cuda), torch.empty(cols, device=cuda)
        got = K.layer_norm_bwd(dy, x, mean, rstd, gamma, dg, db, False, dresid=dres if residual else None,
                               colsum=residual)
        dx, part = got if residual else (got, None)
        want = xd.grad + (dres.double() if residual else 0)
        slack = 2.0**-8 * (want.abs() + (xd.grad.abs() if residual else 0)) + 2.0**-16 * xd.grad.abs().max()
        assert bool(((dx.double() - want).abs() <= slack).all())
        xhat = (x.double() - x.double().mean(1, keepdim=True)) * rstd.double()[:, None]
        for name, have, ref, mag in (("dgamma", dg, gd.grad, (dy.double() * xhat).abs().sum(0)),
                                     ("dbeta", db, bd.grad, dy.double().abs().sum(0))):
            assert bool(((have.double() - ref).abs() <= (rows * 2.0**-23 + 2.0**-18) * mag + 1e-6).all()), name
        if residual:
            sums = K.reduce_partials(part, torch.empty(cols, device=cuda), accumulate=False)
            mag = dx.double().abs().sum(0)
            assert bool(((sums.double() - dx.double().sum(0)).abs() <= rows * 2.0**-23 * mag + 1e-6).all())


@pytest.mark.parametrize("cols", [8, 264, 512, 1536, 2048, 8192])
def test_row_mean_adds_lanes_in_pairs(cuda, cols):
    """A lane adds its columns (eight of every 512) in order; the wave then
    adds lanes 32, 16, 8, 4, 2 and 1 apart, every addition in fp32."""
    rows = 37
    announce(f"layer norm mean order {rows}x{cols}")
    gen = torch.Generator().manual_seed(cols)
    x = (torch.randn(rows, cols, generator=gen) * 2 + 0.5).bfloat16()
    one = torch.ones(cols).bfloat16().to(cuda)
    mean = K.layer_norm_fwd(x.to(cuda), one, one)[1]
    padded = np.zeros((rows, -(-cols // 512) * 512), np.float32)
    padded[:, :cols] = x.float().numpy()
    lanes = np.zeros((rows, 64), np.float32)
    for vec in padded.reshape(rows, -1, 64, 8).transpose(1, 3, 0, 2).reshape(-1, rows, 64):
        lanes = lanes + vec
    for apart in (32, 16, 8, 4, 2, 1):
        lanes = lanes + lanes[:, np.arange(64) ^ apart]
    assert lanes.dtype == np.float32
    assert np.array_equal(mean.cpu().numpy(), lanes[:, 0] / np.float32(cols))
