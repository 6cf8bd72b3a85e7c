"""GPU parity of causal attention on both sides of the lines where two groups
of waves share a block (forward, dQ, and dK/dV up to a head dim of 96): odd
numbers of rows past whole blocks, odd counts of query blocks for the two groups, query blocks whose second group has no keys for some waves, and grids
just above one workgroup per CU.

Outputs and gradients are held to the bounds of the 16-bit roundings of P and
dS (2^-7 / 2^-6 of the largest magnitude in bf16, two bits less in fp16).  The
row statistics are fp32 throughout: scores of up to 128 products carry at most
128 * 2^-24 of their magnitude (below 2^5), so they are held to 2^-12."""

import math

import pytest
import torch

from eth_amd import kernels as K
from oracle import layer as ol
from tests.conftest import announce

pytestmark = pytest.mark.gpu


def _err(out, ref):
    out, ref = out.float().cpu(), ref.float()
    return (out - ref).abs().max().item() / ref.abs().max().item()


@pytest.mark.parametrize("s,b,n,d,dtype", [
    (512, 1, 2, 64, torch.bfloat16),  # one group
    (513, 1, 2, 64, torch.bfloat16),
    (640, 1, 2, 64, torch.float16),
    (640, 1, 2, 128, torch.float16),
    (777, 1, 3, 96, torch.float16),
    (641, 2, 1, 128, torch.bfloat16),
    (1030, 1, 2, 80, torch.bfloat16),
    (1024, 1, 33, 64, torch.bfloat16),  # 264 workgroups: one group
    (1032, 1, 29, 40, torch.bfloat16),  # 261 workgroups, past 1024 rows: two
])
def test_two_groups_of_waves(cuda, s, b, n, d, dtype):
    announce(f"attention groups {dtype} s={s} b={b} n={n} d={d}")
    gen = torch.Generator().manual_seed(s * n + d)
    qkv = torch.randn(s, b, n, 3 * d, generator=gen).to(dtype)
    dout = torch.randn(s, b, n * d, generator=gen).to(dtype)
    qkv_d = qkv.to(cuda)
    q, k, v = torch.split(qkv_d, d, dim=-1)
    out, lse = K.attention_fwd(q, k, v)
    qr, kr, vr = (t.float().requires_grad_(True) for t in torch.split(qkv, d, dim=-1))
    ref = ol.causal_attention(qr, kr, vr)
    half = 2 if dtype == torch.float16 else 0
    assert _err(out, ref.detach()) < 2.0 ** (-7 - half)
    qb, kb = (t.detach().permute(1, 2, 0, 3).reshape(b * n, s, d) for t in (qr, kr))
    scores = qb @ kb.transpose(1, 2).contiguous() / math.sqrt(d)
    scores.masked_fill_(torch.ones(s, s, dtype=torch.bool).triu(1), float("-inf"))
    want = torch.logsumexp(scores, -1) / math.log(2.0)
    assert (lse.cpu() - want).abs().max().item() < 2.0**-12
    ref.backward(dout.float())
    dqkv = torch.empty_like(qkv_d)
    dq, dk, dv = torch.split(dqkv, d, dim=-1)
    K.attention_bwd(q, k, v, out, dout.to(cuda), lse, dq, dk, dv)
    for name, g, r in (("dq", dq, qr.grad), ("dk", dk, kr.grad), ("dv", dv, vr.grad)):
        assert _err(g, r) < 2.0 ** (-6 - half), name
