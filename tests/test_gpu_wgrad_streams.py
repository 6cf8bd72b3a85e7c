"""GPU: weight gradients inside overlapped_wgrad, on the side stream or in
line by their size, accumulate alike in every order."""

import pytest
import torch

from eth_amd import kernels as K
from eth_amd.model import functional as Fn
from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["small first", "large first"])
def test_one_weight_with_small_and_large_contributions(cuda, order):
    """A weight used by a small and a large product in one backward and in
    successive ones: the in-line product waits for the side stream's."""
    announce(f"wgrad streams {order}")
    h = 2048
    gen = torch.Generator(device=cuda).manual_seed(3)
    small, large = 64, 4096
    assert 2.0 * small * h * h < Fn._SIDE_MIN_FLOPS <= 2.0 * large * h * h
    xs = [torch.randn(t, h, device=cuda, generator=gen).bfloat16() for t in (small, large)]
    dys = [torch.randn(t, h, device=cuda, generator=gen).bfloat16() for t in (small, large)]
    if order == "large first":
        xs, dys = xs[::-1], dys[::-1]
    want = torch.zeros(h, h, device=cuda)
    for x, dy in zip(xs, dys):
        K.gemm(dy.t(), x, out=want, accumulate=True)
    w = torch.nn.Parameter(torch.randn(h, h, device=cuda, generator=gen).bfloat16())
    w.main_grad = torch.zeros(h, h, device=cuda)
    for _ in range(3):
        w.main_grad.zero_()
        outs = [Fn.LinearFn.apply(x, w, None) for x in xs]
        with Fn.overlapped_wgrad():
            for o, dy in zip(outs, dys):
                torch.autograd.backward(o, dy)
        assert torch.equal(w.main_grad, want)


def test_join_waits_only_for_new_side_work(cuda):
    announce("side-stream marks")
    mark = K.side_mark()
    with Fn.overlapped_wgrad():
        pass
    assert K.side_mark() == mark
    K.mark_side_launch()
    assert K.side_mark() != mark
