"""GPU: weight gradients inside overlapped_wgrad, on the side stream or in
line by their size, accumulate alike in every order.  A bounded delay queued
on the stream that a later step has to wait for keeps its work pending when
that step is issued, and results are read right after the context."""

import pytest
import torch

from eth_amd import kernels as K
from eth_amd.model import functional as Fn
from tests.conftest import announce

pytestmark = pytest.mark.gpu

DELAY = 2_000_000  # clock ticks: 1 ms at 2 GHz, 20 ms at 100 MHz


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
        with torch.cuda.stream(K.side_stream(w.device)):
            torch.cuda._sleep(DELAY)
        with Fn.overlapped_wgrad():
            for o, dy in zip(outs, dys):
                torch.autograd.backward(o, dy)
        got = w.main_grad.clone()
        assert torch.equal(got, want)


def test_join_waits_only_for_new_side_work(cuda):
    announce("side-stream marks")
    mark = K.side_mark()
    with Fn.overlapped_wgrad():
        pass
    assert K.side_mark() == mark
    K.mark_side_launch()
    assert K.side_mark() != mark


@pytest.mark.parametrize("own_stream", [False, True])
@pytest.mark.parametrize("tokens", [64, 4096])
def test_node_of_another_stream_and_nested_contexts(cuda, tokens, own_stream):
    """One weight used by a product on the context's stream (the default one
    or its own) and one on another stream that is behind; an inner context
    that launches nothing leaves the wait to the outer one."""
    announce(f"wgrad streams nested {tokens} own={own_stream}")
    h = 2048
    gen = torch.Generator(device=cuda).manual_seed(tokens)
    xs = [torch.randn(tokens, h, device=cuda, generator=gen).bfloat16() for _ in range(2)]
    dys = [torch.randn(tokens, h, device=cuda, generator=gen).bfloat16() for _ in range(2)]
    want = torch.zeros(h, h, device=cuda)
    for x, dy in zip(xs, dys):
        K.gemm(dy.t(), x, out=want, accumulate=True)
    w = torch.nn.Parameter(torch.randn(h, h, device=cuda, generator=gen).bfloat16())
    w.main_grad = torch.zeros(h, h, device=cuda)
    home = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    for order in ((0, 1), (1, 0)):
        with torch.cuda.stream(home):
            w.main_grad.fill_(7.0)
            w._eth_main_grad_stale = True  # the first contribution stores
            outs = [Fn.LinearFn.apply(xs[0], w, None)]
            other.wait_stream(home)
            with torch.cuda.stream(other):
                outs.append(Fn.LinearFn.apply(xs[1], w, None))
            torch.cuda.synchronize()
            with Fn.overlapped_wgrad():
                # each of the two streams is behind when it is to be waited for
                with torch.cuda.stream(other if order[0] else home):
                    torch.cuda._sleep(DELAY)
                for i in order:
                    torch.autograd.backward(outs[i], dys[i])
                with Fn.overlapped_wgrad():
                    pass
            got = w.main_grad.clone()
            # (the two sums of one pair of products: fp32 addition commutes)
            assert torch.equal(got, want)
        torch.cuda.synchronize()
