"""Where overlapped_wgrad puts weight gradients, and what waits for what: the
streams and the product are stand-ins that record which earlier products each
one is ordered after, so the order is checked without a GPU."""

import contextlib
import itertools
import types

import pytest
import torch

from eth_amd import kernels as K
from eth_amd.grad_sync.streamed import StreamedGradSync
from eth_amd.model import functional as Fn

DEVICE = torch.device("cuda:0")


class Stream:
    """seen: the products that work issued to it from now on is ordered after."""

    def __init__(self, name):
        self.name, self.device, self.seen = name, DEVICE, set()

    def wait_stream(self, other):
        self.seen |= other.seen


class Operand:
    is_cuda, device = True, DEVICE

    def __init__(self, rows, cols):
        self.shape = (rows, cols)

    def numel(self):
        return self.shape[0] * self.shape[1]

    def t(self):
        return Operand(*self.shape[::-1])

    def record_stream(self, stream):
        pass


class Streams:
    """Stand-ins for the current stream, the side stream and the product."""

    def __init__(self, monkeypatch):
        self.main, self.side, self.other, self.third = (Stream(n) for n in ("main", "side", "other", "third"))
        self.now, self.products = self.main, []
        self.of_handle = dict(enumerate((self.main, self.side, self.other, self.third)))
        for handle, stream in self.of_handle.items():
            stream.handle = handle
        monkeypatch.setattr(torch.cuda, "is_initialized", lambda: True)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: self.now)
        monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: self.now.handle, raising=False)
        monkeypatch.setattr(torch.cuda, "default_stream", lambda device: self.main)
        monkeypatch.setattr(torch.cuda, "ExternalStream", lambda handle, device: self.of_handle[handle])
        monkeypatch.setattr(torch.cuda, "stream", self.on)
        monkeypatch.setattr(K, "_side", {DEVICE: self.side})
        monkeypatch.setattr(K, "gemm", self.product)

    @contextlib.contextmanager
    def on(self, stream):
        before, self.now = self.now, stream
        yield
        self.now = before

    def product(self, a, b, out=None, accumulate=False):
        self.products.append((self.now.name, set(self.now.seen)))
        self.now.seen.add(len(self.products) - 1)

    def contribute(self, weight, stream, large):
        tokens = 4096 if large else 64
        with self.on(stream):
            Fn._wgrad(weight, Operand(tokens, 2048), Operand(tokens, 2048), None, True)

    def assert_chain(self):
        for i, (name, seen) in enumerate(self.products):
            assert seen >= set(range(i)), f"product {i} on {name} is ordered after {sorted(seen)} only"


@pytest.fixture
def streams(monkeypatch):
    return Streams(monkeypatch)


STEPS = list(itertools.product(("main", "other", "third"), (False, True)))


@pytest.mark.parametrize("first", STEPS)
def test_contributions_to_one_weight_are_ordered(monkeypatch, first):
    """Three contributions from nodes of any streams and sizes: each after
    the ones before it, and all before what follows the context."""
    for second, third in itertools.product(STEPS, repeat=2):
        streams, weight = Streams(monkeypatch), types.SimpleNamespace()
        with Fn.overlapped_wgrad():
            for name, large in (first, second, third):
                streams.contribute(weight, getattr(streams, name), large)
        streams.assert_chain()
        assert streams.main.seen == {0, 1, 2}


def test_small_products_stay_on_the_stream_of_the_context(streams):
    weight = types.SimpleNamespace()
    with Fn.overlapped_wgrad():
        streams.contribute(weight, streams.main, False)
        streams.contribute(weight, streams.main, True)
        streams.contribute(weight, streams.other, False)
    streams.contribute(weight, streams.other, False)  # outside: in line
    assert [name for name, _ in streams.products] == ["main", "side", "side", "other"]


@pytest.mark.parametrize("outer_large,inner_large", itertools.product((False, True), repeat=2))
def test_nested_contexts(streams, outer_large, inner_large):
    """An inner context on another stream: its exit and the outer one's each
    cover what was issued before them."""
    weight = types.SimpleNamespace()
    with Fn.overlapped_wgrad():
        streams.contribute(weight, streams.main, outer_large)
        with streams.on(streams.other):
            with Fn.overlapped_wgrad():
                streams.contribute(weight, streams.other, inner_large)
            assert streams.other.seen >= {0, 1}
        streams.contribute(weight, streams.main, outer_large)
        with Fn.overlapped_wgrad():
            pass  # launches nothing: the outer exit still has to wait
    streams.assert_chain()
    assert streams.main.seen == {0, 1, 2}
    assert not Fn._overlap["wgrad"]


def test_exit_on_another_stream(streams):
    weight = types.SimpleNamespace()
    context = Fn.overlapped_wgrad()
    context.__enter__()
    streams.contribute(weight, streams.main, False)
    streams.contribute(types.SimpleNamespace(), streams.main, True)
    with streams.on(streams.other):
        context.__exit__(None, None, None)
    assert streams.other.seen == {0, 1}


def test_contexts_of_two_threads_that_end_in_either_order(streams):
    first, second = Fn.overlapped_wgrad(), Fn.overlapped_wgrad()
    first.__enter__()
    with streams.on(streams.other):
        second.__enter__()
    first.__exit__(None, None, None)
    weight = types.SimpleNamespace()
    with streams.on(streams.other):
        streams.contribute(weight, streams.other, False)
        second.__exit__(None, None, None)
    assert streams.other.seen == {0}
    streams.contribute(weight, streams.main, True)  # outside every context: in line
    assert streams.products[-1][0] == "main"


def test_streamed_sync_waits_for_products_in_line(streams):
    """A bucket completed by a node of another stream is synced after the
    products that stayed on the stream of the step."""
    sync = StreamedGradSync.__new__(StreamedGradSync)
    sync.device, sync.stream, sync.buckets, sync.launched = DEVICE, streams.third, [[]], [False]
    sync.where, sync.params = {}, {}
    sync.ex = types.SimpleNamespace(begin=lambda scale: None, run_bucket=lambda b: None)
    sync.start()
    with Fn.overlapped_wgrad():
        streams.contribute(types.SimpleNamespace(), streams.main, False)
        streams.contribute(types.SimpleNamespace(), streams.other, True)
        with streams.on(streams.other):
            sync._launch(0)
    assert sync.stream.seen == {0, 1}
