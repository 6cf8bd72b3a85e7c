"""The embedding backward's key workspace belongs to one call: two calls that
overlap on the host (two threads, or a call issued from another's launch) must
not sort into the same memory, since the first's rows are added from its keys."""

import torch

from eth_amd import _native as nat
from eth_amd import kernels as K


def test_overlapping_calls_have_their_own_keys(monkeypatch):
    tokens = torch.zeros(2, 8, dtype=torch.int64)
    dout = torch.zeros(8, 2, 16, dtype=torch.bfloat16)
    keys = []

    def call(name, *args):
        assert name == "eth_embedding_bwd"
        workspace = args[5]
        assert workspace not in keys, "a pending call's keys are there"
        keys.append(workspace)
        if len(keys) < 3:  # another thread's call before this one's launches
            K.embedding_bwd(tokens, tokens, dout, torch.zeros(4, 16), torch.zeros(4, 16))

    monkeypatch.setattr(K, "_check_half", lambda *ts: nat.ETH_BF16)
    monkeypatch.setattr(K, "_check_ids", lambda *a: None)
    monkeypatch.setattr(nat, "value", lambda name, *args: 2 * 4 * 16)
    monkeypatch.setattr(nat, "call", call)
    monkeypatch.setattr(nat, "stream_ptr", lambda device=None: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: type("S", (), {"cuda_stream": 0}))
    K.embedding_bwd(tokens, tokens, dout, torch.zeros(4, 16), torch.zeros(4, 16))
    assert len(keys) == 3
