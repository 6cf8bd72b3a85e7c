"""GPU: the embedding backward's sort and run sums at the edges of its key
tiles, key groups and row batches, bit for bit against the ordered oracle."""

import numpy as np
import pytest
import torch

from eth_amd import kernels as K
from oracle import layer as ol
from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,s", [(1, 1), (1, 3), (3, 11), (1, 32), (2, 129), (5, 819), (1, 4096), (1, 4097), (3, 2731)])
def test_runs_match_the_ordered_oracle(cuda, b, s):
    V, P, h = 97, s, 24
    announce(f"embedding runs {b}x{s}")
    rng = np.random.default_rng(b * 10007 + s)
    tokens = rng.integers(0, V, (b, s))
    # runs of 15, 16, 17, 32 and 33 rows, one of a third of all rows, and ids
    # outside the table (clamped)
    flat = tokens.reshape(-1)
    for k, n in enumerate((15, 16, 17, 32, 33)):
        if flat.size > 400:
            at = rng.choice(flat.size, n, replace=False)
            flat[flat == 40 + k] = 0
            flat[at] = 40 + k
    flat[rng.random(flat.size) < 1 / 3] = 7
    if flat.size > 2:
        flat[0], flat[-1] = -5, V + 3
    positions = np.broadcast_to(np.arange(s), (b, s)).copy()
    dout = torch.from_numpy(rng.standard_normal((s, b, h)).astype(np.float32)).bfloat16()
    word = rng.standard_normal((V, h)).astype(np.float32)
    pos = rng.standard_normal((P, h)).astype(np.float32)
    dword, dpos = torch.from_numpy(word.copy()).to(cuda), torch.from_numpy(pos.copy()).to(cuda)
    K.embedding_bwd(torch.from_numpy(tokens).to(cuda), torch.from_numpy(positions).to(cuda), dout.to(cuda), dword, dpos)
    ol.embedding_grad_ordered(tokens, positions, dout.float().numpy(), word, pos)
    assert np.array_equal(dword.cpu().numpy(), word)
    assert np.array_equal(dpos.cpu().numpy(), pos)
