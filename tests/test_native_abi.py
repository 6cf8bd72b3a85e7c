"""CPU: the C-ABI library loads and exports every function include/eth_amd.h
declares; argument validation errors surface as ValueError (no GPU calls)."""

import re
from pathlib import Path

import pytest

from eth_amd import _native as nat

HEADER = Path(__file__).resolve().parents[1] / "include" / "eth_amd.h"


def declared_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"^\s*(?:const\s+)?\w+\s*\*?\s*(eth_\w+)\s*\(", text, flags=re.M)))


def test_header_declares_functions():
    names = declared_functions()
    assert "eth_bucket_pack" in names and "eth_adam_step" in names
    assert len(names) >= 8


def test_library_exports_every_declared_symbol():
    lib = nat.load()
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} declared in eth_amd.h but not exported"
    assert set(declared_functions()) == set(nat.exported_symbols())
    assert lib.eth_abi_version() >= 1


def test_integration_guide_names_every_declared_symbol():
    """The binding guide's export table keeps up with the header: a
    maintainer binding the reference finds every function there."""
    guide = (HEADER.parents[1] / "INTEGRATION.md").read_text()
    missing = [name for name in declared_functions() if f"`{name}`" not in guide]
    assert not missing, f"not in the integration guide: {missing}"


def test_invalid_arguments_raise_value_error_without_gpu():
    with pytest.raises(ValueError, match="unsupported dtype"):
        nat.call("eth_bucket_pack", None, 1, None, 9, None)
    with pytest.raises(ValueError, match="step must be positive"):
        nat.call("eth_adam_step", None, None, 1, 0.9, 0.999, 1e-8, 0, nat.ETH_BF16, None, None, None)
    with pytest.raises(ValueError, match="unscale requires fp32"):
        nat.call("eth_bucket_unpack", None, 1, None, nat.ETH_BF16, 1.0, 0.5, nat.UNPACK_UNSCALE, None, None, 0, None)


def test_struct_layouts_match_header():
    assert nat.CHUNK_DTYPE.itemsize == 40
    assert nat.ADAM_TENSOR_DTYPE.itemsize == 64
    assert nat.ADAM_CHUNK_DTYPE.itemsize == 16
    text = HEADER.read_text()
    assert f"#define ETH_CHUNK_ELEMS {nat.CHUNK_ELEMS}" in text


def test_gemm_plan_covers_the_output():
    """The launches eth_gemm plans: one of three tiles over whole rows or whole
    columns of C, the rest in a second; 256x256 only where that kernel takes
    the C rows."""
    import ctypes
    import random

    def plan(M, N, K, a_k, b_k, ldc, dtype=nat.ETH_BF16):
        out = (ctypes.c_int64 * 4)()
        nat.call("eth_gemm_plan", M, N, K, a_k, b_k, ldc, dtype, out)
        return tuple(out)

    rng = random.Random(7)
    seen = set()
    for _ in range(4000):
        M, N = (int(2 ** rng.uniform(0, 14)) for _ in range(2))
        K = 8 * int(2 ** rng.uniform(0, 11))
        if rng.random() < 0.5:
            N = -(-N // 8) * 8
        a_k, b_k, ldc = rng.randrange(2), rng.randrange(2), N + rng.choice((0, 0, 4, 1))
        tile, m, n, rest = plan(M, N, K, a_k, b_k, ldc)
        assert tile in (64, 128, 256) and 0 < m <= M and 0 < n <= N and (m == M or n == N)
        assert (rest == 0) == ((m, n) == (M, N)) and rest in (0, 64, 128, 256)
        if 256 in (tile, rest):
            assert N % 4 == 0 and ldc % 4 == 0
        if rest:
            assert tile == 256 and m % 256 == 0 or n % 256 == 0
            # whole rounds, but for the last tile row or column of the other side
            assert -(-m // 256) * -(-n // 256) <= -(-M // 256) * -(-N // 256) // 256 * 256
        seen.add((tile, rest > 0, m < M))
    assert {(64, False, False), (128, False, False), (256, False, False), (256, True, True), (256, True, False)} <= seen
    for bad in ((0, 8, 8, 1, 1, 8), (8, 8, 8, 1, 1, 4)):
        with pytest.raises(ValueError):
            plan(*bad)
