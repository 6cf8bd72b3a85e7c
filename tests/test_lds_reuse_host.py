"""A wave that stages 16-bit rows in LDS over its own float sums must have a
compiler barrier between the two: the types differ, so nothing else keeps the
stores behind the loads.  Checked in the unoptimised device IR, where accesses
stand in source order."""

import re
import subprocess

import pytest

from eth_amd import build as eb


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("ir") / "attention.ll"
    flags = [f for f in eb.HIPCC_FLAGS if f != "-O3"] + ["-O0", "-Xclang", "-disable-llvm-passes"]
    subprocess.run([eb.hipcc_path(), *flags, f"-I{eb.INCLUDE}", "--cuda-device-only", "-S", "-emit-llvm",
                    str(eb.CSRC / "attention.hip"), "-o", str(out)], check=True, capture_output=True, timeout=100)
    bodies = re.findall(r"^define [^\n]*@(\w+)\([^\n]*\{\n(.*?)^\}", out.read_text(), re.M | re.S)
    return {name: body for name, body in bodies if re.search(r"attn_bwd_dkdv_(x128_)?kernel\w*8AttnArgsE$", name)}


def test_staging_follows_a_fence(kernels):
    bodies = {name: body for name, body in kernels.items() if "store i16" in body}
    two_groups = [n for n in bodies if "Li2EE" in n]
    assert len(bodies) == 20 and len(two_groups) == 8  # two widths (x two group counts), 128; types and padding
    for name, body in bodies.items():
        first_store, last_store = body.index("store i16"), body.rindex("store i16")
        fences = [m.start() for m in re.finditer(r"call [^\n]*wave_lds_fence", body)]
        assert any(at > last_store for at in fences), f"{name}: rows read back without a fence"
        if name in two_groups:
            barrier = body.rindex("__syncthreads", 0, first_store)
            assert any(barrier < at < first_store for at in fences), f"{name}: rows staged without a fence"
