"""The loop of the decode attention over the positions behind its stages, on the device listing: it asks for the key and the
value row of a position and has nothing to choose, also where the new position comes from LDS."""
import os
import re
import subprocess

import pytest


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    from qfactory import native
    out = tmp_path_factory.mktemp("listing") / "decode.s"
    (source,) = [s for s in native.SOURCES if s.endswith("qfactory_decode.hip")]
    flags = [f for f in native.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    hipcc = os.environ.get("QFACTORY_HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-x", "hip", source, "-o", str(out), *flags, f"-I{native.REPO_INCLUDE}", "--offload-device-only", "-S"],
                   check=True, capture_output=True)
    return out.read_text()


def _loops(body):
    """Lines of every loop: from the label that a branch goes back to up to that branch."""
    lines = body.splitlines()
    at = {line.split(":")[0]: i for i, line in enumerate(lines) if line.startswith(".LBB")}
    for i, line in enumerate(lines):
        branch = re.match(r"\s+s_c?branch\S*\s+(\.LBB\w+)", line)
        if branch and at.get(branch[1], i) < i:
            yield lines[at[branch[1]]:i]


@pytest.mark.parametrize("lanes", [4, 8, 16, 32])
@pytest.mark.parametrize("fused", [0, 1])
def test_the_loop_over_positions_does_not_branch(listing, lanes, fused):
    """Two modes of reading (cached, read once) with one loop each: two loads of 16 bytes, no lane mask set, no LDS row beside them."""
    (body,) = re.findall(r"^(_ZN\w*decode_attention_kernelILi%dELb%dE\w*):(.*?)^\.Lfunc_end" % (lanes, fused), listing, re.M | re.S)
    loops = [loop for loop in _loops(body[1]) if any("_load_dwordx4" in line for line in loop)]
    assert len(loops) == 2
    for loop in loops:
        assert sum("_load_dwordx4" in line for line in loop) % 2 == 0
        assert not any(word in line for line in loop for word in ("saveexec", "ds_read", "s_cbranch_exec", "flat_load")), loop
