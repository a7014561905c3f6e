"""Compiled kernels keep what their source asks of the compiler: aligned vector
stores of operator outputs are nontemporal (two stores of one value in both
branches of an alignment test are easily joined into one plain store)."""
import re
import subprocess

import pytest

from hipacc_amd import build as hb


@pytest.mark.parametrize("stem", ["point", "bilateral"])
def test_aligned_vector_stores_are_nontemporal(stem, tmp_path):
    out = tmp_path / f"{stem}.s"
    subprocess.run([hb.HIPCC, *hb.HIP_FLAGS, "-w", "-S", "--offload-device-only",
                    str(hb.CSRC / f"{stem}.hip"), "-o", str(out)], check=True)
    text = out.read_text()
    kernels = re.findall(r"\n(_ZN2hh\d+\w*_kernel\w+):(.*?)\.Lfunc_end", text, re.S)
    assert len(kernels) >= 14
    plain = [name for name, body in kernels
             if not re.search(r"global_store_\w+ [^\n]* nt\b", body)]
    assert not plain, plain
