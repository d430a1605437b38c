"""What the compiler made of kernels that keep arrays in registers: an array that is indexed by a
run-time value ends up in private memory, without an error and at several times the cost.
"""
import os
import re
import subprocess

import pytest

from contact_amd import build_lib as B


@pytest.fixture(scope="module")
def resources(tmp_path_factory):
    """{kernel: {resource: value}} of kernels.hip, as the compiler reports them."""
    cmd = [B.HIPCC] + B.FLAGS + ["-Rpass-analysis=kernel-resource-usage", "--offload-device-only", "-c",
                                 os.path.join(B.CSRC, "kernels.hip"), "-o", str(tmp_path_factory.mktemp("o") / "k.o")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = {}
    for line in r.stderr.splitlines():
        m = re.search(r"remark:\s*(.*?): (\S+) \[-Rpass-analysis=kernel-resource-usage", line)
        if m and m.group(1) == "Function Name":
            out[m.group(2)] = cur = {}
        elif m:
            cur[m.group(1)] = m.group(2)
    return out


@pytest.mark.parametrize("kernel", ["k_gsb_walk"])
def test_no_private_memory(resources, kernel):
    found = {k: v for k, v in resources.items() if re.search(r"\d%s[EI]" % kernel, k)}
    assert found
    for name, r in found.items():
        print(name, r)
        assert r["ScratchSize [bytes/lane]"] == "0" and r["VGPRs Spill"] == "0"
