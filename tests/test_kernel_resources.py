"""What the compiler reports for kernels that must not use the private stack."""
import re
import subprocess

import pytest

from conftest import ROOT


@pytest.mark.parametrize("source", ["dn_prefill.hip"])
def test_no_private_stack(source):
    """An array indexed by a run-time value goes to scratch memory: every kernel
    here is meant to hold its arrays in registers."""
    from spock_amd import build
    r = subprocess.run([build.HIPCC, *build.FLAGS, "-Rpass-analysis=kernel-resource-usage", "--cuda-device-only", "-c",
                        str(ROOT / "spock_amd" / "csrc" / source), "-o", "/dev/null"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    names = re.findall(r"Function Name: (\S+)", r.stderr)
    sizes = [int(x) for x in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", r.stderr)]
    assert names and len(names) == len(sizes)
    assert not {n: s for n, s in zip(names, sizes) if s}
