"""Private memory of kernels that were written to need none, from the
compiler's resource report.  A choice between an element of a by-value argument
(or of LDS) and a named zero is one of addresses to the compiler: it then
copies the whole argument to private memory in every lane."""
import os
import re
import subprocess

import pytest

from sternheimergw_amd import build


def _private_bytes(src):
    cmd = [build._hipcc(), *build.HIPCC_FLAGS, *build.FILE_FLAGS.get(src, []), "-c",
           os.path.join(build.CSRC, src), "-o", os.devnull,
           "-Rpass-analysis=kernel-resource-usage"]
    out = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                         check=True).stdout
    names = re.findall(r"Function Name: (\S+)", out)
    sizes = [int(s) for s in re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", out)]
    assert names and len(names) == len(sizes)
    return dict(zip(names, sizes))


@pytest.mark.parametrize("src", ["aaa.hip"])
def test_no_private_memory(src):
    used = {k: v for k, v in _private_bytes(src).items() if v}
    assert not used, used
