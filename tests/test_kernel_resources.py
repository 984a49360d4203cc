"""No kernel of the library uses scratch memory (spilled registers or call
frames): the compiler's own report over every kernel source, with the flags
the library is built with."""
import concurrent.futures as cf
import os
import re
import shutil
import subprocess

import pytest

from gfd_amd import builder


def report(src):
    cmd = [builder.HIPCC, "-x", "hip", "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage"]
    r = subprocess.run(cmd + builder.HIP_FLAGS + builder.INCLUDES + ["-c", src, "-o", os.devnull],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    names = re.findall(r"Function Name: (\S+)", r.stderr)
    scratch = re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", r.stderr)
    assert len(names) == len(scratch)
    return [(os.path.basename(src), n, int(s)) for n, s in zip(names, scratch)]


def test_no_kernel_uses_scratch():
    if shutil.which(builder.HIPCC) is None:
        pytest.skip("hipcc not available")
    srcs = [s for s in builder.sources() if os.sep + "kernels" + os.sep in s] + builder.aql_sources()
    with cf.ThreadPoolExecutor(8) as ex:
        kernels = [k for r in ex.map(report, srcs) for k in r]
    assert len(kernels) >= 20
    assert [k for k in kernels if k[2] != 0] == []
