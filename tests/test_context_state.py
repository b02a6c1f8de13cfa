"""What the kernels read belongs to the context that launches them: the sources
keep no table in a device global, whose contents a device reset would take away
from contexts created after it, and no flag that says it was filled (no GPU)."""
import glob
import os
import re

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_no_device_globals():
    src = sorted(glob.glob(os.path.join(ROOT, "oak_amd", "csrc", "*.h*p*")))
    assert len(src) > 10
    for path in src:
        text = open(path).read()
        assert "hipMemcpyToSymbol" not in text, path
        # a __device__ or __constant__ variable at file scope: no parameter list
        for line in text.splitlines():
            assert not re.match(r"^(static )?__(device|constant)__ [^({]*[\];=]", line), (path, line)
