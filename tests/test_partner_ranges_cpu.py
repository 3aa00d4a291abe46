"""The partner ranges of a window link split over a workgroup's wavefronts, from the
engine's own header compiled for the host: for every particle number and split they
cover the partners once, in order, and no range begins or ends past the last one."""
import ctypes
import os
import subprocess

import pytest

from simpimc_amd import build

SOURCE = """
#include "spimc_device.h"
extern "C" int partner_ranges(int N, int qpw, int* out) {
    const int ns = spimc::pair_split<4>(N, qpw);
    for (int k = 0; k < ns; ++k) {
        const int2 q = spimc::pair_range(N, ns, k);
        out[2 * k] = q.x;
        out[2 * k + 1] = q.y;
    }
    return ns;
}
"""


@pytest.fixture(scope="module")
def ranges(tmp_path_factory):
    d = tmp_path_factory.mktemp("ranges")
    (d / "ranges.hip").write_text(SOURCE)
    csrc = os.path.dirname(build.SRC)
    res = subprocess.run([build.HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-shared", "-I", csrc,
                          "-o", str(d / "ranges.so"), str(d / "ranges.hip")], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-2000:]
    fn = ctypes.CDLL(str(d / "ranges.so")).partner_ranges
    out = (ctypes.c_int * 64)()
    return lambda n, qpw: [(out[2 * k], out[2 * k + 1]) for k in range(fn(n, qpw, out))]


@pytest.mark.parametrize("qpw", [64, 128, 256])
def test_ranges_cover_the_partners_once(ranges, qpw):
    for n in range(1, 2200):
        at = 0
        for lo, hi in ranges(n, qpw):
            assert lo == at and lo <= hi <= n, (n, lo, hi)
            at = hi
        assert at == n
