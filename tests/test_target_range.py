"""The byte ranges of IC-GN's target loads (CPU check of the arithmetic).

The integer pass masks the rows beyond a lane's share by an offset that the
buffer's range check refuses.  It must lie past the range of every image that
the library accepts (65,535 px per side, below 2^31 bytes in all, a ROI down to
the last row but one), and must not wrap with the scalar offset that is added
to it.  0x7fffffff does not: the range exceeds 2^31 there."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

SRC = """
#include "twdic_internal.h"
#include <cstdio>
#include <cstdint>
int main()
{
    int bad = 0;
    long long most = 0;
    for (int64_t stride = 8; stride <= 65535; ++stride) {
        const int64_t h = std::min<int64_t>(65535, (((int64_t)1 << 31) - 1) / stride);     // the tallest image
        const int sy0 = 1, rh = (int)h - 2;
        const int64_t want = (int64_t)(sy0 + rh + 3) * stride;
        const uint32_t got = twdic::target_records(sy0, rh, (int)stride);
        const int64_t at = (int64_t)twdic::kNoOffset;
        if ((int64_t)got != want || at < want || at + stride + 1 >= ((int64_t)1 << 32)) ++bad;
        if (want > most) most = want;
    }
    std::printf("%d %lld\\n", bad, most);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc for the HIP headers")
def test_masked_rows_lie_past_every_image(tmp_path):
    src, exe = tmp_path / "range.hip", tmp_path / "range"
    src.write_text("#include <algorithm>\n" + SRC)
    r = subprocess.run(["hipcc", "-std=c++17", "-O1", "--offload-host-only", f"-I{ROOT / 'include'}",
                        f"-I{ROOT / 'tw_amd' / 'csrc'}", str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60).stdout.split()
    assert int(out[0]) == 0
    assert int(out[1]) > 2 ** 31                        # images whose range an int does not hold are accepted
