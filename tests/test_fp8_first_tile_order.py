"""The e4m3 forward whose waves stage their own key tiles has no barrier between a wave's stores to LDS and its reads of what other lanes stored: LDS serves a
wave's requests in the order of the instructions, so the stores have to stand first.  A fence says so to the compiler; this looks at the assembly (device
side only, no GPU needed): all of the first tile's rows are stored before any row is read."""
import os
import re
import subprocess

import pytest

from nvfuserexamples_amd import build as B

SRC = os.path.join(os.path.dirname(B.__file__), "csrc", "fmha_fwd_fp8.hip")


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="needs hipcc")
def test_first_tile_is_stored_before_it_is_read(tmp_path):
    out = tmp_path / "fp8.s"
    subprocess.run([B.HIPCC, *B.HIP_FLAGS, "-S", "--cuda-device-only", SRC, "-o", str(out)], check=True, capture_output=True)
    lines = out.read_text().split("\n")
    seen = 0
    for start, line in enumerate(lines):
        m = re.match(r"^_ZN4fmha19fmha_fwd_fp8_kernelI\w+?Li(64|128)ELb\dELb\dELb1EEE\w+:", line)   # (the last argument: a wave has its own tiles)
        if not m:
            continue
        seen += 1
        body = lines[start:next(i for i in range(start, len(lines)) if lines[i].startswith(".Lfunc_end"))]
        stores = [i for i, l in enumerate(body) if re.match(r"\s+ds_write_b128", l)]
        reads = [i for i, l in enumerate(body) if re.match(r"\s+ds_read_b128", l)]
        rows = 2 * int(m.group(1)) // 16             # 16-byte pieces of K and of V per lane
        assert len([i for i in stores if i < reads[0]]) >= rows, line
    assert seen == 16                                # two output types, two head dims, causal or not, mask or not
