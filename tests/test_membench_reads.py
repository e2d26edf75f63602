"""The LDS microbenchmark reads what it is named for: one instruction per read.

Where a part of a vector is not used, the compiler leaves it out of the read (a
16-byte one becomes two reads of a word), and the figure is not that width's.
Checked on the device assembly of splotch_amd/csrc/membench.hip; needs no GPU.
"""
import os
import re
import subprocess

import pytest

from splotch_amd import build


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_lds_reads_have_their_width(tmp_path):
    out = tmp_path / "membench.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "-S", "--cuda-device-only",
                    os.path.join(build.CSRC, "membench.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text()
    bodies = re.findall(r"^(_Z\w*k_lds_read\w*):(.*?)s_endpgm", text, re.S | re.M)
    assert len(bodies) == 6
    for name, body in bodies:
        width = {"j1E": "b32", "j2E": "b64", "j4E": "b128"}[re.search(r"j[124]E", name).group()]
        reads = re.findall(r"\bds_read\w+", body)
        assert reads == ["ds_read_" + width] * 16, (name, reads)
