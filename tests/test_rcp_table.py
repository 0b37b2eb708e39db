"""The raster kernel's test for hidden records (pf_device.hip, hidden_behind)
allows the emulated x86 reciprocal a relative error of 2^-10; every entry of
its table is within 2^-11 over the whole interval of mantissas it stands
for."""
import os
import re
from fractions import Fraction as F


def test_x86_reciprocal_table_error():
    text = open(os.path.join(os.path.dirname(__file__), "..", "include", "pf_x86_approx.h")).read()
    body = re.search(r"pf_rcp_table\[[^\]]*\]\s*=\s*\{([^}]*)\}", text).group(1)
    table = [int(v, 0) for v in re.findall(r"0x[0-9a-fA-F]+|\d+", body)]
    assert len(table) == 2048
    for i, t in enumerate(table):
        r = F(4096 + t, 8192)                    # for 1 <= x < 2: exponent 253 - 127, 12 mantissa bits
        for x in (F(2048 + i, 2048), F(2048 + i + 1, 2048)):
            assert abs(r * x - 1) <= F(1, 2048), (i, t)
