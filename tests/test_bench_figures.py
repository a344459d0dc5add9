"""What bench.py reads from the committed counter run of a workload."""
import os
import re

import bench


def test_the_roofline_is_of_instructions_issued():
    """Per launch: VALU instructions (the roofline's numerator), time and HBM bytes; no more than the issue
    rate allows."""
    for workload in ("csg256_L10_1920x1080", "capsules64_L9_1024"):
        traffic, path, us, valu = bench.profiled_traffic(workload, "compiled")
        text = open(os.path.join(bench.ROOT, path)).read()
        assert valu == float(re.search(r"^\s+SQ_INSTS_VALU\s+([\d.]+)$", text, re.M).group(1))
        assert traffic > 0 and us > 0
        assert 0 < valu * 64 / us * 1e-6 < bench.PEAK_VALU_UNPACKED_TOPS
    assert bench.profiled_traffic("csg256_L10_1920x1080", "interpreter") == (None,) * 4
    assert bench.profiled_traffic("no such workload", "compiled") == (None,) * 4
