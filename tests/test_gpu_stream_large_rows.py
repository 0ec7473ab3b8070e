"""stream_collide of large MHD FP32 lattices whose rows end inside a cache line:
the only ones of such rows that stream past the cache (nontemporal accesses cell
by cell, the +x stores handed over through LDS), against the oracle. The limit in
bytes is read from the source, so that a changed one fails here."""
import os
import re

import numpy as np
import pytest

from harness import compare_all, make_pair

pytestmark = pytest.mark.gpu

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ionsolver_amd", "csrc", "kernels_lbm.hip")


@pytest.mark.parametrize("shape,q,kw", [
    ((136, 144, 160), 19, dict()),
    ((136, 144, 160), 19, dict(relaxation_time=1, charge_inlet=True)),
    ((272, 96, 152), 15, dict(velocity_set=1)),
], ids=["srt", "trt-inlet", "d3q15"])
def test_mhd_fp32_rows_that_stream(shape, q, kw):
    limit = int(re.search(r"SHARED_BYTES = (\d+)ull << 20", open(SOURCE).read()).group(1)) << 20
    assert shape[0] % 64 != 0 and int(np.prod(shape)) * (2 * q + 7) * 4 > limit
    gpu, orc, info = make_pair(np.random.default_rng(sum(shape)), nx=shape[0], ny=shape[1], nz=shape[2], float_type=2,
                               mhd=True, lod_depth=3, **kw)
    try:
        gpu.initialize()
        orc.initialize()
        for _ in range(2):
            gpu.do_time_step()
            orc.do_time_step()
        assert compare_all(gpu, orc, info) == []
    finally:
        gpu.close()
