"""ion_update_e_b_noalloc captured in a HIP graph: each replay, with other LOD sums
in the buffers than at the capture and the program's own work in between, leaves
the fields of an eager call. Which kernels do the update is decided on the GPU by the
charges (all blocks, half of them, few of them, one not finite)."""
import ctypes

import numpy as np
import pytest
import torch

import ionsolver_amd as I
from harness import make_config
from ionsolver_amd import FieldMode
from test_zz_no_alloc import _FieldBuffers, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [FieldMode.FAST, FieldMode.EXACT], ids=lambda m: m.name)
@pytest.mark.parametrize("shape,D", [((64, 64, 64), 3), ((160, 96, 112), 4), ((32, 32, 32), 2)],
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_replays_match_eager_calls(shape, D, mode):
    cfg = make_config(nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D, float_type=2)
    rng = np.random.default_rng(3)
    arr = inputs(cfg, rng)
    buf = {k: torch.from_numpy(v).cuda() for k, v in arr.items()}
    n = int(np.prod(shape))
    for k in ("e_dyn", "b_dyn"):
        buf[k] = torch.zeros(3 * n, device="cuda")
    ptr, c, lib = _FieldBuffers(**{k: v.data_ptr() for k, v in buf.items()}), cfg._to_c(), I.load_library()

    def call():
        stream = torch.cuda.current_stream().cuda_stream
        assert lib.ion_update_e_b_noalloc(ctypes.byref(c), ctypes.byref(ptr), int(mode), stream) == 0

    lods = []
    for share, value in ((1.0, None), (0.5, None), (0.01, None), (1.0, float("nan"))):
        lod = (0.05 * rng.standard_normal((arr["qu_lod"].size // 4, 4))).astype(np.float32)
        lod[rng.uniform(size=len(lod)) >= share, 0] = 0.0
        if value is not None:
            lod[len(lod) // 2, 0] = value
        lods.append(torch.from_numpy(lod.reshape(-1)).cuda())
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for lod in lods + lods[::-1]:
        buf["qu_lod"].copy_(lod)
        out = []
        for run in (graph.replay, call):
            buf["e_dyn"].zero_()
            buf["b_dyn"].zero_()
            run()
            out.append(torch.cat([buf["e_dyn"], buf["b_dyn"]]).cpu().numpy())
            torch.cuda.synchronize()
        assert np.abs(out[0][np.isfinite(out[0])]).max() > 0
        np.testing.assert_array_equal(out[0], out[1])
