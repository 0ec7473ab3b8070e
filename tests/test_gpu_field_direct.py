"""The FAST direct sum by shifts (the surrogate's training target and judge; fields
without a multilevel plan) is the sum source by source bit for bit: the same
charges with and without further ones too weak to change a sum, which decide
between the two."""
import numpy as np
import pytest

import ionsolver_amd as I
from harness import make_config
from ionsolver_amd import Field
from ionsolver_amd.lbm import FieldMode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,D", [((64, 64, 64), 4), ((80, 112, 48), 4), ((176, 80, 48), 4), ((64, 64, 64), 3), ((88, 56, 72), 3)],
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_raw_sums_do_not_depend_on_the_route(shape, D):
    rng = np.random.default_rng(7)
    n, nd = int(np.prod(shape)), 1 << D
    cfg = make_config(nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D)
    lbm = I.Lbm(cfg)
    try:
        lbm.set_field_mode(FieldMode.FAST)
        flags = np.where(rng.uniform(size=n) < 0.3, 1, 0).astype(np.uint8)
        n_lod = lbm.config.kernel_constants()["n_lod"]
        lo = n_lod - nd ** 3
        lod = np.zeros((n_lod, 4), np.float32)
        some = lo + rng.permutation(nd ** 3)
        few, all_ = some[:nd ** 3 // 2], some[:nd ** 3 * 7 // 8]
        lod[few] = 0.05 * rng.standard_normal((few.size, 4)) + np.array([0.2, 0, 0, 0])
        more = lod.copy()
        more[np.setdiff1d(all_, few)] = (1e-36, 1e-3, -1e-3, 2e-3)
        lbm.write_field(Field.FLAGS, flags)
        lbm.surrogate_create(channels=8)
        out = []
        for q in (lod, more):
            lbm.write_field(Field.QU_LOD, q.reshape(-1))
            lbm.compute_fields()
            out.append(np.concatenate([lbm.read_field(f) for f in (Field.E_DYN, Field.B_DYN)]))
        assert np.abs(out[0]).max() > 0
        assert np.array_equal(out[0], out[1])
    finally:
        lbm.close()
