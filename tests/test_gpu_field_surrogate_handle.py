"""FAST field updates of a handle that has a surrogate (which keeps the raw
source sums), of one that has none, and of the allocation-free entry point:
E_dyn and B_dyn bit-identical, on lattices whose LOD blocks' cells are the sample
points, on ones of columns of cells, and on blocks too uneven for the
multilevel update."""
import numpy as np
import pytest

import ionsolver_amd as I
from harness import make_config
from ionsolver_amd import Field, FieldMode
from test_zz_no_alloc import hip, inputs, no_alloc, with_handle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,D", [((64, 64, 64), 3), ((128, 128, 128), 4), ((176, 112, 208), 4), ((256, 192, 136), 3),
                                     ((512, 64, 64), 4)], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_fields_with_and_without_a_surrogate(shape, D):
    cfg = make_config(nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D, float_type=2)
    arr = inputs(cfg, np.random.default_rng(sum(shape)))
    e_ref, b_ref = with_handle(cfg, arr, FieldMode.FAST)
    assert np.abs(e_ref - arr["e_stat"]).max() > 0
    e, b = no_alloc(hip(), cfg, arr, FieldMode.FAST)
    np.testing.assert_array_equal(e, e_ref)
    np.testing.assert_array_equal(b, b_ref)
    lbm = I.Lbm(cfg)
    try:
        lbm.surrogate_create(channels=8)
        lbm.set_field_mode(FieldMode.FAST)
        for k, f in (("flags", Field.FLAGS), ("qu_lod", Field.QU_LOD), ("e_stat", Field.E_STAT), ("b_stat", Field.B_STAT)):
            lbm.write_field(f, arr[k])
        lbm.compute_fields()
        np.testing.assert_array_equal(lbm.read_field(Field.E_DYN), e_ref)
        np.testing.assert_array_equal(lbm.read_field(Field.B_DYN), b_ref)
    finally:
        lbm.close()
