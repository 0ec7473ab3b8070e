"""Error of the multilevel field update against the sum in float64, held to what
the code gives, on cubic blocks and on uneven ones up to the most uneven that it
takes (16 x 16 x 5 cells).

Tolerance: the near sources are 26 float additions in a row, sqrt(26 / 3) 2^-24 =
1.8e-7; |r|^2 of a far pair is off by up to 2^2.8 of its rounding (a quarter of it
typically: 1.5e-7 of 1/|r|^3, and as much of the sum of charges of both signs); the
interpolation errs by 5e-8, 5e-8 and 1e-8 on its levels; the far sums round at some
1e-7. Together 2.7e-7 in squares, doubled: 5.4e-7. Two points fewer along the axes of one level
would be 40 times 5e-8 on cubic blocks."""
import numpy as np
import pytest

from test_gpu_field_fast import fields, reference, setup

pytestmark = pytest.mark.gpu
TOL = 5.4e-7


@pytest.mark.parametrize("shape,D", [((128, 128, 128), 3), ((128, 128, 128), 4), ((192, 192, 192), 4), ((128, 128, 40), 3),
                                     ((144, 144, 64), 3), ((120, 168, 72), 3), ((208, 208, 80), 4), ((384, 192, 192), 4)],
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_error_of_the_multilevel_update(shape, D):
    cfg, lod, flags, cells = setup(shape, D, 11)
    got, want = fields(cfg, lod, flags)[:, cells], reference(cfg, lod, cells)
    for name, s in (("E", slice(0, 3)), ("B", slice(3, 6))):
        rel = np.linalg.norm(got[s] - want[s]) / np.linalg.norm(want[s])
        print(name, rel, flush=True)
        assert rel < TOL
