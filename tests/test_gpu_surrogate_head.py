"""The head's 128-column tiles whose wavefronts share a row's interpolation along x
(blocks of 16 and 4 cells along x), and those that cannot (12 cells; components
of 192 columns), as the other shapes of the float64 comparison."""
import pytest

from test_gpu_surrogate import test_forward_loss_and_gradients_vs_float64_reference as compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(128, 64, 64), (32, 64, 64), (96, 64, 32), (96, 32, 32)], ids=lambda s: "x".join(map(str, s)))
def test_head_columns(shape):
    compare(shape, 0.1)
