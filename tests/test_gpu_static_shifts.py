"""Static fields summed by shifts (precompute_B, precompute_E), bit-identical to
the oracle's loops over every cell: rows whose length is no multiple of four,
more than one tile of columns, sources in every place of a group of four, more
than one window of rows and of columns, two meshes side by side with different
values, non-finite ones; and, source by source, values that change from cell to
cell and a small lattice."""
import numpy as np
import pytest

import ionsolver_amd as I
import oracle_lib as O
from harness import make_config
from ionsolver_amd import Field

pytestmark = pytest.mark.gpu


def cells(shape):
    z, y, x = np.meshgrid(*(np.arange(n) for n in shape[::-1]), indexing="ij")
    return x.ravel(), y.ravel(), z.ravel()


def sources(kind, shape, rng):
    """(mask, value index) of the source cells."""
    x, y, z = cells(shape)
    nx, ny, nz = shape
    if kind == "box":
        return (x >= 1) & (x < nx - 2) & (y >= 1) & (y < ny - 1) & (z >= nz // 3) & (z < nz // 3 + max(3, nz // 3)), np.zeros(x.size, int)
    if kind == "ring":
        r = np.hypot(x - 0.5 * nx, z - 0.5 * nz)
        return (r > 0.2 * min(nx, nz)) & (r < 0.42 * min(nx, nz)) & (y > 1) & (y < ny - 2), np.zeros(x.size, int)
    if kind == "two":  # touching along x, in the middle of a group of four
        return (y > 0) & (y < ny - 1) & (z % 3 == 1), (x >= nx // 2).astype(int)
    if kind == "dots":
        return rng.uniform(size=x.size) < 0.6, np.zeros(x.size, int)
    return rng.uniform(size=x.size) < 0.2, rng.integers(0, 50, x.size)  # "noise"


@pytest.mark.parametrize("kind", ["box", "ring", "two", "dots", "noise"])
@pytest.mark.parametrize("shape", [(34, 61, 32), (150, 48, 10), (16, 41, 101), (9, 11, 7)], ids=lambda s: "x".join(map(str, s)))
def test_static_fields_match_the_oracle(shape, kind):
    check(shape, kind, 1.0)


@pytest.mark.parametrize("scale", [1e-20, np.inf, np.nan])
def test_values_outside_the_specialised_range(scale):
    check((42, 40, 40), "two", scale)


def check(shape, kind, scale):
    rng = np.random.default_rng(17)
    n = int(np.prod(shape))
    mask, which = sources(kind, shape, rng)
    values = (rng.standard_normal((50, 3)) * np.array([1.0, 2.0, 0.5])).astype(np.float32)
    values[0] *= np.float32(scale)
    for flag in (0x11, 0x05):
        flags = np.where(mask, flag, 0).astype(np.uint8)
        flags[rng.choice(np.flatnonzero(~mask), 3)] = 0x01
        b_dyn = np.zeros((3, n), np.float32)
        b_dyn[:, mask] = values[which[mask]].T
        b_dyn = b_dyn.reshape(-1)
        lbm = I.Lbm(make_config(nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=0, eqb=False, vforce=True))
        try:
            k = lbm.config.kernel_constants()
            lbm.write_field(Field.FLAGS, flags)
            lbm.write_field(Field.B_DYN, b_dyn)
            b_stat, e_stat = np.zeros(3 * n, np.float32), np.zeros(3 * n, np.float32)
            with np.errstate(all="ignore"):
                if flag == 0x11:
                    lbm.precompute_b()
                    psi = O.precompute_b(shape, flags, b_dyn, b_stat, k["kmu0"])
                    if psi.size <= 3 * n:
                        assert np.array_equal(lbm.read_field(Field.E_DYN)[:psi.size], psi, equal_nan=True)
                    assert np.array_equal(lbm.read_field(Field.B_STAT), b_stat, equal_nan=True)
                else:
                    lbm.precompute_e()
                    O.precompute_e(shape, flags, b_dyn, e_stat, k["ke"])
                    assert np.array_equal(lbm.read_field(Field.E_STAT), e_stat, equal_nan=True)
        finally:
            lbm.close()
