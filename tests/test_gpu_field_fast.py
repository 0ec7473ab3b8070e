"""The multilevel field update (fast arithmetic, LOD depth 3 and 4) against the
plain sum over the LOD sources in float64, on lattices whose LOD blocks take
each of its paths: cells as sample points (1 to 4 cells a work-item), columns
of 4 to 8 cells, tiles of part of a block's columns, several z groups, uneven
blocks, blocks too uneven for it (direct sum), sources above the domain, few
sources and non-finite ones (direct sum).

Tolerance: a float sum of m <= 4096 terms taken one after the other errs by
about sqrt(m / 3) 2^-24 = 2e-6 of its size when the terms have one sign (the
direct sum), the interpolation by less than 2e-7; the terms here have both
signs."""
import numpy as np
import pytest

import ionsolver_amd as I
from harness import make_config
from ionsolver_amd import Field, FieldMode

pytestmark = pytest.mark.gpu
TOL = 2e-6


def sources(cfg, lod):
    """(indices, centres, charges, velocities) of the sources the field step reads."""
    nd = 1 << cfg.mhd_lod_depth
    b = np.array([cfg.n_x // nd, cfg.n_y // nd, cfg.n_z // nd], np.float64)
    d = np.arange(len(lod) - nd ** 3, len(lod))
    d = d[lod[d, 0] != 0]
    pos = (np.stack([d % nd, d // nd % nd, d // nd ** 2], 1) + 0.5) * b
    return d, pos, lod[d, 0].astype(np.float64), lod[d, 1:].astype(np.float64)


def reference(cfg, lod, cells):
    """E and B sums [6][len(cells)] in float64, the own LOD block left out."""
    nd = 1 << cfg.mhd_lod_depth
    nx, ny, nz = cfg.n_x, cfg.n_y, cfg.n_z
    d, pos, q, v = sources(cfg, lod)
    x, y, z = cells % nx, cells // nx % ny, cells // (nx * ny)
    own = x // (nx // nd) + (y // (ny // nd) + z // (nz // nd) * nd) * nd
    out = np.zeros((6, len(cells)))
    for i, c in enumerate(np.stack([x, y, z], 1).astype(np.float64)):
        k = d != own[i]
        r = c - pos[k]
        t = q[k] / (r * r).sum(1) ** 1.5
        out[:3, i] = (t[:, None] * r).sum(0)
        out[3:, i] = (t[:, None] * np.cross(v[k], r)).sum(0)
    return out


def fields(cfg, lod, flags):
    lbm = I.Lbm(cfg)
    try:
        lbm.write_field(Field.FLAGS, flags)
        lbm.write_field(Field.QU_LOD, lod.reshape(-1))
        lbm.set_field_mode(FieldMode.FAST)
        lbm.compute_fields()
        k = cfg.kernel_constants()
        e, b = lbm.read_field(Field.E_DYN).reshape(3, -1), lbm.read_field(Field.B_DYN).reshape(3, -1)
        return np.concatenate([e.astype(np.float64) / k["ke"], b.astype(np.float64) / k["kmu"]])
    finally:
        lbm.close()


def setup(shape, D, seed, tail=True, share=1.0):
    rng = np.random.default_rng(seed)
    cfg = make_config(nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D, float_type=2)
    n_lod, top = cfg.kernel_constants()["n_lod"], 8 ** D
    lod = (0.05 * rng.standard_normal((n_lod, 4))).astype(np.float32)
    lod[rng.uniform(size=n_lod) >= share, 0] = 0.0
    if not tail:
        lod[top:] = 0.0
    n = int(np.prod(shape))
    flags = np.where(rng.uniform(size=n) < 0.1, 1, 0).astype(np.uint8)
    fluid = np.flatnonzero(flags == 0)
    cells = np.unique(np.concatenate([rng.choice(fluid, 400), fluid[:20], fluid[-20:]]))
    return cfg, lod, flags, cells


def check(cfg, lod, flags, cells):
    got, want = fields(cfg, lod, flags), reference(cfg, lod, cells)
    assert (got[:, flags == 1] == 0).all()  # solid cells are not written
    for s in (slice(0, 3), slice(3, 6)):
        rel = np.linalg.norm(got[s][:, cells] - want[s]) / np.linalg.norm(want[s])
        assert rel < TOL, rel


SHAPES = [((64, 64, 64), 3), ((48, 48, 48), 4), ((64, 80, 48), 4), ((128, 144, 144), 4), ((160, 160, 160), 4),
          ((176, 112, 208), 4), ((240, 336, 144), 4), ((88, 104, 72), 3), ((256, 192, 136), 3), ((112, 96, 608), 4),
          ((512, 64, 64), 4), ((272, 256, 256), 4)]


@pytest.mark.parametrize("shape,D", SHAPES, ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_fast_field_matches_float64_sum(shape, D):
    check(*setup(shape, D, 5))


@pytest.mark.parametrize("share", [0.004, 0.05, 0.2])
def test_few_sources(share):
    check(*setup((160, 128, 144), 4, 6, tail=False, share=share))


@pytest.mark.parametrize("value", [np.nan, np.inf, 1e35])
@pytest.mark.parametrize("shape,D", [((64, 64, 64), 3), ((160, 160, 160), 4)], ids=["leaf", "cells"])
def test_unbounded_sources_take_the_direct_sum(shape, D, value):
    """A NaN or infinite charge reaches every cell but its own block's; a very
    large one leaves the sums finite."""
    cfg, lod, flags, cells = setup(shape, D, 7)
    nd = 1 << D
    d = nd ** 3 - nd - 3
    lod[d] = (value, 0.01, -0.02, 0.03)
    got = fields(cfg, lod, flags)
    n = np.arange(flags.size)
    x, y, z = n % shape[0], n // shape[0] % shape[1], n // (shape[0] * shape[1])
    own = x // (shape[0] // nd) + (y // (shape[1] // nd) + z // (shape[2] // nd) * nd) * nd == d
    fluid = flags == 0
    assert np.isfinite(got[:, fluid & own]).all()
    if np.isfinite(value):
        check(cfg, lod, flags, cells)
    else:
        assert not np.isfinite(got[:3, fluid & ~own]).all(0).any()
