"""The ways stream_collide reaches its DDFs (lattices that stay in the cache, rows
of whole wavefronts, other rows), against the oracle; cells whose forces
and densities are NaN or leave the formats' range (of infinite ones the oracle's
products with zero direction components are NaN and the kernels' sums are not); and the codes of every finite value."""
import numpy as np
import pytest

import oracle_lib as O
from harness import compare_all, make_config, make_pair, oracle_for, random_inputs, write_both

import ionsolver_amd as I

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,kw", [
    ((192, 120, 120), dict(float_type=2)),
    ((150, 140, 132), dict(float_type=2, relaxation_time=1, ffield=True)),
    ((256, 150, 140), dict(float_type=1)),
    ((181, 172, 175), dict(float_type=0, vforce=False)),
    ((192, 194, 182), dict(float_type=1, velocity_set=1, relaxation_time=1)),
    ((2551, 4403, 1), dict(float_type=1, velocity_set=0)),
    ((128, 96, 96), dict(float_type=2, mhd=True, lod_depth=3)),
    ((104, 112, 104), dict(float_type=2, mhd=True, lod_depth=3)),
    ((136, 144, 152), dict(float_type=2, mhd=True, lod_depth=3)),
    ((192, 112, 112), dict(float_type=1, mhd=True, lod_depth=3)),
    ((152, 136, 112), dict(float_type=0, mhd=True, lod_depth=3, charge_inlet=True)),
    ((64, 3, 1), dict(float_type=1)),
    ((1, 1, 67), dict(float_type=2)),
], ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "-".join(f"{a}{int(b)}" for a, b in v.items()))
def test_lattices_of_every_path(shape, kw):
    gpu, orc, info = make_pair(np.random.default_rng(sum(shape)), nx=shape[0], ny=shape[1], nz=shape[2], **kw)
    try:
        gpu.initialize()
        orc.initialize()
        for _ in range(2):
            gpu.do_time_step()
            orc.do_time_step()
        assert compare_all(gpu, orc, info) == []
    finally:
        gpu.close()


@pytest.mark.parametrize("value", [np.nan, 3e30, -2e38])
@pytest.mark.parametrize("mhd", [False, True])
@pytest.mark.parametrize("float_type", [0, 1])
def test_values_that_are_not_finite(float_type, mhd, value):
    rng = np.random.default_rng(5)
    cfg = make_config(nx=24, ny=16, nz=16, float_type=float_type, mhd=mhd, lod_depth=1, ffield=True)
    gpu = I.Lbm(cfg)
    try:
        orc = oracle_for(gpu.config)
        arrays = random_inputs(gpu.config, rng)
        n = 24 * 16 * 16
        arrays["F"][rng.integers(0, 3 * n, 6)] = value
        arrays["rho"][np.flatnonzero(arrays["flags"] == 2)[:3]] = value
        write_both(gpu, orc, arrays)
        with np.errstate(all="ignore"):
            gpu.initialize()
            orc.initialize()
            names = ["fi", "flags"] + (["ei", "fqi"] if mhd else [])
            for _ in range(2):
                gpu.do_time_step()
                orc.do_time_step()
                assert compare_all(gpu, orc, dict(cfg=gpu.config), names) == []
    finally:
        gpu.close()


@pytest.mark.parametrize("float_type", [0, 1])
def test_codes_of_every_finite_value(float_type):
    encode = O.fp16s_store if float_type == 0 else O.fp16c_encode
    mantissa = np.arange(1 << 23, dtype=np.uint32)
    # every value that has a code of its own or rounds to one, and some of the rest of the range
    for exponent in [*range(90, 130), 1, 45, 135, 180, 239]:
        for sign in (0, 1) if exponent in (99, 111, 112, 113, 127) else (0,):
            x = (np.uint32(sign << 31 | exponent << 23) | mantissa).view(np.float32)
            bad = I.device_codec(float_type, 0, x) != encode(x)
            assert not bad.any(), (exponent, sign, x[bad][:3])
    codes = np.arange(1 << 16, dtype=np.uint16)
    decode = O.fp16s_load if float_type == 0 else O.fp16c_decode
    assert np.array_equal(I.device_codec(float_type, 1, codes).view(np.uint32), decode(codes).view(np.uint32)) or float_type == 0
    if float_type == 0:
        a, b = I.device_codec(0, 1, codes), decode(codes)
        assert np.array_equal(a, b, equal_nan=True)
