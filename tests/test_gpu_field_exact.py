"""The field update in exact arithmetic over all LOD blocks (depth 3 and 4)
against the oracle, every buffer equal: LOD blocks of 1 to 13 cells a side,
uneven ones, sides that are not powers of two; random flags, so that the lanes
of a wavefront are solid and fluid at random; sources above the domain; and the
plain kernels wherever few or non-finite sources send the step there."""
import numpy as np
import pytest

from harness import compare_all, make_pair
from ionsolver_amd import Field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,D", [((16, 16, 16), 4), ((64, 48, 80), 4), ((8, 24, 16), 3), ((24, 16, 40), 3),
                                     ((72, 88, 104), 3), ((32, 32, 64), 3)],
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_exact_steps_match_the_oracle(shape, D):
    gpu, orc, info = make_pair(np.random.default_rng(40), nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D,
                               float_type=2)
    try:
        gpu.initialize()
        orc.initialize()
        for _ in range(2):
            gpu.do_time_step()
            orc.do_time_step()
        assert compare_all(gpu, orc, info) == []
    finally:
        gpu.close()
        orc.close()


@pytest.mark.parametrize("kind", ["all", "few", "nan", "inf", "large"])
@pytest.mark.parametrize("shape,D", [((48, 32, 80), 4), ((40, 24, 56), 3)], ids=["D4", "D3"])
def test_exact_field_of_given_lod_sums(shape, D, kind):
    """compute_fields from written LOD sums, against the float32 sum in the
    reference's order (ascending LOD index), unfused."""
    rng = np.random.default_rng(41)
    gpu, orc, info = make_pair(rng, nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D, float_type=2)
    try:
        nd = 1 << D
        n_lod = gpu.config.kernel_constants()["n_lod"]
        lod = (0.05 * rng.standard_normal((n_lod, 4))).astype(np.float32)
        if kind == "few":
            lod[rng.uniform(size=n_lod) < 0.9, 0] = 0.0
        elif kind != "all":
            lod[nd ** 3 - 2 * nd - 3] = (dict(nan=np.nan, inf=np.inf, large=3e36)[kind], 0.01, -0.02, 0.03)
        gpu.write_field(Field.QU_LOD, lod.reshape(-1))
        gpu.compute_fields()
        got = np.concatenate([gpu.read_field(f).reshape(3, -1) for f in (Field.E_DYN, Field.B_DYN)])
        k = gpu.config.kernel_constants()
        ke, kmu = np.float32(k["ke"]), np.float32(k["kmu"])
        b = [np.float32(n // nd) for n in shape]
        flags = info["arrays"]["flags"] & 0x1F
        cells = rng.choice(np.flatnonzero(flags != 1), 200, replace=False)
        x, y, z = cells % shape[0], cells // shape[0] % shape[1], cells // (shape[0] * shape[1])
        own = x // (shape[0] // nd) + (y // (shape[1] // nd) + z // (shape[2] // nd) * nd) * nd
        s = np.zeros((6, len(cells)), np.float32)
        with np.errstate(all="ignore"):
            for d in range(n_lod - nd ** 3, n_lod):
                q, vx, vy, vz = lod[d]
                if q == 0:
                    continue
                c = [np.float32(i) * w + np.float32(0.5) * w for i, w in zip((d % nd, d // nd % nd, d // nd ** 2), b)]
                r = [p.astype(np.float32) - w for p, w in zip((x, y, z), c)]
                l = np.sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2])
                l3 = l * l * l
                p = [w / l3 for w in r]
                f = [p[0], p[1], p[2], vy * p[2] - vz * p[1], vz * p[0] - vx * p[2], vx * p[1] - vy * p[0]]
                for i in range(6):
                    s[i] = np.where(d == own, s[i], s[i] + q * f[i])
            a = info["arrays"]
            stat = np.concatenate([a["e_stat"].reshape(3, -1), a["b_stat"].reshape(3, -1)])[:, cells]
            want = stat + np.array([ke] * 3 + [kmu] * 3, np.float32)[:, None] * s
        assert np.array_equal(got[:, cells], want, equal_nan=True)
    finally:
        gpu.close()
        orc.close()
