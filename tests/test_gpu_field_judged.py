"""The FAST judge and training target of the surrogate, the direct sum by shifts
or source by source: both leave the same raw sums, and the judge's
residual, whose partial sums the two kernels write between them, agrees with the
explicit one and the fields it leaves with the raw sums, with the route changing
from step to step on one handle."""
import numpy as np
import pytest

import ionsolver_amd as I
from harness import make_config
from ionsolver_amd import Field
from ionsolver_amd.lbm import FieldMode, FieldSolver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,D", [((64, 64, 64), 4), ((80, 112, 48), 4), ((176, 80, 48), 4), ((64, 64, 64), 3), ((88, 56, 72), 3)],
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_raw_sums_are_the_same_by_either_route(shape, D):
    """Half of the LOD blocks charged, and the same with further charges too weak
    to change a sum that has begun (before it they would decide a tie of its first
    rounding: the first charges of the order are strong ones), 7/8 of them charged."""
    rng = np.random.default_rng(7)
    n, nd3 = int(np.prod(shape)), 8 ** D
    lbm = I.Lbm(make_config(nx=shape[0], ny=shape[1], nz=shape[2], mhd=True, lod_depth=D))
    try:
        lbm.set_field_mode(FieldMode.FAST)
        flags = np.where(rng.uniform(size=n) < 0.3, 1, 0).astype(np.uint8)
        n_lod = lbm.config.kernel_constants()["n_lod"]
        lod = np.zeros((n_lod, 4), np.float32)
        some = n_lod - nd3 + rng.permutation(nd3)
        few, all_ = some[:nd3 // 2], some[:nd3 * 7 // 8]
        lod[few] = 0.05 * rng.standard_normal((few.size, 4)) + np.array([0.2, 0, 0, 0])
        more = lod.copy()
        more[np.setdiff1d(all_, few)] = (1e-36, 1e-3, -1e-3, 2e-3)
        lbm.write_field(Field.FLAGS, flags)
        lbm.surrogate_create(channels=8)
        out = []
        for q in (lod, more):
            lbm.write_field(Field.QU_LOD, q.reshape(-1))
            lbm.compute_fields()
            out.append(lbm.read_field(Field.FIELD_SUMS))
        assert np.abs(out[0]).max() > 0
        np.testing.assert_array_equal(out[0], out[1])
    finally:
        lbm.close()


@pytest.mark.parametrize("shape,D", [((64, 64, 64), 4), ((80, 112, 48), 4), ((64, 64, 64), 3), ((128, 128, 128), 4), ((176, 112, 144), 4)],
                         ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else f"D{p}")
def test_judge_of_both_routes(shape, D):
    """The gas at rest under a charge distribution: a step's LOD sums are the cells'
    charges, whose LOD blocks are charged to 1/2 or to 7/8 in turn."""
    rng = np.random.default_rng(23)
    nx, ny, nz = shape
    n, nd = int(np.prod(shape)), 1 << D
    lbm = I.Lbm(make_config(nx=nx, ny=ny, nz=nz, mhd=True, lod_depth=D, graphics=False))
    try:
        lbm.set_field_mode(FieldMode.FAST)
        lbm.write_field(Field.B_STAT, np.full(3 * n, 0.01, np.float32))
        lbm.surrogate_create(channels=8)
        lbm.set_field_solver(FieldSolver.SURROGATE, judge_every=1, tolerance=1.0)
        k = lbm.config.kernel_constants()
        x, y, z = np.arange(n) % nx, np.arange(n) // nx % ny, np.arange(n) // (nx * ny)
        block = x // (nx // nd) + (y // (ny // nd) + z // (nz // nd) * nd) * nd
        charge = 0.05 * rng.standard_normal(nd ** 3) + 0.2
        order = rng.permutation(nd ** 3)
        for share in (0.875, 0.5, 0.875):
            q = np.zeros(nd ** 3)
            q[order[:int(share * nd ** 3)]] = charge[:int(share * nd ** 3)]
            flags = np.where(q[block] == 0, 1, 0).astype(np.uint8)  # blocks without charge are solid
            lbm.write_field(Field.FLAGS, flags)
            lbm.write_field(Field.Q, q[block].astype(np.float32))
            lbm.write_field(Field.U, (0.01 * rng.standard_normal(3 * n)).astype(np.float32))
            lbm.initialize()
            lbm.do_time_step()
            st = lbm.surrogate_stats()
            fused = np.array([st["last_residual_e"], st["last_residual_b"]])
            lod = lbm.read_field(Field.QU_LOD).reshape(-1, 4)
            charged = np.count_nonzero(lod[len(lod) - nd ** 3:, 0])
            # the reference's range of sources ends above the domain
            assert abs(charged / nd ** 3 - share) < 0.15, charged
            assert (charged >= nd ** 3 * 5 // 8) == (share > 0.6)
            fields = lbm.read_field(Field.E_DYN), lbm.read_field(Field.B_DYN)
            lbm.compute_fields()
            explicit = np.array(lbm.surrogate_residual())
            print("judge residual", fused, "explicit", explicit, "charged", charged, flush=True)
            # a float sum of a few cells a work-item, its quotient and square root (the explicit one: network units)
            np.testing.assert_allclose(fused, explicit, rtol=1e-3)
            raw = lbm.read_field(Field.FIELD_SUMS).reshape(2, -1)
            fluid = np.tile(flags == 0, 3)
            stat = lbm.read_field(Field.E_STAT), lbm.read_field(Field.B_STAT)
            for r, s, got, f in zip(raw, stat, fields, (k["ke"], k["kmu"])):
                np.testing.assert_array_equal((s + np.float32(f) * r)[fluid], got[fluid])
    finally:
        lbm.close()
