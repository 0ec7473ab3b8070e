"""Performance cases of the framework: what a program does with it, at the sizes and options it is used with.

Five kinds of work, each through the public entry points:

fluid   ``Lbm.run`` without charges, then rho and u read back (flow studies);
mhd     ``Lbm.run`` with magnetohydrodynamics (fluid, electron gas, charge advection, E/B field every step), then
        u, Q, E and B read back; the field step directly, or by the learned surrogate with the direct one as its judge;
field   one field step on device buffers the caller owns (``ion_update_e_b_noalloc``);
train   one training step of the field surrogate on one charge configuration: LOD sums in, direct field, gradients out;
static  the set-up of a thruster's static fields: magnets and electrodes in, ``precompute_b`` and ``precompute_e``,
        B_stat and E_stat out.

Inputs are made on the GPU from the seed alone. Buffers that are read back lie in pinned host memory that the program
keeps, read through the C entry point ``ion_read_field``.
"""
import ctypes
import math

import torch

import ionsolver_amd as I
from ionsolver_amd import scenarios
from ionsolver_amd.lbm import Field, FieldMode, FieldSolver, FloatType, Lbm, LbmConfig, RelaxationTime, VelocitySet, load_library

DEV = "cuda"
F64 = torch.float64
SETS = {"D2Q9": 9, "D3Q15": 15, "D3Q19": 19}
FLOATS = {"FP32": 4, "FP16S": 2, "FP16C": 2}


# ----------------------------------------------------------------------------------------------------------------------
# The cases
# ----------------------------------------------------------------------------------------------------------------------
def _fluid(name, lattice, store, shape, steps, relax="Srt", channel=False):
    nx, ny, nz = shape
    return dict(name=name, kind="fluid", set=lattice, store=store, nx=nx, ny=ny, nz=nz, steps=steps, relax=relax,
                channel=channel)


def _mhd(name, store, shape, depth, mode, steps, solver="direct", geometry="cylinder"):
    nx, ny, nz = shape
    return dict(name=name, kind="mhd", store=store, nx=nx, ny=ny, nz=nz, depth=depth, mode=mode, steps=steps,
                solver=solver, geometry=geometry)


def _field(name, shape, depth, mode):
    nx, ny, nz = shape
    return dict(name=name, kind="field", nx=nx, ny=ny, nz=nz, depth=depth, mode=mode)


def listed():
    return [
        # the 64^3 Taylor-Green box of the workloads: a step takes some 10 us, so launches count
        _fluid("fluid_64_fp32", "D3Q19", "FP32", (64, 64, 64), 50),
        # a ragged channel with walls, inlet, outlet and a body force, the two-rate collision, 16-bit storage
        _fluid("channel_d3q15_fp16s", "D3Q15", "FP16S", (132, 75, 90), 20, relax="Trt", channel=True),
        # a large box in the storage format of the large runs: memory bound
        _fluid("fluid_256_fp16c", "D3Q19", "FP16C", (256, 256, 256), 20),
        # a small MHD run in the default (exact) field arithmetic, as the tests and first trials use it
        _mhd("mhd_64_exact", "FP32", (64, 64, 64), 3, "exact", 5),
        # the benchmark's default workload: 256^3 FP32, LOD depth 4, direct field in fast arithmetic
        _mhd("mhd_256_fast", "FP32", (256, 256, 256), 4, "fast", 10),
        # a lattice whose LOD blocks (11 x 7 x 13 cells) fit no tile, 16-bit storage, default field arithmetic
        _mhd("mhd_ragged_fp16c", "FP16C", (176, 112, 208), 4, "exact", 2),
        # thruster: tube, inlet and outlet with charge, FP16C, surrogate field, the direct one as judge every 50 steps
        _mhd("thruster_256_fp16c", "FP16C", (256, 256, 256), 4, "fast", 50, solver="surrogate", geometry="tube"),
        # the field step alone on the caller's buffers: the benchmark's lattice, a ragged one, the exact arithmetic
        _field("field_256_fast", (256, 256, 256), 4, "fast"),
        _field("field_ragged_fast", (240, 336, 144), 4, "fast"),
        _field("field_128_exact", (128, 128, 128), 4, "exact"),
        # one step of the surrogate's training loop
        dict(name="train_128", kind="train", nx=128, ny=128, nz=128, depth=4, channels=16),
        # static fields of a thruster with a ring and a disk magnet and two charged plates, at a coarse resolution
        dict(name="static_96", kind="static", nx=96, ny=192, nz=96),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _shape(rng, cells, unit, lo):
    """Three sides, multiples of `unit` of at least `lo`, of about `cells` cells and up to 2 : 1 apart."""
    side = cells ** (1 / 3)
    return [max(lo, unit * round(side * _log(rng, 0.75, 1.33) / unit)) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["fluid", "fluid", "mhd", "mhd", "field", "field", "train", "static"])
    if kind == "fluid":
        lattice = rng.choice(["D2Q9", "D3Q15", "D3Q19", "D3Q19"])
        store = rng.choice(["FP32", "FP16S", "FP16C"])
        cells = int(_log(rng, 64 ** 3, 240 ** 3))
        shape = _shape(rng, cells, 1, 8)
        if lattice == "D2Q9":
            nx = int(math.sqrt(cells) * _log(rng, 0.5, 2.0))
            shape = [nx, max(8, cells // nx), 1]
        c = _fluid("", lattice, store, shape, rng.randint(5, 25), rng.choice(["Srt", "Trt"]), rng.random() < 0.5)
    elif kind == "mhd":
        depth = rng.choice([3, 4])
        shape = _shape(rng, int(_log(rng, 48 ** 3, 180 ** 3)), 2 ** depth, 3 * 2 ** depth)
        c = _mhd("", rng.choice(["FP32", "FP16S", "FP16C"]), shape, depth, rng.choice(["fast", "exact"]),
                 rng.randint(1, 5), geometry=rng.choice(["cylinder", "tube"]))
        if rng.random() < 0.3:
            c.update(solver="surrogate", mode="fast", steps=rng.randint(10, 30))
    elif kind == "field":
        depth = rng.choice([3, 4, 4])
        mode = rng.choice(["fast", "fast", "exact"])
        most = 230 if mode == "fast" else 140
        c = _field("", _shape(rng, int(_log(rng, 48 ** 3, most ** 3)), 2 ** depth, 2 * 2 ** depth), depth, mode)
    elif kind == "train":
        depth = rng.choice([3, 4])
        nx, ny, nz = _shape(rng, int(_log(rng, 48 ** 3, 120 ** 3)), 2 ** depth, 2 * 2 ** depth)
        c = dict(name="", kind="train", nx=nx, ny=ny, nz=nz, depth=depth, channels=rng.choice([8, 16]))
    else:
        n = int(_log(rng, 40, 90))
        c = dict(name="", kind="static", nx=n + rng.randint(0, 6), ny=2 * n + rng.randint(0, 9), nz=n + rng.randint(0, 6))
    del c["name"]
    return c


# ----------------------------------------------------------------------------------------------------------------------
# Inputs
# ----------------------------------------------------------------------------------------------------------------------
def _cells(c):
    return c["nx"] * c["ny"] * c["nz"]


def _coords(c, dtype=torch.float32):
    """x, y, z of the cells, broadcastable to [nz][ny][nx]."""
    return (torch.arange(c["nx"], device=DEV, dtype=dtype)[None, None, :],
            torch.arange(c["ny"], device=DEV, dtype=dtype)[None, :, None],
            torch.arange(c["nz"], device=DEV, dtype=dtype)[:, None, None])


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _uniform(g, lo, hi, n):
    return (lo + (hi - lo) * torch.rand(n, generator=g, device=DEV)).tolist()


def _vortices(c, g, u0):
    """Velocity [3][nz][ny][nx] of a few periodic vortices around the z axis, of random phase, peak about u0."""
    x, y, z = _coords(c)
    u = torch.zeros(3, c["nz"], c["ny"], c["nx"], device=DEV)
    for kx, ky, kz in ((1, 1, 0), (2, 1, 1)):
        if c["nz"] == 1 and kz:
            continue
        px, py, pz = _uniform(g, 0.0, 2 * math.pi, 3)
        ax, ay, az = 2 * math.pi * kx / c["nx"], 2 * math.pi * ky / c["ny"], 2 * math.pi * kz / c["nz"]
        shape = torch.cos(az * z + pz) if kz else 1.0
        u[0] += u0 / (kx + kz) * torch.cos(ax * x + px) * torch.sin(ay * y + py) * shape
        u[1] -= u0 / (kx + kz) * (ax / ay) * torch.sin(ax * x + px) * torch.cos(ay * y + py) * shape
    return u


def _fluid_inputs(c, seed):
    g = _gen(seed)
    u = _vortices(c, g, 0.04)
    rho = torch.ones(c["nz"], c["ny"], c["nx"], device=DEV) + 1e-3 * torch.randn(c["nz"], c["ny"], c["nx"], generator=g,
                                                                                 device=DEV)
    flags = torch.zeros(c["nz"], c["ny"], c["nx"], dtype=torch.uint8, device=DEV)
    if c["channel"]:
        u[0] += 0.03
        flags[:, :, 0] = 2
        flags[:, :, -1] = 2
        flags[:, 0, :] = 1
        flags[:, -1, :] = 1
        x, y, z = _coords(c)
        (cx, cy, cz), r = _uniform(g, 0.3, 0.5, 3), 0.08 * c["ny"]  # an obstacle
        dz = (z - cz * c["nz"]) if c["nz"] > 1 else 0.0
        flags[((x - cx * c["nx"]) ** 2 + (y - cy * c["ny"]) ** 2 + dz ** 2 < r * r).expand_as(flags)] = 1
    return dict(rho=rho, u=u, flags=flags)


FORCE = (1e-5, 2e-6, 0.0)  # body force of the channel


def _fluid_config(c):
    cfg = LbmConfig()
    cfg.velocity_set = VelocitySet[c["set"]]
    cfg.relaxation_time = RelaxationTime[c["relax"]]
    cfg.float_type = FloatType[c["store"]]
    cfg.n_x, cfg.n_y, cfg.n_z = c["nx"], c["ny"], c["nz"]
    cfg.nu = 0.1 / 3.0
    if c["channel"]:
        cfg.ext_equilibrium_boudaries = True
        cfg.ext_volume_force = True
        cfg.f_x, cfg.f_y, cfg.f_z = FORCE
    return cfg


BACKGROUND = 1.0  # charge density of the neutral plasma background
INLET_CHARGE = 0.02


def _mhd_inputs(c, seed):
    """Charge blobs on a neutral plasma background in a slow flow and a magnetic field, around a solid cylinder, or in a
    quartz tube between an inlet and an outlet."""
    g = _gen(seed)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    x, y, z = _coords(c)
    cx, cy, cz = 0.5 * nx, 0.5 * ny, 0.5 * nz
    r2 = (x - cx) ** 2 + (y - cy) ** 2
    flags = torch.zeros(nz, ny, nx, dtype=torch.uint8, device=DEV)
    side = min(nx, ny, nz)
    u = _vortices(c, g, 0.02)
    q = 1e-4 * torch.randn(nz, ny, nx, generator=g, device=DEV)
    for _ in range(8):
        px, py, pz, a, s = _uniform(g, 0.0, 1.0, 5)
        sigma = side * (0.03 + 0.04 * s)
        amp = 0.05 * (0.5 + 0.5 * a) * (1 if px < 0.5 else -1)
        q += amp * torch.exp(-((x - nx * (0.1 + 0.8 * px)) ** 2 + (y - ny * (0.1 + 0.8 * py)) ** 2
                               + (z - nz * (0.1 + 0.8 * pz)) ** 2) / (2 * sigma * sigma))
    q += BACKGROUND
    if c["geometry"] == "cylinder":
        flags[(r2 < (0.156 * side) ** 2).expand_as(flags)] = 1
    else:
        rt = 0.3 * min(nx, ny)
        flags[((r2 >= rt * rt) & (r2 < (rt + 2) ** 2)).expand_as(flags)] = 1
        inside = (r2 < rt * rt)[0]
        u = 0.1 * u
        u[2][inside.expand_as(flags)] = 0.02
        flags[0][inside], flags[-1][inside] = 2, 2
        q[0][inside], q[-1][inside] = BACKGROUND + INLET_CHARGE, BACKGROUND
    q[flags == 1] = 0.0
    rx, ry, rz = x - cx, y - cy, z - cz
    rr = rx * rx + ry * ry + rz * rz + (0.1 * side) ** 2
    m = 0.002 * (0.2 * side) ** 3 * (0.8 + 0.4 * _uniform(g, 0.0, 1.0, 1)[0])  # a dipole of finite size
    k = 3 * m * rz / rr ** 2.5
    b = torch.stack([k * rx, k * ry, k * rz - m / rr ** 1.5 + 0.002])
    return dict(flags=flags, u=u, q=q, b_stat=b)


def _mhd_config(c):
    cfg = LbmConfig()
    cfg.velocity_set = VelocitySet.D3Q19
    cfg.float_type = FloatType[c.get("store", "FP32")]
    cfg.n_x, cfg.n_y, cfg.n_z = c["nx"], c["ny"], c["nz"]
    cfg.nu = 0.1 / 3.0
    cfg.ext_volume_force = True
    cfg.ext_magneto_hydro = True
    cfg.mhd_lod_depth = c["depth"]
    scenarios.use_plasma_units(cfg, BACKGROUND)
    if c.get("geometry") == "tube":
        cfg.ext_equilibrium_boudaries = True
        cfg.ext_charge_inlet = True
    return cfg


def _lod(c, seed, n_lod):
    """Charge and mean velocity of the LOD blocks of a plasma flow, [n_lod][4], the top level first."""
    g = _gen(seed)
    nd = 1 << c["depth"]
    vol = _cells(c) / nd ** 3
    z, y, x = torch.meshgrid(*(torch.arange(nd, device=DEV, dtype=torch.float32),) * 3, indexing="ij")
    q = 1e-4 * math.sqrt(vol) * torch.randn(nd, nd, nd, generator=g, device=DEV)
    for _ in range(8):
        px, py, pz, a, s = _uniform(g, 0.0, 1.0, 5)
        sigma = nd * (0.04 + 0.06 * s)
        q += (1 if a < 0.5 else -1) * 0.02 * vol * torch.exp(-((x - nd * px) ** 2 + (y - nd * py) ** 2 + (z - nd * pz) ** 2)
                                                           / (2 * sigma * sigma))
    top = torch.empty(nd, nd, nd, 4, device=DEV)
    top[..., 0] = q
    for i in range(3):
        k, p = _uniform(g, 1.0, 3.0, 3), _uniform(g, 0.0, 2 * math.pi, 1)[0]
        top[..., 1 + i] = 0.02 * torch.sin(2 * math.pi / nd * (k[0] * x + k[1] * y + k[2] * z) + p)
    buf = torch.zeros(n_lod, 4, device=DEV)
    buf[:nd ** 3] = top.reshape(-1, 4)
    return buf


def _n_lod(depth):
    return sum(8 ** i for i in range(depth + 1))


def _field_inputs(c, seed):
    n = _cells(c)
    g = _gen(seed + 7)
    x, y, z = _coords(c)
    flags = torch.zeros(c["nz"], c["ny"], c["nx"], dtype=torch.uint8, device=DEV)
    flags[((x - 0.5 * c["nx"]) ** 2 + (y - 0.5 * c["ny"]) ** 2 < (0.156 * c["nx"]) ** 2).expand_as(flags)] = 1
    return dict(flags=flags.reshape(-1), q=torch.zeros(n, device=DEV), u=torch.zeros(3 * n, device=DEV),
                qu_lod=_lod(c, seed, _n_lod(c["depth"])).reshape(-1),
                e_stat=1e-6 * torch.randn(3 * n, generator=g, device=DEV),
                b_stat=1e-6 * torch.randn(3 * n, generator=g, device=DEV),
                e_dyn=torch.zeros(3 * n, device=DEV), b_dyn=torch.zeros(3 * n, device=DEV))


def _layers(c):
    """(name, channels of the two inputs, output channels, grid side) of the surrogate's convolutions, in parameter order."""
    C, g = [c["channels"] * k for k in (1, 2, 3, 4)], 1 << c["depth"]
    return [("e0", 8, 0, C[0], g), ("e1", C[0], 0, C[1], g // 2), ("e2", C[1], 0, C[2], g // 4),
            ("e3", C[2], 0, C[3], g // 8), ("d2", C[3], C[2], C[2], g // 4), ("d1", C[2], C[1], C[1], g // 2),
            ("d0", C[1], C[0], C[0], g)]


def _pad32(n):
    return (n + 31) // 32 * 32


def _weights(c, seed):
    """Parameters of a surrogate in the middle of its training, float32, in the order of ``Lbm.surrogate_params``: random
    convolutions; the head's source columns the exact near field of the 26 neighbouring LOD blocks, its feature columns small."""
    g = _gen(seed + 3)
    parts = []
    for _, ca, cb, cout, _ in _layers(c):
        k = 27 * (ca + cb)
        w = torch.zeros(cout, _pad32(k), device=DEV)
        w[:, :k] = torch.randn(cout, k, generator=g, device=DEV) / math.sqrt(k)
        parts.append(w)
    nd = 1 << c["depth"]
    b = [c[s] // nd for s in ("nx", "ny", "nz")]
    cpb, c0 = b[0] * b[1] * b[2], c["channels"]
    gain = cpb ** (2 / 3)
    w = torch.zeros(6, cpb, 27, c0 + 8, dtype=F64, device=DEV)
    w[..., :c0] = 0.01 * torch.randn(6, cpb, 27, c0, generator=g, device=DEV)
    o = torch.arange(cpb, device=DEV, dtype=F64)
    off = torch.stack([o % b[0], (o // b[0]) % b[1], o // (b[0] * b[1])])
    for d in range(27):
        if d == 13:
            continue
        delta = (d % 3 - 1, d // 3 % 3 - 1, d // 9 - 1)
        r = torch.stack([off[i] - (delta[i] + 0.5) * b[i] for i in range(3)])
        K = gain * r / (r * r).sum(0) ** 1.5
        for p in (0, 4):
            for i in range(3):
                w[i, :, d, c0 + p] = K[i]
            for i in range(3):  # B = J x K
                j, k = (i + 1) % 3, (i + 2) % 3
                w[3 + i, :, d, c0 + p + 1 + j] = K[k]
                w[3 + i, :, d, c0 + p + 1 + k] = -K[j]
    head = torch.zeros(6 * cpb, _pad32(27 * (c0 + 8)), device=DEV)
    head[:, :27 * (c0 + 8)] = w.reshape(6 * cpb, -1).float()
    return parts + [head]


def _static_inputs(c, seed):
    """Cells of a ring magnet, a disk magnet and two charged plates; B_dyn holds the magnetisation and the charge, as
    voxelising their meshes leaves it."""
    g = _gen(seed)
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    x, y, z = _coords(c)
    r = torch.sqrt((x - 0.5 * nx) ** 2 + (z - 0.5 * nz) ** 2)
    a = min(nx, nz)
    flags = torch.zeros(nz, ny, nx, dtype=torch.uint8, device=DEV)
    val = torch.zeros(3, nz, ny, nx, device=DEV)
    s = _uniform(g, 0.8, 1.2, 4)
    ring = (r >= 0.33 * a) & (r < 0.4 * a) & (y >= 0.3 * ny) & (y < 0.3 * ny + 0.1 * a)
    disk = (r < 0.15 * a) & (y >= 0.08 * ny) & (y < 0.08 * ny + 0.06 * a)
    for cells, m in ((ring, 0.5 * s[0]), (disk, 1.0 * s[1])):
        cells = cells.expand_as(flags)
        flags[cells] = 0x11
        val[1][cells] = m
        val[0][cells] = 0.1 * m
    for sign, zc, e in ((1, 0.1, s[2]), (-1, 0.9, s[3])):
        plate = ((z - zc * nz).abs() < 1) & ((x - 0.5 * nx).abs() < 0.2 * nx) & ((y - 0.6 * ny).abs() < 0.1 * ny)
        plate = plate.expand_as(flags)
        flags[plate] = 0x05
        val[0][plate] = sign * 1e-3 * e
    return dict(flags=flags, b_dyn=val)


def _static_config(c):
    cfg = LbmConfig()
    cfg.velocity_set = VelocitySet.D3Q19
    cfg.n_x, cfg.n_y, cfg.n_z = c["nx"], c["ny"], c["nz"]
    for k, v in scenarios.PLASMA_UNITS.items():
        setattr(cfg.units, k, v)
    cfg.ext_volume_force = True
    cfg.ext_magneto_hydro = True
    cfg.mhd_lod_depth = 0
    return cfg


# ----------------------------------------------------------------------------------------------------------------------
# The work
# ----------------------------------------------------------------------------------------------------------------------
class _FieldBuffers(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("flags", "q", "u", "qu_lod", "e_stat", "b_stat", "e_dyn", "b_dyn")]


def _write(lbm, arrays):
    names = dict(flags=Field.FLAGS, rho=Field.RHO, u=Field.U, q=Field.Q, b_stat=Field.B_STAT, e_stat=Field.E_STAT,
                 b_dyn=Field.B_DYN)
    for k, v in arrays.items():
        lbm.write_field(names[k], v.reshape(-1).cpu().numpy())


def _outputs(c, fields):
    n = _cells(c)
    return {f: torch.empty(n * (3 if f in ("U", "E_DYN", "B_DYN", "E_STAT", "B_STAT") else 1), pin_memory=True)
            for f in fields}


def _read(lbm, out):
    lib = load_library()
    for f, t in out.items():
        if lib.ion_read_field(lbm._h, int(Field[f]), t.data_ptr(), t.numel() * 4):
            raise I.IonError(lib.ion_last_error().decode())


def prepare(case, seed):
    c = case
    if c["kind"] == "fluid":
        lbm = Lbm(_fluid_config(c))
        _write(lbm, _fluid_inputs(c, seed))
        lbm.initialize()
        return dict(case=c, lbm=lbm, out=_outputs(c, ("RHO", "U")))
    if c["kind"] == "mhd":
        lbm = Lbm(_mhd_config(c))
        _write(lbm, _mhd_inputs(c, seed))
        lbm.set_field_mode(FieldMode.FAST if c["mode"] == "fast" else FieldMode.EXACT)
        if c["solver"] == "surrogate":
            lbm.surrogate_create()
            lbm.set_field_solver(FieldSolver.SURROGATE, judge_every=50, tolerance=0.05)
        lbm.initialize()
        return dict(case=c, lbm=lbm, out=_outputs(c, ("U", "Q", "E_DYN", "B_DYN")))
    if c["kind"] == "field":
        buf = _field_inputs(c, seed)
        cfg = _mhd_config(c)._to_c()
        return dict(case=c, buf=buf, cfg=cfg, ptr=_FieldBuffers(**{k: v.data_ptr() for k, v in buf.items()}),
                    mode=int(FieldMode.FAST if c["mode"] == "fast" else FieldMode.EXACT))
    if c["kind"] == "train":
        lbm = Lbm(_mhd_config(c))
        lbm.set_field_mode(FieldMode.FAST)
        lbm.surrogate_create(channels=c["channels"])
        lbm.set_surrogate_params(torch.cat([w.reshape(-1) for w in _weights(c, seed)]).cpu().numpy())
        return dict(case=c, lbm=lbm, lod=_lod(c, seed, _n_lod(c["depth"])).reshape(-1).cpu().numpy())
    lbm = Lbm(_static_config(c))
    arrays = {k: v.reshape(-1).cpu().numpy() for k, v in _static_inputs(c, seed).items()}
    zero = torch.zeros(3 * _cells(c)).numpy()
    return dict(case=c, lbm=lbm, arrays=arrays, zero=zero, out=_outputs(c, ("E_STAT", "B_STAT")))


def run(state):
    c = state["case"]
    if c["kind"] in ("fluid", "mhd"):
        state["lbm"].run(c["steps"])
        _read(state["lbm"], state["out"])
        return state["out"]
    if c["kind"] == "field":
        lib = load_library()
        stream = torch.cuda.current_stream().cuda_stream
        if lib.ion_update_e_b_noalloc(ctypes.byref(state["cfg"]), ctypes.byref(state["ptr"]), state["mode"], stream):
            raise I.IonError(lib.ion_last_error().decode())
        return dict(e=state["buf"]["e_dyn"], b=state["buf"]["b_dyn"])
    lbm = state["lbm"]
    if c["kind"] == "train":
        lbm.write_field(Field.QU_LOD, state["lod"])
        lbm.compute_fields()
        rel_e, rel_b = lbm.surrogate_train_step(True)
        # float32 quotients of the fields' sums, like the gradients
        return dict(rel=torch.tensor([rel_e, rel_b], dtype=torch.float32), grads=lbm.surrogate_params(grads=True))
    lbm.write_field(Field.FLAGS, state["arrays"]["flags"])
    lbm.write_field(Field.B_DYN, state["arrays"]["b_dyn"])
    lbm.write_field(Field.B_STAT, state["zero"])
    lbm.write_field(Field.E_STAT, state["zero"])
    lbm.precompute_b()
    lbm.precompute_e()
    _read(lbm, state["out"])
    return state["out"]


def work(case):
    """Each distribution is read and written once a step, each field once; operations per cell and direction, and per
    LOD source. A field in fast arithmetic has to sum its 27 nearest sources at each cell (the others may be summed
    for many cells at once); in exact arithmetic every source is added at every cell, in order."""
    c, n = case, _cells(case)
    if c["kind"] == "fluid":
        Q, s = SETS[c["set"]], FLOATS[c["store"]]
        return dict(bytes=c["steps"] * n * (2 * Q * s + 1 + 16) + 16 * n, flops=c["steps"] * n * Q * 15)
    if c["kind"] in ("mhd", "field"):
        per_cell = 27 * 20 if c["mode"] == "fast" or c.get("solver") == "surrogate" else 8 ** c["depth"] * 21
        if c["kind"] == "field":
            return dict(bytes=49 * n, flops=per_cell * n)
        s = FLOATS[c["store"]]
        return dict(bytes=c["steps"] * n * (90 * s + 45 + 49) + 40 * n, flops=c["steps"] * n * (45 * 15 + per_cell))
    if c["kind"] == "train":
        nd = 1 << c["depth"]
        head = 6 * n * _pad32(27 * (c["channels"] + 8))
        conv = sum(g ** 3 * co * 27 * (ca + cb) for _, ca, cb, co, g in _layers(c))
        weights = 6 * n // nd ** 3 * _pad32(27 * (c["channels"] + 8)) + sum(co * 27 * (ca + cb) for _, ca, cb, co, _ in _layers(c))
        return dict(bytes=49 * n + 28 * weights, flops=6 * (head + conv) + 27 * 20 * n)
    a = min(c["nx"], c["nz"])  # magnet and plate cells, each added at each cell, in order
    magnets = math.pi * a ** 3 * ((0.4 ** 2 - 0.33 ** 2) * 0.1 + 0.15 ** 2 * 0.06)
    plates = 4 * 0.4 * c["nx"] * 0.2 * c["ny"]
    return dict(bytes=2 * (13 + 24) * n, flops=n * (magnets * 2 + plates * 6))


# ----------------------------------------------------------------------------------------------------------------------
# The same in 64 bits, in plain torch
# ----------------------------------------------------------------------------------------------------------------------
VELOCITIES = {
    "D2Q9": ((0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0), (1, -1, 0)),
    "D3Q15": ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 1), (1, 1, -1), (1, -1, 1), (-1, 1, 1)),
    "D3Q19": ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (1, 0, 1), (0, 1, 1), (1, -1, 0), (1, 0, -1), (0, 1, -1)),
    "D3Q7": ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)),
}
WEIGHTS = {"D2Q9": (4 / 9, 1 / 9, 1 / 36, 0), "D3Q15": (2 / 9, 1 / 9, 0, 1 / 72), "D3Q19": (1 / 3, 1 / 18, 1 / 36, 0)}
CLAMP = 0.57735027


class _Set64:
    """A velocity set: direction 2 p - 1 is the p-th of VELOCITIES, 2 p its opposite."""

    def __init__(self, name):
        self.v = [(0, 0, 0)]
        for v in VELOCITIES[name][1:]:
            self.v += [v, tuple(-k for k in v)]
        self.w = [WEIGHTS[name][sum(abs(k) for k in v)] for v in self.v] if name in WEIGHTS else None
        self.opp = [0] + [i + 1 if i % 2 else i - 1 for i in range(1, len(self.v))]

    def dot(self, i, u):
        s = 0.0
        for k in range(3):
            if self.v[i][k]:
                s = s + self.v[i][k] * u[k]
        return s

    def eq(self, i, rho, u, uu):
        cu = self.dot(i, u)
        return self.w[i] * (rho * (3 * cu + 4.5 * cu * cu - 1.5 * uu) + (rho - 1))

    def pull(self, f, i):
        """What arrives from direction i (periodic)."""
        x, y, z = self.v[i]
        return torch.roll(f[i], (z, y, x), (0, 1, 2)) if i else f[i]

    def force(self, i, u, F, uF):
        cu, cF = self.dot(i, u), self.dot(i, F)
        return 9 * self.w[i] * (cF * (cu + 1 / 3) - uF / 3)

    def all_eq(self, rho, u):
        uu = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
        return [self.eq(i, rho, u, uu) for i in range(len(self.v))]

    def moments(self, f):
        rho = sum(f) + 1
        u = []
        for k in range(3):
            s = torch.zeros_like(rho)
            for i, v in enumerate(self.v):
                if v[k]:
                    s += v[k] * f[i]
            u.append(s / rho)
        return rho, u

    def collide(self, f, rho, u, F, w, trt=False, eq_cells=None):
        """Relaxes f in place towards the equilibrium of (rho, u) with Guo's forcing."""
        uu = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
        uF = u[0] * F[0] + u[1] * F[1] + u[2] * F[2] if F is not None else None
        wm = 1 / (0.1875 / (1 / w - 0.5) + 0.5) if trt else w
        for i in [0] + list(range(1, len(self.v), 2)):
            j = self.opp[i]
            ei, ej = self.eq(i, rho, u, uu), self.eq(j, rho, u, uu)
            si, sj = (self.force(i, u, F, uF), self.force(j, u, F, uF)) if F is not None else (0.0, 0.0)
            even = 0.5 * (-w * (f[i] + f[j] - ei - ej) + (1 - w / 2) * (si + sj))
            odd = 0.5 * (-wm * (f[i] - f[j] - ei + ej) + (1 - wm / 2) * (si - sj))
            a, b = f[i] + even + odd, f[j] + even - odd
            if eq_cells is not None:
                a, b = torch.where(eq_cells, ei, a), torch.where(eq_cells, ej, b)
            f[i], f[j] = a, b


def _stream(S, f):
    return [S.pull(f, i) for i in range(len(S.v))]


def _after(S, post, pulled, solid):
    """Full-way bounce-back: solid cells turn round what arrives."""
    return [torch.where(solid, pulled[S.opp[i]], post[i]) for i in range(len(S.v))]


def _fluid64(c, seed):
    a = _fluid_inputs(c, seed)
    S = _Set64(c["set"])
    flags, rho, u = a["flags"], a["rho"].to(F64), [t.to(F64) for t in a["u"]]
    solid, eq_cells = flags == 1, (flags == 2) if c["channel"] else None
    u = [torch.where(solid, 0.0, t) for t in u]
    if c["set"] == "D2Q9":
        u[2] = u[2] * 0.0
    w = 1 / (0.1 + 0.5)
    F = [torch.full_like(rho, k) for k in FORCE] if c["channel"] else None
    f = S.all_eq(rho, u)
    for _ in range(c["steps"]):
        pulled = _stream(S, f)
        r, v = S.moments(pulled)
        if eq_cells is not None:
            r, v = torch.where(eq_cells, rho, r), [torch.where(eq_cells, s, t) for s, t in zip(u, v)]
        if F is not None:
            v = [t + 0.5 * k / r for t, k in zip(v, F)]
        v = [t.clamp(-CLAMP, CLAMP) for t in v]
        post = list(pulled)
        S.collide(post, r, v, F, w, c["relax"] == "Trt", eq_cells)
        f = _after(S, post, pulled, solid)
        keep = solid if eq_cells is None else solid | eq_cells
        rho, u = torch.where(keep, rho, r), [torch.where(keep, s, t) for s, t in zip(u, v)]
    return dict(RHO=rho.reshape(-1), U=torch.cat([t.reshape(-1) for t in u]))


def _constants(units):
    """Coulomb's and Biot-Savart's constants and the electron's mass over its charge, in lattice units."""
    m, kg, s, a = (units[k] for k in ("m", "kg", "s", "a"))
    eps0 = 8.8541878128e-12 / (a * a * s ** 4 / (kg * m ** 3))
    mu0 = 1.256637062e-6 / (kg * m / (a * a * s * s))
    return 1 / (4 * math.pi * eps0), mu0, 9.1093837139e-31 / -1.602176634e-19 / (kg / (a * s))


def _sums64(pos, src, weights, own=None, most=1 << 27):
    """sum_s weights[s] / |pos - src|^3 at each position, [len(pos)][columns]; `own`: a source that each position leaves
    out (-1: none). Distances come from exact products of half integers."""
    out = torch.empty(len(pos), weights.shape[1], dtype=F64, device=DEV)
    ss, step = (src * src).sum(1), max(1, most // max(1, len(src)))
    for i in range(0, len(pos), step):
        p = pos[i:i + step]
        r2 = torch.addmm(ss[None, :].expand(len(p), -1), p, src.t(), alpha=-2.0)
        r2 += (p * p).sum(1)[:, None]
        k = torch.where(r2 > 0.1, r2, math.inf).rsqrt_()
        if own is not None:
            o = own[i:i + step]
            at = (o >= 0).nonzero()[:, 0]
            k[at, o[at]] = 0.0
        out[i:i + step] = (k * k * k) @ weights
    return out


def _coulomb64(pos, src, q, v, own=None):
    """E and B sums (without their constants) at the positions, [6][len(pos)]: q r / r^3 and q v x r / r^3."""
    J = q[:, None] * v
    S = _sums64(pos, src, torch.cat([q[:, None], q[:, None] * src, J, torch.cross(J, src, dim=1)], 1), own)
    E = S[:, :1] * pos - S[:, 1:4]
    B = torch.cross(S[:, 4:7], pos, dim=1) - S[:, 7:10]
    return torch.cat([E, B], 1).t()


def _lod_field64(c, top):
    """Field sums [6][nz][ny][nx] of the LOD sums top[8^depth][4]. The field step reads the LOD indices from
    n_lod - 8^depth on, and leaves out a cell's own block."""
    nd = 1 << c["depth"]
    lo = _n_lod(c["depth"]) - nd ** 3
    b = [c[s] // nd for s in ("nx", "ny", "nz")]
    d = torch.arange(lo, nd ** 3, device=DEV)
    src = torch.stack([(d % nd + 0.5) * b[0], (d // nd % nd + 0.5) * b[1], (d // nd ** 2 + 0.5) * b[2]], 1).to(F64)
    x, y, z = _coords(c, torch.int64)
    own = (x // b[0] + nd * (y // b[1] + nd * (z // b[2]))).reshape(-1) - lo
    shape = (c["nz"], c["ny"], c["nx"])
    pos = torch.stack([t.expand(shape).reshape(-1) for t in (x, y, z)], 1).to(F64)
    t = top[lo:].to(F64)
    return _coulomb64(pos, src, t[:, 0], t[:, 1:], own).reshape(6, *shape)


def _mhd64(c, seed):
    nd = 1 << c["depth"]
    if _cells(c) * 8 ** c["depth"] * c["steps"] > 8e11:
        return None  # too long in 64 bits
    a = _mhd_inputs(c, seed)
    S, D7 = _Set64("D3Q19"), _Set64("D3Q7")
    ke, mu0, kkge = _constants(scenarios.PLASMA_UNITS)
    kmu, w, wq = mu0 / (4 * math.pi), 1 / (0.1 + 0.5), 0.4
    flags = a["flags"]
    solid, eq_cells = flags == 1, (flags == 2) if c["geometry"] == "tube" else None
    u = [torch.where(solid, 0.0, t.to(F64)) for t in a["u"]]
    q = torch.where(solid, 0.0, a["q"].to(F64))
    rho = torch.ones_like(q)
    b_stat = [t.to(F64) for t in a["b_stat"]]
    E, B = [torch.zeros_like(q) for _ in range(3)], list(b_stat)

    def a_eq(Q, u):
        out = [0.25 * (Q - 1)]
        for k in range(3):
            out += [0.5 * Q * u[k] + 0.125 * (Q - 1), -0.5 * Q * u[k] + 0.125 * (Q - 1)]
        return out

    def pick(x, y):
        return y if eq_cells is None else torch.where(eq_cells, x, y)

    def cross(p, r):
        return [p[1] * r[2] - p[2] * r[1], p[2] * r[0] - p[0] * r[2], p[0] * r[1] - p[1] * r[0]]

    f, h = S.all_eq(rho, u), a_eq(q, u)
    e = S.all_eq(torch.where(solid, 0.0, torch.full_like(q, BACKGROUND)), u)
    for _ in range(c["steps"]):
        pf, pe, ph = _stream(S, f), _stream(S, e), _stream(D7, h)
        r, v = S.moments(pf)
        r, v = pick(rho, r), [pick(s, t) for s, t in zip(u, v)]
        re, ve = S.moments(pe)
        rq = pick(q, sum(ph) + 1)  # inlet and outlet cells hold their charge
        charge = rq - re
        qeq = a_eq(rq, v)
        nh = [pick(k, (1 - wq) * p + wq * k) for p, k in zip(ph, qeq)]
        Fe = [-re * (x + y) for x, y in zip(E, cross(ve, B))]
        ve = [(t + 0.5 * k / (re * kkge)).clamp(-CLAMP, CLAMP) for t, k in zip(ve, Fe)]
        ne = list(pe)
        S.collide(ne, re, ve, Fe, w, eq_cells=eq_cells)
        F = [rq * (x + y) for x, y in zip(E, cross(v, B))]
        # LOD sums: charge, and mean velocity over the block's cells
        live = ~solid
        top = torch.stack([torch.where(live, t, 0.0).reshape(nd, c["nz"] // nd, nd, c["ny"] // nd, nd, c["nx"] // nd)
                           .sum((1, 3, 5)).reshape(-1) for t in (charge, *v)], 1)
        top[:, 1:] /= _cells(c) / nd ** 3
        v = [(t + 0.5 * k / r).clamp(-CLAMP, CLAMP) for t, k in zip(v, F)]
        nf = list(pf)
        S.collide(nf, r, v, F, w, eq_cells=eq_cells)
        f, e, h = _after(S, nf, pf, solid), _after(S, ne, pe, solid), _after(D7, nh, ph, solid)
        keep = solid if eq_cells is None else solid | eq_cells
        rho, u, q = torch.where(keep, rho, r), [torch.where(keep, s, t) for s, t in zip(u, v)], torch.where(keep, q, charge)
        sums = _lod_field64(c, top)
        E = [torch.where(solid, s, ke * t) for s, t in zip(E, sums[:3])]
        B = [torch.where(solid, s, x + kmu * t) for s, x, t in zip(B, b_stat, sums[3:])]
    flat = [torch.cat([t.reshape(-1) for t in k]) for k in (u, E, B)]
    return dict(U=flat[0], Q=q.reshape(-1), E_DYN=flat[1], B_DYN=flat[2])


def _field64(c, seed):
    a = _field_inputs(c, seed)
    ke, mu0, _ = _constants(scenarios.PLASMA_UNITS)
    sums = _lod_field64(c, a["qu_lod"].reshape(-1, 4)[:8 ** c["depth"]]).reshape(6, -1)
    solid = a["flags"] == 1
    out = {}
    for name, k, part in (("e", ke, sums[:3]), ("b", mu0 / (4 * math.pi), sums[3:])):
        out[name] = torch.where(solid, 0.0, a[name + "_stat"].to(F64).reshape(3, -1) + k * part).reshape(-1)
    return out


def _train64(c, seed):
    nd, c0 = 1 << c["depth"], c["channels"]
    lo = _n_lod(c["depth"]) - nd ** 3
    top = _lod(c, seed, _n_lod(c["depth"]))[:nd ** 3]
    b = [c[s] // nd for s in ("nx", "ny", "nz")]
    cpb = b[0] * b[1] * b[2]
    gain = cpb ** (2 / 3)
    # the network's input: charge and current over their largest values, as a bf16 value and its bf16 remainder
    J = top[:, :1] * top[:, 1:]
    sq, sj = top[:, 0].abs().max(), J.abs().max()
    x = torch.cat([top[:, :1] / sq, J / sj], 1)
    x[:lo] = 0.0
    hi = x.bfloat16().float()
    x = torch.cat([hi, (x - hi).bfloat16().float()], 1).to(F64)  # [voxel][8]
    x = x.t().reshape(1, 8, nd, nd, nd)
    P = [w.to(F64).requires_grad_() for w in _weights(c, seed)]

    def columns(t):
        """[voxels][27 * channels] of the 3^3 neighbourhoods, the neighbour slowest."""
        g, ch = t.shape[-1], t.shape[1]
        p = torch.nn.functional.pad(t, (1,) * 6)
        nb = [p[0, :, dz:dz + g, dy:dy + g, dx:dx + g] for dz in range(3) for dy in range(3) for dx in range(3)]
        return torch.stack(nb).reshape(27 * ch, -1).t()

    def conv(i, t):
        col, g = columns(t), t.shape[-1]
        return (col @ P[i][:, :col.shape[1]].t()).t().reshape(1, -1, g, g, g)

    def pool(t):
        return torch.nn.functional.avg_pool3d(t, 2)

    def up(t):
        return t.repeat_interleave(2, 2).repeat_interleave(2, 3).repeat_interleave(2, 4)

    e0 = conv(0, x)
    e1 = conv(1, pool(e0))
    e2 = conv(2, pool(e1))
    e3 = conv(3, pool(e2))
    d2 = conv(4, torch.cat([up(e3), e2], 1))
    d1 = conv(5, torch.cat([up(d2), e1], 1))
    d0 = conv(6, torch.cat([up(d1), e0], 1))
    col = columns(torch.cat([d0, x], 1))
    y = (col @ P[7][:, :col.shape[1]].t()).reshape(nd ** 3, 6, cpb)
    # far field: every source outside the block's 3^3 neighbourhood at 3^3 points of the block, interpolated
    d = torch.arange(lo, nd ** 3, device=DEV)
    sb = torch.stack([d % nd, d // nd % nd, d // nd ** 2], 1)
    bt = torch.tensor(b, device=DEV, dtype=F64)
    src = (sb + 0.5) * bt
    t = top[lo:].to(F64)
    q, v = t[:, 0], t[:, 1:]
    k3 = (torch.arange(3, device=DEV, dtype=F64) + 0.5) / 3
    pts = torch.stack([k3[p] for p in torch.meshgrid(*(torch.arange(3, device=DEV),) * 3, indexing="ij")[::-1]], -1).reshape(27, 3)
    blk = torch.arange(nd ** 3, device=DEV)
    bb = torch.stack([blk % nd, blk // nd % nd, blk // nd ** 2], 1)
    far = torch.empty(nd ** 3, 6, 27, dtype=F64, device=DEV)
    near = ((bb[:, None] - sb[None]).abs() <= 1).all(-1)
    for p in range(27):
        pos = bb * bt + pts[p] * bt - 0.5
        r = pos[:, None] - src[None]
        k = torch.where(near, 0.0, (r * r).sum(-1) ** -1.5) * q
        far[:, :3, p] = (k[..., None] * r).sum(1)
        far[:, 3:, p] = (k[..., None] * torch.cross(v[None].expand_as(r), r, dim=-1)).sum(1)
    L = []
    for n in b:
        s = (torch.arange(n, device=DEV, dtype=F64) - (0.5 * n / 3 - 0.5)) / (n / 3)
        L.append(torch.stack([0.5 * (s - 1) * (s - 2), -s * (s - 2), 0.5 * s * (s - 1)]))
    inter = torch.einsum("iz,jy,kx->ijkzyx", L[2], L[1], L[0]).reshape(27, cpb)
    scale = torch.tensor([1 / sq.double()] * 3 + [1 / sj.double()] * 3, device=DEV, dtype=F64)[None, :, None] * gain
    y = y + (far.reshape(-1, 27) @ inter).reshape(nd ** 3, 6, cpb) * scale
    raw = _lod_field64(c, top).reshape(6, nd, b[2], nd, b[1], nd, b[0]).permute(1, 3, 5, 0, 2, 4, 6).reshape(nd ** 3, 6, cpb)
    want = raw * scale
    rel = [((y - want)[:, s] ** 2).sum() / (want[:, s] ** 2).sum() for s in (slice(0, 3), slice(3, 6))]
    (rel[0] + rel[1]).backward()
    return dict(rel=torch.stack([r.detach().sqrt() for r in rel]), grads=torch.cat([p.grad.reshape(-1) for p in P]))


def _static64(c, seed):
    a = _static_inputs(c, seed)
    ke, mu0, _ = _constants(scenarios.PLASMA_UNITS)
    flags, val = a["flags"], a["b_dyn"].to(F64)
    shape = (c["nz"], c["ny"], c["nx"])

    def cells(mask):
        at = mask.nonzero()
        return at.flip(1).to(F64), val[:, at[:, 0], at[:, 1], at[:, 2]].t()

    src, M = cells(flags == 0x11)
    padded = [torch.arange(n + 2, device=DEV, dtype=F64) - 1 for n in shape]
    pos = torch.stack(torch.meshgrid(*padded, indexing="ij")[::-1], -1).reshape(-1, 3)
    S = _sums64(pos, src, torch.cat([M, (M * src).sum(1, keepdim=True)], 1))
    psi = ((S[:, :3] * pos).sum(1) - S[:, 3]).reshape(*(n + 2 for n in shape)) / (4 * math.pi)
    free = (flags & 1) == 0
    B = [-mu0 * 0.5 * g for g in (psi[1:-1, 1:-1, 2:] - psi[1:-1, 1:-1, :-2], psi[1:-1, 2:, 1:-1] - psi[1:-1, :-2, 1:-1],
                                  psi[2:, 1:-1, 1:-1] - psi[:-2, 1:-1, 1:-1])]
    src, Q = cells(flags == 0x05)
    x, y, z = _coords(c, F64)
    pos = torch.stack([t.expand(shape).reshape(-1) for t in (x, y, z)], 1)
    S = _sums64(pos, src, torch.cat([Q[:, :1], Q[:, :1] * src], 1))
    E = (ke * (S[:, :1] * pos - S[:, 1:])).t().reshape(3, *shape)
    flat = [torch.cat([torch.where(free, t, 0.0).reshape(-1) for t in k]) for k in (E, B)]
    return dict(E_STAT=flat[0], B_STAT=flat[1])


def exact(case, seed):
    return {"fluid": _fluid64, "mhd": _mhd64, "field": _field64, "train": _train64, "static": _static64}[case["kind"]](case, seed)
