"""Each launch form of the step kernels against the FP64 oracle, at the sizes
where the form changes or its last block is partial.

FP64 lattices: every population bit-identical (the kernels keep the
reference's evaluation order).  Float storage: relative L2 error of the
velocity at most 1e-5 of the oracle's, the bar of every float comparison in
this suite.
"""
import numpy as np
import pytest

from ch4g import abi, Lattice
from oracle import Oracle
import configs

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return np.sqrt(((a - b) ** 2).sum() / (b * b).sum())


def run(x, steps):
    x.initial_conditions()
    x.step(steps)
    return x


# Block orders (step_order): FP64 beyond 1.5 GiB and float beyond 320 MiB of
# state go in groups of 64 blocks with non-temporal stores where these are
# whole lines; 113-wide float rows and 500-wide ones (no whole lines) take the
# linear grid, 128-wide ones the row grid.  Block counts that are no multiple
# of 64 leave a partial last group.
@pytest.mark.parametrize("shape,precision", [
    ((113, 97, 103), abi.FP32_DEV), ((128, 95, 93), abi.FP32_DEV), ((500, 49, 47), abi.FP32_DEV),
    ((140, 139, 141), abi.FP64), ((256, 97, 111), abi.FP64)], ids=str)
def test_streamed_block_order(shape, precision):
    cfg = configs.rb2d(*shape, Ra=1e6, precision=precision, seed=5)
    o = run(Oracle(cfg.copy(precision=abi.FP64)), 4)
    lat = Lattice(cfg)
    lat.set_fusion(False)
    run(lat, 4)
    if precision == abi.FP64:
        (p, g), (po, go) = lat.get_populations(), o.get_populations()
        assert np.array_equal(p, po) and np.array_equal(g, go)
    else:
        err = rel_l2(lat.hydro_fields()["u"], o.hydro_fields()["u"])
        print(f"  {shape}: L2 rel err of u {err:.2e}")
        assert err <= 1e-5
    lat.close()


# 3-D two-step launches below 2^21 nodes: in cache (96^3), streamed with rows
# that are no whole lines (plain stores) or half lines, a channel, partial
# tiles in x and y and a shorter last z range.  Equal, bit for bit, to the same
# lattice advanced one step per launch.
@pytest.mark.parametrize("shape,channel", [((96, 96, 96), False), ((125, 113, 101), False), ((208, 63, 90), False),
                                           ((113, 113, 113), True)], ids=str)
def test_small_3d_two_step_launches(shape, channel):
    from ch4g import workloads
    cfg = workloads.channel3d(*shape) if channel else configs.rb2d(*shape, Ra=1e6, precision=abi.FP32_DEV, seed=5)
    two, one = Lattice(cfg), Lattice(cfg)
    one.set_fusion(False)
    assert (two.steps_per_launch(), one.steps_per_launch()) == (2, 1)
    for lat in (two, one):
        run(lat, 8)
    for a, b in zip(two.get_populations(), one.get_populations()):
        assert np.array_equal(a, b)
    two.close()
    one.close()


# FP64 two-step launches.  2-D: one tile that is narrower and one that is
# shorter than 32 x 4, exact tiles, partial tiles in x and y, a streamed lattice
# with non-temporal stores, a channel.  3-D of few columns (slabs of rows): one
# row more than the last slab, fewer rows than a slab, exact slabs, two rows a
# slab.  3-D: whole tiles with non-temporal stores; partial
# tiles in x and y and a shorter last z range; a channel in cache (61: one
# narrow tile) and one streamed with rows that are no whole lines.  Random
# populations, so that every direction differs; equal, bit for bit, to the same
# lattice advanced one step per launch.
@pytest.mark.parametrize("shape,channel", [((20, 3, 1), False), ((64, 32, 1), False), ((45, 27, 1), False),
                                           ((1040, 630, 1), False), ((130, 61, 1), True), ((4, 15, 4), True),
                                           ((1, 3, 2), False), ((5, 10, 7), False), ((8, 64, 8), False),
                                           ((96, 80, 112), False), ((93, 79, 110), False), ((125, 113, 101), False),
                                           ((61, 61, 240), True), ((113, 113, 113), True)], ids=str)
def test_fp64_two_step_launches(shape, channel):
    from ch4g import workloads
    if channel:
        cfg = workloads.channel3d(*shape, precision=abi.FP64)
    else:
        cfg = configs.rb2d(*shape, Ra=1e6, precision=abi.FP64, seed=5)
    two, one = Lattice(cfg), Lattice(cfg)
    one.set_fusion(False)
    assert (two.steps_per_launch(), one.steps_per_launch()) == (2, 1)
    two.initial_conditions()
    p, g = two.get_populations()
    rng = np.random.default_rng(3)
    p = p * (1.0 + 1e-2 * rng.uniform(-1, 1, p.shape))
    if not channel:
        g = g * (1.0 + 1e-2 * rng.uniform(-1, 1, g.shape))
    for lat in (two, one):
        lat.set_populations(p, None if channel else g)
        lat.step(1)
        lat.step(7)
        lat.step(34)
    for a, b in zip(two.get_populations(), one.get_populations()):
        assert np.array_equal(a, b)
    two.close()
    one.close()


# FP64 2-D lattices in one batch, two steps per launch and a single one for odd
# counts: narrower than a tile, exact tiles, partial tiles, a channel, and a
# float lattice beside them.  Equal, bit for bit, to each alone in single steps.
def test_fp64_batched_two_steps():
    from ch4g import step_batch, workloads
    cfgs = [configs.rb2d(20, 3, 1, Ra=1e4, seed=3), configs.rb2d(64, 32, 1, Ra=1e5, seed=4),
            configs.rb2d(45, 27, 1, Ra=1e5, seed=5), workloads.channel3d(130, 61, 1, precision=abi.FP64),
            configs.rb2d(96, 48, 1, Ra=1e5, precision=abi.FP32_DEV, seed=6)]
    many, one = [Lattice(c) for c in cfgs], [Lattice(c) for c in cfgs]
    for lat in many + one:
        run(lat, 1)
    for lat in one:
        lat.set_fusion(False)
    for n in (1, 7, 10, 2):
        step_batch(many, n)
        for a, b in zip(many, one):
            b.step(n)
            for x, y in zip(a.get_populations(), b.get_populations()):
                assert np.array_equal(x, y), (n, a.cfg.NX)
    for lat in many + one:
        lat.close()


# The averages' and rulers' marches: fewer rows, columns or planes than one
# wave covers, a last wave, row group, z chunk and unit that are partial
# (1 x 300 x 2048: 16 rows per wave of the plane sums, two of the column sums,
# several units per block).  Tolerance: sums of up to N terms in another
# order, N eps of the largest member (614400 * 2.2e-16 = 1.4e-10 at most).
@pytest.mark.parametrize("shape", [(3, 5, 2), (64, 3, 1), (65, 7, 33), (130, 41, 70), (1, 300, 2048)], ids=str)
def test_diagnostics_at_partial_waves(shape):
    cfg = configs.rb2d(*shape, Ra=1e4, seed=9, noise=0.05)
    o, lat = run(Oracle(cfg), 3), run(Lattice(cfg), 3)
    eps = cfg.nodes() * 2.3e-16
    got, want = lat.dump_averages(), o.dump_averages()
    flux = max(abs(want[k]) for k in want if k not in ("x", "y", "z"))
    for k in want:
        assert abs(got[k] - want[k]) <= eps * max(abs(want[k]), flux), (k, got[k], want[k])
    for r, w in zip(lat.dump_rulers(), o.dump_rulers()[1:]):
        a, b = r.view(np.float64).reshape(len(r), -1), w.view(np.float64).reshape(len(w), -1)
        assert np.abs(a - b).max() <= eps * np.abs(b).max()
    lat.close()


# FP64 collisions leave out products by zero velocity components; what those
# products do to numbers that are not finite has to remain: populations equal
# to the oracle's, NaN where it has NaN, infinities included.
@pytest.mark.parametrize("cfg", [configs.rb2d(20, 9, 5, Ra=1e4), configs.rb2d(64, 8, 3, Ra=1e4),
                                 configs.poiseuille(12, 10, 6, tau=0.8), configs.hit(10, les="local")],
                         ids=["rb_dense", "rb_rows", "channel", "hit_les"])
def test_fp64_numbers_that_are_not_finite(cfg):
    rng = np.random.default_rng(3)
    w = np.array([1 / 3] + [1 / 18] * 6 + [1 / 36] * 12)
    shape = (cfg.NZ, cfg.NY, cfg.NX)
    p = w * (1.0 + 0.01 * rng.standard_normal(shape + (19,)))
    g = w * (0.5 + 0.01 * rng.standard_normal(shape + (19,)))
    p[1, 2, 3, 0], p[2, 4, 9, 7], p[0, 5, 6, 3], p[2, 7, 1, 12] = np.inf, np.nan, 1e300, -np.inf
    g[1, 6, 7, 5], g[0, 3, 3, 0], g[2, 1, 8, 16] = np.inf, np.nan, -1e300
    lat, o = Lattice(cfg), Oracle(cfg)
    for x in (lat, o):
        x.set_populations(p, g if cfg.has(abi.LB_TEMPERATURE) else None)
        x.step(2)
    for a, b in zip(lat.get_populations(), o.get_populations()):
        assert np.array_equal(a, b, equal_nan=True)
    assert np.isnan(o.get_populations()[0]).any()
    lat.close()


# Records read back in chunks of 65536 live particles: one particle, chunk
# edges, particles dropped (x = -1e-18 wraps onto the upper face) at the
# edges, all of them, and a caller's array shorter than the live count.
@pytest.mark.parametrize("n,dead", [(1, []), (1, [0]), (65536, []), (65537, [0, 65536]), (131073, [65535, 65536, 70000])],
                         ids=str)
def test_particle_records_in_chunks(n, dead):
    import ctypes as C
    lat = Lattice(configs.poiseuille(8, 8, 8, tau=0.8, g=0.0))
    lat.initial_conditions()
    lat.particles_init(abi.make_particle_config(abi.LAGRANGE_WRAP, 1))
    rng = np.random.default_rng(n)
    a = np.zeros(n, dtype=abi.particle_dtype())
    for k in a.dtype.names:
        a[k] = rng.uniform(1.0, 7.0, n)
    a["name"], a["tau_drag"] = np.arange(n), 0.0
    for k in ("vx_old", "vy_old", "vz_old"):  # tracers of a fluid at rest stay where they are
        a[k] = 0.0
    a["x"][dead] = -1e-18
    lat.set_particles(a)
    back = lat.particles()
    assert all(np.array_equal(back[k], a[k]) for k in a.dtype.names)
    lat.step(1)
    alive = np.setdiff1d(np.arange(n), dead)
    back = lat.particles()
    assert np.array_equal(back["name"], alive) and np.array_equal(back["y"], a["y"][alive])
    assert np.array_equal(back["jump_time"], a["jump_time"][alive])
    short = np.zeros(max(len(alive) // 2, 1) + 1, dtype=a.dtype)
    got = C.c_int64()
    cap = len(short) - 1
    assert lat._L.ch4g_get_particles(lat.handle, short.ctypes.data, cap, C.byref(got)) == 0
    assert got.value == len(alive)
    m = min(cap, len(alive))
    assert np.array_equal(short[:m], back[:m]) and not short[-1:].view(np.float64).any()
    lat.close()


# HIT tables made ahead (batches of 1, 2, 4, 8, 8, ... steps in a call, cut at
# its end): calls of every length to past three batches, one step at a time,
# and new phases between calls give the same states, bit for bit, and the
# oracle's phases; also with the drand48 stream on the device (randomly
# oriented particles draw from it between two steps' walks).
@pytest.mark.parametrize("shape,draws", [(12, False), (19, False), (12, True)], ids=str)
def test_hit_tables_ahead(shape, draws):
    cfg = configs.hit(shape, tau=0.55, amp=1e-4, les=False)
    calls = [1, 2, 3, 7, 8, 9, 15, 16, 17, 31]
    if draws:
        flags = (abi.LAGRANGE_ADD_TRACER | abi.LAGRANGE_WRAP | abi.LAGRANGE_GRADIENT | abi.LAGRANGE_ADDEDMASS |
                 abi.LAGRANGE_ORIENTATION | abi.LAGRANGE_ORIENTATION_JEFFREY)
        pc = abi.make_particle_config(flags, 50, aspect_ratio=(2, 0.5, 4.0), flags2=abi.LAGRANGE_ORIENTATION_RANDOM)

    def advance(x, single):
        x.initial_conditions()
        if draws:
            x.particles_init(pc)
        for n in calls:
            if single:
                for _ in range(n):
                    x.step(1)
            else:
                x.step(n)
        return x

    a, b, o = advance(Lattice(cfg), False), advance(Lattice(cfg), True), advance(Oracle(cfg), False)
    np.testing.assert_array_equal(a.hit_phases(), o.hit_phases())
    np.testing.assert_array_equal(b.hit_phases(), o.hit_phases())
    pa, pb = a.get_populations()[0], b.get_populations()[0]
    assert np.array_equal(pa, pb)
    new = o.hit_phases()[::-1] * 0.5 + 0.125
    for x in (a, b):
        x.set_hit_phases(new)
    a.step(5)
    for _ in range(5):
        b.step(1)
    assert np.array_equal(a.get_populations()[0], b.get_populations()[0])
    a.close()
    b.close()


# The interpolation with gradients, eight lanes a particle: counts around a wave
# (8) and a block (32), particles on and beside the walls and the periodic faces,
# fluid and temperature together, fluid alone, and walls of the fluid only (the
# two fields read apart).  FP64: every field as the oracle's, bit for bit.
@pytest.mark.parametrize("n", [1, 7, 33])
@pytest.mark.parametrize("kind", ["both", "fluid", "apart"])
def test_gradient_interpolation_counts(kind, n):
    cfg = configs.rb2d(12, 10, 7, Ra=1e4, seed=5, noise=0.05)
    if kind == "fluid":
        cfg = configs.poiseuille(12, 10, 7, tau=0.8, g=1e-4)
    if kind == "apart":
        cfg.flags &= ~abi.TEMPERATURE_BC_Y
    flags = abi.LAGRANGE_WRAP | abi.LAGRANGE_GRADIENT | abi.LAGRANGE_ADDEDMASS
    rng = np.random.default_rng(n)
    a = np.zeros(n, dtype=abi.particle_dtype())
    a["name"], a["tau_drag"], a["beta_coeff"] = np.arange(n), 5.0, 0.8
    for axis, m in (("x", 12.0), ("y", 10.0), ("z", 7.0)):
        a[axis] = rng.uniform(0.0, m, n)
    a["y"][:2], a["x"][2:4], a["z"][4:6] = (0.2, 9.9)[:min(n, 2)], (0.1, 11.9)[:max(0, min(n - 2, 2))], \
        (0.1, 6.9)[:max(0, min(n - 4, 2))]
    got = []
    for x in (Oracle(cfg), Lattice(cfg)):
        x.initial_conditions()
        x.particles_init(abi.make_particle_config(flags, 1, tau_drag=(1, 5.0, 5.0), beta_coeff=(1, 0.8, 0.8)))
        x.set_particles(a)
        x.step(6)
        got.append(x.particles())
    for f in abi.PARTICLE_FIELDS:
        assert np.array_equal(got[0][f], got[1][f], equal_nan=True), f


# FP64 members of a batch that take one step per launch there (k_step_batch64:
# linear and row grids, with and without temperature, temperature alone, the
# local-strain closure; lattices of few columns, two of them; streamed in groups
# of blocks with non-temporal stores) and a z-marching lattice on its own branch
# beside them.  Random populations; equal, bit for bit, to each alone in single
# steps, for odd and even counts.
@pytest.mark.parametrize("kind", ["small", "les", "branch", "streamed"])
def test_fp64_batched_single_steps(kind):
    from ch4g import step_batch, workloads
    rb, ch = configs.rb2d, workloads.channel3d

    def les(cfg):
        cfg.flags |= abi.FLUID_LES | abi.FLUID_LES_LOCAL_STRAIN
        if cfg.has(abi.LB_TEMPERATURE):
            cfg.flags |= abi.TEMPERATURE_LES
        cfg.les_cs = 0.1
        return cfg

    conduction = rb(40, 12, 9, Ra=1e4)
    conduction.flags &= ~(abi.LB_FLUID | abi.TEMPERATURE_BUOYANCY | abi.FLUID_BC_Y)
    cfgs = {"small": [rb(48, 40, 30, Ra=1e5), rb(64, 24, 20, Ra=1e5), ch(40, 24, 20, precision=abi.FP64),
                      ch(128, 20, 12, precision=abi.FP64), conduction, ch(4, 16, 4, precision=abi.FP64),
                      rb(5, 10, 7, Ra=1e4)],
            "les": [les(rb(20, 14, 9, Ra=1e5)), les(rb(64, 9, 5, Ra=1e5)), les(ch(61, 17, 8, precision=abi.FP64))],
            "branch": [rb(96, 80, 112, Ra=1e6), ch(24, 20, 16, precision=abi.FP64), ch(8, 24, 6, precision=abi.FP64)],
            "streamed": [les(rb(128, 160, 130, Ra=1e6))]}[kind]
    many, one = [Lattice(c) for c in cfgs], [Lattice(c) for c in cfgs]
    two = [lat.steps_per_launch() == 2 for lat in many]
    assert two == {"small": [False] * 5 + [True] * 2, "les": [False] * 3, "branch": [True, False, True],
                   "streamed": [False]}[kind]
    rng = np.random.default_rng(8)
    for a, b in zip(many, one):
        b.set_fusion(False)
        a.initial_conditions()
        p, g = (x * (1.0 + 1e-2 * rng.uniform(-1, 1, x.shape)) for x in a.get_populations())
        for lat in (a, b):
            lat.set_populations(p, g if a.cfg.has(abi.LB_TEMPERATURE) else None)
            lat.step(1)
    for n in (1, 7, 10) if kind != "streamed" else (3,):
        step_batch(many, n)
        for a, b in zip(many, one):
            b.step(n)
            for x, y in zip(a.get_populations(), b.get_populations()):
                assert np.array_equal(x, y), (n, a.cfg.NX, a.cfg.NY, a.cfg.NZ)
            assert np.isfinite(a.get_populations()[0]).all()
    for lat in many + one:
        lat.close()


# Records of few particles (formed on the host), some dropped, rows in cell order.
@pytest.mark.parametrize("n,dead", [(100, [0, 7, 99]), (600, []), (601, [600])], ids=str)
def test_few_particle_records(n, dead):
    test_particle_records_in_chunks(n, dead)


# The same for lattices narrower than a wave, several groups of rows in one:
# every power of two and its neighbours, with a partial last group.
@pytest.mark.parametrize("shape", [(1, 3, 1), (1, 200, 130), (2, 131, 3), (5, 70, 33), (8, 67, 9), (17, 37, 5),
                                   (32, 9, 4), (33, 10, 4)], ids=str)
def test_diagnostics_of_narrow_lattices(shape):
    test_diagnostics_at_partial_waves(shape)
