"""The host side of libch4g.so with the HIP runtime replaced by hip_stub.cpp
(host memory, no kernel runs, launches counted by name): what is launched,
allocated and given back, and what happens when an allocation fails.  Each case
is a program of its own, so that the stub stays out of this process."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = f"""
import ctypes as C, sys
sys.path[:0] = [{os.path.join(ROOT, 'ch4-project_amd')!r}, {HERE!r}]
S = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
S.stub_launches.restype = S.stub_streams_made.restype = S.stub_captures.restype = C.c_long
S.stub_live_bytes.restype = S.stub_peak_bytes.restype = C.c_size_t
S.stub_fail.argtypes = [C.c_size_t, C.c_long, C.c_long]
import numpy as np
from ch4g import abi, footprint_bytes, Lattice, serve, step_batch, workloads
import configs

def started(cfg, n=1):
    lat = Lattice(cfg)
    lat.initial_conditions()
    lat.step(n)
    return lat

def launches(part=b"k_"):
    return S.stub_launches(part)
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = tmp_path_factory.mktemp("stub") / "hip_stub.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub.cpp"), "-o", str(so)], check=True)
    return str(so)


@pytest.fixture
def run(stub):
    def go(code):
        r = subprocess.run([sys.executable, "-c", PRELUDE + code, stub], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return go


# Ensembles of FP64 3-D lattices of few columns: one batched launch per step for
# all of them on the batch's stream, whatever their number; one alone keeps its
# two steps per launch.
@pytest.mark.parametrize("n", [2, 3, 32])
def test_few_column_ensembles_share_their_launches(run, n):
    run(f"""
lats = [started(workloads.channel3d(*s, tau=1.0, precision=abi.FP64)) for s in
        [(4, 64, 4), (8, 24, 6), (8, 64, 8)] * 11][:{n}]
S.stub_reset()
step_batch(lats, 7)
assert launches(b"k_step_batch64") == launches() == 7, launches()
assert S.stub_streams_made() == 1, S.stub_streams_made()
S.stub_reset()
step_batch(lats[:1], 7)
assert launches(b"k_step2y_fp64") == 3 and launches() == 4, launches()
""")


# A served stream (arrivals, odd shares, a rebuilt table, jobs of every group)
# captures no graph while jobs run together.
def test_served_chunks_are_launched_not_captured(run):
    run("""
cfgs = [workloads.rb2d(48, 24, 1, Ra=2e5, precision=abi.FP64), workloads.channel3d(8, 24, 6, precision=abi.FP64),
        workloads.rb2d(96, 48, 1, Ra=1e6), workloads.channel3d(40, 24, 20)]
jobs = []
for i, cfg in enumerate(cfgs):
    j = abi.Job()
    j.cfg, j.nsteps, j.arrival_s = cfg, 60 - 7 * i, 0.001 * i
    jobs.append(j)
for schedule in (abi.SCHEDULE_LOCKSTEP, abi.SCHEDULE_PROPORTIONAL):
    done = serve([abi.Job.from_buffer_copy(j) for j in jobs], mode=abi.SERVE_BATCHED, chunk_steps=7,
                 use_graphs=True, schedule=schedule)
    assert all(d.status == 0 for d in done)
    assert S.stub_captures() == 0 and launches(b"k_step_batch32") > 0 and launches(b"k_step2_batch64") > 0
""")


# Lattices on branches of their own share a bounded number of streams.
def test_branches_share_streams(run):
    run("""
lats = [started(workloads.channel3d(64, 64, 256)) for _ in range(20)]
assert lats[0].steps_per_launch() == 2
S.stub_reset()
step_batch(lats, 4)
assert launches(b"k_step2z_fp32") == launches() == 40
assert S.stub_streams_made() <= 1 + 8, S.stub_streams_made()
""")


# A served job never holds more than the budget, the second lag array of two
# steps per launch included; where only that does not fit, it takes single steps.
@pytest.mark.parametrize("mode", ["SERVE_BATCHED", "SERVE_SEQUENTIAL"])
@pytest.mark.parametrize("precision", ["FP64", "FP32_DEV"])
def test_served_job_stays_in_its_budget(run, mode, precision):
    run(f"""
cfg = workloads.rb2d(1024, 512, 1, Ra=1e6, precision=abi.{precision})
real = 8 if cfg.precision == abi.FP64 else 4
tables = 1 << 18  # of the batch
need = footprint_bytes(cfg) + 40 * cfg.nodes() + (1 << 20)
for extra, two in ((0, False), (real * cfg.nodes() + tables, True)):
    job = abi.Job()
    job.cfg, job.nsteps = cfg, 9
    S.stub_reset()
    done = serve([job], mode=abi.{mode}, hbm_budget=need + extra)
    assert done[0].status == 0
    assert S.stub_peak_bytes() <= need + extra, (S.stub_peak_bytes(), need + extra)
    assert (launches(b"k_step2") > 0) == two
job = abi.Job()
job.cfg, job.nsteps = cfg, 9
assert serve([job], mode=abi.{mode}, hbm_budget=need - 1)[0].status < 0
""")


# No memory for the second lag array: single steps in that call, two per launch
# again once there is room; ch4g_set_fusion's setting is the caller's alone.
def test_two_steps_return_when_memory_does(run):
    run("""
for cfg in (workloads.rb2d(512, 128, 1, precision=abi.FP64), workloads.rb2d(512, 128, 1, precision=abi.FP32_DEV)):
    lat = started(cfg)
    S.stub_fail(4 * cfg.nodes(), 0, 1000)
    S.stub_reset()
    lat.step(70)
    assert launches(b"k_step2") == 0 and launches(b"k_step_fp") > 0 and lat.itime == 71
    step_batch([lat], 5)
    assert launches(b"k_step2") == 0 and launches(b"k_step_batch") == 5
    S.stub_fail(0, 0, 0)
    S.stub_reset()
    lat.step(70)
    assert launches(b"k_step_fp") == 0 and launches(b"k_step2_fp") == 16 + 3 and lat.itime == 146
    S.stub_reset()
    step_batch([lat], 4)
    assert launches(b"k_step2_batch") == launches() == 2
    lat.close()
""")


# Particle records where the device has no room for the read-back buffers: the
# same records, rows read one at a time; nothing is left over from the failed
# allocation, and the buffers come once there is room.
def test_particle_records_without_device_memory(run):
    run("""
lat = started(configs.poiseuille(8, 8, 8, tau=0.8, g=0.0), 0)
lat.particles_init(abi.make_particle_config(abi.LAGRANGE_WRAP, 1))
rng = np.random.default_rng(5)
a = np.zeros(70001, dtype=abi.particle_dtype())
for k in a.dtype.names:
    a[k] = rng.uniform(1.0, 7.0, len(a))
lat.set_particles(a)
before = S.stub_live_bytes()
for first in (0, 1, 2):
    S.stub_fail(0, first, 1)
    back = lat.particles()
    if first == 0:
        assert np.array_equal(back, a)
        short = np.zeros(11, dtype=a.dtype)
        n = C.c_int64()
        S.stub_fail(0, 0, 1)
        assert lat._L.ch4g_get_particles(lat.handle, short.ctypes.data, 10, C.byref(n)) == 0
        assert n.value == len(a) and np.array_equal(short[:10], a[:10]) and not short[10:].view(np.float64).any()
        assert S.stub_live_bytes() == before
        assert launches(b"k_records") == 0
kept = S.stub_live_bytes() - before
assert a.dtype.itemsize * 65536 + 16 * len(a) <= kept <= a.dtype.itemsize * 65536 + 16 * len(a) + (1 << 20), kept
S.stub_fail(0, 0, 0)
lat.particles()
assert S.stub_live_bytes() - before == kept
""")


# An allocation that fails among several leaves nothing behind, and a retry gets
# all of them (no call goes on with some of its buffers).
@pytest.mark.parametrize("call,buffers", [("lat.hydro_fields()", 5), ("lat.dump_averages()", 5),
                                          ("lat.get_populations()", 2)])
def test_failed_allocations_are_taken_back(run, call, buffers):
    run(f"""
for k in range({buffers}):
    lat = started(workloads.rb2d(64, 32, 1, precision=abi.FP64), 3)
    live, own = S.stub_live_bytes(), lat.device_bytes
    S.stub_fail(0, k, 1)
    try:
        {call}
        raise SystemExit("call without its memory")
    except Exception as e:
        assert "hipMalloc" in str(e), e
    assert (S.stub_live_bytes(), lat.device_bytes) == (live, own)
    {call}
    lat.close()
""")


def test_particles_without_memory_leave_the_lattice(run):
    run("""
flags = (abi.LAGRANGE_WRAP | abi.LAGRANGE_GRADIENT | abi.LAGRANGE_ADDEDMASS | abi.LAGRANGE_TWOWAY_MOMENTUM)
for k in range(8):
    lat = started(configs.poiseuille(8, 8, 8, tau=0.8, g=0.0), 0)
    lat.particles_init(abi.make_particle_config(flags, 3, tau_drag=(1, 5.0, 5.0), beta_coeff=(1, 0.8, 0.8)))
    S.stub_fail(0, k, 1)
    try:
        lat.set_particles(np.ones(50, dtype=abi.particle_dtype()))
        raise SystemExit("particles without their memory")
    except Exception as e:
        assert "hipMalloc" in str(e), e
    S.stub_reset()
    lat.step(3)
    assert launches() == launches(b"k_step") > 0 and lat.particles_count() == 0
    lat.close()
""")


# FP64 2-D lattices whose rows leave their tiles mostly idle take two steps per
# launch only while their launches are small, alone and in a batch.
def test_thin_2d_lattices_take_single_steps(run):
    run("""
def steps(nx, ny):
    return Lattice(workloads.rb2d(nx, ny, 1, precision=abi.FP64)).steps_per_launch()

for nx, ny in ((1, 64), (2, 1000), (1, 30000), (4, 5000), (8, 20000), (16, 10000), (33, 4000), (36, 1000), (97, 1000)):
    assert steps(nx, ny) == 1, (nx, ny)
for nx, ny in ((3, 64), (16, 1000), (33, 256), (20, 16000), (32, 16000), (40, 4000), (65, 16000), (97, 4000), (100, 1000),
               (129, 1000), (512, 256)):
    assert steps(nx, ny) == 2, (nx, ny)
for n, two in ((3, True), (16, False)):
    lats = [started(workloads.rb2d(6, 300, 1, precision=abi.FP64)) for _ in range(n)]
    wide = started(workloads.rb2d(64, 32, 1, precision=abi.FP64))
    S.stub_reset()
    step_batch(lats + [wide], 8)
    assert launches(b"k_step2_batch64") == 4 and launches(b"k_step_batch64") == (0 if two else 8)
""")


# FP64 single steps beyond the cached sizes go in groups of blocks with
# non-temporal stores (fifth template argument), below them with plain ones.
def test_fp64_streamed_single_steps_use_streaming_stores(run):
    run("""
for n, streamed in ((64, 0), (100, 1), (112, 1)):
    cfg = configs.hit(n, les=False) if n == 112 else workloads.rb2d(n, n, n, precision=abi.FP64)
    lat = started(cfg)
    lat.set_fusion(False)
    S.stub_reset()
    lat.step(2)
    t = 0 if n == 112 else 1
    dense = 1 if n % 64 else 0
    assert launches(f"k_step_fp64ILb0ELb1ELb{t}ELb{dense}ELb{streamed}E".encode()) == launches() == 2
    lat.close()
""")


# A few particles are read back without kernels or device buffers.
@pytest.mark.parametrize("n,kernels", [(1, False), (600, False), (601, True)])
def test_few_particle_records_are_formed_on_the_host(run, n, kernels):
    run(f"""
lat = started(configs.poiseuille(8, 8, 8, tau=0.8, g=0.0), 0)
lat.particles_init(abi.make_particle_config(abi.LAGRANGE_WRAP, 1))
a = np.zeros({n}, dtype=abi.particle_dtype())
for i, k in enumerate(a.dtype.names):
    a[k] = 1000.0 * i + np.arange({n})
lat.set_particles(a)
S.stub_reset()
live = S.stub_live_bytes()
back = lat.particles()
assert (launches() > 0) == {kernels} and (S.stub_live_bytes() > live) == {kernels}
assert {kernels} or np.array_equal(back, a)
""")
