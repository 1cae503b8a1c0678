"""Host side of the stepping calls (mpd_capi.cpp), compiled for the CPU against
a stand-in for the HIP runtime and the kernels (tests/standin): what a call
enqueues, what it waits for, and what it leaves behind when a resident run
stops short or an allocation fails."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

import lattice_microbes_amd as lmx
from lattice_microbes_amd import _lib, build, models

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.skipif(not (shutil.which(build.HIPCC) or os.path.exists(build.HIPCC)), reason="no hipcc")


@pytest.fixture(scope="module")
def standin_library(tmp_path_factory):
    out = tmp_path_factory.mktemp("standin")
    objs = []
    for src in (os.path.join(build.CSRC, "mpd_capi.cpp"), os.path.join(HERE, "standin", "hip_standin.cpp")):
        objs.append(str(out / (os.path.basename(src) + ".o")))
        subprocess.run([build.HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-fPIC", "-ffp-contract=off", "-w",
                        "-I" + os.path.join(build.ROOT, "include"), "-I" + build.CSRC, "-c", "-x", "hip", src,
                        "-o", objs[-1]], check=True)
    so = str(out / "libstandin.so")
    subprocess.run([build.CXX, "-shared", "-Wl,-z,defs", *objs, "-o", so], check=True)
    lib = ctypes.CDLL(so)
    for name, (res, args) in _lib.SIGNATURES.items():
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = res, args
    lib.standin_log.restype = ctypes.c_char_p
    lib.standin_cost.argtypes = [ctypes.c_char_p, ctypes.c_double]
    lib.standin_resident_limit.argtypes = [ctypes.c_uint32]
    return lib


@pytest.fixture
def lib(standin_library, monkeypatch):
    monkeypatch.setattr(_lib, "_lib", standin_library)
    standin_library.standin_reset()
    yield standin_library
    standin_library.standin_reset()


def log(lib):
    """The log since the last look at it."""
    lines = lib.standin_log().decode().split("\n")[:-1]
    lib.standin_clear_log()
    return lines


def small(words=False, **kw):
    """A solver whose calls of four steps and more are resident runs."""
    spec = models.bimolecular(shape=(16, 16, 16), nA=50, nB=50, seed=1, **kw)
    if words:
        spec.lattice = spec.lattice.astype(np.uint32)
    s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, seed=3)
    return spec, s


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
def test_a_run_that_did_nothing_does_not_pack_the_lattice(lib, words):
    """A resident run that found too many particles leaves them where they
    were, with empty slots before occupied ones: the first step made up for it
    reads every plane."""
    spec, s = small(words)
    p, q = ctypes.c_void_p(), ctypes.c_void_p()
    _lib.check(lib.lmx_device_lattice(s._h, ctypes.byref(p), ctypes.byref(q)))
    lib.standin_resident_limit(0)
    log(lib)
    s.runTimesteps(5)
    lines = log(lib)
    assert [l for l in lines if l.startswith("resident")] == ["resident t=0 steps=5 packed=0"]
    boxes = [l for l in lines if l.startswith("box")]
    assert [l.split()[:3] for l in boxes] == [["box", f"t={t}", f"packed={int(t > 0)}"] for t in range(5)]
    s.close()


def test_a_run_that_ended_packs_the_lattice(lib):
    spec, s = small()
    p, q = ctypes.c_void_p(), ctypes.c_void_p()
    _lib.check(lib.lmx_device_lattice(s._h, ctypes.byref(p), ctypes.byref(q)))
    log(lib)
    s.runTimesteps(5)
    s.runTimesteps(1)
    lines = log(lib)
    assert "resident t=0 steps=5 packed=0" in lines
    assert [l.split()[:3] for l in lines if l.startswith("box")] == [["box", "t=5", "packed=1"]]
    s.close()


def test_missing_steps_run_on_the_solvers_device(lib):
    """New parameters first make up for the steps that an earlier run left
    out, on the solver's device, whichever is current."""
    spec = models.bimolecular(shape=(16, 16, 16), nA=50, nB=50, seed=1)
    s = lmx.MpdRdmeSolver(1)
    spec.load_into(s, seed=3)
    lib.standin_resident_limit(2)
    s.runTimesteps(6, synchronize=False)
    other = lmx.MpdRdmeSolver(0)
    log(lib)
    _lib.check(lib.lmx_initialize(s._h, 0, 9, 1e-6, _lib.OVERFLOW_CLASSIC, _lib.BOUNDARY_PERIODIC))
    lines = log(lib)
    assert lines[0] == "device 1"
    assert [l.split()[1] for l in lines if l.startswith("box")] == ["t=2", "t=3", "t=4", "t=5"]
    other.close()
    s.close()


@pytest.mark.parametrize("rebuilt", ["model", "lattice"])
@pytest.mark.parametrize("then", ["synchronize", "overflow_stats", "unresolved", "initialize"])
def test_a_rebuild_launches_no_old_step_with_new_shapes(lib, rebuilt, then):
    """A resident run stopped short, nothing has looked at it yet, and the
    model is replaced, or a new lattice refused: the missing steps run with
    the old model and lattice, and none after that."""
    spec, s = small()
    lib.standin_resident_limit(2)
    s.runTimesteps(6, synchronize=False)
    log(lib)
    if rebuilt == "model":
        big = models.random_model(shape=(8, 8, 8), P=8, nS=40, nST=2, R=30, density=0.01, seed=2)
        s.buildModel(big.nS, big.R, big.initial_counts(), big.types, big.K, big.S, big.D, 1)
    else:
        big = models.bimolecular(shape=(64, 64, 64), nA=50, nB=50, seed=1)
        with pytest.raises(lmx.InvalidArgException, match="diffusion coefficient is too high"):
            s.buildDiffusionModel(big.nST, big.DF * 1e6, big.RL, 64, 64, 64, big.P, 1, big.spacing, big.lattice,
                                  big.sites, True)
    want = [f"box t={t} packed=1 N={spec.N} R={spec.R}" for t in (2, 3, 4, 5)]
    assert [l for l in log(lib) if l.startswith(("box", "sweep", "fused", "resident"))] == want
    {"synchronize": s.synchronize, "overflow_stats": s.getOverflowStats, "unresolved": s.getUnresolvedOverflows,
     "initialize": lambda: s.initialize(0, spec.parameters(3))}[then]()
    assert not [l for l in log(lib) if l.startswith(("box", "sweep", "fused", "resident"))]
    s.close()


def test_reports_survive_a_failed_allocation(lib):
    """A model of more species than the counts' buffers hold, and no memory for
    larger ones: the lattice is refused, and the calls that report through
    those buffers still work."""
    spec, s = small()
    big = models.random_model(shape=(8, 8, 8), P=8, nS=300, nST=1, R=0, density=0.0, seed=2)
    s2 = lmx.IntMpdRdmeSolver(0)
    s2.initialize(0, big.parameters(3))
    s2.buildModel(big.nS, big.R, big.initial_counts(), big.types, big.K, big.S, big.D, 1)
    lib.standin_pinned_fails(1)
    with pytest.raises(lmx.LmxError) as e:
        s2.buildDiffusionModel(big.nST, big.DF, big.RL, 8, 8, 8, big.P, 4, big.spacing, big.lattice.astype(np.uint32),
                               big.sites, True)
    assert e.value.code == _lib.ERR_NOMEM
    log(lib)
    s2.synchronize()
    assert [l for l in log(lib) if l.startswith("report")] == ["report"]
    s2.close()
    s.close()


def test_calls_behind_a_resident_run_do_not_wait(lib):
    """Steps of any number, from either list, and a new rate are accepted
    behind a resident run without a wait or a blocking copy."""
    spec, s = small()
    s.runTimesteps(8)
    s.runTimesteps(8, synchronize=False)
    log(lib)
    s.runTimesteps(2, synchronize=False)
    _lib.check(lib.lmx_run_steps_static(s._h, 3))
    _lib.check(lib.lmx_run_steps_static(s._h, 8))
    s.setReactionRate(0, 0.5)
    lines = log(lib)
    assert not {"sync", "copy"} & set(lines), lines
    s.synchronize()
    assert s.timestep == 29
    s.close()


def test_steps_behind_a_run_that_stopped_short(lib):
    """They run from where the device stands, a later resident run does
    nothing, and the missing steps follow when the state is looked at."""
    spec, s = small()
    lib.standin_resident_limit(2)
    log(lib)
    s.runTimesteps(6, synchronize=False)
    s.runTimesteps(1, synchronize=False)
    s.runTimesteps(5, synchronize=False)
    _lib.check(lib.lmx_run_steps_static(s._h, 1))
    assert [l.split()[:2] for l in log(lib) if l.startswith(("box", "resident"))] == [
        ["resident", "t=0"], ["box", "t=2"], ["resident", "t=7"], ["box", "t=3"]]
    s.synchronize()
    assert [l.split()[1] for l in log(lib) if l.startswith("box")] == [f"t={t}" for t in range(4, 13)]
    assert s.timestep == 13
    s.close()


def test_missing_steps_keep_the_old_rate(lib):
    """New tables are uploaded after the steps that an earlier run left out."""
    spec, s = small()
    lib.standin_resident_limit(2)
    s.runTimesteps(6, synchronize=False)
    s.setReactionRate(0, 0.5)
    log(lib)
    s.runTimesteps(2)
    lines = [l.split()[:2] for l in log(lib) if l.startswith(("box", "tables"))]
    assert lines == [["box", f"t={t}"] for t in range(2, 6)] + [["tables"]] + [["box", "t=6"], ["box", "t=7"]]
    s.close()


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
def test_static_list_is_the_byte_lattices(lib, words):
    """Solvers of the uint32 lattice share no list, so their calls may overlap."""
    spec, s = small(words)
    log(lib)
    _lib.check(lib.lmx_run_steps_static(s._h, 1))
    lines = log(lib)
    assert any(l.startswith("box") for l in lines) and ("static list" in lines) == (not words)
    s.close()


@pytest.mark.parametrize("n,resident", [(3000, True), (3001, False), (4000, False)])
@pytest.mark.parametrize("by", ["build", "set", "set_native"])
def test_crowded_small_lattices_are_counted(lib, n, resident, by):
    """More particles than sites: a lattice of 500 sites is run in one block
    only if its particles are few, however the lattice was set."""
    rng = np.random.default_rng(1)
    spec = models.random_model(shape=(10, 10, 5), P=16, nS=3, nST=1, R=0, density=0.0, seed=1)
    lattice = np.zeros(500 * 16, np.uint8)
    lattice[rng.permutation(lattice.size)[:n]] = 1
    lattice = lattice.reshape(10, 10, 5, 16)
    s = lmx.MpdRdmeSolver(0)
    if by == "build":
        spec.lattice = lattice
    spec.load_into(s, seed=1)
    if by == "set":
        s.setLattice(lattice)
    elif by == "set_native":
        packed = np.zeros((4, 5, 10, 10), np.uint32)
        for (x, y, z), c in np.ndenumerate((lattice != 0).sum(axis=3)):
            for j in range(c):
                packed[j // 4, z, y, x] |= np.uint32(1 << (8 * (j % 4)))
        s.setLatticeNative(packed)
    log(lib)
    s.runTimesteps(8)
    assert any(l.startswith("resident") for l in log(lib)) == resident
    s.close()


@pytest.mark.parametrize("cost,limit,steps,resident,best", [
    (dict(resident=1, box=16, sweep=10, fused=5), None, 8, True, 1.0),
    (dict(resident=1, box=16, sweep=10, fused=5), None, 2, True, 1.0),   # shorter than any resident run
    (dict(resident=7, box=16, sweep=10, fused=5), None, 8, False, 5.0),
    (dict(resident=1, box=16, sweep=10, fused=15), 3, 8, False, 10.0),    # a block that is full takes no time
])
def test_autotune_times_the_resident_run(lib, cost, limit, steps, resident, best):
    """The run that calls of four steps and more would be is what the other
    shapes have to beat."""
    spec, s = small()
    for kind, ms in cost.items():
        lib.standin_cost(kind.encode(), float(ms))
    if limit is not None:
        lib.standin_resident_limit(limit)
    assert s.autotune(steps=steps)["ms_per_step"] == pytest.approx(best)
    lib.standin_resident_limit(0xFFFFFFFF)
    log(lib)
    assert s.timestep == 0
    s.runTimesteps(5)
    lines = log(lib)
    assert any(l.startswith("resident") for l in lines) == resident
    assert s.timestep == 5
    s.close()


@pytest.mark.parametrize("threads,sweeps", [(0, False), (256, False), (512, True)])
def test_default_tile_threads_by_their_number(lib, threads, sweeps):
    """256 threads are the default and leave the members' routes alone, also
    after another size was set."""
    ens = lmx.Ensemble(0, graph=False)
    few, many = small()[1], lmx.MpdRdmeSolver(0)
    models.bimolecular(shape=(64, 64, 64), nA=5000, nB=50, seed=1).load_into(many, seed=2)
    for s in (few, many):
        ens.add(s)
    ens.set_tile_threads(1024)
    ens.set_tile_threads(threads)
    log(lib)
    ens.run(5)
    kinds = {l.split()[0] for l in log(lib)} & {"resident", "box", "sweep"}
    assert kinds == ({"sweep"} if sweeps else {"resident", "box"})
    assert few.timestep == many.timestep == 5
    ens.close()


@pytest.mark.parametrize("steps", [2, 8])
def test_batch_autotune_times_the_resident_runs(lib, steps):
    """Also when asked for fewer steps than a run in one block takes."""
    ens = lmx.Ensemble(0, graph=False)
    spec, s = small()
    ens.add(s)
    for kind, ms in dict(resident=1, box=16, sweep=10).items():
        lib.standin_cost(kind.encode(), float(ms))
    assert ens.autotune(steps=steps) == {"reaction_list": True, "tile_threads": 256, "ms_per_step": 1.0}
    log(lib)
    ens.run(5)
    assert {l.split()[0] for l in log(lib)} & {"resident", "box", "sweep"} == {"resident"}
    ens.close()


@pytest.mark.parametrize("box,boxes", [(5, True), (20, False)])
def test_autotune_tells_boxes_from_tiles(lib, box, boxes):
    """The other options read the same for the boxed step and the row tiles."""
    s = lmx.MpdRdmeSolver(0)
    models.bimolecular(shape=(64, 64, 64), nA=5000, nB=50, seed=1).load_into(s, seed=2)
    for kind, ms in dict(box=box, sweep=10, fused=15).items():
        lib.standin_cost(kind.encode(), float(ms))
    tuned = s.autotune()
    assert (tuned["path"], tuned["yz_kernel"], tuned["fuse_reaction"]) == (_lib.PATH_SWEEPS, 0, True)
    assert tuned["boxes"] == boxes
    for option, value in ((_lib.OPT_MARCH_SEGMENT, 4), (_lib.OPT_FORCE_GENERIC, 1), (_lib.OPT_YZ_KERNEL, 3),
                          (_lib.OPT_FUSED_ZSEG, 7), (_lib.OPT_FUSE_REACTION, 0), (_lib.OPT_BOXES, 1)):
        s.setLaunchOption(option, value)
        assert s.getLaunchOption(option) == value
    with pytest.raises(lmx.InvalidArgException):
        s.getLaunchOption(99)
    s.close()


def _crowded(shape, P, density, spot, words, R):
    """Uniform particles, one a site, and a cube of 32^3 sites (at most) with
    `spot` a site."""
    spec = models.bimolecular(shape=shape, nA=1, nB=1, P=P, seed=1)
    if not R:
        spec = models.random_model(shape=shape, P=P, nS=3, nST=1, R=0, density=0.0, seed=1)
    rng = np.random.default_rng(3)
    first = rng.random(shape) < density
    if spot:
        first[:32, :32, :32] = rng.random(first[:32, :32, :32].shape) < spot
    spec.lattice = np.zeros(shape + (P,), np.uint32 if words else np.uint8)
    spec.lattice[..., 0] = first
    return spec


@pytest.mark.parametrize("shape,P,density,spot,words,R,boxes", [
    ((96, 96, 96), 8, 0.5, 0, False, 2, True),
    ((160, 160, 100), 8, 0.5, 0, False, 2, False),
    ((160, 160, 100), 8, 0.2, 0, False, 2, True),
    ((160, 160, 100), 8, 0.01, 0.6, False, 2, False),
    ((96, 96, 96), 8, 0.01, 0.6, False, 2, True),
    ((63, 61, 151), 8, 0.5, 0, False, 2, False),
    ((63, 61, 151), 8, 0.3, 0, False, 2, True),
    ((160, 160, 100), 16, 0.8, 0, False, 2, True),
    ((63, 61, 151), 16, 0.5, 0, False, 2, True),
    ((95, 93, 91), 16, 0.01, 0.9, False, 2, False),
    ((96, 96, 96), 4, 0.5, 0, False, 2, True),
    ((96, 96, 96), 4, 0.45, 0, False, 0, False),
    ((96, 96, 96), 4, 0.3, 0, False, 0, True),
    ((96, 96, 96), 8, 0.5, 0, True, 2, False),
    ((96, 96, 96), 8, 0.2, 0, True, 2, True),
    ((95, 93, 91), 8, 0.01, 0.6, True, 2, True),
    ((32, 32, 32), 8, 0.5, 0, True, 2, True),
])
def test_crowded_lattices_step_in_what_is_faster(lib, shape, P, density, spot, words, R, boxes):
    """Both sides of each line of the rule for the smallest boxes that fit."""
    spec = _crowded(shape, P, density, spot, words, R)
    s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
    spec.load_into(s, seed=2)
    log(lib)
    s.runTimesteps(1)
    assert [l.split()[0] for l in log(lib) if l.startswith(("box", "sweep"))] == ["box" if boxes else "sweep"]
    s.close()


@pytest.mark.parametrize("edge,n,steps,resident", [(64, 2048, 3, False), (64, 2048, 4, True), (64, 2049, 7, False),
                                                   (64, 2049, 8, True), (160, 2049, 4, True)])
def test_short_calls_of_more_particles_than_two_a_thread(lib, edge, n, steps, resident):
    """Alone on a small lattice; beside others in an ensemble they run in one
    block from four steps on."""
    s = lmx.MpdRdmeSolver(0)
    models.bimolecular(shape=(edge,) * 3, nA=n // 2, nB=n - n // 2, seed=1).load_into(s, seed=2)
    log(lib)
    s.runTimesteps(steps)
    assert any(l.startswith("resident") for l in log(lib)) == resident
    ens = lmx.Ensemble(0, graph=False)
    ens.add(s)
    log(lib)
    ens.run(steps)
    assert any(l.startswith("resident") for l in log(lib)) == (steps >= 4)
    ens.close()


@pytest.mark.parametrize("words", [False, True], ids=["byte", "uint32"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 1, 1), (5, 3, 7), (8, 4, 6)])
@pytest.mark.parametrize("P", [4, 8, 16])
def test_host_lattice_writes(lib, shape, P, words):
    """Row-major writes pack every site's particles in their order; native
    writes stay as they are, and whether a site has an empty slot before an
    occupied one, in one word or across words, is seen at every site; a
    species that the model does not have is refused wherever it stands."""
    rng = np.random.default_rng(P + len(shape))
    spec = models.random_model(shape=shape, P=P, nS=5, nST=1, R=0, density=0.0, seed=1)
    s = (lmx.IntMpdRdmeSolver if words else lmx.MpdRdmeSolver)(0)
    if words:
        spec.lattice = spec.lattice.astype(np.uint32)
    spec.load_into(s, seed=1)
    rm = np.where(rng.random(shape + (P,)) < 0.4, rng.integers(1, 6, shape + (P,)), 0).astype(spec.lattice.dtype)
    packed = np.zeros_like(rm)
    for at in np.ndindex(*shape):
        v = rm[at][rm[at] != 0]
        packed[at][:v.size] = v
    s.setLattice(rm)
    np.testing.assert_array_equal(s.getLattice(), packed)

    def native(lattice):
        z = lattice.transpose(2, 1, 0, 3)
        w = z if words else np.ascontiguousarray(z).view(np.uint32)
        return np.ascontiguousarray(np.moveaxis(w, 3, 0)).astype(np.uint32)

    def first_step_reads_as_packed():
        log(lib)
        s.runTimesteps(1)
        return "packed=1" in [l for l in log(lib) if l.startswith(("box", "sweep"))][0]

    s.setLatticeNative(native(packed))
    np.testing.assert_array_equal(s.getLatticeNative(), native(packed))
    assert first_step_reads_as_packed()
    for trial in range(8):
        one = np.zeros_like(rm)
        at = tuple(int(rng.integers(0, k)) for k in shape)
        slot = int(rng.integers(1, P))
        one[at][slot] = 3
        one[at][:slot] = 1
        s.setLatticeNative(native(one))
        assert first_step_reads_as_packed()
        one[at][int(rng.integers(0, slot))] = 0
        s.setLatticeNative(native(one))
        assert not first_step_reads_as_packed()
        one[at][slot] = 6
        for write, lattice in ((s.setLatticeNative, native(one)), (s.setLattice, one)):
            with pytest.raises(lmx.InvalidArgException, match="invalid species"):
                write(lattice)
    s.close()


def test_timed_steps_include_those_a_resident_run_left_out(lib):
    spec, s = small()
    for kind, ms in dict(resident=1, box=16).items():
        lib.standin_cost(kind.encode(), float(ms))
    assert s.timeSteps(6)[0] == pytest.approx(6.0)
    lib.standin_resident_limit(2)
    assert s.timeSteps(6)[0] == pytest.approx(2 * 1.0 + 4 * 16.0)
    assert s.timestep == 12
    s.close()


def test_timed_batch_steps_include_those_a_resident_run_left_out(lib):
    ens = lmx.Ensemble(0, graph=False)
    members = [small()[1] for _ in range(2)]
    for s in members:
        ens.add(s)
    for kind, ms in dict(resident=1, box=16).items():
        lib.standin_cost(kind.encode(), float(ms))
    lib.standin_resident_limit(2)
    assert ens.time_steps(6) == pytest.approx(2 * (2 * 1.0 + 4 * 16.0))
    assert [s.timestep for s in members] == [6, 6]
    ens.close()
