"""What the engine's host code allocates and launches, on the CPU: libsjf runs against
tests/host/fake_hip.cpp, a stand-in for the HIP runtime that records launches (no kernel runs),
knows which memory is live and can fail a chosen allocation.  Each case runs in a process of its
own, since the stand-in has to be loaded before libsjf.
"""
import ctypes as C
import os
import shutil
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def fake_path(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    out = str(tmp_path_factory.mktemp("fake_hip") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "host", "fake_hip.cpp"), "-o", out],
                   check=True, capture_output=True, text=True)
    return out


def run_case(fake, name, *args):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), fake, name, *map(str, args)], cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]


class Fake:
    def __init__(self, path):
        self.lib = C.CDLL(path, mode=C.RTLD_GLOBAL)
        for f, res in (("fake_log", C.c_char_p), ("fake_last_kernel", C.c_char_p), ("fake_live_bytes", C.c_double),
                       ("fake_host_bytes", C.c_double),
                       ("fake_steps", C.c_long), ("fake_refused", C.c_long), ("fake_source_entries", C.c_long), ("fake_source_shared", C.c_long), ("fake_allocations", C.c_long),
                       ("fake_last_table", C.c_size_t)):
            getattr(self.lib, f).restype = res
        self.lib.fake_fail_at.argtypes = [C.c_long]
        self.lib.fake_last_table.argtypes = [C.c_char_p, C.c_size_t]

    def __getattr__(self, name):
        return getattr(self.lib, "fake_" + name)

    def table(self):
        """The argument table of the last fused step."""
        buf = C.create_string_buffer(self.lib.fake_last_table(None, 0))
        self.lib.fake_last_table(buf, len(buf))
        return buf.raw


# ---- DFT launches -------------------------------------------------------------------------------

def case_dft_launch(fake, source):
    """Many (component, cell) pairs at one frequency beside one cell at 64: more threads than one grid
    dimension takes, whether or not the source could share the launch."""
    from sim_juncs_amd.engine import Engine

    n = 236
    e = Engine((n, n, n), 0.01)
    at = 0.01 * (n // 2 if source == "inside" else 1)
    e.add_source("Ex", [at - 0.005, at, at] * 2, freq=1.0, width=1.0, t_end=10.0)
    e.add_dft((8, 8, 8), (n, n, n), ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"), [1.0])
    e.add_dft((6, 6, 6), (7, 7, 7), ("Ex",), np.linspace(0.5, 1.5, 64))
    pairs = 6 * (n - 8) ** 3 + 1
    assert pairs * 64 >= 2 ** 32
    e.step(2)
    assert fake.refused() == 0 and fake.steps() == 2
    log = [line for line in fake.log().decode().split("\n") if "k_dft<" in line or "k_source_dft<" in line]
    assert len(log) == 2 and all("k_dft<" in line for line in log), log
    assert all(f" {-(-pairs // 256)} 64 1 x 256" in line for line in log), log


@pytest.mark.parametrize("source", ["inside", "outside"])
def test_dft_of_many_values_and_many_frequencies_is_launched(fake_path, source):
    run_case(fake_path, "dft_launch", source)


# ---- sources ------------------------------------------------------------------------------------

def case_shared_cells(fake, which):
    """No launch has two threads add to one value: sources that share cells go out one after another."""
    from sim_juncs_amd.engine import Engine

    shape, periodic = (12, 11, 14), (0, 0, 0)
    if which == "thin":
        shape, periodic = (1, 1, 14), (1, 1, 0)
    e = Engine(shape, 0.1, periodic=periodic)
    pulse = dict(freq=1.0, width=0.3, t_start=-1.0, t_end=2.0)
    sheet = [0.0, 0.0, 0.6, 0.1 * shape[0], 0.1 * shape[1], 0.6]
    expect = 1
    if which == "thin":
        e.add_source("Ex", [0.03, 0.07, 0.63] * 2, **pulse)
    else:
        comps = {"electric": ("Ex",) * 3, "magnetic": ("Hy",) * 3, "mixed": ("Ex", "Ey", "Ex", "Hx", "Hx")}[which]
        for c in comps:
            e.add_source(c, sheet, **pulse)
        e.add_source(comps[0], [0.55, 0.55, 0.6] * 2, **pulse)
        e.add_source(comps[0], [0.5, 0.5, 1.1] * 2, **pulse)  # apart from the sheets
        expect = 4 if which != "mixed" else 3 + 2
    e.add_dft((0, 0, 13), shape, ("Ex",), [1.0])
    e.step(2)
    launches = [x for x in fake.log().decode().split("\n") if "k_source" in x]
    assert fake.source_shared() == 0 and fake.source_entries() > 0
    assert len(launches) == 2 * expect, launches


@pytest.mark.parametrize("which", ["electric", "magnetic", "mixed", "thin"])
def test_sources_that_share_cells_do_not_share_a_launch(fake_path, which):
    run_case(fake_path, "shared_cells", which)


# ---- allocations that fail ----------------------------------------------------------------------

SHAPE = (10, 9, 12)


def case_failed_allocation(fake):
    """A call that runs out of memory before it has changed anything fails alone: the next step runs
    and is not reported as failed (its launches ask for the last error)."""
    from sim_juncs_amd import materials as M
    from sim_juncs_amd._lib import EngineError
    from sim_juncs_amd.engine import Engine

    words = np.zeros(SHAPE, np.uint32)
    calls = {
        "materials": lambda e: e.set_materials(words, [M.AU.scaled(1.0)]),
        "dft": lambda e: e.add_dft((1, 1, 1), (3, 3, 3), ("Ex",), [1.0]),
        "flux": lambda e: e.dft_flux(0, 2),
        "monitors": lambda e: e.reserve_steps(100),
        "adjoint": lambda e: e.adjoint_run(4, 2, (5, 4, 6), 8),
    }
    for name, call in calls.items():
        with Engine(SHAPE, 0.02) as e:
            if name == "flux":
                e.add_dft((0, 0, 6), SHAPE[:2] + (7,), ("Ex", "Ey", "Hx", "Hy"), [1.0])
            if name == "monitors":
                e.add_monitors("Ex", [[0.1, 0.1, 0.1]])
            if name == "adjoint":
                e.set_design_eps((2, 2, 2), (4, 4, 4), np.full((2, 2, 2), 3.0))
                e.reserve_steps(1)
            else:
                e.step(1)
            fake.fail_at(0)
            with pytest.raises(EngineError):
                call(e)
            fake.fail_at(-1)
            before = fake.steps()
            e.step(1)
            assert fake.steps() == before + 1, name


def test_a_failed_allocation_is_not_reported_by_the_next_step(fake_path):
    run_case(fake_path, "failed_allocation")


def case_no_leak(fake):
    """Each allocation of each of these calls fails in turn: the call can be made again, and nothing is
    left once the engine is closed."""
    from sim_juncs_amd import materials as M
    from sim_juncs_amd._lib import EngineError
    from sim_juncs_amd.engine import Engine

    def engine():
        e = Engine(SHAPE, 0.02, precision="fp64")
        e.set_materials(_blocks([0, 1]), [M.VACUUM, M.AU.scaled(1.0)])
        e.set_pml([2] * 6)
        e.set_design_eps((2, 2, 2), (4, 4, 4), np.full((2, 2, 2), 3.0))
        for c in ("Ex", "Hy"):
            e.add_source(c, [0.1, 0.1, 0.1] * 2, freq=1.0, width=1.0, t_end=10.0)
        e.add_monitors("Ex", [[0.1, 0.1, 0.1]])
        return e

    calls = {
        "dft": lambda e: e.add_dft((1, 1, 1), (3, 3, 3), ("Ex",), [1.0]),
        "step": lambda e: e.step(2),
        "record": lambda e: e.adjoint_run(4, 0, (5, 4, 6), 8),
        "checkpoints": lambda e: e.adjoint_run(4, 2, (5, 4, 6), 8),
    }
    engine().close()
    none = fake.live_bytes()
    for name, call in calls.items():
        with engine() as e:
            start = fake.allocations()
            call(e)
            count = fake.allocations() - start
        assert count >= 3
        for k in range(count):
            with engine() as e:
                fake.fail_at(k)
                with pytest.raises(EngineError):
                    call(e)
                fake.fail_at(-1)
                call(e)
            assert fake.live_bytes() == none, (name, k)


def test_calls_that_run_out_of_memory_leave_nothing_behind(fake_path):
    run_case(fake_path, "no_leak")


# ---- material changes that fail -----------------------------------------------------------------

def _blocks(ids):
    w = np.zeros(SHAPE, np.uint32)
    for q, m in enumerate(ids):
        w[q::len(ids)] = m * 0x010101
    return w


def _changes():
    """name -> (calls that come first, the call that is made to fail)"""
    from sim_juncs_amd import materials as M

    vac, sio2, au, drude = M.VACUUM, M.SIO2.scaled(1.0), M.AU.scaled(1.0), M.AU_REFERENCE_AS_RUN.scaled(1.0)

    def mats(*lut):
        return lambda e: e.set_materials(_blocks(range(len(lut))), list(lut))

    def pml(e):
        e.set_pml([2] * 6)
        e.set_pml_dispersion(1.25)

    maps = lambda e: e.set_eps_maps(np.full((3,) + SHAPE, 2.0))  # noqa: E731
    design = lambda e: e.set_design_eps((2, 2, 2), (5, 6, 7), np.full((3, 4, 5), 3.0))  # noqa: E731
    return {
        "first": ([], mats(vac, au)),
        "more poles": ([mats(vac, drude)], mats(vac, sio2, au)),
        "more materials": ([mats(vac, au)], mats(vac, sio2, au, drude, sio2)),
        "folded": ([pml, mats(vac, sio2)], mats(vac, sio2, au)),
        "fold": ([lambda e: e.set_pml([2] * 6), mats(vac, au)], lambda e: e.set_pml_dispersion(1.25)),
        "first maps": ([], maps),
        "maps": ([mats(vac, au)], maps),
        "no maps": ([mats(vac, au), maps], lambda e: e.set_eps_maps(None)),
        "first design": ([], design),
        "design": ([mats(vac, au)], design),
        "design of maps": ([maps], design),
    }


def _pointers(table):
    """Which words of an argument table are pointers (the stand-in's range is far above any size)."""
    w = np.frombuffer(table[:len(table) // 8 * 8], np.uint64)
    return [i for i, v in enumerate(w) if 1 << 40 < v < 1 << 47]


def case_failed_change(fake, precision):
    from sim_juncs_amd._lib import EngineError
    from sim_juncs_amd.engine import Engine

    for name, (before, change) in _changes().items():
        def engine():
            e = Engine(SHAPE, 0.02, precision=precision)
            for f in before:
                f(e)
            if name == "fold":  # set before the first step: tables that are built, no step
                e.reserve_steps(1)
            else:
                e.step(1)
            return e

        with engine() as e:  # how it ends when nothing fails
            start = fake.allocations()
            change(e)
            count = fake.allocations() - start
            e.step(1)
            want = _pointers(fake.table())
        assert count > 0 or name == "no maps"
        for k in range(count):
            with engine() as e:
                old, steps = fake.table(), fake.steps()
                fake.fail_at(k)
                with pytest.raises(EngineError):
                    change(e)
                fake.fail_at(-1)
                try:
                    e.step(1)
                except EngineError:
                    assert fake.steps() == steps, (name, k)  # refused: nothing ran
                else:  # the state before the call
                    assert fake.last_stale() == 0 and (fake.table() == old or name == "fold"), (name, k)
                    if name == "fold":
                        continue
                change(e)  # memory is there again
                e.step(1)
                assert fake.last_stale() == 0 and _pointers(fake.table()) == want, (name, k)
    assert fake.bad_copies() == 0


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_material_changes_that_run_out_of_memory_leave_no_stale_tables(fake_path, precision):
    run_case(fake_path, "failed_change", precision)


def case_refused_twins(fake):
    """More than 255 materials with their PML twins: refused, and the earlier map stays whole."""
    from sim_juncs_amd import materials as M
    from sim_juncs_amd._lib import EngineError
    from sim_juncs_amd.engine import Engine

    e = Engine(SHAPE, 0.02)
    e.set_materials(_blocks([1, 0]), [M.VACUUM, M.AU.scaled(1.0)])
    e.set_pml([2] * 6)
    e.set_pml_dispersion(1.25)
    e.step(1)
    old, live = fake.table(), fake.live_bytes()
    with pytest.raises(EngineError, match="twins"):
        e.set_materials(_blocks([7, 8]), [M.SIO2.scaled(1.0)] * 200)
    e.step(1)
    assert fake.table() == old and fake.live_bytes() == live
    e.set_design_eps((2, 2, 2), (5, 6, 7), np.full((3, 4, 5), 3.0))
    assert fake.first_word() == 0x010101  # the words that belong to the LUT in use


def test_refused_materials_leave_the_earlier_ones(fake_path):
    run_case(fake_path, "refused_twins")


def case_failed_pml(fake, precision):
    """The same for sjf_set_pml, on engines whose tables are built, with and without an earlier PML."""
    from sim_juncs_amd import materials as M
    from sim_juncs_amd._lib import EngineError
    from sim_juncs_amd.engine import Engine

    def thin(e):
        e.set_pml([1, 0, 2, 2, 0, 1])

    def folded(e):
        e.set_materials(_blocks([0, 1]), [M.VACUUM, M.AU.scaled(1.0)])
        e.set_pml_dispersion(1.25)

    for before in ([], [thin], [folded], [thin, folded]):
        def engine():
            e = Engine(SHAPE, 0.02, precision=precision)
            for f in before:
                f(e)
            e.reserve_steps(1)
            return e

        with engine() as e:
            start = fake.allocations()
            e.set_pml([2, 1, 2, 2, 3, 1])
            count = fake.allocations() - start
            e.step(1)
            want = _pointers(fake.table())
        assert count >= 3
        for k in range(count):
            with engine() as e:
                steps = fake.steps()
                fake.fail_at(k)
                with pytest.raises(EngineError):
                    e.set_pml([2, 1, 2, 2, 3, 1])
                fake.fail_at(-1)
                with pytest.raises(EngineError, match="incomplete"):
                    e.step(1)
                assert fake.steps() == steps
                e.set_pml([2, 1, 2, 2, 3, 1])
                e.step(1)
                assert fake.last_stale() == 0 and _pointers(fake.table()) == want, k
    # layers too large for one buffer range are refused before anything changes
    with Engine((700, 700, 230), 0.02, precision="fp64") as e:
        e.set_pml([0, 0, 0, 0, 2, 2])
        e.step(0)
        live = fake.live_bytes()
        with pytest.raises(EngineError, match="2 GiB"):
            e.set_pml([0, 0, 0, 0, 60, 60])
        assert fake.live_bytes() == live
        e.step(1)
        assert fake.last_stale() == 0
    assert fake.bad_copies() == 0


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_a_pml_that_runs_out_of_memory_leaves_no_stale_tables(fake_path, precision):
    run_case(fake_path, "failed_pml", precision)


# ---- pole state ---------------------------------------------------------------------------------

def case_pole_memory(fake, precision):
    """A second array of pole state is there for Lorentz poles alone."""
    from sim_juncs_amd import materials as M
    from sim_juncs_amd.engine import Engine

    one = (4 if precision == "fp32" else 8) * 3 * np.prod(SHAPE)  # one slot of one array
    used = {}
    for name, metal in (("drude", M.AU_REFERENCE_AS_RUN), ("lorentz", M.SIO2)):
        with Engine(SHAPE, 0.02, precision=precision) as e:
            e.set_materials(_blocks([0, 1]), [M.VACUUM, metal.scaled(1.0)])
            used[name] = fake.live_bytes()
            e.step(2)
            e.step(1)
            assert fake.last_stale() == 0
    assert used["lorentz"] - used["drude"] == one


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_drude_media_hold_one_array_of_pole_state(fake_path, precision):
    run_case(fake_path, "pole_memory", precision)


# ---- batches ------------------------------------------------------------------------------------

def case_batch_form(fake, precision, lines, cells, form, threads):
    from sim_juncs_amd.engine import Batch, Engine

    engines = []
    for nz in map(int, lines.split(",")):
        n = round((float(cells) / nz) ** 0.5)
        engines.append(Engine((n, n, nz), 0.02, precision=precision))
    b = Batch(engines)
    b.step(1)
    kernel = {"rows": "k_step_rows<", "lines": "k_step<", "passes": "k_step_z<"}[form]
    assert kernel in fake.last_kernel().decode()
    assert b.launch_info()[0] == int(threads)


@pytest.mark.parametrize("precision,lines,cells,form,threads", [
    ("fp32", "100,500", 1.5e6, "rows", 1024), ("fp32", "256,300", 1.5e6, "lines", 320),
    ("fp64", "100,200", 1.5e6, "rows", 512), ("fp64", "128,200", 1.5e6, "lines", 256),
    ("fp64", "100,300", 1.5e6, "lines", 320), ("fp64", "100,300", 2e5, "rows", 640),
    ("fp64", "120,255,257", 1.5e6, "lines", 320), ("fp64", "60,60,60,300", 1.5e6, "rows", 640),
    ("fp64", "64,513", 2e5, "passes", 256),
])
def test_default_form_of_a_batch(fake_path, precision, lines, cells, form, threads):
    """Thread rows where they were measured to be faster: FP64 workgroups above 512 threads spill."""
    run_case(fake_path, "batch_form", precision, lines, cells, form, threads)


def case_reverse_chunk(fake, precision, count, shape, groups):
    from sim_juncs_amd.engine import Batch, Engine

    shape = tuple(map(int, shape.split(",")))
    engines = []
    for _ in range(int(count)):
        e = Engine(shape, 0.02, precision=precision)
        lo = tuple(n // 2 for n in shape)
        e.set_design_eps(lo, tuple(n + 2 for n in lo), np.full((2, 2, 2), 3.0))
        engines.append(e)
    b = Batch(engines)
    b.adjoint_run(3, [(1, 1, 1)] * len(engines), [8] * len(engines))
    assert b.adjoint_kernel_info()[2] == int(groups)


@pytest.mark.parametrize("precision,count,shape,groups", [
    # 3 tiles of 16 rows each: one round of 3-plane chunks on 256 places (12 planes: 48 workgroups)
    ("fp32", 4, "48,48,48", 4 * 3 * 16),
    # 15 tiles of 9 rows: 12 planes fill the chip more than twice
    ("fp32", 4, "128,128,96", 4 * 15 * 11),
    # 10 tiles of 7 rows in workgroups of 8 waves, 12 waves to a CU without poles
    ("fp64", 2, "64,64,64", 2 * 10 * 11),
])
def test_default_chunk_of_a_batched_reverse_launch(fake_path, precision, count, shape, groups):
    """Small batches take chunks short enough to fill the chip once."""
    run_case(fake_path, "reverse_chunk", precision, count, shape, groups)


def case_chunk(fake, precision, shape, xchunk):
    from sim_juncs_amd.engine import Engine

    e = Engine(tuple(map(int, shape.split(","))), 0.02, precision=precision)
    assert e.launch_info()["xchunk"] == int(xchunk)
    e.step(1)
    assert fake.last_grid() == e.launch_info()["groups"]


@pytest.mark.parametrize("precision,shape,xchunk", [
    ("fp32", "43,46,320", 3),    # five wavefronts: three workgroups to a CU, 768 places
    ("fp32", "40,43,384", 4),    # six: two
    ("fp32", "44,46,512", 4),    # eight: two, as the registers alone say
    ("fp64", "32,35,300", 5),    # five at three per SIMD: one
    ("fp64", "45,48,180", 3),    # three wavefronts pack as the registers say
    ("fp64", "125,128,320", 32),  # one round would save too little
    ("fp32", "6,2000,300", 6),   # more rows than places: whole lines
])
def test_default_chunk_of_one_row_tiles(fake_path, precision, shape, xchunk):
    """Chunks that run in one round of the workgroups a CU really holds."""
    run_case(fake_path, "chunk", precision, shape, xchunk)


def case_store_hint(fake, precision, shape, maps, hint):
    """Sides of the line (300 MB) from which stores take the non-temporal hint."""
    from sim_juncs_amd.engine import Engine

    shape = tuple(map(int, shape.split(",")))
    e = Engine(shape, 0.02, precision=precision)
    if maps == "maps":
        e.set_eps_maps(np.full((3,) + shape, 2.0))
    e.step(1)
    assert fake.last_kernel().decode().split(">")[0].endswith(hint.lower())


@pytest.mark.parametrize("precision,shape,maps,hint", [
    # cells x (96 fields, 4 words, 24 maps) bytes in FP64, x (48, 4, 12) in FP32
    ("fp64", "136,136,136", "maps", True), ("fp64", "136,136,136", "no", False),  # 312 MB, 241 MB
    ("fp64", "132,132,136", "maps", False),                                       # 294 MB
    ("fp32", "170,170,166", "maps", True), ("fp32", "170,170,166", "no", False),  # 307 MB, 230 MB
    ("fp32", "166,166,168", "maps", False),                                       # 296 MB
])
def test_eps_maps_count_in_what_a_step_touches(fake_path, precision, shape, maps, hint):
    run_case(fake_path, "store_hint", precision, shape, maps, hint)


def case_store_scenes(fake, index):
    import test_gpu_store_hint as g

    from sim_juncs_amd.engine import Batch

    precision, shape, count, tile, kernel = g.CASES[int(index)]
    grouped = g.engines(precision, shape, count)
    (single,) = g.engines(precision, shape, 1)
    g.alone(single, tile)
    single.step(1)
    threads = fake.last_block()
    off = fake.last_kernel().decode()
    b = Batch(grouped)
    if tile:
        b.set_tile(*tile)
    b.step(1)
    on = fake.last_kernel().decode()
    assert kernel in off and off.split(">")[0].endswith("false"), off
    assert kernel in on and on.split(">")[0].endswith("true"), on
    assert off.replace("false", "true") == on and fake.last_block() == threads


@pytest.mark.parametrize("index", range(6))
def test_scenes_lie_on_either_side_of_the_store_line(fake_path, index):
    """The scenes of test_gpu_store_hint.py run the kernels that it means to compare."""
    run_case(fake_path, "store_scenes", index)


def case_reverse_hint(fake, shape, hint):
    from sim_juncs_amd.engine import Batch, Engine

    shape = tuple(map(int, shape.split(",")))
    for batch in (False, True):
        e = Engine(shape, 0.02, precision="fp64")
        e.set_design_eps((2, 2, 2), (4, 4, 4), np.full((2, 2, 2), 3.0))
        fake.clear_log()
        if batch:
            b = Batch([e])
            b.adjoint_run(2, [(1, 1, 1)], [8])
            b.close()
        else:
            e.adjoint_run(2, 0, (1, 1, 1), 8)
        e.close()
        names = {x.split(">")[0] for x in fake.log().decode().split("\n") if "k_adj_step" in x}
        assert len(names) == 1 and names.pop().endswith(hint.lower()), batch


@pytest.mark.parametrize("shape,hint", [("70,70,300", False), ("110,110,300", True)])  # 147 and 363 MB
def test_reverse_stores_follow_the_forward_line_alone_and_in_a_batch(fake_path, shape, hint):
    run_case(fake_path, "reverse_hint", shape, hint)


# ---- read-outs ----------------------------------------------------------------------------------

def case_pinned_memory(fake):
    """Read-outs keep at most 16 MiB of pinned memory however many engines read, and none without one."""
    from sim_juncs_amd.engine import Engine

    most, kept = 16 << 20, []
    for _ in range(2):
        engines = [Engine((128, 128, 80), 0.02) for _ in range(6)]  # 10 MB of FP64 values per component
        for e in engines:
            e.step(1)
            e.read_field("Ex")
            e.get_field("Ey", (0.1, 0.1, 0.1))
            e.read_field("Hz", (3, 3, 3), (100, 90, 20))
            kept.append(fake.host_bytes())
        for e in engines:
            e.close()
        assert 0 < max(kept) <= most and fake.host_bytes() == 0


def test_read_outs_share_their_pinned_memory(fake_path):
    run_case(fake_path, "pinned_memory")


if __name__ == "__main__":
    sys.path[:0] = [ROOT, HERE]
    globals()["case_" + sys.argv[2]](Fake(sys.argv[1]), *sys.argv[3:])
