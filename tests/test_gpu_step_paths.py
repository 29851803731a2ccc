"""The fused step where its paths part: z lines around a wavefront's 64 cells, segments of one
material, of several and of design voxels, Drude and Lorentz pole state over odd and even step
counts, grids that end with a full tile, the default z passes and non-temporal stores.

Tolerances are those of the other parity tests: FP64 rounding (1e-10 relative L2) and the FP32
workload tolerance (1e-4) against the FP64 oracle.
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from sim_juncs_amd import materials as M
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Batch, Engine

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-10, "fp32": 1e-4}


def rel(a, b):
    n = np.linalg.norm(b)
    return np.linalg.norm(a - b) / (n if n > 0 else 1.0)


def scene(shape, media, precision, periodic, seed=0):
    """`media`: "segments" (whole z lines of gold and of SiO2 beside mixed ones), "drude" (the same
    with a Drude metal and no Lorentz pole), "design" (a design box over them), "metal" (one material
    with poles in every cell)."""
    rng = np.random.default_rng(seed + sum(shape))
    gold = M.AU_REFERENCE_AS_RUN if media == "drude" else M.AU
    lut = [M.VACUUM, M.SIO2_CONST if media == "drude" else M.SIO2.scaled(1.0), gold.scaled(1.0)]
    ids = np.zeros(tuple(shape) + (3,), dtype=np.int64)
    if media == "metal":
        lut, ids = [lut[2]], ids
    else:
        ids[:, shape[1] // 2:] = 2                   # one-material segments with poles
        ids[:, :1, shape[2] // 3:] = 1               # a material boundary within a segment
        ids[shape[0] // 2:, 1:2] = rng.integers(0, 3, size=ids[shape[0] // 2:, 1:2].shape)
    pml = None if any(periodic) else ([1, 1, 1, 1, 2, 2] if min(shape) > 3 else None)
    scn = scenario.Scenario(name=f"{media}{shape}", shape=tuple(shape), dx=0.02, precision=precision,
                            periodic=periodic, matw=scenario.pack(ids), lut=lut)
    if pml:
        scn.pml = (pml, 1e-15, 2.0)
    if media == "design":
        lo = [n // 3 for n in shape]
        hi = [min(n, l + 5) for n, l in zip(shape, lo)]
        scn.design = (lo, hi, rng.uniform(1.5, 4.0, size=tuple(h - l for l, h in zip(lo, hi))))
    scn.sources = [scenario.plane_source(shape, scn.dx, shape[2] // 2,
                                         scenario.gaussian_pulse(0.8, 2.0, 0.3, start_fs=0.0))]
    return scn, rng


@pytest.mark.parametrize("media", ["segments", "drude", "design", "metal"])
@pytest.mark.parametrize("precision,shape,periodic,tile", [
    ("fp64", (6, 8, 63), (0, 0, 0), None), ("fp32", (6, 8, 64), (0, 0, 0), None),
    ("fp64", (6, 9, 65), (0, 0, 0), ("thread_rows", 3, 6)),    # three full tiles of one chunk
    ("fp32", (7, 8, 65), (0, 0, 0), ("thread_rows", 4, 1)),    # one-plane chunks
    ("fp64", (7, 6, 64), (0, 0, 0), ("register_rows", 1, 1)),
    ("fp32", (5, 6, 130), (1, 1, 1), ("register_rows", 1, 2)),
    ("fp64", (5, 6, 130), (1, 0, 1), None), ("fp32", (6, 7, 130), (0, 1, 0), None),
    ("fp64", (5, 4, 200), (0, 0, 0), None), ("fp32", (5, 4, 300), (0, 0, 0), None),  # one register row
    ("fp64", (4, 4, 520), (0, 0, 0), None),                    # 256-cell passes
    ("fp32", (4, 4, 1030), (0, 0, 0), None),                   # 128-cell passes
    ("fp64", (1, 1, 65), (0, 0, 0), None), ("fp32", (2, 3, 1), (0, 0, 0), None),
])
def test_step_paths_match_oracle(precision, shape, periodic, tile, media):
    scn, rng = scene(shape, media, precision, periodic)
    eng, orc = scn.make(Engine, precision=precision), scn.make(Oracle)
    if tile:
        eng.set_tile(*tile)
    print(f"[case] {scn.name} {precision} {periodic} {eng.launch_info()}", flush=True)
    for c in range(6):
        f = rng.standard_normal(shape)
        if precision == "fp32":
            f = f.astype(np.float32).astype(np.float64)
        eng.write_field(c, f)
        orc.write_field(c, f)
    for n in (1, 12, 9):  # odd and even counts: either of two buffers is the current one
        eng.step(n)
        orc.step(n)
        errs = [rel(eng.read_field(c), orc.read_field(c)) for c in range(6)]
        assert max(errs) < TOL[precision], (n, errs)
    eng.close()


@pytest.mark.parametrize("form", ["register_rows", "thread_rows"])
def test_nontemporal_stores_of_a_large_set_change_no_bits(form):
    """Eight FP32 boxes below the 300 MB working set from which stores take the non-temporal hint
    alone (43-45 MB of fields each), above it together, step to the same bits."""
    scns = [scenario.plain_box(n=96, steps=0, precision="fp32", seed=i) for i in range(8)]
    assert sum(48 * s.cells for s in scns) > 300e6
    for s in scns:
        s.sources[0].update(scenario.gaussian_pulse(0.8, 2.0, 0.3, start_fs=0.0))
    print("[case] non-temporal stores", form, flush=True)
    grouped = [s.make(Engine) for s in scns]
    b = Batch(grouped)
    b.set_tile(form, 8)
    b.step(40)
    for s, g in zip(scns, grouped):
        e = s.make(Engine)
        e.set_tile(form, 1 if form == "register_rows" else 9, 8)
        e.step(40)
        for c in range(6):
            assert np.array_equal(e.read_field(c), g.read_field(c)), c
        assert np.abs(e.read_field("Ex")).max() > 0
        e.close()
    b.close()
    for g in grouped:
        g.close()
