"""The row-of-threads reverse tile gives the bits of the one-row tile: z lines around a wavefront's 64
cells, workgroups of one wavefront to the largest, tiles that end with the grid or past it, one-plane
chunks, PML layers on each axis alone and on all, periodic axes, Drude-only and Lorentz media, and the
default tile on either side of the size from which it takes rows of threads.

No tolerance: both forms spell out the same operations in the same order."""
import numpy as np
import pytest

from sim_juncs_amd import materials as M
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Batch, Engine

pytestmark = pytest.mark.gpu


def scene(shape, precision, pml=None, periodic=(0, 0, 0), drude=False, seed=2):
    rng = np.random.default_rng(seed)
    lut = [M.VACUUM, M.SIO2_CONST if drude else M.SIO2.scaled(1.0),
           (M.AU_REFERENCE_AS_RUN if drude else M.AU).scaled(1.0)]
    ids = np.zeros(tuple(shape) + (3,), dtype=np.int64)
    ids[:, shape[1] // 2:, shape[2] // 2:] = 2
    ids[shape[0] // 2:, :, : shape[2] // 3] = 1
    scn = scenario.Scenario(name=f"adjoint{shape}", shape=tuple(shape), dx=0.02, precision=precision,
                            periodic=periodic, matw=scenario.pack(ids), lut=lut)
    if pml:
        scn.pml = (pml, 1e-15, 2.0)
    lo = [max(0, n // 2 - 2) for n in shape]
    hi = [min(n, l + 3) for n, l in zip(shape, lo)]
    scn.design = (lo, hi, rng.uniform(1.5, 4.0, size=tuple(h - l for l, h in zip(lo, hi))))
    scn.sources = [scenario.plane_source(shape, scn.dx, max(0, shape[2] // 2 - 4),
                                         scenario.gaussian_pulse(0.8, 1.5, 0.3, start_fs=0.0))]
    scn.meta = dict(gap=tuple(n // 2 for n in shape), nd=int(np.prod(scn.design[2].shape)))
    return scn


def run(scn, tile, steps=45):
    eng = scn.make(Engine, precision=scn.precision)
    if tile:
        eng.set_adjoint_tile(*tile)
    J, g = eng.adjoint_run(steps, 0, scn.meta["gap"], scn.meta["nd"])
    info = eng.adjoint_kernel_info()
    eng.close()
    assert np.abs(g).max() > 0 and np.isfinite(g).all()
    return J, g, info


@pytest.mark.parametrize("pml,periodic,drude", [
    ([3] * 6, (0, 0, 0), False), ([3, 3, 0, 0, 0, 0], (0, 0, 0), False), ([0, 0, 3, 3, 0, 0], (0, 0, 0), True),
    ([0, 0, 0, 0, 3, 3], (1, 1, 0), False), (None, (1, 1, 1), True), (None, (0, 0, 0), False),
])
@pytest.mark.parametrize("precision,shape,rows,xc", [
    ("fp64", (10, 8, 62), 5, 3), ("fp64", (10, 12, 70), 6, 10), ("fp64", (9, 8, 64), 4, 1), ("fp64", (7, 9, 20), 8, 2),
    ("fp64", (8, 7, 250), 1, 4), ("fp32", (10, 9, 65), 14, 4), ("fp32", (8, 8, 128), 7, 1), ("fp32", (7, 7, 300), 2, 3),
    ("fp32", (6, 8, 512), 1, 6), ("fp32", (9, 10, 6), 9, 5),
])
def test_rows_of_threads_give_the_bits_of_one_row(precision, shape, rows, xc, pml, periodic, drude):
    if min(shape) < 7:
        pml = [min(p, 1) for p in pml] if pml else None
    scn = scene(shape, precision, pml, periodic, drude)
    print("[case] reverse rows", shape, precision, pml, periodic, drude, rows, xc, flush=True)
    J0, g0, _ = run(scn, ("register_rows", 1, 4))
    J1, g1, info = run(scn, ("thread_rows", rows, xc))
    assert info[1:] == (-(-(rows + 1) * shape[2] // 64) * 64, -(-shape[1] // rows) * -(-shape[0] // xc))
    assert J0 == J1 and np.array_equal(g0, g1)


@pytest.mark.parametrize("precision,shape,threads", [
    ("fp32", (52, 52, 52), 64),      # below 12 MB of fields: one row per workgroup
    ("fp32", (64, 62, 64), 896),     # five tiles of 13 rows
    ("fp64", (40, 60, 100), 512),
    ("fp32", (20, 12, 900), 960),    # a row and its halo do not fit a workgroup
])
def test_default_reverse_tile_gives_the_same_bits_alone_and_in_a_batch(precision, shape, threads):
    scns = [scene(shape, precision, [3] * 6, seed=s) for s in (2, 3)]
    print("[case] default reverse tile", shape, precision, flush=True)
    ref = [run(s, ("register_rows", 1, 4), steps=20) for s in scns]
    own = [run(s, None, steps=20) for s in scns]
    assert own[0][2][1] == threads
    engs = [s.make(Engine, precision=precision) for s in scns]
    b = Batch(engs)
    J, g = b.adjoint_run(20, [s.meta["gap"] for s in scns], [s.meta["nd"] for s in scns], 0)
    b.close()
    for i, e in enumerate(engs):
        assert np.array_equal(own[i][1], ref[i][1]) and np.array_equal(g[i], ref[i][1]), i
        e.close()
