"""Material words prepared on the device: the order of the set-up calls, PML twins, design voxels,
refused words, and the pole count that sjf_step_bytes reports."""
import itertools

import numpy as np
import pytest

from oracle.oracle import Oracle
from sim_juncs_amd import materials as M
from sim_juncs_amd import scenario
from sim_juncs_amd._lib import EngineError
from sim_juncs_amd.engine import Engine

pytestmark = pytest.mark.gpu

LUT = [M.VACUUM, M.SIO2.scaled(1.0), M.AU.scaled(1.0), M.MaterialSpec(2.13)]


def setup(sim, shape, order, fold, design):
    rng = np.random.default_rng(sum(shape))
    ids = rng.integers(0, len(LUT), size=tuple(shape) + (3,))
    ids[:, : shape[1] // 2] = 1
    lo = [n // 2 - 1 for n in shape]
    hi = [n // 2 + 1 for n in shape]
    eps = rng.uniform(1.5, 4.0, size=(2, 2, 2))
    calls = dict(m=lambda: sim.set_materials(scenario.pack(ids), LUT), p=lambda: sim.set_pml([2, 1, 0, 2, 2, 3]),
                 f=lambda: sim.set_pml_dispersion(fold), d=lambda: sim.set_design_eps(lo, hi, eps))
    for c in order:
        if c != "d" or design:
            calls[c]()
    sim.add_source(**scenario.plane_source(shape, 0.02, shape[2] // 2,
                                           scenario.gaussian_pulse(0.8, 2.0, 0.3, start_fs=0.0)))
    if design:
        ids[tuple(slice(l, h) for l, h in zip(lo, hi))] = 255
    return ids


@pytest.mark.parametrize("shape", [(7, 8, 65), (6, 6, 130)])
@pytest.mark.parametrize("fold,design", [(1.25, True), (1.25, False), (0.0, True)])
def test_set_up_calls_in_any_order_match_oracle(shape, fold, design):
    # materials write the whole map: the design box comes after them
    orders = [o for o in itertools.permutations("mpfd") if o.index("m") < o.index("d")][::3]
    orc = Oracle(shape, 0.02, precision="fp64")
    ids = setup(orc, shape, "mpfd", fold, design)
    orc.step(25)
    pml = [(2, 1), (0, 2), (2, 3)]
    slab = np.zeros(shape, dtype=bool)
    for d, (lo, hi) in enumerate(pml):
        i = np.arange(shape[d]).reshape([-1 if q == d else 1 for q in range(3)])
        slab |= np.broadcast_to((i < lo) | (i >= shape[d] - hi), shape)
    npol = np.array([len(m.poles) for m in LUT] + [0] * 252)
    ndrude = np.array([sum(p.drude for p in m.poles) for m in LUT] + [0] * 252)
    poles = np.where(slab[..., None] & (fold > 0), ndrude[ids], npol[ids]).sum()
    cells = int(np.prod(shape))
    expect = cells * (12 * 8 + 4) + 3 * 8 * poles + (8 * 8 if design else 0) + \
        sum(8 * 8 * sum(p) * cells // n for p, n in zip(pml, shape))
    for order in orders:
        eng = Engine(shape, 0.02, precision="fp64")
        setup(eng, shape, order, fold, design)
        print("[case] set-up", shape, order, fold, design, flush=True)
        assert eng.step_bytes() == expect
        eng.step(25)
        for c in range(6):
            ref = orc.read_field(c)
            assert np.linalg.norm(eng.read_field(c) - ref) <= 1e-10 * max(np.linalg.norm(ref), 1e-300), (order, c)
        eng.close()


def test_refused_words_leave_the_materials_as_they_were():
    shape = (6, 7, 66)
    eng, orc = Engine(shape, 0.02, precision="fp64"), Oracle(shape, 0.02, precision="fp64")
    setup(eng, shape, "mpf", 1.25, False)
    setup(orc, shape, "mpf", 1.25, False)
    print("[case] refused words", flush=True)
    bad = np.zeros(shape, dtype=np.uint32)
    bad[5, 6, 65] = 0x040000  # an id past the list, in the last cell
    with pytest.raises(EngineError, match="id >= n_mat"):
        eng.set_materials(bad, LUT)
    bad[0, 0, 3] = 0x00ff00   # a design id before there is a design box, in an earlier cell
    with pytest.raises(EngineError, match="before sjf_set_design_eps"):
        eng.set_materials(bad, LUT)
    bad[0, 0, 3] = 0xff0400   # an id past the list comes first within the cell
    with pytest.raises(EngineError, match="id >= n_mat"):
        eng.set_materials(bad, LUT)
    eng.step(20)
    orc.step(20)
    for c in range(6):
        ref = orc.read_field(c)
        assert np.linalg.norm(eng.read_field(c) - ref) <= 1e-10 * max(np.linalg.norm(ref), 1e-300), c
    eng.close()
