"""DFT accumulation where a wavefront's (component, cell) pairs end, cross regions or cross from E to H,
regions with different numbers of frequencies, and step counters advanced by the source, the DFT or a
launch of their own, over graph replays and single steps; FP64 rounding (1e-10) against the oracle."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("source", [True, False])
@pytest.mark.parametrize("regions", [
    [], [((3, 3, 9), (4, 4, 10), ("Ez",), 1)], [((0, 0, 9), (8, 8, 10), ("Ex", "Hy"), 3)],      # 64 pairs a component
    [((0, 0, 9), (7, 9, 10), ("Ex", "Ey", "Hx", "Hz"), 2), ((2, 2, 12), (3, 3, 13), ("Hx",), 5),
     ((1, 0, 14), (10, 11, 15), ("Ey", "Hy"), 1)],
    [((0, 0, 4), (10, 11, 7), ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"), 4)],  # holds the source cells: two launches
])
def test_dft_regions_match_oracle(regions, source):
    shape = (10, 11, 17)
    scn = scenario.Scenario(name="dft", shape=shape, dx=0.02, precision="fp64", periodic=(0, 0, 0))
    if source:
        scn.sources = [scenario.plane_source(shape, scn.dx, 5, scenario.gaussian_pulse(0.8, 1.0, 0.3, start_fs=0.0))]
    scn.dfts = [(lo, hi, comps, np.linspace(0.7, 1.5, nf)) for lo, hi, comps, nf in regions]
    eng, orc = scn.make(Engine), scn.make(Oracle)
    rng = np.random.default_rng(4)
    for c in range(6):
        f = rng.standard_normal(shape)
        eng.write_field(c, f)
        orc.write_field(c, f)
    print("[case] dft regions", len(regions), source, flush=True)
    for n in (1, 2, 70, 1):  # single steps and replays of the captured graph
        eng.step(n)
        orc.step(n)
    for c in range(6):
        ref = orc.read_field(c)
        assert np.linalg.norm(eng.read_field(c) - ref) <= 1e-10 * np.linalg.norm(ref)
    for i in range(len(regions)):
        a, b = eng.read_dft(i), orc.read_dft(i)
        assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b), i
    eng.close()
