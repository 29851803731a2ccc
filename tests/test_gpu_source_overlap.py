"""Sources that inject into the same values add up: sheets on one plane (two colours, or two polarisations
of one pulse), points on a sheet, magnetic ones, and one source whose images on a periodic axis of one
cell are the same cell; against the FP64 oracle (1e-10 relative, FP32 1e-4) and the same bits every time.
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Batch, Engine

pytestmark = pytest.mark.gpu


def scene(kind, precision):
    shape, periodic = ((14, 12, 30), (0, 0, 0)) if kind != "thin" else ((1, 1, 30), (1, 1, 0))
    scn = scenario.Scenario(name=kind, shape=shape, dx=0.02, precision=precision, periodic=periodic,
                            pml=([0, 0, 0, 0, 4, 4], 1e-15, 2.0))

    def pulse(wavelength, cep):
        return scenario.gaussian_pulse(wavelength, 1.5, cep, start_fs=-3.0)

    def sheet(comp, wavelength, cep, z=10):
        return scenario.plane_source(shape, scn.dx, z, pulse(wavelength, cep), comp=comp)

    def point(comp, x, y, z, wavelength):
        return dict(comp=comp, box=[x * scn.dx, y * scn.dx, z * scn.dx] * 2, **pulse(wavelength, 0.2))

    if kind == "electric":
        scn.sources = [sheet("Ex", 0.8, 0.1), sheet("Ex", 0.6, 0.9), sheet("Ey", 0.8, 0.4), point("Ex", 6.3, 5.2, 10, 0.7)]
    elif kind == "magnetic":
        scn.sources = [sheet("Hy", 0.8, 0.1), sheet("Hy", 0.6, 0.9), point("Hy", 6.3, 5.2, 10.4, 0.7), sheet("Ex", 0.7, 0.0)]
    else:
        scn.sources = [point("Ex", 0.3, 0.6, 10.2, 0.8), point("Hz", 0.2, 0.7, 14.3, 0.6)]
    scn.dfts = [((0, 0, 20), shape[:2] + (21,), ("Ex", "Hy"), [1.2])]
    return scn


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["electric", "magnetic", "thin"])
def test_sources_on_the_same_cells_add_up(kind, precision):
    scn = scene(kind, precision)
    print("[case] source overlap", kind, precision, flush=True)
    o = scn.make(Oracle)
    o.step(90)
    ref = [o.read_field(c) for c in range(6)]
    engines = [scn.make(Engine) for _ in range(3)]
    engines[0].step(90)
    engines[1].set_graph(10)
    engines[1].step(90)
    b = Batch([engines[2]])
    b.step(90)
    for c in range(6):
        family = max(np.linalg.norm(ref[q]) for q in (range(3) if c < 3 else range(3, 6)))
        got = engines[0].read_field(c)
        assert family > 0 and np.linalg.norm(got - ref[c]) <= (1e-10 if precision == "fp64" else 1e-4) * family, c
        for e in engines[1:]:
            assert np.array_equal(e.read_field(c), got), c
    spectrum = o.read_dft(0)
    assert np.linalg.norm(engines[0].read_dft(0) - spectrum) <= (1e-10 if precision == "fp64" else 1e-4) * np.linalg.norm(spectrum)
    b.close()
    for e in engines:
        e.close()
