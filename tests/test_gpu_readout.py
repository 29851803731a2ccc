"""Read-outs that pass through the pinned stage in chunks of 4 MiB: one value, a partial chunk, an
exact multiple of it and more than two, for whole components, boxes, DFT regions and points."""
import numpy as np
import pytest

from oracle.oracle import Oracle
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 7), (64, 64, 128), (128, 64, 128), (67, 131, 150)])
def test_components_and_boxes_come_back_as_written(shape, precision):
    rng = np.random.default_rng(5)
    eng = Engine(shape, 0.02, precision=precision)
    vals = [rng.standard_normal(shape).astype(np.float32 if precision == "fp32" else np.float64) for _ in range(6)]
    for c, v in enumerate(vals):
        eng.write_field(c, v)
    print("[case] read-out", shape, precision, flush=True)
    for c in (5, 0, 2):
        assert np.array_equal(eng.read_field(c), vals[c])
        for lo, hi in (((0, 0, 0), shape), ([n // 3 for n in shape], [n // 3 + 1 for n in shape]),
                       ([n // 2 for n in shape], shape), ((0, 0, 0), [max(1, n - 1) for n in shape])):
            box = vals[c][tuple(slice(l, h) for l, h in zip(lo, hi))]
            assert np.array_equal(eng.read_field(c, lo, hi), box), (c, lo, hi)
    eng.close()


def test_dft_regions_and_points_match_oracle():
    shape = (90, 80, 14)
    scn = scenario.Scenario(name="read", shape=shape, dx=0.02, precision="fp64", periodic=(0, 0, 0))
    scn.sources = [scenario.plane_source(shape, scn.dx, 4, scenario.gaussian_pulse(0.8, 1.0, 0.3, start_fs=0.0))]
    freqs = np.linspace(0.7, 1.5, 20)
    # 2 * 20 * 90 * 80 values: two chunks and a part; 1 * 1 * 1: one value
    scn.dfts = [((0, 0, 8), (90, 80, 9), ("Ex", "Hy"), freqs), ((3, 4, 9), (4, 5, 10), ("Ex",), freqs[:1])]
    pts = np.array(shape) * scn.dx * np.array([[0.5] * 3, [0.013, 0.991, 0.7], [0.0] * 3, [1.0] * 3])
    scn.monitors = [("Ex", pts), ("Hy", pts)]
    eng, orc = scn.make(Engine), scn.make(Oracle)
    print("[case] dft read-out", flush=True)
    eng.step(29)
    got = [np.array([eng.get_field(c, p) for p in pts]) for c in ("Ex", "Hy")]
    eng.step(1)
    orc.step(30)
    for i in range(2):
        a, b = eng.read_dft(i), orc.read_dft(i)
        assert a.shape == b.shape and a.dtype == np.complex128 and np.abs(b).max() > 0
        assert np.linalg.norm(a - b) < 1e-10 * np.linalg.norm(b)
    last = orc.read_monitors()[-1].reshape(2, len(pts))  # sampled at the start of the last step
    for c, g, ref in zip(("Ex", "Hy"), got, last):
        assert np.abs(g - ref).max() <= 1e-10 * np.abs(orc.read_field(c)).max()
    eng.close()
