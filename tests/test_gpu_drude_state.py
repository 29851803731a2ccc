"""FP32 Drude media hold one array of pole state, updated in place: the adjoint run that records and the
one that checkpoints and recomputes give the same bits (the state is saved and restored whole), and
both agree with the FP64 engine within the FP32 tolerance of the gradient tests (1e-4 relative).
Forward steps of such media are compared with the oracle in test_gpu_step_paths.py.
"""
import numpy as np
import pytest

from sim_juncs_amd import materials as M
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,tile", [
    ((14, 12, 20), ("thread_rows", 5, 4)), ((12, 10, 70), ("register_rows", 1, 3)), ((8, 9, 130), ("register_rows", 2, 8)),
])
def test_gradients_of_drude_media(shape, tile):
    rng = np.random.default_rng(sum(shape))
    ids = np.zeros(shape + (3,), dtype=np.int64)
    ids[:, : shape[1] // 2, shape[2] // 2:] = 1
    lo = tuple(n // 2 - 2 for n in shape)
    scn = scenario.Scenario(name="drude", shape=shape, dx=0.02, matw=scenario.pack(ids),
                            lut=[M.VACUUM, M.AU_REFERENCE_AS_RUN.scaled(1.0)], pml=([2] * 6, 1e-15, 2.0),
                            design=(lo, tuple(l + 3 for l in lo), rng.uniform(1.5, 4.0, size=(3, 3, 3))))
    scn.sources = [scenario.plane_source(shape, scn.dx, shape[2] // 2 - 6, scenario.gaussian_pulse(0.8, 1.5, 0.4, start_fs=0.0))]
    gap = tuple(n // 2 + 1 for n in shape)
    print("[case] drude gradients", shape, tile, flush=True)
    got = {}
    for precision, every in (("fp32", 0), ("fp32", 7), ("fp32", 4), ("fp64", 0)):
        e = scn.make(Engine, precision=precision)
        e.set_tile(*tile)
        got[precision, every] = e.adjoint_run(61, every, gap, 27)
        e.close()
    J, g = got["fp32", 0]
    J64, g64 = got["fp64", 0]
    assert np.abs(g64).max() > 0
    for every in (7, 4):
        assert got["fp32", every][0] == J and np.array_equal(got["fp32", every][1], g), every
    assert abs(J - J64) <= 1e-4 * abs(J64)
    assert np.linalg.norm(g - g64) <= 1e-4 * np.linalg.norm(g64)
