"""Read-outs of several engines from several threads at a time take pinned buffers of their own: each
gives what the same engine gives alone, for values of one buffer, of several and single points."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from sim_juncs_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
def test_read_outs_from_threads(precision):
    shapes = [(120, 100, 70), (33, 20, 17), (96, 110, 90), (5, 6, 7)]
    print("[case] read-outs from threads", precision, shapes, flush=True)
    engines, values = [], []
    for i, shape in enumerate(shapes):
        e = Engine(shape, 0.02, precision=precision)
        v = np.random.default_rng(i).standard_normal(shape).astype(np.float32).astype(np.float64)
        e.write_field("Ey", v)
        engines.append(e)
        values.append(v)

    def read(i):
        e, v = engines[i], values[i]
        hi = tuple(n - 1 for n in e.shape)
        at = np.array([1.0, 1.5, 1.0]) * e.dx  # the Ey point of cell (1, 1, 1)
        for _ in range(20):
            assert np.array_equal(e.read_field("Ey"), v)
            assert np.array_equal(e.read_field("Ey", (1, 2, 3), hi), v[1:-1, 2:-1, 3:-1])
            assert abs(e.get_field("Ey", at) - v[1, 1, 1]) <= 1e-12 * max(1.0, np.abs(v).max())

    with ThreadPoolExecutor(len(shapes)) as pool:
        for f in [pool.submit(read, i) for i in range(len(shapes))]:
            f.result()
    for e in engines:
        e.close()
