"""DFT regions whose launch has more threads than one grid dimension takes: many (component, cell)
pairs at one frequency beside one cell at 64 frequencies.  The sums are those of small regions over
the same field, bit for bit: every accumulator is summed by one thread in the order of the steps.
"""
import numpy as np
import pytest

from sim_juncs_amd.engine import Engine

pytestmark = pytest.mark.gpu

COMPS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")


def test_sums_of_many_values_and_many_frequencies():
    n = 226
    freqs = np.linspace(0.5, 1.5, 64)
    assert 64 * 6 * n ** 3 >= 2 ** 32
    print("[case] large DFT launch", n, flush=True)
    reads = []
    for large in (True, False):
        e = Engine((n, n, n), 0.01)
        e.add_source("Ex", [1.13, 1.13, 1.13] * 2, freq=1.0, width=0.02, t_start=-0.1, t_end=0.3)
        box = ((0, 0, 0), (n, n, n)) if large else ((100, 110, 105), (120, 115, 125))
        a = e.add_dft(*box, COMPS, [1.1])
        b = e.add_dft((112, 113, 114), (113, 114, 115), ("Ez",), freqs)
        e.step(6)
        v = e.read_dft(a)
        reads.append((v[:, :, 100:120, 110:115, 105:125] if large else v, e.read_dft(b)))
        e.close()
    assert np.abs(reads[1][0]).max() > 0 and np.abs(reads[1][1]).max() > 0
    for x, y in zip(*reads):
        assert np.array_equal(x, y)
