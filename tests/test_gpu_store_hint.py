"""Stores with the non-temporal cache hint change no bits: engines whose step touches too little for it
alone, and enough together, step to the same bits alone and as one batch, in every form that has both
kinds of store (FP64 pairs of auxiliaries go out as two of them).

That the hint is off alone and on together is asserted for these same scenes, on the CPU, by
test_host_runtime.py (test_scenes_lie_on_either_side_of_the_store_line): a line that moves fails there.
"""
import numpy as np
import pytest

from sim_juncs_amd import materials as M
from sim_juncs_amd import scenario
from sim_juncs_amd.engine import Batch, Engine

# precision, shape, engines, tile of the batch (None: the default, here z passes), kernel
CASES = [
    ("fp32", (96, 96, 96), 8, ("register_rows", 8), "k_step<"),
    ("fp32", (96, 96, 96), 8, ("thread_rows", 8), "k_step_rows<"),
    ("fp64", (96, 96, 96), 3, ("register_rows", 8), "k_step<"),
    ("fp64", (96, 96, 96), 3, ("thread_rows", 8), "k_step_rows<"),
    ("fp32", (50, 40, 1100), 3, None, "k_step_z<"),
    ("fp64", (40, 40, 600), 4, None, "k_step_z<"),
]


def scene(precision, shape):
    ids = np.zeros(shape + (3,), dtype=np.uint8)
    ids[:, :, shape[2] // 2:] = 1
    ids[shape[0] // 3: shape[0] // 2, :, shape[2] // 4: shape[2] // 2] = 2
    return scenario.Scenario(name="store_hint", shape=shape, dx=0.02, precision=precision, matw=scenario.pack(ids),
                             lut=[M.VACUUM, M.SIO2.scaled(1.0), M.AU.scaled(1.0)], pml=([6] * 6, 1e-15, 2.0))


def engines(precision, shape, count):
    scn = scene(precision, shape)
    return [scn.make(Engine) for _ in range(count)]


def alone(e, tile):
    """The batch's tile on an engine of its own (the default fills a workgroup with thread rows)."""
    if tile:
        e.set_tile(tile[0], 1 if tile[0] == "register_rows" else (1024 if e.precision == "fp32" else 512) // e.shape[2] - 1,
                   tile[1])


@pytest.mark.gpu
@pytest.mark.parametrize("precision,shape,count,tile,kernel", CASES)
def test_the_store_hint_changes_no_bits(precision, shape, count, tile, kernel):
    print("[case] store hint", precision, shape, count, tile, flush=True)
    grouped = engines(precision, shape, count)

    def fill(e, seed):
        rng = np.random.default_rng(seed)
        for c in range(6):
            e.write_field(c, rng.standard_normal(shape).astype(np.float32))

    for i, e in enumerate(grouped):
        fill(e, i)
    b = Batch(grouped)
    if tile:
        b.set_tile(*tile)
    b.step(7)
    for i in (0, count - 1):
        (e,) = engines(precision, shape, 1)
        alone(e, tile)
        fill(e, i)
        e.step(7)
        for c in range(6):
            a = e.read_field(c)
            assert np.isfinite(a).all() and np.array_equal(a, grouped[i].read_field(c)), (i, c)
        e.close()
    b.close()
    for e in grouped:
        e.close()
