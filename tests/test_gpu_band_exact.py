"""The exact band path (scalar cells too coarse for the box dilation: every
surface particle walks its own box) against the oracle, bit for bit: particle
counts around the 8-particle step and the per-wave group sizes, boxes clamped
at the grid's faces, rows that straddle two mask words, and particles spread so
widely that a step's boxes do not fit its LDS window."""
import numpy as np
import pytest

from fluidsurfacereconstructiongpu_amd import datasets as ds
from tests import parity

pytestmark = pytest.mark.gpu

CASES = {
    "one": lambda: ds.scattered(n=1, extent=0.2),
    "step": lambda: ds.scattered(n=8, extent=0.1, ratio=2),
    "step+1": lambda: ds.scattered(n=9, extent=0.1, ratio=2),
    "wave+1": lambda: ds.scattered(n=65, extent=0.2, ratio=3),
    "spread": lambda: ds.scattered(n=3001, extent=2.9, ratio=1),
    "group16": lambda: ds.scattered(n=40013, extent=1.9, ratio=2),
    "block-ratio1": lambda: ds.small_block(13, 9, 7, ratio=1),
    "block-ratio2": lambda: ds.small_block(70, 21, 33, ratio=2),
    "block-ratio3": lambda: ds.small_block(45, 30, 11, ratio=3),
    # group 64: more than 64 x 4096 particles
    "block-group64": lambda: ds.small_block(82, 66, 54, ratio=2),
}


@pytest.mark.parametrize("name", list(CASES))
def test_exact_band_matches_oracle(torch_cuda, name):
    print(f"\n[gpu case] exact band {name}", flush=True)
    fr = CASES[name]()
    rec, res = parity.run_gpu(fr, "zb05")
    buf = parity.gpu_buffers(rec, fr, res.stats)
    ref = parity.Stage(fr, "zb05")
    assert res.stats["num_surface_particles"] == int(ref.flags.sum())
    assert res.stats["band_exceptions"] == int(ref.flags.sum())
    assert np.array_equal(buf["flags"], ref.flags)
    assert np.array_equal(buf["band"], ref.band)
    assert np.array_equal(buf["index"], ref.index)
