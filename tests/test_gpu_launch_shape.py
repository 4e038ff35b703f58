"""The limit on the workgroups per CU of the band class (fsr_set_launch_shape, and
what fsr_autotune chooses) holds for the exact band pass: it limits the launch,
never raises it past the 6 workgroups that are resident, and leaves the band as
it is."""
import numpy as np
import pytest

from fluidsurfacereconstructiongpu_amd import datasets as ds
from fluidsurfacereconstructiongpu_amd.reconstructor import Reconstructor
from tests import launches

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("limit", [0, 1, 4, 6, 9])
def test_band_limit_reaches_exact_pass(torch_cuda, limit):
    print(f"\n[gpu case] band class limit {limit}", flush=True)
    fr = ds.small_block(30, 20, 17, ratio=2)
    rec = Reconstructor("zb05")
    rec.run(fr)
    bits = rec.buffer("band_bits", np.uint32, rec.ctx.buffer_ptr("band_bits")[1])
    launches.set_workgroups(rec, band=limit)
    res = rec.run(fr)
    assert res.stats["band_exceptions"] > 0
    assert np.array_equal(rec.buffer("band_bits", np.uint32, bits.size), bits)
    k = launches.find(launches.frame_launches(torch_cuda, rec, fr), "k_band_exceptions")
    assert k.grid == (launches.num_cus(torch_cuda) * min(limit or 6, 6), 1, 1)
