"""Reconstructor.run and run_indexed around the sizes where the upload changes
form (nothing, one particle, just below and above the staged size), and their
rerun after an overflow, which puts the sorted particles back in order: the same
bits as a run whose buffers were large enough, on host arrays and on device
tensors, and the particles as a plain upload sorts them."""
import numpy as np
import pytest

from fluidsurfacereconstructiongpu_amd import datasets as ds
from fluidsurfacereconstructiongpu_amd import reconstructor as rc

pytestmark = pytest.mark.gpu

EDGE = (rc._STAGE_FLOATS - 64) // 4


def outputs(rec, fr, indexed, cap, pos=None, dens=None):
    if indexed:
        phi, vtx, nrm, idx, stats = rec.run_indexed(fr, cap, cap, pos=pos, dens=dens)
        out = [phi, vtx, nrm, idx]
    else:
        res = rec.run(fr, cap, pos=pos, dens=dens)
        stats = res.stats
        out = [res.phi, *res.soup()]
    out += [rec.pos_sorted, rec.dens_sorted]
    return [t.cpu().numpy().tobytes() for t in out], stats


@pytest.mark.parametrize("indexed", [False, True])
@pytest.mark.parametrize("n", [1, 257, EDGE - 1, EDGE, EDGE + 16, EDGE + 17, 50001])
def test_upload_and_rerun(torch_cuda, n, indexed):
    print(f"\n[gpu case] run host path {n} indexed={indexed}", flush=True)
    torch = torch_cuda
    fr = ds.scattered(n=n, extent=0.02 * n ** (1 / 3), ratio=2)
    rec = rc.Reconstructor("zb05")
    cap = 64 * n + 4096
    want, stats = outputs(rec, fr, indexed, cap)
    assert not stats["overflow"] and stats["num_mesh_vertices"] > 0
    dev = lambda a: torch.from_numpy(a).cuda()
    for pos, dens in ((None, None), (dev(fr.pos), dev(fr.dens))):
        got, st = outputs(rc.Reconstructor("zb05"), fr, indexed, 1, pos, dens)
        assert got == want and not st["overflow"]
    # another frame through the same staging buffer, then the first again
    outputs(rec, ds.scattered(n=max(1, n // 2), extent=0.3, ratio=2), indexed, cap)
    assert outputs(rec, fr, indexed, cap)[0] == want
