"""The neighbour kernels treat a chunk (64 particles or vertices of one hash
cell) with one wave, or share it among the 4 waves of a workgroup when the frame
has few chunks; and they deal a short chunk list out to the waves, or fetch from
counters.  All forms evaluate the same candidates in the same order, so a
frame's outputs are the same bits: a launch limit of one workgroup per CU moves
these frames from the shared form and the dealt list to the others."""
import ctypes

import numpy as np
import pytest

from fluidsurfacereconstructiongpu_amd import datasets as ds
from fluidsurfacereconstructiongpu_amd.reconstructor import Reconstructor

pytestmark = pytest.mark.gpu

# about 900 to 2500 chunks each: above 3 x 256, the limit with one workgroup
# per CU, and below the limit of the default launch
FRAMES = {
    "lattice36": lambda m, scale: ds.jittered_lattice(n_side=36, grid_res=96, scale=scale,
                                                      method=m, cell=0.0055),
    # chunks with remainders of every size, and particles on their own
    "dam": lambda m, scale: ds.dam_break(n_target=61_003, block=(64, 32, 32), spacing=0.0125,
                                         grid_res=104, method=m, scale=scale),
}
FRAMES["small"] = lambda m, scale: ds.jittered_lattice(n_side=17, grid_res=56, scale=scale,
                                                       method=m)
CASES = [("yu13", "lattice36"), ("yu13", "dam"), ("zb05", "small"), ("zb05", "dam"),
         ("akinci12", "small"), ("akinci12", "dam")]


def frame_outputs(fr, method, per_cu):
    rec = Reconstructor(method)
    shape = (ctypes.c_uint32 * 4)(*([per_cu] * 4))
    assert rec.ctx.lib.fsr_set_launch_shape(rec.ctx.handle, shape) == 0
    res = rec.run(fr)
    tri, nrm = res.soup()
    out = dict(phi=res.phi, tri=tri, nrm=nrm)
    out = {k: v.cpu().numpy().view(np.uint32).copy() for k, v in out.items()}
    out["flags"] = rec.buffer("surface_flags", np.uint32, fr.n)
    if method == "yu13":
        out["mean"] = rec.buffer("mean_pos", np.uint32, 4 * fr.n)
        out["G"] = rec.buffer("g_matrices", np.uint32, 9 * res.stats["num_involved_particles"])
    else:
        _, cap = rec.ctx.buffer_ptr("field_work")
        w = rec.buffer("field_work", np.uint32, cap)
        out["work"] = w[: np.nonzero(w == 0xFFFFFFFF)[0][0]]
    return out, res.stats


@pytest.mark.parametrize("method,name", CASES)
def test_shared_and_wave_chunks_agree(torch_cuda, method, name):
    print(f"\n[gpu case] shared chunks {method} {name}", flush=True)
    fr = FRAMES[name](method, 1.3 if method == "yu13" else 1.0)
    shared, st = frame_outputs(fr, method, 0)
    wave, st1 = frame_outputs(fr, method, 1)
    assert st == st1
    for k in shared:
        assert np.array_equal(shared[k], wave[k]), k
    if name == "small" and method == "zb05":
        assert 3 * 256 < len(shared["work"]) // 3 <= 3 * 6 * 256
