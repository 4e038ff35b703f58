"""Reconstructor.run and run_indexed with arrays that hold the frame's particles in
another form than (N, 3) and (N,): one density per row of a column, a position as
a column vector, more densities than particles.  Below and above the size up to
which the upload is staged they give the frame's outputs, and the particles come
back in the form that they were given in.  What is no array stays refused."""
import dataclasses

import numpy as np
import pytest

from fluidsurfacereconstructiongpu_amd import datasets as ds
from fluidsurfacereconstructiongpu_amd import reconstructor as rc

pytestmark = pytest.mark.gpu

EDGE = (rc._STAGE_FLOATS - 64) // 4
FORMS = {
    "column": lambda fr: dict(dens=fr.dens[:, None]),
    "vectors": lambda fr: dict(pos=fr.pos[:, :, None]),
    "longer": lambda fr: dict(dens=np.concatenate([fr.dens, np.full(7, -5.0, np.float32)])),
}


def outputs(fr, indexed, cap):
    rec = rc.Reconstructor("zb05")
    if indexed:
        phi, vtx, nrm, idx, stats = rec.run_indexed(fr, cap, cap)
        out = [phi, vtx, nrm, idx]
    else:
        res = rec.run(fr, cap)
        out, stats = [res.phi, *res.soup()], res.stats
    assert not stats["overflow"] and stats["num_mesh_vertices"] > 0
    return [t.cpu().numpy().tobytes() for t in out], rec


@pytest.mark.parametrize("indexed", [False, True])
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("n", [257, EDGE + 17])
def test_forms(torch_cuda, n, form, indexed):
    print(f"\n[gpu case] run array forms {n} {form} indexed={indexed}", flush=True)
    fr = ds.scattered(n=n, extent=0.02 * n ** (1 / 3), ratio=2)
    fr.dens = np.random.default_rng(3).uniform(900.0, 1100.0, n).astype(np.float32)
    cap = 64 * n + 4096
    want, rec = outputs(fr, indexed, cap)
    other = dataclasses.replace(fr, **FORMS[form](fr))
    got, rec2 = outputs(other, indexed, cap)
    assert got == want
    assert rec2.pos_sorted.shape == other.pos.shape and rec2.dens_sorted.shape == other.dens.shape
    assert rec2.pos_sorted.cpu().numpy().tobytes() == rec.pos_sorted.cpu().numpy().tobytes()
    dens = rec2.dens_sorted.cpu().numpy().ravel()
    assert np.array_equal(dens[:n], rec.dens_sorted.cpu().numpy())
    assert np.all(dens[n:] == -5.0)


@pytest.mark.parametrize("n", [257, EDGE + 17])
def test_host_tensors_are_refused(torch_cuda, n):
    print(f"\n[gpu case] run array forms {n} tensors", flush=True)
    fr = ds.scattered(n=n, extent=0.02 * n ** (1 / 3), ratio=2)
    other = dataclasses.replace(fr, pos=torch_cuda.from_numpy(fr.pos))
    with pytest.raises(TypeError):
        rc.Reconstructor("zb05").run(other)


@pytest.mark.parametrize("n", [257, EDGE + 17])
def test_too_few_values_are_refused(torch_cuda, n):
    print(f"\n[gpu case] run array forms {n} too few", flush=True)
    fr = ds.scattered(n=n, extent=0.02 * n ** (1 / 3), ratio=2)
    for short in (dict(dens=fr.dens[:1]), dict(dens=fr.dens[:-1]), dict(pos=fr.pos[:, :2].copy())):
        with pytest.raises(ValueError):
            rc.Reconstructor("zb05").run(dataclasses.replace(fr, **short))


@pytest.mark.parametrize("indexed", [False, True])
@pytest.mark.parametrize("form", ["column", "longer", "spare rows", "part"])
def test_rerun_restores_given_tensors(torch_cuda, form, indexed):
    """The rerun after an overflow puts device tensors back in order whatever their
    form: the same bits as a run with room from the start."""
    print(f"\n[gpu case] rerun forms {form} indexed={indexed}", flush=True)
    n = 5003
    fr = ds.scattered(n=n, extent=0.02 * n ** (1 / 3), ratio=2)
    fr.dens = np.random.default_rng(3).uniform(900.0, 1100.0, n).astype(np.float32)

    def run(cap):
        pos, dens = torch_cuda.from_numpy(fr.pos).cuda(), torch_cuda.from_numpy(fr.dens).cuda()
        spare = torch_cuda.full((7,), -5.0, device="cuda")
        if form == "column":
            dens = dens[:, None]
        elif form == "longer":
            dens = torch_cuda.cat([dens, spare])
        elif form == "spare rows":
            dens = torch_cuda.cat([dens, spare]).view(-1, 10)   # 5,010 in rows of 10
        else:   # inside a larger buffer
            dens = torch_cuda.cat([spare, dens, spare])[7:7 + n]
        rec = rc.Reconstructor("zb05")
        if indexed:
            phi, vtx, nrm, idx, stats = rec.run_indexed(fr, cap, cap, pos=pos, dens=dens)
            out = [phi, vtx, nrm, idx]
        else:
            res = rec.run(fr, cap, pos=pos, dens=dens)
            out, stats = [res.phi, *res.soup()], res.stats
        assert rec.dens_sorted is dens and not stats["overflow"]
        return [t.cpu().numpy().tobytes() for t in out + [pos, dens]]

    assert run(1) == run(64 * n + 4096)
