"""Every form of the neighbour kernels' work split, with the form asserted: a chunk
(64 particles or vertices of one hash cell) shared by a workgroup's waves or a wave
each, the chunks dealt out or fetched from counters, and the build for long lists.
All evaluate the same candidates in the same order, so a frame's outputs are the
same bits under every limit of workgroups per CU.  The form follows from the chunk
count (from the hash cells, the field's work record or the band), the launch's grid and the limit that the
kernel is given, both read from the recorded launch."""
import numpy as np
import pytest

from fluidsurfacereconstructiongpu_amd import datasets as ds
from fluidsurfacereconstructiongpu_amd.autograd import SurfaceField
from fluidsurfacereconstructiongpu_amd.reconstructor import Batch, Reconstructor
from tests import launches

pytestmark = pytest.mark.gpu

LATTICE = {
    "lattice13": lambda m, s: ds.jittered_lattice(n_side=13, grid_res=64, method=m, scale=s),
    "lattice17": lambda m, s: ds.jittered_lattice(n_side=17, grid_res=56, method=m, scale=s),
    "lattice24": lambda m, s: ds.jittered_lattice(n_side=24, grid_res=80, method=m, scale=s),
    "lattice36": lambda m, s: ds.jittered_lattice(n_side=36, grid_res=96, method=m, scale=s,
                                                  cell=0.0055),
    "scattered": lambda m, s: (ds.scattered(n=20_011, extent=0.5, ratio=3, method=m)
                               if m == "yu13" else ds.scattered(n=30_011, extent=1.0, ratio=2)),
    "dam": lambda m, s: ds.dam_break(n_target=61_003, block=(64, 32, 32), spacing=0.0125,
                                     grid_res=104, method=m, scale=s),
}
# kernel -> index of its chunk limit for the shared form
LIMIT_ARG = {"k_field_zb05I": 3, "k_smooth_mcI": 10, "k_covariance_mcI": 2, "k_field_anisoI": 1}
# the forms of (field) or (smoothing, covariance, field) per limit
ZB05 = [
    ("lattice17", {0: ["shared dealt"], 1: ["dealt"]}),
    ("lattice24", {0: ["shared counters"], 1: ["counters"]}),
    ("scattered", {0: ["counters"], 1: ["counters"]}),
]
YU13 = [
    ("lattice13", {0: ["shared", "shared", "shared dealt"]}),
    ("lattice36", {0: ["shared", "shared", "shared counters"], 1: ["dealt", "dealt", "counters"]}),
    ("scattered", {0: ["shared", "shared", "shared counters"], 2: ["counters", "dealt", "shared counters"],
                   1: ["counters", "counters", "counters"]}),
    ("dam", {0: ["shared", "shared", "shared counters"], 1: ["long", "counters", "counters"]}),
]


def chunks(counts) -> int:
    return int(((counts.astype(np.int64) + 63) // 64).sum())


def field_chunks(fr, index, radius) -> int:
    """Chunks of the band vertices per hash cell, the grid padded by radius cells (but
    for vertices within rounding of a cell's face)."""
    rx, ry, _ = fr.sc.res
    f = np.float32
    n = [r + 2 * radius for r in fr.sp.res]
    key = 0
    for axis, v in ((2, index // (rx * ry)), (1, index // rx % ry), (0, index % rx)):
        x = f(fr.sc.min[axis]) + v.astype(f) * f(fr.sc.cell)
        c = np.trunc((x - f(fr.sp.min[axis])) / f(fr.sp.cell)).astype(np.int64)
        key = key * n[axis] + np.clip(c, -radius, fr.sp.res[axis] - 1 + radius) + radius
    return chunks(np.bincount(key))


def form(launch, nch, limit) -> str:
    grid = launch.grid[0]
    if "Lb0E" in launch.name:
        return "long"
    dealt = lambda units: (nch + 63) // 64 <= units * (grid // 64)
    if nch > limit:
        return "dealt" if dealt(4) else "counters"
    if "k_field" not in launch.name:
        return "shared"
    return "shared dealt" if dealt(1) else "shared counters"


def run(torch, fr, method, per_cu):
    rec = Reconstructor(method)
    launches.set_workgroups(rec, field=per_cu, aniso=per_cu)
    res = rec.run(fr)
    out = [t.cpu().numpy().view(np.uint32).copy() for t in (res.phi, *res.soup())]
    if method == "yu13":
        out.append(rec.buffer("mean_pos", np.uint32, 4 * fr.n))
        out.append(rec.buffer("g_matrices", np.uint32, 9 * res.stats["num_involved_particles"]))
        r = rec.buffer("cell_ranges", np.uint32, 2 * fr.sp.count).reshape(-1, 2).astype(np.int64)
        index = rec.buffer("band_index", np.uint32, res.stats["num_band_vertices"])
        inv = rec.buffer("involve_counts", np.uint32, fr.sp.count)
        kernels = [("k_smooth_mcI", chunks(np.where(r[:, 0] == 0xFFFFFFFF, 0, r[:, 1] - r[:, 0]))),
                   ("k_covariance_mcI", chunks(inv)),
                   ("k_field_anisoI", field_chunks(fr, index.astype(np.int64), 2))]
    else:
        work = rec.buffer("field_work", np.uint32, rec.ctx.buffer_ptr("field_work")[1])
        kernels = [("k_field_zb05I", np.nonzero(work == 0xFFFFFFFF)[0][0] // 3)]
    got = launches.frame_launches(torch, rec, fr, {k: [LIMIT_ARG[k]] for k, _ in kernels})
    forms = []
    for name, nch in kernels:
        k = launches.find(got, name)
        forms.append(form(k, nch, k.args[LIMIT_ARG[name]]))
    return out, forms


@pytest.mark.parametrize("method,name,by_limit", [("zb05", *c) for c in ZB05] +
                         [("akinci12", "lattice24", {0: [], 1: []})] + [("yu13", *c) for c in YU13])
def test_forms_give_the_same_bits(torch_cuda, method, name, by_limit):
    print(f"\n[gpu case] chunk forms {method} {name}", flush=True)
    fr = LATTICE[name](method, 1.3 if method == "yu13" else 1.0)
    want = None
    for per_cu, forms in by_limit.items():
        got, took = run(torch_cuda, fr, method, per_cu)
        if forms:
            assert took == forms, (per_cu, took)
        want = want or got
        for a, b in zip(want, got):
            assert np.array_equal(a, b), per_cu


@pytest.mark.parametrize("method", ["zb05", "yu13"])
def test_long_build_in_a_batch(torch_cuda, method):
    """Four frames in flight: past 131,072 particles together they take the build
    for long lists, one at a time the one for few chunks."""
    print(f"\n[gpu case] chunk forms batch {method}", flush=True)
    fr = LATTICE["lattice36"](method, 1.3 if method == "yu13" else 1.0)
    assert fr.n <= 131_072 < 4 * fr.n
    rec = Reconstructor(method)
    res = rec.run(fr)
    phi, T = res.phi.cpu().numpy(), res.stats["num_mesh_vertices"]
    tri = res.tri_pos[:T].cpu().numpy()
    batch = Batch(method, [fr] * 4, lanes=4, cap_factor=T / fr.n + 1.0)
    batch.run()
    torch_cuda.cuda.synchronize()
    assert not batch.grow_overflowed()
    for b in batch.bufs:
        assert b["phi"].cpu().numpy().tobytes() == phi.tobytes()
        assert b["tri"][:T].cpu().numpy().tobytes() == tri.tobytes()
    batch.close()


def test_adjoint_gather_dealt_and_fetched(torch_cuda):
    print("\n[gpu case] chunk forms adjoint", flush=True)
    torch = torch_cuda
    fr = ds.lattice_ball(n_target=60_001, grid_res=96)
    cus = launches.num_cus(torch)
    grads = []
    for per_cu in (0, 1):
        sf = SurfaceField(fr)
        launches.set_workgroups(sf.rec, field=per_cu)
        pos = torch.from_numpy(fr.pos).cuda().requires_grad_(True)
        phi, soup = sf(pos)
        r = sf.rec.buffer("cell_ranges", np.uint32, 2 * fr.sp.count).reshape(-1, 2).astype(np.int64)
        nch = chunks(np.where(r[:, 0] == 0xFFFFFFFF, 0, r[:, 1] - r[:, 0]))
        # one chunk per workgroup at most, or not
        assert ((nch + 63) // 64 <= (per_cu or 6) * cus // 64) == (per_cu == 0)
        w = torch.linspace(-1.0, 1.0, phi.numel(), device="cuda")
        (g,) = torch.autograd.grad([phi, soup], pos, [w, torch.ones_like(soup)])
        grads.append(g.cpu().numpy().tobytes())
        sf.close()
    assert grads[0] == grads[1]
