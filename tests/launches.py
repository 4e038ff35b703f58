"""The kernels that a frame launches, read from a stream capture that is never
replayed: names, grids and scalar arguments, for the tests of host rules whose
choice does not show in a frame's outputs."""
from __future__ import annotations

import ctypes
import dataclasses


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class _KernelNodeParams(ctypes.Structure):
    """hipKernelNodeParams (hip_runtime_api.h)."""

    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", _Dim3), ("params", ctypes.POINTER(ctypes.c_void_p)),
                ("shared", ctypes.c_uint32)]


@dataclasses.dataclass
class Launch:
    name: str       # mangled
    grid: tuple
    args: list      # the kernel's arguments as u32, None for those not asked for


_THREAD_LOCAL = 1   # hipStreamCaptureModeThreadLocal
_KERNEL = 0         # hipGraphNodeTypeKernel


def recorded(torch, enqueue, u32_args=None) -> list:
    """Launches of enqueue(stream), in no particular order.  u32_args: kernel name
    part -> indices of its 32-bit arguments to read.  Everything that enqueue needs
    must be allocated (run the frame once before)."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p

    def ok(rc):
        assert rc == 0, "HIP error %d" % rc

    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    s = ctypes.c_void_p(stream.cuda_stream)
    graph = ctypes.c_void_p()
    ok(hip.hipStreamBeginCapture(s, _THREAD_LOCAL))
    try:
        enqueue(stream)
    finally:
        ok(hip.hipStreamEndCapture(s, ctypes.byref(graph)))
    out = []
    try:
        count = ctypes.c_size_t()
        ok(hip.hipGraphGetNodes(graph, None, ctypes.byref(count)))
        nodes = (ctypes.c_void_p * count.value)()
        ok(hip.hipGraphGetNodes(graph, nodes, ctypes.byref(count)))
        for node in nodes[: count.value]:
            node = ctypes.c_void_p(node)
            kind = ctypes.c_int()
            ok(hip.hipGraphNodeGetType(node, ctypes.byref(kind)))
            if kind.value != _KERNEL:
                continue
            p = _KernelNodeParams()
            ok(hip.hipGraphKernelNodeGetParams(node, ctypes.byref(p)))
            name = hip.hipKernelNameRefByPtr(ctypes.c_void_p(p.func), s).decode()
            args = []
            for part, indices in (u32_args or {}).items():
                if part in name:
                    args = [None] * (max(indices) + 1)
                    for i in indices:
                        args[i] = ctypes.cast(p.params[i], ctypes.POINTER(ctypes.c_uint32))[0]
            out.append(Launch(name, (p.grid.x, p.grid.y, p.grid.z), args))
    finally:
        ok(hip.hipGraphDestroy(graph))
    return out


def frame_launches(torch, rec, fr, u32_args=None) -> list:
    """Launches of one frame of the Reconstructor, which has run it before."""
    pos = torch.from_numpy(fr.pos).cuda()
    dens = torch.from_numpy(fr.dens).cuda()
    cap = int(rec._tri.shape[0])
    return recorded(torch, lambda s: rec.launch(fr, pos, dens, cap, stream=s), u32_args)


def find(launches: list, part: str) -> Launch:
    hits = [x for x in launches if part in x.name]
    assert len(hits) == 1, (part, [x.name for x in launches])
    return hits[0]


def set_workgroups(rec, field=0, mc=0, aniso=0, band=0) -> None:
    """The context's limits on the workgroups per CU, per kernel class (0: none)."""
    shape = (ctypes.c_uint32 * 4)(field, mc, aniso, band)
    assert rec.ctx.lib.fsr_set_launch_shape(rec.ctx.handle, shape) == 0


def num_cus(torch) -> int:
    return torch.cuda.get_device_properties(0).multi_processor_count
