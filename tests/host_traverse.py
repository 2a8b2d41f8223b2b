"""The library's traversal compiled for the host (tests/host/traverse.cpp), for
scenes of one mesh under one instance, and the path state's size."""
import ctypes as C
import os
import subprocess

import numpy as np

from ymrt_amd import abi

_HERE = os.path.dirname(os.path.abspath(__file__))
_lib = None


def lib():
    global _lib
    if _lib is None:
        path = os.path.join(_HERE, "_build", "libhost_traverse.so")
        if not os.path.exists(path):
            subprocess.check_call(["make", "-s", "-C", os.path.join(_HERE, "host")])
        L = C.CDLL(path)
        vp, u32 = C.c_void_p, C.c_uint32
        L.ht_mesh.restype = L.ht_nodes.restype = vp
        L.ht_mesh.argtypes = [vp, u32, vp]
        L.ht_free.argtypes = L.ht_nodes.argtypes = [vp]
        L.ht_max_stack.restype = L.ht_node_count.restype = u32
        L.ht_max_stack.argtypes = L.ht_node_count.argtypes = [vp]
        L.ht_trace.restype = C.c_int
        L.ht_trace.argtypes = [vp, vp, u32, C.c_int, C.c_int, vp, vp]
        L.ht_visit.argtypes = [vp, vp, u32, C.c_int, vp]
        L.ht_path_bytes.restype = C.c_uint64
        _lib = L
    return _lib


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


class Mesh:
    """The mesh and instance transform of sa, which holds one instance."""

    def __init__(self, sa):
        it, = sa.instances
        assert it["geometry_type"] == abi.GEOMETRY_MESH
        m = sa.meshes[it["mesh"]]
        pos = np.ascontiguousarray(np.asarray(m["pos"], np.float32)[np.asarray(m["pidx"])].reshape(-1, 9))
        w2o = np.ascontiguousarray(np.asarray(it["w2o"], np.float32)[:3])
        self._h = lib().ht_mesh(_ptr(pos), len(pos), _ptr(w2o))
        self.max_stack = lib().ht_max_stack(self._h)

    def __del__(self):
        if getattr(self, "_h", None):
            lib().ht_free(self._h)

    def trace(self, rays, any=False, ring=False):
        """(hits (n, 4) or flags (n,), visits (n, 2), the most stack entries
        that a ray held at once)."""
        out = np.empty((len(rays),) if any else (len(rays), 4), np.uint32)
        visits = np.empty((len(rays), 2), np.uint32)
        rays = np.ascontiguousarray(rays)
        deepest = lib().ht_trace(self._h, _ptr(rays), len(rays), int(any), int(ring), _ptr(out), _ptr(visits))
        return out, visits, deepest


def nodes(lo, hi, child):
    """128-B-aligned node records of boxes (n, 4, 3) and child codes (n, 4)."""
    n = len(lo)
    buf = np.zeros(n * 32 + 32, np.float32)
    skip = (-buf.ctypes.data % 128) // 4
    rec = buf[skip:skip + n * 32].reshape(n, 32)
    for a in range(3):
        rec[:, 8 * a:8 * a + 4] = lo[:, :, a]
        rec[:, 8 * a + 4:8 * a + 8] = hi[:, :, a]
    rec[:, 24:28] = child.astype(np.uint32).view(np.float32)
    return rec


def visit(recs, rays, park):
    out = np.empty((len(rays), 4), np.uint32)
    lib().ht_visit(_ptr(recs), _ptr(rays), len(rays), int(park), _ptr(out))
    return out
