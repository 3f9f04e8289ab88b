"""Thin host-side driver of libdiso_hip.so for torch tensors.

`Extractor` is the counterpart of the reference's engine objects (CuMC, src/cumc.h:70-139;
CUDualMC, src/cudualmc.h:70-150): it owns the scan control workspace of each stream it has run
on (zero-filled once, grown on demand) and runs the count / emit / backward passes on the
current torch stream. Per-call state (the segment bases the backward needs) is returned to the
caller instead of being kept inside the object, so one extractor can serve many grids whose
backward runs later (autograd, activation checkpointing).
"""
import ctypes

import torch

from . import _lib

_DTYPES = {torch.float32: _lib.F32, torch.float64: _lib.F64}


class Counted:
    """Result of the counting pass: segment bases on the device and the totals on the host.
    After emission it also holds what a DMC backward needs from the forward: the quads and one
    byte of patch information per DMC vertex."""

    __slots__ = ("seg", "n_verts", "n_faces", "n_crossing", "flags", "dims", "iso", "flags_in", "quads", "vinfo",
                 "spec")

    def __init__(self, seg, totals, dims, iso, flags_in):
        self.seg = seg
        self.n_verts = int(totals.n_verts)
        self.n_faces = int(totals.n_faces)
        self.n_crossing = int(totals.n_crossing)
        self.flags = int(totals.flags)
        self.dims = dims
        self.iso = iso
        self.flags_in = flags_in
        self.quads = None
        self.vinfo = None
        self.spec = None  # (verts, faces, vinfo) already emitted into buffers these counts fit

    @property
    def empty_grid(self):
        """The reference wrapper's early-out: min(sdf) >= iso or max(sdf) <= iso
        (diso/__init__.py:49,103)."""
        both = _lib.TOTAL_HAS_BELOW | _lib.TOTAL_HAS_ABOVE
        return (self.flags & both) != both

    @property
    def has_nan(self):
        return bool(self.flags & _lib.TOTAL_HAS_NAN)


def _ptr(t):
    return ctypes.c_void_p(0 if t is None else t.data_ptr())


def _prefix(buf, n):
    """The first n rows of `buf` as a tensor of their own over the same memory. Not a view (as
    buf[:n] would be): autograd forbids in-place edits of views made inside a custom Function's
    forward, and callers may edit the returned vertices in place."""
    size = (n,) + tuple(buf.shape[1:])
    return torch.empty(0, dtype=buf.dtype, device=buf.device).set_(buf.untyped_storage(), buf.storage_offset(), size,
                                                                    buf.stride())


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(device):
    """The current HIP stream of `device` as a raw handle (the direct query when torch has it:
    the public one costs some ten microseconds per call)."""
    if _raw_stream is not None:
        return ctypes.c_void_p(_raw_stream(device.index if device.index is not None else torch.cuda.current_device()))
    return ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)


def _capturing():
    return torch.cuda.is_current_stream_capturing()


class Extractor:
    def __init__(self, algo, dtype):
        if dtype not in _DTYPES:
            raise ValueError(f"diso_amd: dtype must be torch.float32 or torch.float64, got {dtype}")
        self.algo = algo
        self.dtype = dtype
        self.code = _DTYPES[dtype]
        self._ctl = {}  # (device, stream) -> control block (ctl_for)
        self._first = {}  # device -> the first of them, for captures
        self._guess = {}  # (device, dims, flags) -> (vertices, faces) of the last call
        self._need = {}  # (dims, flags) -> workspace bytes (_sizes)
        self._at = {}  # (dims, flags) -> offset of the totals (_totals_at)
        _lib.lib()  # fail loudly now if the HIP library is not there

    def check_grid(self, grid, name="grid"):
        if not isinstance(grid, torch.Tensor):
            raise TypeError(f"{name} must be a torch.Tensor")
        if grid.device.type != "cuda":
            raise RuntimeError(f"{name} must be a CUDA tensor")
        if grid.dtype != self.dtype:
            raise RuntimeError(f"{name} type must match the {'mc' if self.algo == _lib.MC else 'dmc'} class")

    def _sizes(self, dims, flags):
        """Workspace bytes of a grid: the segment workspace, what of it a backward with these flags
        keeps, and the control block (asked once per dims and flags)."""
        key = (dims, flags)
        got = self._need.get(key)
        if got is None:
            L = _lib.lib()
            seg = L.diso_seg_bytes(*dims, flags & ~_lib.FLAG_RECOMPUTE)
            got = (seg, L.diso_seg_bytes(*dims, flags) if flags & _lib.FLAG_RECOMPUTE else seg,
                   L.diso_ctl_bytes(*dims, flags))
            if min(got) < 0:
                _lib.check(min(got), "workspace sizing")
            if len(self._need) >= 256:
                self._need.clear()
            self._need[key] = got
        return got

    def _totals_at(self, dims, flags):
        """Offset of the totals in the segment workspace (asked once per dims and flags)."""
        got = self._at.get((dims, flags))
        if got is None:
            got = _lib.lib().diso_totals_offset(*dims, flags)
            if got < 0:
                _lib.check(got, "workspace sizing")
            if len(self._at) >= 256:
                self._at.clear()
            self._at[(dims, flags)] = got
        return got

    def ctl_for(self, device, dims, flags, capturing=False, stream=None):
        """The control block of the current stream. One per stream, because consecutive calls may use
        it only in stream order: a forward returns as soon as its totals are known, while blocks of
        its count may still be reading and clearing the block's words. A capture takes the device's
        first block, which is kept as long as this object (or, without one, a block that each replay
        clears)."""
        need = self._sizes(dims, flags)[2]
        key = (device.index, (_stream(device) if stream is None else stream).value)
        if not capturing:
            ctl = self._ctl.get(key)
            if ctl is not None and ctl.numel() >= need:
                return ctl
            capturing = _capturing()
        first = self._first.get(device.index)
        if first is not None and first.numel() < need:
            first = None
        if capturing and first is not None:
            return first
        # New blocks start zero-filled; the scan keeps them consistent from then on (its words carry
        # their call's epoch, so not even a timed-out call needs a reset).
        ctl = torch.zeros(max(need, 1 << 16) * 5 // 4, dtype=torch.uint8, device=device)
        if not capturing:
            if first is None:
                self._first[device.index] = ctl
            if len(self._ctl) >= 64:
                self._ctl.clear()  # many streams: start over (freed memory goes back to its own stream)
            self._ctl[key] = ctl
        return ctl

    def _extract(self, grid, deform, iso, flags, verts=None, faces=None, vinfo=None):
        """diso_extract: the counting pass, and behind it the emission into the given buffers (none: no
        emission). Waits only for the counts, which the counting kernel writes to host memory."""
        dims = tuple(grid.shape)
        dev = grid.device
        nseg, _, need = self._sizes(dims, flags)
        seg = torch.empty(nseg, dtype=torch.uint8, device=dev)
        stream = _stream(dev)
        ctl = self._ctl.get((dev.index, stream.value))
        if ctl is None or ctl.numel() < need:
            ctl = self.ctl_for(dev, dims, flags, stream=stream)
        tot = _lib.Totals()
        vp, vcap, fp, fcap, ip = 0, 0, 0, 0, 0
        if verts is not None:
            vp, vcap, fp, fcap = verts.data_ptr(), verts.shape[0], faces.data_ptr(), faces.shape[0]
            ip = 0 if vinfo is None else vinfo.data_ptr()
        rc = _lib.lib().diso_extract(self.algo, self.code, grid.data_ptr(), 0 if deform is None else deform.data_ptr(),
                                     *dims, iso, flags, seg.data_ptr(), nseg, ctl.data_ptr(), ctl.numel(), vp, vcap, fp,
                                     fcap, ip, tot, stream)
        _lib.check(rc, "extraction")
        return Counted(seg, tot, dims, iso, flags)

    def count(self, grid, iso, flags):
        """The counting pass alone."""
        return self._extract(grid, None, float(iso), flags)

    def count_speculative(self, grid, deform, iso, flags):
        """The counting pass, and, when an earlier call on a grid of these dims gives a size
        estimate, the emission queued right behind it into buffers of that size plus a margin: the
        host then waits only for the counts, so its work until the next launch overlaps the emission
        instead of leaving the device idle. If the counts fit, `counted.spec` holds the emitted
        buffers (emit() returns views of them); otherwise emit() runs the emission again at the exact
        size (the queued one writes nothing when the counts exceed its capacities)."""
        dev = grid.device
        key = (dev.index, tuple(grid.shape), flags)
        guess = self._guess.get(key)
        if guess is None:
            counted = self.count(grid, iso, flags)
        else:
            dmc = self.algo == _lib.DMC
            vcap, fcap = guess[0] + guess[0] // 4 + 1024, guess[1] + guess[1] // 4 + 1024
            verts = torch.empty((vcap, 3), dtype=self.dtype, device=dev)
            faces = torch.empty((fcap, 4 if dmc else 3),
                                dtype=torch.int64 if flags & _lib.FLAG_INDEX64 else torch.int32, device=dev)
            vinfo = torch.empty(vcap, dtype=torch.uint8, device=dev) if dmc else None
            counted = self._extract(grid, deform, iso, flags, verts, faces, vinfo)
            if counted.n_verts <= vcap and counted.n_faces <= fcap:
                counted.spec = (verts, faces, vinfo)
        self._remember(key, counted.n_verts, counted.n_faces)
        return counted

    def _remember(self, key, n_verts, n_faces):
        if len(self._guess) >= 64 and key not in self._guess:
            self._guess.clear()  # many different grids: start over
        self._guess[key] = (n_verts, n_faces)

    def _scratch(self, counted, device):
        n = _lib.lib().diso_scratch_bytes(self.algo, self.code, counted.n_crossing)
        if n < 0:
            _lib.check(n, "scratch sizing")
        return torch.empty(max(n, 1), dtype=torch.uint8, device=device), n

    def emit(self, grid, deform, counted, flags):
        """Vertices [V,3] and faces ([F,3] MC triangles / [Q,4] DMC quads) of a counted grid."""
        L = _lib.lib()
        dmc = self.algo == _lib.DMC
        k = 4 if dmc else 3
        idx = torch.int64 if flags & _lib.FLAG_INDEX64 else torch.int32
        if counted.spec is not None:  # emitted already (count_speculative): exact-size prefixes
            v, f, vi = counted.spec
            counted.spec = None
            verts, faces = _prefix(v, counted.n_verts), _prefix(f, counted.n_faces)
            vinfo = vi
        else:
            verts = torch.empty((counted.n_verts, 3), dtype=self.dtype, device=grid.device)
            faces = torch.empty((counted.n_faces, k), dtype=idx, device=grid.device)
            vinfo = torch.empty(counted.n_verts, dtype=torch.uint8, device=grid.device) if dmc else None
            rc = L.diso_emit(self.algo, self.code, _ptr(grid), _ptr(deform), *counted.dims, counted.iso, flags,
                             _ptr(counted.seg), counted.seg.numel(), _ptr(verts), counted.n_verts, _ptr(faces),
                             counted.n_faces, _ptr(vinfo), _stream(grid.device))
            _lib.check(rc, "emit pass")
        if dmc:
            counted.quads, counted.vinfo = faces, vinfo
        if flags & _lib.FLAG_RECOMPUTE:
            # The backward will re-derive the classification from the samples: keep only the
            # segment bases and release the stored classification.
            counted.seg = counted.seg[:self._sizes(counted.dims, flags)[1]].clone()
        return verts, faces

    def backward(self, grid, deform, counted, flags, adj_verts, adj_grid, adj_deform):
        """Writes (or, with FLAG_ACCUMULATE, adds) d(sum(adj_verts*verts))/d(grid, deform)."""
        check_backward_shapes(counted.dims, grid, deform, adj_grid, adj_deform)
        L = _lib.lib()
        adj_verts = adj_verts.contiguous()
        if adj_verts.dtype != self.dtype:
            raise RuntimeError("adj_verts type must match the extractor's dtype")
        if adj_verts.shape != (counted.n_verts, 3):
            raise ValueError(f"adj_verts must have shape ({counted.n_verts}, 3), got {tuple(adj_verts.shape)}")
        dmc = self.algo == _lib.DMC
        quads = counted.quads if dmc else None
        if dmc and quads is None:
            raise RuntimeError("DMC backward needs the quads of its forward")
        if dmc:
            # the quads' index width decides how the backward reads them
            flags = (flags & ~_lib.FLAG_INDEX64) | (_lib.FLAG_INDEX64 if quads.dtype == torch.int64 else 0)
        scratch, nscratch = self._scratch(counted, grid.device)
        rc = L.diso_backward(self.algo, self.code, _ptr(grid), _ptr(deform), *counted.dims, counted.iso, flags,
                             _ptr(counted.seg), counted.seg.numel(), _ptr(quads), counted.n_faces if dmc else 0,
                             _ptr(counted.vinfo if dmc else None), _ptr(adj_verts), counted.n_verts,
                             _ptr(adj_grid), _ptr(adj_deform), _ptr(scratch), nscratch, _stream(grid.device))
        _lib.check(rc, "backward pass")


def check_backward_shapes(dims, grid, deform, adj_grid, adj_deform):
    """The backward writes dims worth of gradients: the grid, the gradient buffers and (with
    deform) the deform must have the forward's dims, or the kernels would address memory outside
    them. Raises RuntimeError (the reference binding's error type) otherwise."""
    dims = tuple(int(d) for d in dims)
    if tuple(grid.shape) != dims:
        raise RuntimeError(f"grid has shape {tuple(grid.shape)}, the forward's was {dims}")
    if adj_grid is None or tuple(adj_grid.shape) != dims:
        raise RuntimeError(f"adj_grid must have shape {dims}, got {None if adj_grid is None else tuple(adj_grid.shape)}")
    if deform is not None:
        want = dims + (3,)
        if tuple(deform.shape) != want:
            raise RuntimeError(f"deform must have shape {want}, got {tuple(deform.shape)}")
        if adj_deform is None or tuple(adj_deform.shape) != want:
            raise RuntimeError(f"adj_deform must have shape {want}, got "
                               f"{None if adj_deform is None else tuple(adj_deform.shape)}")


def split_quads(verts, quads):
    """DiffDMC quad -> triangle split on the GPU (diso_split; diso/__init__.py:117-147):
    [Q,4] quads -> [2Q,3] int64 triangles, first-cut quads first."""
    if verts.device.type != "cuda" or quads.device.type != "cuda":
        raise RuntimeError("split_quads: verts and quads must be CUDA tensors")
    if verts.dtype not in _DTYPES:
        raise RuntimeError(f"split_quads: verts must be float32 or float64, got {verts.dtype}")
    if quads.dtype not in (torch.int32, torch.int64) or quads.dim() != 2 or quads.shape[1] != 4:
        raise ValueError("split_quads: quads must be an int32/int64 [Q, 4] tensor")
    L = _lib.lib()
    nq = int(quads.shape[0])
    tris = torch.empty((2 * nq, 3), dtype=torch.int64, device=verts.device)
    if nq == 0:
        return tris
    verts = verts.detach().contiguous()
    quads = quads.contiguous()
    nbytes = L.diso_split_scratch_bytes(nq)
    if nbytes < 0:
        _lib.check(nbytes, "split sizing")
    with torch.cuda.device(verts.device):
        scratch = torch.empty(nbytes, dtype=torch.uint8, device=verts.device)
        flags = _lib.FLAG_INDEX64 if quads.dtype == torch.int64 else 0
        rc = L.diso_split(_DTYPES[verts.dtype], _ptr(verts), int(verts.shape[0]), _ptr(quads), nq, flags, _ptr(tris),
                          2 * nq, _ptr(scratch), nbytes, _stream(verts.device))
    _lib.check(rc, "split")
    return tris
