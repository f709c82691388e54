"""Weight containers and the device weight cache.

``WeightStore`` mirrors the subset of the reference's ``WeightFile``
(cv3cpu/io/weights.py:94-215) the models use: ``get``, ``get_f32``, ``entry``,
``__contains__``, ``keys`` and ``meta``.  Quantised entries are built with a
configurable QTensor class so one store can feed either this package or a
NumPy restatement.

Device copies of weights are cached per host object (the reference's
``WeightFile.get`` returns the same object for a name, io/weights.py:153-165)
and released by ``weakref.finalize`` when the host object goes away, the
analogue of ``WeightFile.evict`` (io/weights.py:182-205).  Only read-only
arrays (mmap views, or arrays a store has frozen) and QTensors are cached; a
writeable array is re-uploaded on every call because it may change.
"""

from __future__ import annotations

import ctypes
import threading
import weakref
from dataclasses import dataclass
from typing import Dict, Optional

import numpy as np

from . import _lib
from .device import DeviceArray, to_device


@dataclass
class DeviceQ:
    kind_code: int
    q: DeviceArray
    scales: DeviceArray
    scale_code: int
    kp: int
    block: int
    n: int
    k: int


_CACHE: Dict[int, object] = {}
_UPLOAD = threading.Lock()   # one upload per weight object when several threads miss at once


def _remember(obj, value):
    key = id(obj)
    _CACHE[key] = value
    weakref.finalize(obj, _CACHE.pop, key, None)
    return value


def device_qtensor(qt) -> DeviceQ:
    """Device copy of a QTensor's payload and scales (cached per object)."""
    hit = _CACHE.get(id(qt))
    if hit is not None:
        return hit
    with _UPLOAD:
        hit = _CACHE.get(id(qt))
        return hit if hit is not None else _upload_qtensor(qt)


def _upload_qtensor(qt) -> DeviceQ:
    kind = {"q8": _lib.KIND_Q8, "q4": _lib.KIND_Q4}[qt.kind]
    sdt = np.dtype(qt.scales.dtype)
    sc_code = _lib.F16 if sdt == np.float16 else _lib.F32
    q = qt.q if isinstance(qt.q, DeviceArray) else to_device(np.ascontiguousarray(qt.q))
    s = qt.scales if isinstance(qt.scales, DeviceArray) else to_device(np.ascontiguousarray(qt.scales))
    kp = int(qt.scales.shape[1]) * int(qt.block)
    d = DeviceQ(kind, q, s, sc_code, kp, int(qt.block), int(qt.shape[0]), int(qt.shape[1]))
    return _remember(qt, d)


def device_f32(arr) -> DeviceArray:
    """Device float32 copy of a host weight (cached if the array is read-only)."""
    if isinstance(arr, DeviceArray):
        return arr
    if isinstance(arr, np.ndarray) and not arr.flags.writeable:
        hit = _CACHE.get(id(arr))
        if hit is not None:
            return hit
        with _UPLOAD:
            hit = _CACHE.get(id(arr))
            return hit if hit is not None else _remember(arr, to_device(arr, np.float32))
    return to_device(np.asarray(arr), np.float32)


@dataclass
class DevicePlanes:
    """A linear weight laid out for ``cv3_linear_rows_planes``."""
    kind_code: int
    frag: DeviceArray
    scales_ptr: Optional[int]
    block: int
    scales: Optional[DeviceArray] = None


def device_planes(weight, dev) -> Optional[DevicePlanes]:
    """The matrix cores' layout of a weight whose device copy is ``dev`` (a DeviceArray or DeviceQ), made
    beside that copy on first use and kept and released with it.  None for what the plane linear does not
    take, for K up to 512 (two launches: 10.7 us against 8.6 of the one float32 kernel at K = 256, within 15 %
    of each other either way at 512, 13.5 against 21.5 at 1024, whatever m; q8 more), for a first use inside
    a capture (packing waits for the device), for weights that are not cached: a writeable array, or one
    that lives on the device (its owner may write to it between calls), for a weight whose planes found no
    memory (6 bytes a float32 weight, 2 a code), and for one with a row too small for them (cv3_x3_rows_fit)."""
    quantised = isinstance(dev, DeviceQ)
    if quantised:
        cached = not isinstance(weight.q, DeviceArray) and not isinstance(weight.scales, DeviceArray)
        n, k, block = dev.n, dev.k, dev.block
        cached = cached and (block in (32, 64) or block >= k) and dev.kp % 16 == 0
    else:
        cached = isinstance(weight, np.ndarray) and not weight.flags.writeable and weight.ndim == 2
        n, k = (dev.shape if cached else (0, 1))
        block = k
    if not cached or k % 64 or n % 4 or not n or k <= 512:
        return None
    key = ("planes", id(weight))
    hit = _CACHE.get(key)
    if hit is not None:
        return hit or None
    with _UPLOAD:
        hit = _CACHE.get(key)
        if hit is None:
            capturing = ctypes.c_int()
            _lib.call("stream_capturing", None, ctypes.addressof(capturing))
            if capturing.value:
                return None
            hit = _CACHE[key] = _pack_planes(dev, n, k, block) or False
            weakref.finalize(weight, _CACHE.pop, key, None)
    return hit or None


def _pack_planes(dev, n: int, k: int, block: int) -> Optional[DevicePlanes]:
    ne, ns = ctypes.c_int64(), ctypes.c_int64()
    quantised = isinstance(dev, DeviceQ)
    if quantised:
        _lib.call("code_planes_elems", n, k, block, ctypes.addressof(ne), ctypes.addressof(ns))
    else:
        _lib.call("x3_frag_elems", n, k, ctypes.addressof(ne))
    try:
        if not quantised:
            fit = ctypes.c_int()
            _lib.call("x3_rows_fit", dev.ptr, n, k, k, ctypes.addressof(fit), None)
            if not fit.value:
                return None
        frag = DeviceArray((ne.value,), np.uint16)
        scales = DeviceArray((ns.value,)) if quantised else None
    except _lib.HIPError:
        return None
    if quantised:
        _lib.call("pack_code_planes", dev.kind_code, dev.q.ptr, n, k, dev.scales.ptr, dev.scale_code, dev.kp, block, 0,
                  0, frag.ptr, scales.ptr, None)
        out = DevicePlanes(dev.kind_code, frag, scales.ptr, block, scales)
    else:
        _lib.call("split_x3_frag", dev.ptr, n, k, k, frag.ptr, None)
        out = DevicePlanes(_lib.KIND_F32, frag, None, k)
    _lib.call("stream_sync", None)   # another thread's stream may read it next
    return out


class WeightStore:
    """In-memory weight container with the reference WeightFile's read API.

    ``tensors`` maps names to float arrays or to quantised records
    ``{"kind", "q", "scales", "shape", "block", "orig_shape"}``.
    """

    def __init__(self, tensors: Dict[str, object], meta: Optional[dict] = None, qtensor_cls=None):
        from .quant import QTensor
        self._t = {}
        for name, v in tensors.items():
            if isinstance(v, np.ndarray):
                v = np.ascontiguousarray(v)
                v.flags.writeable = False
            self._t[name] = v
        self.meta = dict(meta or {})
        self._qcls = qtensor_cls or QTensor
        self._objs: Dict[str, object] = {}

    def keys(self):
        return self._t.keys()

    def __contains__(self, name):
        return name in self._t

    def raw(self, name):
        return self._t[name]

    def get(self, name):
        if name in self._objs:
            return self._objs[name]
        v = self._t[name]
        if isinstance(v, dict):
            v = self._qcls(v["kind"], v["q"], v["scales"], tuple(v["shape"]), int(v["block"]),
                           tuple(v["orig_shape"]) if v.get("orig_shape") is not None else None)
        self._objs[name] = v
        return v

    def get_f32(self, name):
        v = self.get(name)
        if hasattr(v, "dequant"):
            out = v.dequant()
            if v.orig_shape is not None:
                out = out.reshape(v.orig_shape)
            return np.asarray(out, dtype=np.float32)
        return np.asarray(v, dtype=np.float32)

    def entry(self, name):
        v = self._t[name]
        if isinstance(v, dict):
            shape = v.get("orig_shape") or v["shape"]
            return {"shape": list(shape), "kind": v["kind"]}
        return {"shape": list(np.shape(v)), "kind": str(np.asarray(v).dtype)}

    def with_qtensor(self, qtensor_cls) -> "WeightStore":
        """Same tensors, QTensors built from ``qtensor_cls``."""
        return WeightStore(self._t, self.meta, qtensor_cls)
