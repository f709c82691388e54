"""Re-entrancy of the drop-in ops and stream safety of the caching allocator.

* The reference calls the quantised GEMV from a pool of min(4, cpu) threads
  (cv3cpu/quant.py:139-153,192-197).  Here four host threads call
  ``cv3amd.ops.linear`` at once, each on its own stream, on weights they share
  (one device upload per weight object); every result meets the oracle.
* A block freed while its thread's stream is being captured belongs to the
  graph: it is not handed out again until the graph is destroyed.
"""

import threading
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


def test_linear_from_four_threads(gpu):
    import oracle.ops as rops
    import oracle.quant as rquant
    import cv3amd.ops as ops
    import cv3amd.quant as quant
    rng = np.random.default_rng(11)
    w8 = rng.standard_normal((4864, 896), dtype=np.float32) * np.float32(0.02)
    q, s, _ = rquant.quantize_q8(w8, 896, np.float32)
    qb, sb, _ = rquant.quantize_q8(w8, 64, np.float16)
    dev_w = {"pc": quant.QTensor("q8", q, s, (4864, 896), 896), "blk": quant.QTensor("q8", qb, sb, (4864, 896), 64)}
    ref_w = {"pc": rquant.QTensor("q8", q, s, (4864, 896), 896), "blk": rquant.QTensor("q8", qb, sb, (4864, 896), 64)}
    wf = rng.standard_normal((1024, 1024), dtype=np.float32) * np.float32(0.02)
    wf.flags.writeable = False
    bias = rng.standard_normal(1024, dtype=np.float32) * np.float32(0.02)
    # (weight key, rows): the GEMV regime (m <= 4) and the MFMA GEMM
    jobs = [(key, m, seed) for seed in range(6) for key, m in (("pc", 1), ("blk", 3), ("f32", 200), ("pc", 64))]
    barrier = threading.Barrier(4)
    threads = set()

    def run(job):
        key, m, seed = job
        if seed == 0:
            barrier.wait(timeout=60)    # the first four jobs start together, one per thread
        threads.add(threading.get_ident())
        x = np.random.default_rng(100 + seed).standard_normal((m, 896 if key != "f32" else 1024), dtype=np.float32)
        if key == "f32":
            got, want = ops.linear(x, wf, bias), rops.linear(x, wf, bias)
        else:
            got, want = ops.linear(x, dev_w[key]), rops.linear(x, ref_w[key])
        return key, m, seed, rel_err(got, want)

    print(f"[threads] {len(jobs)} linear calls from 4 host threads", flush=True)
    with ThreadPoolExecutor(4) as ex:
        results = list(ex.map(run, jobs))
    assert len(threads) == 4      # four threads, hence four per-thread streams
    for key, m, seed, e in results:
        assert e < 1e-5, f"{key} m={m} seed={seed}: rel err {e:.2e}"
    print(f"[threads] worst rel err {max(r[3] for r in results):.2e}", flush=True)


def test_block_freed_during_capture_belongs_to_the_graph(gpu):
    from cv3amd import _lib
    from cv3amd.device import DeviceArray, Graph, synchronize
    nbytes = 3 << 20
    a = DeviceArray((nbytes // 4,)).zero_()
    pa = a.ptr
    g = Graph()
    with g:
        _lib.call("fill_zero", a.ptr, a.nbytes, None)   # the graph writes a ...
        del a                                           # ... and a is dropped while capturing
    synchronize()
    b = DeviceArray((nbytes // 4,))
    assert b.ptr != pa, "a block the graph refers to was handed out again"
    g.launch()
    g.launch()
    synchronize()
    in_use0, cached0 = _lib.mem_stats()
    del g                                               # the graph goes: its block returns to the cache
    synchronize()
    in_use1, cached1 = _lib.mem_stats()
    assert in_use0 - in_use1 == nbytes and cached1 - cached0 == nbytes
    del b


def test_record_stream_orders_reuse(gpu):
    """A block written on a side stream and freed from the thread's stream is reused only
    behind the side stream's work: the value written there is never overwritten early."""
    from cv3amd import _lib
    from cv3amd.device import DeviceArray, Stream, synchronize
    n = 1 << 22
    src = DeviceArray((n,)).copy_from(np.full(n, 7.0, np.float32))
    side = Stream()
    for _ in range(5):
        tmp = DeviceArray((n,))
        tmp.record_stream(side)
        dst = DeviceArray((n,))
        dst.record_stream(side)
        _lib.call("copy_d2d", tmp.ptr, src.ptr, tmp.nbytes, side.handle)
        _lib.call("copy_d2d", dst.ptr, tmp.ptr, tmp.nbytes, side.handle)
        del tmp                        # its block may be reused below, behind the side stream
        over = DeviceArray((n,)).zero_()
        _lib.call("stream_sync", side.handle)
        synchronize()
        assert float(dst.numpy().min()) == 7.0
        del over, dst


def test_block_freed_at_home_waits_for_its_stream(gpu):
    """A block freed on the one stream that used it goes back to that stream at once, and to another
    thread's stream only when the first has run dry."""
    import cv3amd.ops as ops
    from cv3amd import _lib
    from cv3amd.device import DeviceArray, synchronize, to_device
    nbytes = 37 << 20   # a size class of its own, with nothing cached in it
    synchronize()
    _lib.call("empty_cache")
    rng = np.random.default_rng(2)
    x = to_device(rng.normal(size=(3000, 1024)).astype(np.float32))
    w = rng.normal(size=(4096, 1024)).astype(np.float32)
    w.flags.writeable = False
    ops.linear(x, w)
    synchronize()

    def fresh():
        a = DeviceArray((nbytes,), np.uint8)
        return a, a.ptr

    with ThreadPoolExecutor(1) as other:
        other.submit(lambda: DeviceArray((16,))).result()   # the other thread's stream exists
        a, ptr = fresh()
        for _ in range(200):     # some 20 ms of work
            y = ops.linear(x, w)
        a.zero_()
        del a
        a, again = fresh()
        assert again == ptr
        del a
        b, elsewhere = other.submit(fresh).result()
        assert elsewhere != ptr
        synchronize()
        c, late = other.submit(fresh).result()
        assert late == ptr
        del b, c, y


def _rows_planes(x, w, y, stream):
    """ops.linear's plane call on an explicit stream, without a bias: x [m, k], w the cached float32 weight."""
    from cv3amd import _lib, weights
    n, k = w.shape
    p = weights.device_planes(w, weights.device_f32(w))
    _lib.call("linear_rows_planes", p.kind_code, x.ptr, x.shape[0], k, k, p.frag.ptr, p.scales_ptr, p.block, n, None,
              y.ptr, n, None, stream.handle if stream is not None else None)


def _plane_linear_case(seed, m=2500, k=1024, n=2048):
    from cv3amd.device import to_device
    import cv3amd.ops as ops
    rng = np.random.default_rng(seed)
    w = rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)
    w.flags.writeable = False
    xs = [to_device(rng.standard_normal((m, k), dtype=np.float32)) for _ in range(2)]
    return w, xs, [ops.linear(x, w).numpy() for x in xs]


def test_call_scratch_is_ordered_on_its_own_stream(gpu):
    """A linear on a stream that is not the thread's splits its rows into scratch that the thread's stream gave
    back a moment ago, or the other way round: each waits for the other's use of it."""
    from cv3amd.device import DeviceArray, Stream, synchronize
    w, (x0, x1), (want0, want1) = _plane_linear_case(5)
    side = Stream()
    y = [DeviceArray(want0.shape) for _ in range(4)]
    synchronize()
    for _ in range(8):
        _rows_planes(x0, w, y[0], None)
        _rows_planes(x1, w, y[1], side)
        _rows_planes(x0, w, y[2], None)
        _rows_planes(x1, w, y[3], side)
        _sync(side)
        synchronize()
        for got, want in zip(y, (want0, want1, want0, want1)):
            np.testing.assert_array_equal(got.numpy(), want)
            got.zero_()
        synchronize()


def _sync(stream):
    from cv3amd import _lib
    _lib.call("stream_sync", stream.handle)


def test_call_scratch_on_a_capturing_stream_belongs_to_the_graph(gpu):
    """The same call captured on such a stream, while the thread's own is not: eager calls of the same shape
    between the replays never share its scratch."""
    import ctypes
    from cv3amd import _lib
    from cv3amd.device import DeviceArray, Stream, synchronize
    w, (x0, x1), (want0, want1) = _plane_linear_case(6)
    side = Stream()
    y, z = DeviceArray(want0.shape), DeviceArray(want0.shape)
    synchronize()
    _rows_planes(x0, w, y, side)    # the stream has scratch of its own in the cache
    _sync(side)
    _lib.call("graph_begin", side.handle)
    _rows_planes(x0, w, y, side)
    x = ctypes.c_void_p()
    _lib.call("graph_end", side.handle, ctypes.addressof(x))
    for _ in range(4):
        y.zero_()
        synchronize()
        _lib.call("graph_launch", x.value, side.handle)
        for _ in range(3):
            _rows_planes(x1, w, z, None)
        _sync(side)
        synchronize()
        np.testing.assert_array_equal(y.numpy(), want0)
        np.testing.assert_array_equal(z.numpy(), want1)
    synchronize()
    in_use, _ = _lib.mem_stats()
    _lib.call("graph_destroy", x.value)
    assert _lib.mem_stats()[0] < in_use     # the scratch was the graph's until now


def test_block_dropped_during_another_streams_capture_belongs_to_its_graph(gpu):
    """A block recorded on a stream under capture and dropped meanwhile, from a thread whose own stream is not
    capturing, stays with that graph."""
    import ctypes
    from cv3amd import _lib
    from cv3amd.device import DeviceArray, Stream, synchronize
    nbytes = 5 << 20
    side = Stream()
    a = DeviceArray((nbytes // 4,)).record_stream(side)
    pa = a.ptr
    synchronize()
    _lib.call("graph_begin", side.handle)
    _lib.call("fill_zero", a.ptr, a.nbytes, side.handle)
    del a
    x = ctypes.c_void_p()
    _lib.call("graph_end", side.handle, ctypes.addressof(x))
    b = DeviceArray((nbytes // 4,)).copy_from(np.ones(nbytes // 4, np.float32))
    assert b.ptr != pa, "a block the graph refers to was handed out again"
    for _ in range(2):
        _lib.call("graph_launch", x.value, side.handle)
        _sync(side)
    assert float(b.numpy().min()) == 1.0
    in_use0, _ = _lib.mem_stats()
    _lib.call("graph_destroy", x.value)
    assert in_use0 - _lib.mem_stats()[0] == nbytes
    del b


def test_refused_allocation_leaves_the_capture_and_the_thread_whole(gpu):
    """A capture takes memory from the cache only.  An allocation that finds none raises; the thread's stream goes on
    afterwards, and captures again."""
    from cv3amd import _lib
    from cv3amd.device import DeviceArray, Graph, synchronize, to_device
    a = to_device(np.arange(1024, dtype=np.float32))
    synchronize()
    _lib.call("empty_cache")
    with pytest.raises(_lib.HIPError, match="capture"):
        with Graph():
            a.zero_()
            DeviceArray((91 << 20,), np.uint8)
    np.testing.assert_array_equal(a.numpy(), np.arange(1024))    # captured, not run
    with Graph() as g:
        a.zero_()
    g.launch()
    assert not a.numpy().any()
