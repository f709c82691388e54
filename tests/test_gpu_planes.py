"""Linears, norms and attention on activations held as bfloat16 planes in fragment order.

The planes of a float32 value are the rounding chain test_gpu_x3.py pins bit for bit, and reproduce it to
2^-24; so every result is compared with float64 (or the oracle) at the bar of the other float32 kernels,
max |error| / max |reference| <= 1e-5.  Shapes sit at the edges of the 32-row fragments, of each kernel's
tile (32 x 32 up to 128 x 128) and of its K ranges; that every tile of the shape rule runs for every kind of
weight is asked of the rule itself (test_every_tile_of_the_rule, test_prompt_on_every_tile).
"""

import ctypes

import numpy as np
import pytest

from conftest import rel_err
import oracle.ops as ref
import oracle.quant as rquant

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def lib(gpu):
    from cv3amd import _lib
    from cv3amd.device import to_device, empty
    return _lib, to_device, empty


def elems(lib, m, k):
    ne = ctypes.c_int64()
    lib[0].call("x3_frag_elems", m, k, ctypes.byref(ne))
    return ne.value


def to_planes(lib, a):
    _lib, to_device, empty = lib
    m, k = a.shape
    out = empty((elems(lib, m, k),), np.uint16)
    d = to_device(np.ascontiguousarray(a, np.float32))
    _lib.call("split_x3_frag", d.ptr, m, k, k, out.ptr, None)
    return out


def from_planes(p, m, k):
    """The float32 rows of a plane buffer (hi + mid + lo, exact in float64)."""
    mb = -(-m // 32)
    with np.errstate(invalid="ignore"):    # rows past m are whatever the memory held
        f = (p.numpy().astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    f = f.reshape(3, mb, k // 16, 2, 32, 8)                   # plane, block, step, lane half, row, k
    return f.sum(0).transpose(0, 3, 1, 2, 4).reshape(mb * 32, k)[:m]


def ptr(d):
    return d.ptr if d is not None else None


# (rows, K, N): one row, fragment and tile edges, few rows to many
SHAPES = [(1, 128, 32), (31, 256, 68), (33, 1024, 96), (65, 320, 1024), (97, 1024, 3072), (302, 2048, 1024),
          (500, 1024, 1024), (700, 1024, 3072), (1001, 1024, 2048), (1500, 1024, 1028), (2100, 1024, 3072)]
KINDS = ["f32", "q8_rows", "q8_block"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_linear_from_planes(lib, m, k, n, kind):
    _lib, to_device, empty = lib
    if kind == "q8_block" and k < 256:
        pytest.skip("64-code blocks need K >= 256")
    rng = np.random.default_rng([m, k, n])
    x = rng.normal(size=(m, k)).astype(np.float32)
    w = (0.02 * rng.normal(size=(n, k))).astype(np.float32)
    b = rng.normal(size=n).astype(np.float32)
    xp, bd = to_planes(lib, x), to_device(b)
    if kind == "f32":
        wd, w64 = to_planes(lib, w), w.astype(np.float64)
        run = lambda *a: _lib.call("linear_x3_planes", xp.ptr, m, k, wd.ptr, n, *a)  # noqa: E731
    else:
        block = 64 if kind == "q8_block" else k
        sdt = np.float16 if kind == "q8_block" else np.float32
        q, s, kp = rquant.quantize_q8(w, block, sdt)
        w64 = (q.astype(np.float64).reshape(n, -1, block) * s.astype(np.float64)[:, :, None]).reshape(n, -1)[:, :k]
        qd, sd = to_device(np.ascontiguousarray(q)), to_device(np.ascontiguousarray(s))
        nc, ns = ctypes.c_int64(), ctypes.c_int64()
        _lib.call("code_planes_elems", n, k, block, ctypes.byref(nc), ctypes.byref(ns))
        wd, st = empty((nc.value,), np.uint16), empty((ns.value,))
        _lib.call("pack_code_planes", _lib.KIND_Q8, qd.ptr, n, k, sd.ptr, _lib.F16 if sdt == np.float16 else _lib.F32,
                  kp, block, 0, 0, wd.ptr, st.ptr, None)
        run = lambda *a: _lib.call("linear_code_planes", xp.ptr, m, k, wd.ptr, st.ptr, block, n, *a)  # noqa: E731
    want = x.astype(np.float64) @ w64.T + b
    y = empty((m, n))
    run(bd.ptr, y.ptr, n, None, None, 0, None)
    assert rel_err(y.numpy(), want) < TOL
    if n % 16:
        return
    # the gated residual, in place, and an activation straight into planes
    h, gate = rng.normal(size=(m, n)).astype(np.float32), rng.normal(size=n).astype(np.float32)
    hd, gd = to_device(h), to_device(gate)
    epi = _lib.epilogue(residual=hd.ptr, ld_res=n, gate=gd.ptr, gate_stride=0, rows_per_gate=1)
    run(bd.ptr, hd.ptr, n, None, ctypes.byref(epi), 0, None)
    assert rel_err(hd.numpy(), h + gate * want) < TOL
    yp = empty((elems(lib, m, n),), np.uint16)
    run(bd.ptr, None, 0, yp.ptr, ctypes.byref(_lib.epilogue("gelu_tanh")), 0, None)
    assert rel_err(from_planes(yp, m, n), ref.gelu_tanh(want)) < TOL


def tile_of(lib, kind, m, k, n):
    """(tile, tiles, row blocks, column blocks, through LDS) of the shape rule."""
    _lib = lib[0]
    v = [ctypes.c_int() for _ in range(5)]
    code = _lib.KIND_F32 if kind == "f32" else _lib.KIND_Q4 if kind == "q4" else _lib.KIND_Q8
    block = {"f32": 1, "q8_rows": k, "q8_block": 64, "q4": 32}[kind]
    _lib.call("plane_linear_tile", code, block, m, k, n, *(ctypes.addressof(a) for a in v))
    return tuple(a.value for a in v)


def shape_for(lib, kind, tile, k):
    """The least work whose shape takes the tile, its last row and column blocks partial: rows 32 j + 1, columns
    32 j + 16."""
    found = [(m * n, m, n) for n in (1040, 1168, 2064, 3088, 9744) for m in range(33, 4000, 32)
             if tile_of(lib, kind, m, k, n)[0] == tile]
    return min(found)[1:] if found else None


@pytest.mark.parametrize("tile", range(6))
@pytest.mark.parametrize("kind", ["f32", "q8_rows", "q8_block", "q4"])
def test_every_tile_of_the_rule(lib, kind, tile):
    """Each tile with each kind of weight, at both tails of its K loops (K / 64 even and odd; thirds for the
    float32 ring of three): float rows, a gated residual in place, GELU into planes."""
    _lib, to_device, empty = lib
    assert tile_of(lib, kind, 1, 1024, 1024)[1] == 6
    ran = 0
    for k in (896, 832, 960, 2048, 2112):
        shape = shape_for(lib, kind, tile, k)
        if shape is None:
            continue
        m, n = shape
        ran += 1
        rng = np.random.default_rng([m, k, n])
        x, w = rng.normal(size=(m, k)).astype(np.float32), (0.02 * rng.normal(size=(n, k))).astype(np.float32)
        b = rng.normal(size=n).astype(np.float32)
        xp, bd = to_planes(lib, x), to_device(b)
        if kind == "f32":
            wd, w64 = to_planes(lib, w), w.astype(np.float64)
            run = lambda *a: _lib.call("linear_x3_planes", xp.ptr, m, k, wd.ptr, n, *a)  # noqa: E731
        else:
            import cv3amd.quant as quant
            block = {"q8_rows": k, "q8_block": 64, "q4": 32}[kind]
            sdt = np.float32 if kind == "q8_rows" else np.float16
            q, s, kp = quant.quantize_q4(w) if kind == "q4" else quant.quantize_q8(w, block, sdt)
            name, code = ("q4", _lib.KIND_Q4) if kind == "q4" else ("q8", _lib.KIND_Q8)
            w64 = quant.QTensor(name, q, s, (n, k), block).dequant().astype(np.float64)
            qd, sd = to_device(np.ascontiguousarray(q)), to_device(np.ascontiguousarray(s))
            nc, ns = ctypes.c_int64(), ctypes.c_int64()
            _lib.call("code_planes_elems", n, k, block, ctypes.byref(nc), ctypes.byref(ns))
            wd, st = empty((nc.value,), np.uint16), empty((ns.value,))
            _lib.call("pack_code_planes", code, qd.ptr, n, k, sd.ptr, _lib.F32 if kind == "q8_rows" else _lib.F16, kp, block,
                      0, 0, wd.ptr, st.ptr, None)
            run = lambda *a: _lib.call("linear_code_planes", xp.ptr, m, k, wd.ptr, st.ptr, block, n, *a)  # noqa: E731
        want = x.astype(np.float64) @ w64.T + b
        print(f"[tile] {kind} {tile} m={m} k={k} n={n}", flush=True)
        y = empty((m, n))
        run(bd.ptr, y.ptr, n, None, None, 0, None)
        assert rel_err(y.numpy(), want) < TOL
        h, gate = rng.normal(size=(m, n)).astype(np.float32), rng.normal(size=n).astype(np.float32)
        hd, gd = to_device(h), to_device(gate)
        epi = _lib.epilogue(residual=hd.ptr, ld_res=n, gate=gd.ptr, gate_stride=0, rows_per_gate=1)
        run(bd.ptr, hd.ptr, n, None, ctypes.byref(epi), 0, None)
        assert rel_err(hd.numpy(), h + gate * want) < TOL
        if kind != "q4":    # no GELU with 32-code blocks
            yp = empty((elems(lib, m, n),), np.uint16)
            run(bd.ptr, None, 0, yp.ptr, ctypes.byref(_lib.epilogue("gelu_tanh")), 0, None)
            assert rel_err(from_planes(yp, m, n), ref.gelu_tanh(want)) < TOL
    assert ran, "no shape takes this tile: delete it from the rule"


@pytest.mark.parametrize("profile,kind", [("per_channel", "q8_rows"), ("balanced", "q8_block"), ("tiny", "q4")])
def test_prompt_on_every_tile(lib, profile, kind):
    """Prompt lengths at which the four projections together take every tile that any length up to 1000 takes, so
    that the prompt's own epilogues (rotary into the cache, SwiGLU into planes) run on each, against the decode's
    rows."""
    import cv3amd.quant as quant
    from cv3amd import synth
    from cv3amd.qwen2 import DeviceQwen2
    from cv3amd.weights import WeightStore
    shapes = dict(qkv=(896, 1152), o=(896, 896), gate_up=(896, 9728), down=(4864, 896))

    def tiles(t):
        return {(p, tile_of(lib, kind, t, k, n)[0]) for p, (k, n) in shapes.items()}

    reach = {t: tiles(t) for t in range(1, 1001, 16)}
    left, lengths = set().union(*reach.values()), []
    while left:
        t = max(reach, key=lambda a: (len(reach[a] & left), -a))
        lengths.append(t)
        left -= reach[t]
    print(f"[tile] prompt {profile}: lengths {lengths}", flush=True)
    tensors = synth.quantize_store(synth.qwen2_tensors(layers=1), profile, quant.quantize_q8, quant.quantize_q4)
    lms = [DeviceQwen2(WeightStore(dict(tensors), synth.qwen2_meta(layers=1), quant.QTensor), cap=1024, prompt_planes=on)
           for on in (True, False)]
    for t in lengths:
        x = np.random.default_rng(t).normal(size=(t, 896)).astype(np.float32)
        got = []
        for lm in lms:
            lm.prefill(x, 0)
            got.append((lm.logits.numpy(), lm.k_cache.numpy()[:, :, :t], lm.v_cache.numpy()[:, :, :t]))
        for a, b in zip(*got):
            assert rel_err(a, b) < TOL


@pytest.mark.parametrize("rows_per_batch,m", [(151, 302), (29, 58), (400, 400)])
def test_rotary_from_planes(lib, rows_per_batch, m):
    """The DiT's partial rotary on q and k (columns 0..63 of each 256 here), as the plane linear without it
    followed by the rotary kernel."""
    _lib, to_device, empty = lib
    from cv3amd.dit import dit_rope_tables
    rng = np.random.default_rng(m)
    k = D = 256
    xp, wd = (to_planes(lib, rng.normal(size=(r, k)).astype(np.float32)) for r in (m, 3 * D))
    c, s = (to_device(a) for a in dit_rope_tables(rows_per_batch, 64))
    y, z = empty((m, 3 * D)), empty((m, 3 * D))
    epi = _lib.epilogue(rope=(c.ptr, s.ptr, rows_per_batch, D, 64, 2 * D))
    _lib.call("linear_x3_planes", xp.ptr, m, k, wd.ptr, 3 * D, None, y.ptr, 3 * D, None, ctypes.byref(epi), 0, None)
    _lib.call("linear_x3_planes", xp.ptr, m, k, wd.ptr, 3 * D, None, z.ptr, 3 * D, None, None, 0, None)
    for col in (0, D):
        _lib.call("rope_pairs", z.ptr + 4 * col, 3 * D, m, rows_per_batch, 64, c.ptr, s.ptr, None)
    assert rel_err(y.numpy(), z.numpy()) < 1e-6   # the same products; two roundings and a fused multiply-add apart


@pytest.mark.parametrize("rows,cols", [(1, 16), (33, 896), (5, 1008), (100, 1024), (64, 528)])
def test_norms_into_planes(lib, rows, cols):
    _lib, to_device, empty = lib
    rng = np.random.default_rng(cols)
    x = (3 + 5 * rng.normal(size=(rows, cols))).astype(np.float32)
    sh, sc = (rng.normal(size=cols).astype(np.float32) for _ in range(2))
    xd, shd, scd = to_device(x), to_device(sh), to_device(sc)
    p = empty((elems(lib, rows, cols),), np.uint16)
    _lib.call("layer_norm_planes", xd.ptr, p.ptr, rows, cols, 1e-6, shd.ptr, scd.ptr, None)
    assert rel_err(from_planes(p, rows, cols), ref.layer_norm(x, None, None, 1e-6) * (1 + sc) + sh) < TOL
    _lib.call("rms_norm_planes", xd.ptr, scd.ptr, p.ptr, rows, cols, 1e-6, None)
    assert rel_err(from_planes(p, rows, cols), ref.rms_norm(x, sc, 1e-6)) < TOL


@pytest.mark.parametrize("batch,n", [(2, 37), (1, 64), (2, 151)])
def test_attention_into_planes(lib, batch, n):
    """Bit for bit the planes of what cv3_attention_x3 writes as float32."""
    _lib, to_device, empty = lib
    h, d = 3, 64
    rng = np.random.default_rng(n)
    qkv = to_device(rng.normal(size=(batch * n, 3 * h * d)).astype(np.float32))
    S3 = ctypes.c_int64 * 3
    st, os_ = S3(n * 3 * h * d, d, 3 * h * d), S3(n * h * d, d, h * d)
    args = (qkv.ptr, qkv.ptr + 4 * h * d, qkv.ptr + 8 * h * d)
    y, p = empty((batch * n, h * d)), empty((elems(lib, batch * n, h * d),), np.uint16)
    _lib.call("attention_x3", *args, y.ptr, batch, h, h, n, n, d, st, st, st, os_, 0.125, 0, 0, 0, None)
    _lib.call("attention_x3_planes", *args, p.ptr, batch, h, h, n, n, d, st, st, st, 0.125, 0, 0, 0, None)
    got, want = from_planes(p, batch * n, h * d), y.numpy().astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -24 * np.abs(want))


def test_plane_linear_refuses_what_it_cannot_read(lib):
    _lib, to_device, empty = lib
    a = empty((4096,))
    for m, k, n in ((4, 96, 32), (4, 64, 32), (4, 128, 30)):
        with pytest.raises(NotImplementedError):
            _lib.call("linear_x3_planes", a.ptr, m, k, a.ptr, n, None, a.ptr, n, None, None, 0, None)
    with pytest.raises(ValueError):
        _lib.call("linear_x3_planes", a.ptr + 4, 4, 128, a.ptr, 32, None, a.ptr, 32, None, None, 0, None)


@pytest.mark.parametrize("profile,t,pos0", [("per_channel", 1, 0), ("per_channel", 33, 7), ("balanced", 130, 0),
                                            ("tiny", 65, 1), ("tiny", 1, 40), ("per_channel", 321, 0),
                                            ("balanced", 500, 20), ("tiny", 300, 0)])
def test_prompt_on_code_planes(gpu, profile, t, pos0):
    """DeviceQwen2.prefill on code planes against the same method's float32 route (its former only one, pinned
    to the oracle by test_gpu_decode.py): logits, the appended cache rows and the position, at fragment and
    tile edges, one row, and on top of cached rows, for every storage profile."""
    import cv3amd.quant as quant
    from cv3amd import synth
    from cv3amd.qwen2 import DeviceQwen2
    from cv3amd.weights import WeightStore
    tensors = synth.quantize_store(synth.qwen2_tensors(layers=2), profile, quant.quantize_q8, quant.quantize_q4)
    rng = np.random.default_rng(t)
    x = rng.normal(size=(t, 896)).astype(np.float32)
    k, v = (rng.normal(size=(2, 2, pos0, 64)).astype(np.float32) for _ in range(2))
    got = []
    for planes in (True, False):
        d = DeviceQwen2(WeightStore(dict(tensors), synth.qwen2_meta(layers=2), quant.QTensor), cap=576)
        assert d._prompt is not None
        if not planes:
            d._prompt = None
        if pos0:
            d.fill_cache(k, v)
        d.prefill(x, pos0)
        got.append([d.logits.numpy(), d.k_cache.numpy(), d.v_cache.numpy()])
        assert int(d.ints.numpy()[0]) == pos0 + t - 1
    for a, b in zip(*got):
        assert rel_err(a, b) < TOL
    assert not got[0][1][:, :, pos0 + t:].any() and not got[0][2][:, :, pos0 + t:].any()


@pytest.mark.parametrize("why", ["asked", "memory"])
def test_prompt_without_its_planes(gpu, monkeypatch, why):
    """The LM without the prompt's second copy of the body, by choice or for want of memory: the same logits from
    the decode's rows."""
    import cv3amd.quant as quant
    from cv3amd import _lib, qwen2, synth
    from cv3amd.weights import WeightStore
    tensors = synth.quantize_store(synth.qwen2_tensors(layers=2), "per_channel", quant.quantize_q8, quant.quantize_q4)
    store = WeightStore(dict(tensors), synth.qwen2_meta(layers=2), quant.QTensor)
    x = np.random.default_rng(8).normal(size=(37, 896)).astype(np.float32)
    full = qwen2.DeviceQwen2(store, cap=64)
    body, rows = 2 * (1152 * 896 + 896 * 896 + 9728 * 896 + 896 * 4864), 2 * (1152 + 896 + 9728 + 896)
    assert full.prompt_nbytes == 2 * body + 4 * rows + 4 * 2 * 1152    # codes, a scale a row, the bias of qkv
    if why == "memory":
        real = qwen2._Stacked.planes

        def planes(self, *a):
            if self.k == 4864:
                raise _lib.HIPError("hipMalloc failed")
            return real(self, *a)
        monkeypatch.setattr(qwen2._Stacked, "planes", planes)
    bare = qwen2.DeviceQwen2(store, cap=64, prompt_planes=why != "asked")
    assert bare._prompt is None and bare.prompt_nbytes == 0
    full.prefill(x, 0)
    bare.prefill(x, 0)
    assert rel_err(bare.logits.numpy(), full.logits.numpy()) < TOL


@pytest.mark.parametrize("kind", ["f32", "q8_rows", "q8_block", "q4"])
@pytest.mark.parametrize("m,k,n", [(5, 576, 64), (33, 896, 1152), (130, 1024, 68), (331, 1024, 2048), (40, 4864, 896)])
def test_drop_in_linear_on_planes(lib, m, k, n, kind):
    """ops.linear with a cached weight against float64, and rows with an infinity, a NaN and the largest
    float against the float32 kernels (a weight that lives on the device keeps those)."""
    import cv3amd.ops as ops
    import cv3amd.quant as quant
    _lib, to_device, empty = lib
    rng = np.random.default_rng([m, k, n])
    x, w = rng.normal(size=(m, k)).astype(np.float32), (0.02 * rng.normal(size=(n, k))).astype(np.float32)
    b = rng.normal(size=n).astype(np.float32)
    w[w == 0] = 0.01
    if kind == "f32":
        w.flags.writeable = False
        wc, wd, w64 = w, to_device(w), w.astype(np.float64)
    else:
        if kind == "q4":
            q, s, _ = quant.quantize_q4(w)
            block = 32
        else:
            block = 64 if kind == "q8_block" else k
            q, s, _ = quant.quantize_q8(w, block, np.float16 if kind == "q8_block" else np.float32)
        name = "q4" if kind == "q4" else "q8"
        wc = quant.QTensor(name, q, s, (n, k), block)
        wd = quant.QTensor(name, to_device(q), to_device(s), (n, k), block)
        w64 = wc.dequant().astype(np.float64)
    assert rel_err(ops.linear(x, wc, b), x.astype(np.float64) @ w64.T + b) < TOL
    x[1, 3], x[2, 5], x[3, 7], x[4, k - 1] = np.inf, -np.inf, np.nan, np.finfo(np.float32).max
    got, want = ops.linear(to_device(x), wc, b).numpy(), ops.linear(to_device(x), wd, b).numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    for r in range(m):
        if ok[r].any():
            assert np.abs(got[r] - want[r])[ok[r]].max() <= TOL * np.abs(want[r][ok[r]]).max()


@pytest.mark.parametrize("m,k,n", [(5, 576, 64), (40, 640, 96), (331, 1024, 2048), (1500, 1024, 1152)])
def test_drop_in_linear_with_a_weight_past_bfloat16(lib, m, k, n):
    """A cached float32 weight with infinities, a NaN and values between the largest bfloat16 and the largest
    float: what the float32 kernel gives (a weight that lives on the device keeps it), whatever the row count."""
    import cv3amd.ops as ops
    _lib, to_device, empty = lib
    rng = np.random.default_rng([m, k, n])
    x, w = rng.normal(size=(m, k)).astype(np.float32), (0.02 * rng.normal(size=(n, k))).astype(np.float32)
    top = np.finfo(np.float32).max
    w[1, 3], w[2, 5], w[3, 7], w[7, 0] = np.inf, -np.inf, np.nan, np.inf
    w[4, 9], w[5, k - 1], w[6, 64], w[n - 1, 33] = top, -top, 3.395e38, 3.3961775e38
    x[:, [9, k - 1, 64, 33]] *= np.float32(0.1)     # finite products: |x| < 1
    x[0, :] = 0.0                                   # 0 * inf
    x[2, 9] = 4.0                                   # and one past the range
    w.flags.writeable = False
    b = rng.normal(size=n).astype(np.float32)
    xd, wd = to_device(x), to_device(w)
    got, want = ops.linear(xd, w, b).numpy(), ops.linear(xd, wd, b).numpy()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    ok = np.isfinite(want)
    assert ok[:, 4].any() and np.isinf(want[2, 4]) and np.isnan(want[0, 1])
    for c in range(n):
        r = ok[:, c]
        if r.any():
            assert np.abs(got[r, c].astype(np.float64) - want[r, c]).max() <= TOL * np.abs(want[r, c].astype(np.float64)).max()
    # and the planes themselves: exact
    p = to_planes(lib, w)
    back, finite = from_planes(p, n, k), np.isfinite(w)
    np.testing.assert_array_equal(back[finite], w[finite].astype(np.float64))
    np.testing.assert_array_equal(back[np.isinf(w)], w[np.isinf(w)])


@pytest.mark.parametrize("kind", ["f32", "q8_rows", "q8_block", "q4"])
@pytest.mark.parametrize("m,k,n", [(5, 640, 64), (70, 1024, 96), (1500, 640, 1152)])
def test_drop_in_linear_below_the_planes_range(lib, m, k, n, kind):
    """Rows, and rows of a float32 weight, whose planes hold fewer than 24 bits: within the float32 kernels' error
    of float64 (their sums of k terms; 9e-7 measured), row by row, beside ordinary rows and zeros."""
    import cv3amd.ops as ops
    import cv3amd.quant as quant
    _lib, to_device, empty = lib
    rng = np.random.default_rng([m, k])
    x, w = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(n, k)).astype(np.float32)
    for r, e in enumerate((0, -89, -104, -111, -116)):
        x[r] *= np.float32(2.0 ** e)
    x[m - 1, :k // 2] = 0.0
    if kind == "f32":
        small = w.copy()
        small[1] *= np.float32(2.0 ** -118)
        small[2] = 0.0
        cases = [(w, w.astype(np.float64)), (small, small.astype(np.float64))]
        for a, _ in cases:
            a.flags.writeable = False
    else:
        if kind == "q4":
            q, s, _ = quant.quantize_q4(w)
            block = 32
        else:
            block = 64 if kind == "q8_block" else k
            q, s, _ = quant.quantize_q8(w, block, np.float16 if kind == "q8_block" else np.float32)
        t = quant.QTensor("q4" if kind == "q4" else "q8", q, s, (n, k), block)
        cases = [(t, t.dequant().astype(np.float64))]
    for a, w64 in cases:
        got, want = ops.linear(to_device(x), a).numpy(), x.astype(np.float64) @ w64.T
        for r in range(m):
            for c0, c1 in ((0, 1), (1, 2), (2, 3), (3, n)):
                if np.abs(want[r, c0:c1]).max() > 1e-36:    # float32's own subnormals aside
                    assert rel_rows(got[r, c0:c1], want[r, c0:c1], x[r], w64[c0:c1]) < 2e-6, (r, c0)
        assert not got[:, 2].any() or w64[2].any()


def rel_rows(got, want, x, w64):
    """max |error| over sum |x| |w|, the scale that rounding errors of a sum follow."""
    return float((np.abs(got - want) / (np.abs(x.astype(np.float64)) @ np.abs(w64).T)).max())


def test_drop_in_linear_first_used_in_a_capture(lib):
    """A weight that a capture meets first keeps the float32 kernel there; its planes come with the next
    eager call, and both give the same layer."""
    import cv3amd.ops as ops
    from cv3amd.device import Graph
    _lib, to_device, empty = lib
    rng = np.random.default_rng(4)
    w = (0.02 * rng.normal(size=(96, 640))).astype(np.float32)
    w.flags.writeable = False
    x = to_device(rng.normal(size=(40, 640)).astype(np.float32))
    ops.linear(x.rows(0, 2), w)   # the weight is on the device, its planes are not
    [empty((40, 96)) for _ in range(3)]   # results to be had from the cache: a capture allocates nothing
    out = []
    with Graph() as g:
        out.append(ops.linear(x, w))
    g.launch()
    assert rel_err(out[0].numpy(), x.numpy().astype(np.float64) @ w.T.astype(np.float64)) < TOL
    eager = ops.linear(x, w)
    assert rel_err(eager.numpy(), x.numpy().astype(np.float64) @ w.T.astype(np.float64)) < TOL
    with Graph() as h:
        out.append(ops.linear(x, w))
    for r in range(3):
        x.copy_from(rng.normal(size=(40, 640)).astype(np.float32))
        want = ops.linear(x, w).numpy()
        h.launch()
        np.testing.assert_array_equal(out[1].numpy(), want)


def test_captured_linears_find_their_scratch(lib):
    """A capture cannot allocate: its linears share the one piece of scratch in the cache, and with none there
    they run the float32 kernels, as they do when memory is short.  Replays with eager calls between them."""
    import cv3amd.ops as ops
    from cv3amd.device import Graph, synchronize
    _lib, to_device, empty = lib
    rng = np.random.default_rng(9)
    m, k, n = 700, 1024, 2048    # 5.6 MB of results, 4.3 of scratch: size classes of their own
    w = (0.02 * rng.normal(size=(n, k))).astype(np.float32)
    w.flags.writeable = False
    xs = [to_device(rng.normal(size=(m, k)).astype(np.float32)) for _ in range(3)]
    want = [x.numpy().astype(np.float64) @ w.T.astype(np.float64) for x in xs]
    ops.linear(xs[0], w)         # the weight's planes are there
    for scratch in (1, 0):
        synchronize()
        _lib.call("empty_cache")
        eager = [ops.linear(x, w) for x in xs] if scratch else [empty((m, n)) for _ in xs]
        del eager                # three results in the cache, and one piece of scratch or none
        with Graph() as g:
            out = [ops.linear(x, w) for x in xs]
        for _ in range(3):
            for y in out:
                y.zero_()
            g.launch()
            other = ops.linear(xs[2], w).numpy()
            for y, a in zip(out, want):
                assert rel_err(y.numpy(), a) < TOL
            assert rel_err(other, want[2]) < TOL
        if scratch:
            np.testing.assert_array_equal(out[2].numpy(), other)
        del out, y, g


def _from_planes(p: np.ndarray, t: int, c: int) -> np.ndarray:
    """(3, blocks, c / 16, 64, 8) bfloat16 fragments -> (t, c) float64 (hi + mid + lo)."""
    b = -(-t // 32)
    with np.errstate(invalid="ignore"):   # rows past t are not written
        v = (p.astype(np.uint32) << 16).view(np.float32).astype(np.float64).reshape(3, b, c // 16, 2, 32, 8).sum(0)
    return v.transpose(0, 3, 1, 2, 4).reshape(b * 32, c)[:t]


@pytest.mark.parametrize("c,k,d", [(16, 4, 2), (64, 3, 1), (64, 11, 5), (80, 4, 3), (128, 7, 3), (256, 11, 1), (256, 11, 5)])
@pytest.mark.parametrize("t", [1, 31, 65, 440, 8231])
def test_vocoder_conv_on_planes(lib, t, c, k, d):
    """Snake planes, then the causal conv with each of its outputs, at the edges of the three tiles."""
    _lib, to_device, empty = lib
    if t > 1000 and c > 64:
        t = 4000 + c     # 64-row tiles, their channels in passes
    rng = np.random.default_rng([t, c, k])
    x, add = rng.normal(size=(t, c)).astype(np.float32), rng.normal(size=(t, c)).astype(np.float32)
    w = (rng.normal(size=(c, c, k)) / np.sqrt(c * k)).astype(np.float32)
    bias, a1, a2 = (rng.uniform(0.2, 1.5, size=c).astype(np.float32) for _ in range(3))

    def snake(v, a):
        return v + np.sin(a.astype(np.float64) * v) ** 2 / (a.astype(np.float64) + 1e-9)

    ne = ctypes.c_int64()
    _lib.call("x3_frag_elems", c, k * c, ctypes.addressof(ne))
    frag, wd = empty((ne.value,), np.uint16), to_device(np.ascontiguousarray(w.transpose(0, 2, 1)))
    _lib.call("split_x3_frag", wd.ptr, c, k * c, k * c, frag.ptr, None)
    planes = [empty((3 * -(-t // 32) * 32 * c,), np.uint16) for _ in range(3)]
    xd, ad, a1d, a2d, bd, total = to_device(x), to_device(add), to_device(a1), to_device(a2), to_device(bias), empty((t, c))
    P = ctypes.c_void_p * 2
    _lib.call("snake_planes", xd.ptr, ad.ptr, total.ptr, t, c, 1e-9, 2, P(a1d.ptr, a2d.ptr),
              P(planes[0].ptr, planes[1].ptr), None)
    np.testing.assert_array_equal(total.numpy(), x + add)
    s64 = (x + add).astype(np.float64)
    assert rel_err(_from_planes(planes[0].numpy(), t, c), snake(s64, a1)) < 1e-6
    assert rel_err(_from_planes(planes[1].numpy(), t, c), snake(s64, a2)) < 1e-6
    xin = np.vstack([np.zeros(((k - 1) * d, c)), _from_planes(planes[0].numpy(), t, c)])
    want = bias + sum(xin[j * d:j * d + t] @ w[:, :, j].T.astype(np.float64) for j in range(k))
    y = empty((t, c))
    _lib.call("conv_planes", planes[0].ptr, t, c, frag.ptr, c, k, d, bd.ptr, None, y.ptr, None, 1e-9, None, None)
    assert rel_err(y.numpy(), want) < 1e-6
    # in place on the residual, and the next conv's planes
    _lib.call("conv_planes", planes[0].ptr, t, c, frag.ptr, c, k, d, bd.ptr, total.ptr, total.ptr, a2d.ptr, 1e-9,
              planes[2].ptr, None)
    assert rel_err(total.numpy(), want + s64) < 1e-6
    assert rel_err(_from_planes(planes[2].numpy(), t, c), snake(want + s64, a2)) < 2e-6


def test_vocoder_mean_leaky(lib):
    _lib, to_device, empty = lib
    rng = np.random.default_rng(0)
    xs = [rng.normal(size=(7, 36)).astype(np.float32) for _ in range(4)]
    ds, y = [to_device(x) for x in xs], empty((7, 36))
    for n in (1, 2, 3, 4):
        _lib.call("mean_leaky", n, (ctypes.c_void_p * n)(*(d.ptr for d in ds[:n])), y.ptr, y.size, 0.1, None)
        v = sum(xs[1:n], xs[0]) / np.float32(n)
        np.testing.assert_allclose(y.numpy(), np.where(v >= 0, v, np.float32(0.1) * v), rtol=2e-7)
    with pytest.raises(NotImplementedError):
        _lib.call("mean_leaky", 1, (ctypes.c_void_p * 1)(ds[0].ptr + 4), y.ptr, 4, 0.1, None)
