"""GPU parity of quantized_conv (q8_quantized_conv) against the CPU oracle.

int32 accumulators and fp32 dequantized outputs are compared bit for bit.
The cases cover the device paths (the direct kernel for short contractions
of little work, else a GEMM), groups / depthwise, strides, asymmetric
padding, dilation, batch > 1 (images in one GEMM whose epilogue scatters
columns to images, with 16-byte and with per-element stores), spatial ranks
1 to 3, the byte-gather im2col (channels per group not a multiple of 16) and
the channel-last frame, each GEMM kernel and tile behind them (the route is
asserted where a case is for one), passes over parts of a batch, a split of
K, misaligned weights and workspaces; zero points and ui8 operands; then the whole pipeline QuantizationPass builds
for a conv (quantize input, quantize kernel, quantized_conv, dequantize).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    from mlfw_amd import ops as O
    from mlfw_amd import _lib
    _lib.call("q8_init", 0)
    return O


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


def same_bits(a, b):
    a = np.ascontiguousarray(a)
    b = np.ascontiguousarray(b)
    assert a.shape == b.shape, (a.shape, b.shape)
    av = a.view(np.uint8).reshape(-1, a.itemsize)
    bv = b.view(np.uint8).reshape(-1, b.itemsize)
    bad = np.nonzero(np.any(av != bv, axis=1))[0]
    if bad.size:
        i = bad[0]
        raise AssertionError(f"{bad.size} of {a.size} differ; first at flat {i}: "
                             f"{a.reshape(-1)[i]!r} vs {b.reshape(-1)[i]!r}")


CASES = [
    # x shape, w shape, strides, padding, dilation, groups      path
    ((1, 3, 8, 8), (16, 3, 3, 3), [1, 1], [[0, 0], [0, 0]], [1, 1], 1),      # direct (Kc 27)
    ((1, 3, 8, 8), (16, 3, 3, 3), [2, 2], [[1, 1], [1, 1]], [1, 1], 1),      # direct
    ((2, 32, 9, 7), (8, 8, 3, 2), [2, 1], [[1, 2], [0, 1]], [2, 1], 4),      # direct (Kc 48), groups
    ((1, 64, 10), (64, 1, 3), [1], [[1, 1]], [2], 64),                       # depthwise 1-D
    ((2, 64, 12, 12), (32, 64, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),  # GEMM (Kc 576)
    ((1, 20, 11, 13), (48, 10, 3, 3), [1, 2], [[0, 2], [1, 0]], [1, 1], 2),  # GEMM, Kc 90 -> 96, groups
    ((3, 16, 7, 9), (8, 16, 2, 3), [1, 1], [[1, 0], [0, 0]], [2, 1], 1),     # 8 outputs, Kc 96
    ((1, 8, 6, 5, 7), (24, 8, 2, 3, 2), [1, 2, 1], [[1, 0], [0, 1], [1, 1]], [1, 1, 2], 1),  # 3-D
    ((1, 256, 14, 14), (300, 256, 1, 1), [1, 1], [[0, 0], [0, 0]], [1, 1], 1),  # 1x1, tile edges
    # batched im2col + column-blocked GEMM (N > 1, Og > 16)
    ((3, 20, 12, 12), (48, 10, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 2),  # groups, Kc 90 -> 96
    ((5, 256, 14, 14), (300, 256, 1, 1), [1, 1], [[0, 0], [0, 0]], [1, 1], 1),  # P 196, edges
    ((4, 32, 6, 10), (40, 32, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),   # P 60, tile straddles
    ((2, 64, 11, 11), (32, 64, 3, 3), [1, 1], [[0, 0], [0, 0]], [1, 1], 1),  # P 81: element stores
    ((3, 512, 7, 7), (64, 512, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),  # P 49, Kc 4608
    # channel-last frame (Cg % 16 == 0) beyond the cases above
    ((2, 32, 9, 11), (48, 16, 3, 2), [2, 1], [[1, 2], [0, 1]], [1, 2], 2),   # groups, stride, dilation
    ((2, 16, 5, 6, 7), (32, 16, 2, 3, 2), [1, 2, 1], [[1, 0], [0, 1], [1, 1]], [1, 1, 2], 1),  # 3-D
    ((3, 64, 9, 9), (40, 64, 1, 1), [2, 2], [[0, 0], [0, 0]], [1, 1], 1),    # 1x1 at stride 2
    ((2, 48, 6, 6), (24, 48, 1, 1), [1, 1], [[1, 1], [0, 2]], [1, 1], 1),    # 1x1 padded: frame is B
    # few tiles, longer contractions
    ((2, 64, 9, 9), (48, 64, 5, 5), [1, 1], [[2, 2], [2, 2]], [1, 1], 1),    # Kc 1600, K % 128 = 64
    ((2, 256, 6, 6), (96, 128, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 2),  # Kc 1152, groups
]


@pytest.mark.parametrize("case", CASES)
def test_quantized_conv_int32(ops, oracle, case):
    xs, ws, st, pd, dl, g = case
    rng = np.random.default_rng(sum(xs) + 13 * g)
    x = rng.integers(-128, 128, xs).astype(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    print(f"conv case x{xs} w{ws} s{st} p{pd} d{dl} g{g}", flush=True)
    got = ops.quantized_conv(dev(x), dev(w), st, pd, dl, g)
    same_bits(host(got), oracle.quantized_conv(x, w, st, pd, dl, g))


@pytest.mark.parametrize("case", CASES)
def test_quantized_conv_prepacked_weight(ops, oracle, case):
    """A constant weight prepacked once (q8_conv_weight_taps: tap-major,
    w_taps[o][t * Cg + c] = w[o][c][t]) gives the same bits as the per-call
    permutation, on every path that reads it; weights without a tap-major
    form (Cg % 16 != 0, one kernel position) report None."""
    xs, ws, st, pd, dl, g = case
    rng = np.random.default_rng(sum(xs) + 17 * g)
    x = rng.integers(-128, 128, xs).astype(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    wt = ops.conv_weight_taps(dev(w), g)
    kn = int(np.prod(ws[2:]))
    if ws[1] % 16 != 0 or kn < 2:
        assert wt is None
        return
    O, Cg = ws[0], ws[1]
    same_bits(host(wt), w.reshape(O, Cg, kn).transpose(0, 2, 1).reshape(-1))
    for s_out in (None, 1e-4):
        got = ops.quantized_conv(dev(x), dev(w), st, pd, dl, g, s_out=s_out, w_taps=wt)
        acc = oracle.quantized_conv(x, w, st, pd, dl, g)
        want = acc if s_out is None else oracle.dequantize(acc.reshape(-1), s_out).reshape(acc.shape)
        same_bits(host(got), want)


@pytest.mark.parametrize("case", CASES[:2] + CASES[4:6] + CASES[9:])
def test_quantized_conv_dequant_epilogue(ops, oracle, case):
    xs, ws, st, pd, dl, g = case
    rng = np.random.default_rng(sum(ws))
    x = rng.integers(-128, 128, xs).astype(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    s_out = (2.5 / 127) * (0.07 / 127)
    got = ops.quantized_conv(dev(x), dev(w), st, pd, dl, g, s_out=s_out)
    acc = oracle.quantized_conv(x, w, st, pd, dl, g)
    want = oracle.dequantize(acc.reshape(-1), s_out).reshape(acc.shape)
    same_bits(host(got), want)


@pytest.mark.parametrize("case", [CASES[0], CASES[2], CASES[4], CASES[7]])
@pytest.mark.parametrize("x_u8,w_u8", [(False, False), (True, False), (True, True)])
def test_quantized_conv_zero_points_and_ui8(ops, oracle, case, x_u8, w_u8):
    """input_zero_point / kernel_zero_point and ui8 operands (the direct
    kernel), int32 bit for bit; a padded tap adds 0."""
    xs, ws, st, pd, dl, g = case
    rng = np.random.default_rng(len(xs) * 13 + g + 2 * x_u8 + w_u8)
    x = rng.integers(0, 256, xs).astype(np.uint8)
    w = rng.integers(0, 256, ws).astype(np.uint8)
    x = x if x_u8 else x.view(np.int8)
    w = w if w_u8 else w.view(np.int8)
    for zpx, zpw in ((0, 0), (128, 0), (3, -2), (128, 128)):
        print(f"conv zp {xs} {ws} x_u8={x_u8} w_u8={w_u8} zp=({zpx},{zpw})", flush=True)
        want = oracle.quantized_conv(x, w, st, pd, dl, g, zpx, zpw)
        got = ops.quantized_conv(dev(x), dev(w), st, pd, dl, g, zpx=zpx, zpw=zpw)
        same_bits(host(got), want)


def test_conv_pipeline_of_the_quantization_pass(ops, oracle):
    """quantize(input), quantize(kernel), quantized_conv, dequantize -- the op
    sequence pass.test.js:428-441 pins -- on fp32 data, both quantizes with the
    compiled op's arithmetic (quant_math.ts:16-27) and calibrated per-tensor
    symmetric scales, output scale input_scale * kernel_scale in f64."""
    r = oracle.Rng(41)
    x = r.normal((2, 64, 10, 10))
    w = r.normal((32, 64, 3, 3), 0.0, 0.05)
    sx = oracle.scale_per_tensor(x)
    sw = oracle.scale_per_tensor(w)
    xq = oracle.quantize(x.reshape(-1), sx).reshape(x.shape)
    wq = oracle.quantize(w.reshape(-1), sw).reshape(w.shape)
    s_out = sx * sw
    acc = oracle.quantized_conv(xq, wq, [1, 1], [[1, 1], [1, 1]], [1, 1], 1)
    want = oracle.dequantize(acc.reshape(-1), s_out).reshape(acc.shape)
    xq_d = ops.quantize(dev(x), sx)
    wq_d = ops.quantize(dev(w), sw)
    same_bits(host(xq_d), xq)
    same_bits(host(wq_d), wq)
    got = ops.quantized_conv(xq_d, wq_d, [1, 1], [[1, 1], [1, 1]], [1, 1], 1, s_out=s_out)
    same_bits(host(got), want)


def test_conv_workspace_is_reused(ops, oracle):
    """A caller-owned workspace serves consecutive calls on one stream."""
    rng = np.random.default_rng(3)
    x = rng.integers(-128, 128, (1, 64, 9, 9)).astype(np.int8)
    w = rng.integers(-128, 128, (40, 64, 3, 3)).astype(np.int8)
    ws = torch.empty(1 << 20, dtype=torch.int8, device=DEV)
    a = ops.quantized_conv(dev(x), dev(w), [1, 1], [[0, 0], [0, 0]], workspace=ws)
    b = ops.quantized_conv(dev(x[:, :, :5, :5].copy()), dev(w), [1, 1], [[0, 0], [0, 0]], workspace=ws)
    same_bits(host(a), oracle.quantized_conv(x, w, [1, 1], [[0, 0], [0, 0]]))
    same_bits(host(b), oracle.quantized_conv(x[:, :, :5, :5].copy(), w, [1, 1], [[0, 0], [0, 0]]))


AFFINE = [
    # x shape, w shape, strides, padding, dilation, groups
    ((2, 64, 12, 11), (32, 64, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),   # frame path
    ((3, 96, 9, 9), (80, 32, 3, 3), [2, 1], [[1, 2], [0, 1]], [1, 2], 3),     # groups of one launch, 80 / 3 rows
    ((5, 48, 7, 7), (9, 16, 5, 5), [1, 1], [[2, 2], [2, 2]], [1, 1], 3),      # 3 output channels per group
    ((4, 32, 8, 8), (40, 32, 1, 1), [1, 1], [[0, 0], [0, 0]], [1, 1], 1),     # 1 x 1
    ((2, 10, 11, 13), (48, 10, 3, 3), [1, 2], [[0, 2], [1, 0]], [1, 1], 1),   # im2col, Kc 90
    ((2, 20, 11, 13), (6, 10, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 2),    # im2col, groups
    ((1, 16, 6, 5, 7), (24, 16, 2, 3, 2), [1, 2, 1], [[1, 0], [0, 1], [1, 1]], [1, 1, 2], 1),  # 3-D
    ((8, 3, 56, 56), (32, 3, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),     # Kc 27, large: im2col
    ((2, 512, 7, 7), (80, 512, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),   # 36 stages, few tiles
    ((64, 64, 14, 14), (192, 64, 3, 3), [1, 1], [[1, 1], [1, 1]], [1, 1], 1),  # more tiles than 2 per CU
]


@pytest.mark.parametrize("case", AFFINE)
@pytest.mark.parametrize("x_u8,w_u8,zpx,zpw", [(True, False, 117, 0), (False, False, -128, 0), (True, True, 3, 130),
                                               (False, False, 0, 0), (True, False, 300, 0)])
def test_quantized_conv_affine_paths(ops, oracle, case, x_u8, w_u8, zpx, zpw):
    """The GEMM paths with zero points and ui8 operands (and, symmetric, the
    same shapes), bit for bit; zpx = 300 has no ui8 code and runs direct."""
    xs, ws, st, pd, dl, g = case
    if np.prod(xs) * np.prod(ws) > 1 << 33 and zpx not in (117, 0):
        pytest.skip("large shape: one affine and one symmetric run")
    if ws[0] % g:
        ws = (ws[0] // g * g, *ws[1:])
    rng = np.random.default_rng(sum(xs) + zpx + 256 + 2 * x_u8)
    x = rng.integers(0, 256, xs).astype(np.uint8)
    w = rng.integers(0, 256, ws).astype(np.uint8)
    x = x if x_u8 else x.view(np.int8)
    w = w if w_u8 else w.view(np.int8)
    print(f"conv affine {xs} {ws} g{g} u8=({x_u8},{w_u8}) zp=({zpx},{zpw})", flush=True)
    want = oracle.quantized_conv(x, w, st, pd, dl, g, zpx, zpw)
    same_bits(host(ops.quantized_conv(dev(x), dev(w), st, pd, dl, g, zpx=zpx, zpw=zpw)), want)
    s_out = 1.7e-4
    got = host(ops.quantized_conv(dev(x), dev(w), st, pd, dl, g, zpx=zpx, zpw=zpw, s_out=s_out))
    same_bits(got, (want.astype(np.float64) * s_out).astype(np.float32))


def test_conv_affine_without_workspace(ops, oracle):
    """An affine conv still runs with no workspace (the direct kernel), as a
    caller that never brought one expects, with the same bits."""
    import ctypes as C
    from mlfw_amd import _lib as L
    rng = np.random.default_rng(5)
    x = rng.integers(0, 256, (2, 64, 9, 9)).astype(np.uint8)
    w = rng.integers(-128, 128, (24, 64, 3, 3)).astype(np.int8)
    out = torch.empty((2, 24, 9, 9), dtype=torch.int32, device=DEV)
    arr = lambda v: (C.c_int64 * len(v))(*v)  # noqa: E731
    dx, dw = dev(x), dev(w)
    L.call("q8_quantized_conv_ex", C.c_void_p(dx.data_ptr()), L.Q8_U8, C.c_void_p(dw.data_ptr()), L.Q8_I8, 2,
           arr(x.shape), arr(w.shape), arr([1, 1]), arr([1, 1]), arr([1, 1]), arr([1, 1]), 1, 99, 0, L.Q8_I32, 0.0,
           None, 0, C.c_void_p(out.data_ptr()), None)
    same_bits(host(out), oracle.quantized_conv(x, w, [1, 1], [[1, 1], [1, 1]], [1, 1], 1, 99, 0))


def conv_call(x, w, st, pd, g=1, s_out=None, zpx=0, ws_bytes=None, ws_shift=0, w_shift=0, taps=None):
    """quantized_conv through the C ABI with a workspace of ws_bytes (the size
    asked for when None) that starts ws_shift bytes past an aligned address,
    the weight w_shift bytes past one; the bytes around the workspace are
    checked afterwards."""
    import ctypes as C
    from mlfw_amd import _lib as L
    d = x.ndim - 2
    arr = lambda v: (C.c_int64 * len(v))(*v)  # noqa: E731
    lo, hi = [p[0] for p in pd], [p[1] for p in pd]
    geom = (d, arr(x.shape), arr(w.shape), arr(st), arr(lo), arr(hi), arr([1] * d), g)
    if ws_bytes is None:
        need = C.c_size_t(0)
        L.call("q8_quantized_conv_workspace", *geom, C.byref(need))
        ws_bytes = need.value
    GUARD = 4096
    buf = torch.full((GUARD + ws_shift + ws_bytes + GUARD,), 0x5a, dtype=torch.uint8, device=DEV)
    wbuf = torch.zeros(w.size + 64, dtype=torch.uint8, device=DEV)
    wbuf[w_shift:w_shift + w.size] = dev(w.view(np.uint8).reshape(-1))
    shape = (x.shape[0], w.shape[0], *[(x.shape[2 + i] + lo[i] + hi[i] - w.shape[2 + i]) // st[i] + 1 for i in range(d)])
    out = torch.empty(shape, dtype=torch.int32 if s_out is None else torch.float32, device=DEV)
    dx = dev(x)
    p = lambda t, off=0: C.c_void_p(t.data_ptr() + off)  # noqa: E731
    kind, s = (L.Q8_I32, 0.0) if s_out is None else (L.Q8_F32, s_out)
    code = {np.dtype(np.int8): L.Q8_I8, np.dtype(np.uint8): L.Q8_U8}
    ws = p(buf, GUARD + ws_shift) if ws_bytes else None
    print(f"conv C ABI x{x.shape} w{w.shape} g{g} ws={ws_bytes}+{ws_shift} w+{w_shift}", flush=True)
    if taps is not None:
        L.call("q8_quantized_conv_prepacked", p(dx), p(wbuf, w_shift), p(taps), *geom, zpx, 0, kind, s, ws, ws_bytes,
               p(out), None)
    else:
        L.call("q8_quantized_conv_ex", p(dx), code[x.dtype], p(wbuf, w_shift), code[w.dtype], *geom, zpx, 0, kind, s, ws,
               ws_bytes, p(out), None)
    got = host(out)
    b = host(buf)
    assert (b[:GUARD + ws_shift] == 0x5a).all() and (b[GUARD + ws_shift + ws_bytes:] == 0x5a).all(), "workspace overrun"
    return got


@pytest.mark.parametrize("ws_shift,w_shift", [(0, 1), (0, 8), (1, 0), (15, 3)])
@pytest.mark.parametrize("xs,ws,pd", [((1, 16, 112, 112), (64, 16, 1, 3), [[0, 0], [1, 1]]),   # short, frame
                                      ((1, 16, 6000), (64, 16, 3), [[1, 1]]),
                                      ((2, 16, 6000), (128, 16, 2), [[0, 0]]),
                                      ((2, 64, 9, 9), (48, 64, 3, 3), [[1, 1], [1, 1]]),       # frame
                                      ((3, 10, 9, 11), (24, 10, 3, 3), [[1, 1], [1, 0]])])     # matrix
@pytest.mark.parametrize("u8", [False, True])
def test_conv_misaligned_weight_and_workspace(ops, oracle, xs, ws, pd, u8, ws_shift, w_shift):
    """A weight (a view into a larger blob) and a workspace at any byte
    address: the same bits, and nothing written outside a workspace of exactly
    the size asked for."""
    rng = np.random.default_rng(sum(xs) + ws_shift)
    x = rng.integers(0, 256, xs).astype(np.uint8)
    x = x if u8 else x.view(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    st, zp = [1] * (len(xs) - 2), 77 if u8 else 0
    got = conv_call(x, w, st, pd, zpx=zp, ws_shift=ws_shift, w_shift=w_shift)
    same_bits(got, oracle.quantized_conv(x, w, st, pd, [1] * len(st), 1, zp, 0))


@pytest.mark.parametrize("xs,ws,pd,g,u8", [((5, 64, 28, 28), (64, 64, 3, 3), [[1, 1], [1, 1]], 1, False),
                                           ((4, 96, 28, 28), (96, 32, 3, 3), [[1, 1], [1, 1]], 3, False),
                                           ((4, 96, 28, 28), (96, 32, 3, 3), [[1, 1], [1, 1]], 3, True),
                                           ((6, 20, 40, 40), (48, 10, 3, 3), [[1, 1], [1, 0]], 2, False),
                                           ((6, 20, 40, 40), (48, 10, 3, 3), [[1, 1], [1, 0]], 2, True)])
def test_conv_in_several_passes(ops, oracle, xs, ws, pd, g, u8):
    """A workspace for one image of one group, for an odd share of the batch
    and for all of it but a byte: the passes over images and groups give the
    same bits and stay inside it."""
    import ctypes as C
    from mlfw_amd import _lib as L
    rng = np.random.default_rng(sum(xs))
    x = rng.integers(0, 256, xs).astype(np.uint8)
    x = x if u8 else x.view(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    zp = 77 if u8 else 0
    want = oracle.quantized_conv(x, w, [1, 1], pd, [1, 1], g, zp, 0)
    arr = lambda v: (C.c_int64 * len(v))(*v)  # noqa: E731
    need = C.c_size_t(0)
    lo, hi = [p[0] for p in pd], [p[1] for p in pd]
    L.call("q8_quantized_conv_workspace", 2, arr(xs), arr(ws), arr([1, 1]), arr(lo), arr(hi), arr([1, 1]), g, C.byref(need))
    P = [xs[2 + i] + lo[i] + hi[i] - ws[2 + i] + 1 for i in range(2)]
    kc = ws[1] * ws[2] * ws[3]
    one = ((xs[2] + lo[0] + hi[0]) * (xs[3] + lo[1] + hi[1]) * ws[1] + (ws[0] * kc + 255) // 256 * 256
           if ws[1] % 16 == 0 else P[0] * P[1] * ((kc + 15) // 16 * 16))
    for size in (one, (one + need.value) // 2, need.value - 1):
        same_bits(conv_call(x, w, [1, 1], pd, g, zpx=zp, ws_bytes=size), want)


# Symmetric convs in few groups whose product fills the chip with 128 x 128 tiles
# run a group at a time through the direct-to-LDS GEMM; smaller ones, more
# groups, ragged outputs, 1 x 1 kernels and affine ones all groups in one launch
GROUPED = [((44, 128, 28, 28), (256, 64, 3, 3), 2, False, "conv 128x128"),
           ((22, 128, 27, 29), (480, 64, 3, 3), 2, False, "conv 128x128"),
           ((43, 128, 28, 28), (300, 64, 3, 3), 2, False, "any conv"),
           ((20, 128, 28, 28), (256, 64, 3, 3), 2, False, "any conv"),
           ((43, 192, 28, 28), (384, 64, 3, 3), 3, False, "any conv"),
           ((44, 128, 28, 28), (256, 64, 3, 3), 2, True, "any conv"),
           ((86, 128, 28, 28), (256, 64, 1, 1), 2, False, "any conv")]


@pytest.mark.parametrize("xs,ws,g,u8,route", GROUPED)
def test_conv_large_groups(ops, oracle, xs, ws, g, u8, route):
    rng = np.random.default_rng(sum(xs) + sum(ws))
    x = rng.integers(0, 256, xs).astype(np.uint8)
    x = x if u8 else x.view(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    pad = ws[2] // 2
    pd, zp = [[pad, pad]] * 2, 77 if u8 else 0
    want = oracle.quantized_conv(x, w, [1, 1], pd, [1, 1], g, zp, 0)
    wt = None if u8 or pad == 0 else ops.conv_weight_taps(dev(w), g)
    for taps in {None, wt}:
        got = ops.quantized_conv(dev(x), dev(w), [1, 1], pd, groups=g, zpx=zp, w_taps=taps)
        assert ops.last_gemm().startswith(route), ops.last_gemm()
        same_bits(host(got), want)
    got = ops.quantized_conv(dev(x), dev(w), [1, 1], pd, groups=g, zpx=zp, s_out=1.7e-4)
    same_bits(host(got), (want.astype(np.float64) * 1.7e-4).astype(np.float32))


# 1 x 1 convs on either side of one 32 x 32 tile per CU (256), whole and ragged
POINTWISE = [((8, 64, 14, 14), 64, "any conv 32x32"), ((16, 256, 28, 28), 64, "qgemm 64x64"),
             ((11, 80, 27, 29), 33, "qgemm 64x64"), ((1, 2048, 28, 28), 512, "ring"), ((5, 48, 30, 30), 96, "qgemm"),
             ((2, 96, 45, 46), 65, "qgemm")]


@pytest.mark.parametrize("xs,o,route", POINTWISE)
@pytest.mark.parametrize("w_shift", [0, 1])
def test_conv_pointwise(ops, oracle, xs, o, route, w_shift):
    rng = np.random.default_rng(sum(xs) + o)
    x = rng.integers(-128, 128, xs).astype(np.int8)
    w = rng.integers(-128, 128, (o, xs[1], 1, 1)).astype(np.int8)
    want = oracle.quantized_conv(x, w, [1, 1], [[0, 0], [0, 0]], [1, 1], 1)
    got = conv_call(x, w, [1, 1], [[0, 0], [0, 0]], w_shift=w_shift)
    assert ops.last_gemm().startswith("any conv" if w_shift else route), ops.last_gemm()
    same_bits(got, want)
    got = conv_call(x, w, [1, 1], [[0, 0], [0, 0]], w_shift=w_shift, s_out=1.7e-4)
    same_bits(got, (want.astype(np.float64) * 1.7e-4).astype(np.float32))


# Few tiles over a long contraction: K split over workgroups, its partial sums
# behind the rest of the workspace; without room for them, unsplit
SPLIT_K = [((1, 256, 13, 13), (3, 256, 7, 7), 1), ((2, 1024, 7, 7), (66, 1024, 3, 3), 1),
           ((1, 1280, 7, 9), (40, 640, 3, 3), 2), ((1, 2048, 7, 7), (16, 2048, 3, 3), 1),
           ((1, 108, 9, 9), (17, 108, 7, 7), 1), ((3, 300, 6, 5), (34, 150, 5, 7), 2)]


@pytest.mark.parametrize("xs,ws,g", SPLIT_K)
@pytest.mark.parametrize("u8", [False, True])
def test_conv_split_k(ops, oracle, xs, ws, g, u8):
    import ctypes as C
    from mlfw_amd import _lib as L
    rng = np.random.default_rng(sum(xs) + u8)
    x = rng.integers(0, 256, xs).astype(np.uint8)
    x = x if u8 else x.view(np.int8)
    w = rng.integers(-128, 128, ws).astype(np.int8)
    pd, zp = [[ws[2] // 2] * 2, [ws[3] // 2] * 2], 77 if u8 else 0
    want = oracle.quantized_conv(x, w, [1, 1], pd, [1, 1], g, zp, 0)
    same_bits(conv_call(x, w, [1, 1], pd, g, zpx=zp), want)
    assert ops.last_gemm().startswith("any conv split"), ops.last_gemm()
    same_bits(conv_call(x, w, [1, 1], pd, g, zpx=zp, s_out=1.7e-4), (want.astype(np.float64) * 1.7e-4).astype(np.float32))
    arr = lambda v: (C.c_int64 * len(v))(*v)  # noqa: E731
    need = C.c_size_t(0)
    p = arr([q[0] for q in pd])
    L.call("q8_quantized_conv_workspace", 2, arr(xs), arr(ws), arr([1, 1]), p, p, arr([1, 1]), g, C.byref(need))
    same_bits(conv_call(x, w, [1, 1], pd, g, zpx=zp, ws_bytes=need.value - 4096), want)
    assert ops.last_gemm().startswith("any"), ops.last_gemm()


# Each GEMM kernel and tile behind a conv (256 CUs): x, outputs, kernel edge,
# stride, pad, ui8 input, route
TILES = [((21, 64, 28, 28), 64, 3, 1, 1, False, "conv 64x64"), ((21, 256, 28, 28), 64, 3, 1, 1, False, "conv 64x64"),
         ((43, 256, 28, 28), 130, 3, 1, 1, False, "conv 128x128"), ((43, 64, 28, 28), 130, 3, 1, 1, False, "conv 128x128"),
         ((11, 3, 112, 112), 64, 7, 2, 3, False, "qgemm 64x64"), ((11, 3, 111, 113), 33, 7, 2, 3, False, "qgemm 64x64"),
         ((11, 3, 112, 112), 64, 7, 2, 3, True, "any 64x64"), ((8, 64, 28, 28), 64, 3, 1, 1, True, "any conv 64x64 k4"),
         ((9, 96, 27, 28), 61, 3, 1, 1, False, "any conv 64x64 k4"), ((21, 64, 28, 28), 64, 3, 1, 1, True, "any conv 64x64 k2"),
         ((22, 96, 27, 28), 61, 3, 1, 1, False, "any conv 64x64 k2"), ((21, 16, 28, 28), 64, 3, 1, 1, False, "any conv 64x64 k1"),
         ((21, 16, 28, 28), 63, 3, 1, 1, True, "any conv 64x64 k1"),
         ((32, 128, 28, 28), 128, 3, 1, 1, True, "any conv 128x128 k2"), ((33, 96, 27, 28), 127, 3, 1, 1, False, "any conv 128x128 k2"),
         ((42, 96, 28, 28), 128, 3, 1, 1, True, "any conv 128x128 k1"), ((44, 96, 27, 29), 125, 3, 1, 1, False, "any conv 128x128 k1")]


@pytest.mark.parametrize("xs,o,k,st,pad,u8,route", TILES)
def test_conv_tiles(ops, xs, o, k, st, pad, u8, route):
    """int32 and fp32 outputs, weights as given and prepacked, against a
    float64 convolution on the CPU (exact: sums below 2^53)."""
    rng = np.random.default_rng(sum(xs) + o)
    x = rng.integers(0, 256, xs).astype(np.uint8)
    x = x if u8 else x.view(np.int8)
    w = rng.integers(-128, 128, (o, xs[1], k, k)).astype(np.int8)
    zp = 117 if u8 else 0
    print(f"conv tiles {route} x{xs} o{o} k{k}", flush=True)
    want = torch.nn.functional.conv2d(torch.from_numpy(x.astype(np.float64) - zp), torch.from_numpy(w.astype(np.float64)),
                                      stride=st, padding=pad).numpy().astype(np.int32)
    dx, dw, pd = dev(x), dev(w), [[pad, pad]] * 2
    wt = None if u8 else ops.conv_weight_taps(dw)
    for taps in {None, wt}:
        got = ops.quantized_conv(dx, dw, [st, st], pd, zpx=zp, w_taps=taps)
        assert ops.last_gemm().startswith(route), ops.last_gemm()
        same_bits(host(got), want)
        got = ops.quantized_conv(dx, dw, [st, st], pd, zpx=zp, w_taps=taps, s_out=1.7e-4)
        same_bits(host(got), (want.astype(np.float64) * 1.7e-4).astype(np.float32))
