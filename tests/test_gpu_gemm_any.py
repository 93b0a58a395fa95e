"""The GEMM for any K and alignment and the affine quantized_dot of the same
kernel (csrc/q8_gemm_any.hip) against the oracle, at the sizes where they can
go wrong: rows shorter than a 16-byte chunk, the chunk and stage remainders
of K, tile edges, the three groupings of a tile's K stages, misaligned
operands, every output form.  Integer and fp32 results bit for bit."""
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


def dev(a, shift=0):
    """On the device, `shift` bytes past an aligned address."""
    flat = torch.zeros(a.size + 64, dtype=torch.uint8, device=DEV)
    flat[shift:shift + a.size] = torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).to(DEV)
    t = flat[shift:shift + a.size].view(a.shape)
    return t.view(torch.int8) if a.dtype == np.int8 else t


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# K: below a chunk, a chunk and one past, stage edges, several stages with a remainder
KS = [1, 3, 15, 17, 31, 127, 129, 255, 300, 1001]
# M, N: one element, tile edges, one tile column: K of 64 and more takes a 32 x
# 32 tile with K split over 8 waves, shorter rows a thread per output (the
# tiled kernel: test_tiled)
MNS = [(1, 1), (16, 65), (17, 64), (63, 129), (130, 68)]


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("M,N", MNS)
def test_any_k(ops, oracle, M, N, K):
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    print(f"any M={M} N={N} K={K}", flush=True)
    acc = oracle.quantized_dot(A, B, 1)
    np.testing.assert_array_equal(host(ops.quantized_dot(dev(A), dev(B))), acc)
    sA, sB = rng.uniform(1e-3, 0.05, M), rng.uniform(1e-4, 0.02, N)
    bias = rng.uniform(-1, 1, N).astype(np.float32)
    want = oracle.epilogue(acc, "rowcol", sA, sB, bias=bias, act="silu")
    d = [torch.from_numpy(v).to(DEV) for v in (sA, sB, bias)]
    got = host(ops.qlinear(dev(A), d[0], dev(B), d[1], bias=d[2], act="silu"))
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("M,N,K", [(1030, 1070, 1001), (2100, 1070, 901), (2100, 2300, 900), (70, 3000, 250)])
@pytest.mark.parametrize("u8,zpA,zpB", [(False, 0, 0), (True, 121, 0), (True, 3, -5)])
def test_large_tiles(ops, oracle, M, N, K, u8, zpA, zpB):
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(0, 256, (M, K)).astype(np.uint8)
    A = A if u8 else A.view(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    np.testing.assert_array_equal(host(ops.quantized_dot(dev(A), dev(B), zpA, zpB)),
                                  oracle.quantized_dot(A, B, 1, zpA, zpB))


@pytest.mark.parametrize("M,N,K", [(5, 70, 64), (100, 70, 256), (1, 33, 10)])
@pytest.mark.parametrize("shift", [1, 2, 8])
def test_misaligned_operands(ops, oracle, M, N, K, shift):
    rng = np.random.default_rng(shift + K)
    A = rng.integers(0, 256, (M, K)).astype(np.uint8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    for a, zp in ((A.view(np.int8), 0), (A, 0), (A, 77)):
        got = host(ops.quantized_dot(dev(a, shift), dev(B, 16 - shift), zp, 0))
        np.testing.assert_array_equal(got, oracle.quantized_dot(a, B, 1, zp, 0))


@pytest.mark.parametrize("M,N,K", [(20, 30, 7), (100, 129, 130), (3, 64, 33)])
def test_int8_output(ops, oracle, M, N, K):
    rng = np.random.default_rng(K)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    sA, sB = rng.uniform(1e-3, 0.05, M), rng.uniform(1e-4, 0.02, N)
    y = oracle.epilogue(oracle.quantized_dot(A, B, 1), "rowcol", sA, sB, act="relu")
    s_next = float(np.abs(y).max() / 127.0) or 1.0
    got = host(ops.qlinear_requant(dev(A), torch.from_numpy(sA).to(DEV), dev(B), torch.from_numpy(sB).to(DEV),
                                   s_next, act="relu"))
    np.testing.assert_array_equal(got, oracle.quantize(y.reshape(-1), s_next).reshape(M, N))


# Short rows over many outputs, on either side of the line between one thread
# per output and tiles: skinny and square, below and above a 16-byte chunk
SHORT_ROWS = [(300, 300, 1, "tiny"), (300, 301, 15, "tiny"), (500, 400, 17, "any"), (20000, 10, 15, "tiny"),
              (60000, 10, 17, "any"), (20000, 10, 17, "tiny"), (1, 90000, 33, "tiny"), (90000, 1, 33, "tiny"), (16, 9000, 3, "tiny"),
              (64, 8192, 15, "tiny"), (64, 8192, 17, "any"), (50000, 3, 3, "tiny"), (2048, 2047, 3, "any"),
              (5, 7, 9, "tiny")]


@pytest.mark.parametrize("M,N,K,route", SHORT_ROWS)
def test_short_rows(ops, oracle, M, N, K, route):
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(0, 256, (M, K)).astype(np.uint8)
    B = rng.integers(0, 256, (N, K)).astype(np.uint8)
    print(f"short rows M={M} N={N} K={K}", flush=True)
    i8 = A.view(np.int8), B.view(np.int8)
    acc = oracle.quantized_dot(*i8, 1)
    np.testing.assert_array_equal(host(ops.quantized_dot(dev(i8[0]), dev(i8[1]))), acc)
    assert ops.last_gemm().startswith(route)
    sA, sB = rng.uniform(1e-3, 0.05, M), rng.uniform(1e-4, 0.02, N)
    bias = rng.uniform(-1, 1, N).astype(np.float32)
    want = oracle.epilogue(acc, "rowcol", sA, sB, bias=bias, act="relu")
    d = [torch.from_numpy(v).to(DEV) for v in (sA, sB, bias)]
    got = host(ops.qlinear(dev(i8[0]), d[0], dev(i8[1]), d[1], bias=d[2], act="relu"))
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    for a, b, za, zb in ((A, i8[1], 121, 0), (i8[0], B, -3, 128), (A, B, 7, 250), (i8[0], i8[1], 0, 5)):
        np.testing.assert_array_equal(host(ops.quantized_dot(dev(a), dev(b), za, zb)),
                                      oracle.quantized_dot(a, b, 1, za, zb))


def test_more_tiles_than_a_launch_holds(ops):
    """One row by 2^30 columns and more: tiles of 64 columns would be 2^24
    workgroups of 256 threads, a thread per output still fits a launch."""
    N = (1 << 30) + 1000
    g = torch.Generator(device=DEV).manual_seed(1)
    B = torch.randint(-128, 128, (N, 1), device=DEV, generator=g, dtype=torch.int8)
    A = torch.full((1, 1), -77, dtype=torch.int8, device=DEV)
    print(f"one row by {N} columns", flush=True)
    out = ops.quantized_dot(A, B)
    assert ops.last_gemm() == "tiny"
    for i in range(0, N, 1 << 28):                      # exact int32 products, a slice at a time
        assert torch.equal(out[0, i:i + (1 << 28)], B[i:i + (1 << 28), 0].to(torch.int32) * -77)


# Affine products with aligned operands on either side of the line between one
# launch and passes around the symmetric kernels: flips, row sums of A and B,
# the correction; a few tokens (GEMV) and many (GEMM)
AFFINE_ROUTES = [(4, 256, 256, "A", "any"), (4, 256, 4096, "A", "any"), (1, 4096, 11008, "A", "gemv"),
                 (16, 1024, 11008, "A", "gemv"), (4, 4096, 4096, "csB", "any"), (1, 1024, 11008, "B", "gemv"),
                 (1, 32000, 4096, "rsA", "any"), (1, 4096, 11008, "rsA", "gemv"), (1, 1024, 11008, "csB", "gemv"), (8, 1024, 1024, "all", "any"),
                 (17, 4096, 4096, "A", "any"), (512, 4096, 4096, "A", ("qgemm", "ring")), (512, 4096, 4096, "rsA", "any"),
                 (2048, 1024, 1024, "A", "any"), (2048, 4096, 1024, "A", ("qgemm", "ring")),
                 (1024, 4000, 16384, "csB", ("qgemm", "ring")),
                 (1024, 4000, 8192, "all", "any"), (256, 8200, 4096, "B", "any")]
AFFINE_KINDS = {"A": (1, 0, 128, 0), "B": (0, 1, 0, 128), "rsA": (0, 0, 0, 3), "csB": (0, 0, 3, 0), "all": (1, 1, 121, 7)}


@pytest.mark.parametrize("M,N,K,kind,route", AFFINE_ROUTES)
def test_affine_routes(ops, oracle, M, N, K, kind, route):
    ua, ub, za, zb = AFFINE_KINDS[kind]
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(0, 256, (M, K)).astype(np.uint8)
    B = rng.integers(0, 256, (N, K)).astype(np.uint8)
    A, B = (A if ua else A.view(np.int8)), (B if ub else B.view(np.int8))
    print(f"affine {kind} M={M} N={N} K={K}", flush=True)
    got = host(ops.quantized_dot(dev(A), dev(B), za, zb))
    assert ops.last_gemm().startswith(route), ops.last_gemm()
    want = (A.astype(np.float64) - za) @ (B.astype(np.float64) - zb).T      # exact: sums below 2^53
    np.testing.assert_array_equal(got, want.astype(np.int64).astype(np.int32))


# The tiled kernel in each of its forms (256 CUs): K below a chunk, just past a
# stage, with remainders; quads and single columns stored
TILED = [(4096, 2047, 1, "any 64x64 k1"), (2048, 2048, 15, "any 64x64 k1"), (700, 801, 129, "any 64x64 k1"),
         (2100, 1071, 300, "any 64x64 k1"), (700, 804, 257, "any 64x64 k4"), (701, 801, 300, "any 64x64 k4"),
         (640, 900, 1001, "any 64x64 k4"), (1030, 1072, 257, "any 64x64 k2"), (1030, 1071, 1001, "any 64x64 k2"),
         (2100, 1072, 769, "any 128x128 k2"), (2099, 1071, 901, "any 128x128 k2"),
         (2100, 2300, 769, "any 128x128 k1"), (2101, 2303, 1001, "any 128x128 k1")]


@pytest.mark.parametrize("M,N,K,route", TILED)
def test_tiled(ops, oracle, M, N, K, route):
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(0, 256, (M, K)).astype(np.uint8)
    B = rng.integers(0, 256, (N, K)).astype(np.uint8)
    dot = lambda a, b, za=0, zb=0: ((a.astype(np.float64) - za) @ (b.astype(np.float64) - zb).T).astype(np.int64).astype(np.int32)  # noqa: E731  exact: sums below 2^53
    Ai, Bi = A.view(np.int8), B.view(np.int8)
    print(f"tiled {route} M={M} N={N} K={K}", flush=True)
    for a, b, za, zb in ((Ai, Bi, 0, 0), (A, Bi, 121, 0), (Ai, B, -3, 130), (A, B, 7, 250)):
        np.testing.assert_array_equal(host(ops.quantized_dot(dev(a), dev(b), za, zb)), dot(a, b, za, zb))
        assert ops.last_gemm() == route, ops.last_gemm()
    acc = dot(Ai, Bi)
    sA, sB = rng.uniform(1e-3, 0.05, M), rng.uniform(1e-4, 0.02, N)
    bias = rng.uniform(-1, 1, N).astype(np.float32)
    da, db, dbias = (torch.from_numpy(v).to(DEV) for v in (sA, sB, bias))
    for act in ("none", "relu", "silu"):
        want = oracle.epilogue(acc, "rowcol", sA, sB, bias=bias, act=act)
        got = host(ops.qlinear(dev(Ai), da, dev(Bi), db, bias=dbias, act=act))
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    y = oracle.epilogue(acc, "rowcol", sA, sB, act="relu")
    s_next = float(np.abs(y).max() / 127.0)
    got = host(ops.qlinear_requant(dev(Ai), da, dev(Bi), db, s_next, act="relu"))
    np.testing.assert_array_equal(got, oracle.quantize(y.reshape(-1), s_next).reshape(M, N))
