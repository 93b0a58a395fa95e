"""The deep-ring GEMM (csrc/q8_gemm_ring.hip) against the oracle: each of its
tiles, reached by the sizes the dispatch gives it, with partial tiles on both
edges, K remainders of a stage (16 bytes to a whole one), fewer stages than
the ring is deep and stage counts its K groups do not divide, and every output
form.  Integer and fp32 results bit for bit."""
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


# 256 CUs: the smallest tile with at most 256 tiles is taken
SHAPES = [(17, 33, 144), (100, 70, 256), (64, 300, 1040), (33, 65, 2064),       # 32 x 32
          (128, 2100, 144), (126, 2101, 400), (100, 2100, 1168),               # 64 x 32
          (20, 8300, 272), (32, 8299, 1040),                                   # 32 x 64
          (64, 8300, 1040), (200, 3001, 1168),                                 # 64 x 64
          (130, 5500, 1040), (97, 9000, 1136),                                 # 128 x 64
          (64, 16500, 1040), (40, 16601, 1056),                                # 64 x 128
          (512, 4200, 1040), (300, 6001, 1152)]                                # 128 x 128


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_ring(ops, oracle, M, N, K):
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    print(f"ring M={M} N={N} K={K}", flush=True)
    acc = oracle.quantized_dot(A, B, 1)
    dA, dB = dev(A), dev(B)
    np.testing.assert_array_equal(host(ops.quantized_dot(dA, dB)), acc)
    sA, sB = rng.uniform(1e-3, 0.05, M), rng.uniform(1e-4, 0.02, N)
    bias = rng.uniform(-1, 1, N).astype(np.float32)
    y = oracle.epilogue(acc, "rowcol", sA, sB, bias=bias, act="relu")
    got = host(ops.qlinear(dA, dev(sA), dB, dev(sB), bias=dev(bias), act="relu"))
    np.testing.assert_array_equal(got.view(np.uint32), y.view(np.uint32))
    s_next = float(np.abs(y).max() / 127.0) or 1.0
    q = host(ops.qlinear_requant(dA, dev(sA), dB, dev(sB), s_next, bias=dev(bias), act="relu"))
    np.testing.assert_array_equal(q, oracle.quantize(y.reshape(-1), s_next).reshape(M, N))


def test_ring_under_capture(ops, oracle):
    """Replayed from a graph, with the kernel's own eager calls between."""
    rng = np.random.default_rng(3)
    A = rng.integers(-128, 128, (48, 1024)).astype(np.int8)
    B = rng.integers(-128, 128, (500, 1024)).astype(np.int8)
    acc = oracle.quantized_dot(A, B, 1)
    dA, dB = dev(A), dev(B)
    out = torch.empty((48, 500), dtype=torch.int32, device=DEV)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        ops.quantized_dot(dA, dB, out=out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        ops.quantized_dot(dA, dB, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        np.testing.assert_array_equal(host(out), acc)
        np.testing.assert_array_equal(host(ops.quantized_dot(dA, dB)), acc)


# Either side of each tile's least number of 128-byte stages (256 CUs), K
# ending inside the last one
ROUTES = [(256, 1024, 384, "qgemm"), (48, 1000, 400, "ring 32x32 k4"),
          (96, 4090, 640, "qgemm"), (96, 4090, 656, "ring 64x32 k4"),
          (20, 11000, 384, "qgemm"), (20, 11001, 400, "ring 32x64 k4"),
          (64, 11008, 896, "qgemm"), (61, 11008, 1008, "ring 64x64 k2"),
          (130, 5500, 2416, "qgemm"), (130, 5501, 2448, "ring 128x64 k2"),
          (64, 16500, 1920, "qgemm"), (63, 16500, 2000, "ring 64x128 k2"),
          (512, 4200, 6000, "qgemm"), (511, 4201, 6032, "ring 128x128 k1"),
          (100, 16500, 3968, "qgemm"), (100, 16499, 4000, "ring 128x128 k1"), (1024, 4096, 4096, "qgemm")]


@pytest.mark.parametrize("M,N,K,route", ROUTES)
def test_ring_from_its_first_stages_on(ops, oracle, M, N, K, route):
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    sA, sB = rng.uniform(1e-3, 0.05, M), rng.uniform(1e-4, 0.02, N)
    bias = rng.uniform(-1, 1, N).astype(np.float32)
    print(f"ring route M={M} N={N} K={K}", flush=True)
    acc = (A.astype(np.float64) @ B.T.astype(np.float64)).astype(np.int32)   # exact: sums below 2^53
    dA, dB, da, db, dbias = dev(A), dev(B), dev(sA), dev(sB), dev(bias)
    np.testing.assert_array_equal(host(ops.quantized_dot(dA, dB)), acc)
    assert ops.last_gemm().startswith(route)
    y = oracle.epilogue(acc, "rowcol", sA, sB, bias=bias, act="relu")
    got = host(ops.qlinear(dA, da, dB, db, bias=dbias, act="relu"))
    np.testing.assert_array_equal(got.view(np.uint32), y.view(np.uint32))
    s_next = float(np.abs(y).max() / 127.0)
    q = host(ops.qlinear_requant(dA, da, dB, db, s_next, bias=dbias, act="relu"))
    np.testing.assert_array_equal(q, oracle.quantize(y.reshape(-1), s_next).reshape(M, N))
