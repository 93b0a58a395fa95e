"""The small-call routes against the oracle: the one-launch per-tensor
quantize at the edges of its range (with zeros, NaN and infinities, and
misaligned tensors on the general route), the dot4 GEMV of long rows and
SiLU * up + quantize on either side of its row-length limits."""
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


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("n", [1, 3, 4, 255, 4096, 4097, 65537, 98304, 98305])
@pytest.mark.parametrize("kind", ["normal", "zeros", "nan", "inf", "tiny"])
def test_quantize_per_tensor_small(ops, oracle, n, kind):
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    if kind == "zeros":
        x[:] = -0.0
    elif kind == "nan":
        x[::2] = np.nan
    elif kind == "inf":
        x[n // 2] = -np.inf
    elif kind == "tiny":
        x *= np.float32(1e-42)
    s = oracle.scale_per_tensor(x)
    want = oracle.quantize(x, s)
    for shift in (0, 1):
        buf = torch.empty(n + 1, device=DEV)
        d = buf[shift:shift + n]
        d.copy_(torch.from_numpy(x))
        q, sc = ops.quantize_per_tensor(d)
        assert host(sc)[0] == s or (np.isnan(s) and np.isnan(host(sc)[0])), (kind, n)
        np.testing.assert_array_equal(host(q), want)


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("N,K", [(5, 8208), (70, 12288), (33, 12304), (10, 16400), (7, 20480), (9, 20496)])
def test_gemv_long_rows(ops, oracle, M, N, K):
    rng = np.random.default_rng(M + N + K)
    A = rng.integers(-128, 128, (M, K)).astype(np.int8)
    B = rng.integers(-128, 128, (N, K)).astype(np.int8)
    got = ops.quantized_dot(torch.from_numpy(A).to(DEV), torch.from_numpy(B).to(DEV))
    np.testing.assert_array_equal(host(got), oracle.quantized_dot(A, B, 1))


@pytest.mark.parametrize("M", [1, 3, 300])
@pytest.mark.parametrize("K", [4096, 4100, 8192, 8196, 11008, 12288, 12292, 13376, 20480, 20484])
def test_silu_rows(ops, oracle, M, K):
    rng = np.random.default_rng(M + K)
    gu = (rng.standard_normal((M, 2 * K)) * 4).astype(np.float32)
    gu[0, K - 1] = np.inf
    gu[M - 1, K // 2] = np.nan
    h = oracle.silu_mul(np.ascontiguousarray(gu[:, :K]), np.ascontiguousarray(gu[:, K:]))
    s = oracle.scales_per_token(h)
    want = oracle.quantize_rows(h, s)
    d = torch.from_numpy(gu).to(DEV)
    h_out = torch.empty(M, K, device=DEV)
    for g, u in ((d[:, :K], d[:, K:]), (d[:, :K].contiguous(), d[:, K:].contiguous())):
        q, sc = ops.silu_mul_quantize(g, u, h_out)
        np.testing.assert_array_equal(host(h_out), h)
        np.testing.assert_array_equal(host(sc), s)
        np.testing.assert_array_equal(host(q), want)
