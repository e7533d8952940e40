"""ovh_linear's one-launch form for few rows, on both sides of its size rules, for
any K up to 2048 (whole, ragged and single blocks), odd N and strides, unaligned
rows, values the short quantiser hands back to the general one, and operands that
overlap (which keep the two-launch form).

Bar: bit equality with quantise + linear_q as calls of their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ovnative_amd
    ovnative_amd.load()
    torch.cuda.set_device(0)
    yield
    torch.cuda.synchronize()


def same(a, b):
    return torch.equal(a.contiguous().view(torch.int32), b.contiguous().view(torch.int32))


def _weight(rng, N, K):
    import ovnative_amd as ov
    return ov.Weight.from_host(rng.integers(-127, 128, (N, K)).astype(np.int8),
                               rng.uniform(1e-4, 1e-3, N).astype(np.float32))


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 1), (1, 1024, 2048), (16, 33, 31), (17, 31, 33), (40, 1024, 2048), (15, 130, 1025),
    (65, 77, 333), (128, 1024, 2048), (129, 1024, 2048), (512, 512, 1024), (513, 512, 1024),
    (333, 1501, 1000), (337, 1537, 1000), (512, 1024, 1024), (40, 100, 2049), (300, 1024, 640)])
def test_one_launch_linear(M, N, K, offset):
    import ovnative_amd as ov
    rng = np.random.default_rng(M + N + K)
    w = _weight(rng, N, K)
    flat = torch.from_numpy(rng.standard_normal(M * K + offset).astype(np.float32)).cuda()
    A = flat[offset:].view(M, K)
    # rows of zeros, of one value, tiny, huge, and outside the finite values
    for r, v in enumerate((0.0, 3.5, 1e-44, 1e-36, 1e37, 3e38, float("inf"), float("nan"))):
        if r + 1 < M:
            A[r + 1] = v if r < 2 else A[r + 1] * v
        if r + 20 < M:
            A[r + 20, K // 2] = v
    C0 = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).cuda()
    aq, asc = ov.s8_nk_quantize(A)
    assert same(ov.linear(A, w), ov.linear_q(aq, asc, w))
    assert same(ov.linear(A, w, C=C0.clone(), accumulate=True),
                ov.linear_q(aq, asc, w, C=C0.clone(), accumulate=True))


# rows loaded value by value, on both sides of the lines between 32 columns, 128
# columns and two launches
@pytest.mark.parametrize("M,N,K", [(128, 1024, 1001), (129, 1024, 1001), (480, 1024, 1001),
                                   (481, 1024, 1001), (512, 1024, 850), (513, 1024, 850),
                                   (256, 1024, 767), (257, 1024, 767)])
def test_one_launch_linear_odd_rows(M, N, K):
    test_one_launch_linear(M, N, K, 0)


def test_leading_dimension_and_overlap():
    """Columns past N of a wider C stay as they are; C over A still gives
    A + linear(A) of the old A."""
    import ovnative_amd as ov
    rng = np.random.default_rng(3)
    M, K = 48, 256
    w = _weight(rng, K, K)
    A = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).cuda()
    want = ov.linear_q(*ov.s8_nk_quantize(A), w)
    wide = torch.full((M, K + 7), 9.0, device="cuda")
    ov.linear(A, w, C=wide)
    assert same(wide[:, :K], want) and bool((wide[:, K:] == 9.0).all())
    x = A.clone()
    ov.linear(x, w, C=x, accumulate=True)
    assert same(x, ov.linear_q(*ov.s8_nk_quantize(A), w, C=A.clone(), accumulate=True))


def test_graph_capture():
    """The one-launch call in a captured graph, replayed on new values."""
    import ovnative_amd as ov
    rng = np.random.default_rng(4)
    M, N, K = 40, 1024, 2048
    w = _weight(rng, N, K)
    A, C = torch.zeros((M, K), device="cuda"), torch.zeros((M, N), device="cuda")
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        ov.linear(A, w, C=C)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ov.linear(A, w, C=C)
    for _ in range(3):
        A.copy_(torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert same(C, ov.linear(A, w))
