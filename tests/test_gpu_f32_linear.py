"""The fp32 linear at the edges of its kernels: fewer k steps than the ring has
stages (odd and even), tiles of one row and one column, both sides of the
64- / 128-row tile switch, the one-pass row split and the general one (other K,
rows that are not 16-byte aligned), and rows of zeros.

Bar: |C - float64| <= 2^-18 sum_k |A W| per output, the operator's own bar
(22-bit operands, lo*lo dropped, fp32 sums)."""
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


@pytest.mark.parametrize("offset", [0, 1], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("M,N,K", [(1, 8200, 1024), (63, 130, 16), (64, 129, 48), (65, 128, 64),
                                   (130, 300, 80), (129, 1, 256), (6, 257, 512), (1536, 200, 768),
                                   (1537, 200, 256), (2050, 131, 1024),
                                   # few products, rows of more than 80 n tiles: by whole
                                   # n tiles, in 64 and 128 rows
                                   (70, 1100, 128), (1600, 1100, 77), (65, 1100, 144),
                                   (64, 10241, 160), (200, 10369, 256), (520, 10369, 256),
                                   (520, 10240, 256), (1537, 10241, 130)])
def test_linear_f32_edges(M, N, K, offset):
    import ovnative_amd as ov
    g = torch.Generator().manual_seed(M + N + K)
    flat = torch.randn(M * K + offset, generator=g)
    A = flat.cuda()[offset:].view(M, K)  # contiguous, 4 bytes past 16-byte alignment if offset
    if M > 2:
        A[1] = 0.0
        A[2] *= 1e-30
    W = (torch.randn((K, N), generator=g) * 0.02).numpy()
    w = ov.Weight.from_host_f32(W, layout=1)
    Wd = torch.from_numpy(W).cuda().double()
    want, bound = A.double() @ Wd, 2.0 ** -18 * (A.double().abs() @ Wd.abs())
    got = ov.linear_f32(A, w).double()
    assert ((got - want).abs() <= bound).all()
    C0 = torch.randn((M, N), generator=g).cuda()
    add = ov.linear_f32(A, w, C=C0.clone(), accumulate=True).double()
    # one more fp32 rounding
    assert ((add - (C0.double() + want)).abs() <= bound + 2.0 ** -23 * add.abs()).all()
