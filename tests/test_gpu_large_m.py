"""The large-M GEMM form (gemm_wide.hip) and the SiLU epilogue's short forms, on
both sides of every switch and with values outside the short forms' range.

Bars: bit equality.  Sampled rows against the oracle; every row against the same
rows run a few hundred at a time (the small-M kernels); the SiLU launch against
the projections and silu_mul_quantize as calls of their own."""
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


def bits(t):
    return t.contiguous().view(torch.int32 if t.dtype == torch.float32 else torch.uint8)


def same(a, b):
    return torch.equal(bits(a), bits(b))


def _weight(rng, N, K):
    import ovnative_amd as ov
    q = rng.integers(-127, 128, (N, K)).astype(np.int8)
    s = rng.uniform(1e-4, 1e-3, N).astype(np.float32)
    return ov.Weight.from_host(q, s), q, s


# N odd (a last tile of one weight row), M one past a 64- and a 128-row tile, K of
# one, two and more 128-k chunks; 1024 rows with 480 tiles or more, 2048 with 1000
@pytest.mark.parametrize("M,N,K", [(1024, 3841, 128), (1025, 3841, 256), (2047, 2049, 1024),
                                   (2048, 4096, 384), (2049, 3841, 1024), (8200, 1000, 640)])
def test_large_m_form(oracle, M, N, K):
    import ovnative_amd as ov
    rng = np.random.default_rng(M + N + K)
    w, q, s = _weight(rng, N, K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    aq, asc = ov.s8_nk_quantize(torch.from_numpy(A).cuda())
    C0 = torch.from_numpy(rng.standard_normal((M, N)).astype(np.float32)).cuda()
    got = ov.linear_q(aq, asc, w)
    add = ov.linear_q(aq, asc, w, C=C0.clone(), accumulate=True)
    at = ov.tile_major(aq)
    assert same(ov.linear_q_tiled(at, asc, w, M), got)
    assert same(ov.linear_q_tiled(at, asc, w, M, C=C0.clone(), accumulate=True), add)
    for r in range(0, M, 500):  # the same rows through the small-M kernels
        e = min(r + 500, M)
        assert same(ov.linear_q(aq[r:e].contiguous(), asc[r:e].contiguous(), w), got[r:e]), r
    assert same(got + C0, add)
    rows = sorted({0, 1, 63, 64, 127, 128, M - 65, M - 2, M - 1})
    oq, osc = oracle.quantize(A[rows])
    want = oracle.linear_q(oq, osc, q, s)
    assert same(got[rows], torch.from_numpy(want).cuda())


# the large-M form's own range of K (768 and more, 512 from 4096 rows) on both sides,
# and what it leaves to the other tiles at 1024 rows and at 10240 columns
@pytest.mark.parametrize("M,N,K", [(1025, 3841, 768), (1025, 3841, 640), (4097, 4097, 512),
                                   (4095, 4097, 512), (1087, 6145, 768), (1089, 6145, 768),
                                   (1030, 6145, 1536), (1089, 10241, 768), (1089, 10240, 768)])
def test_large_m_form_by_k(oracle, M, N, K):
    test_large_m_form(oracle, M, N, K)


def test_large_m_form_slices():
    """Slices that end inside a 128-row tile, into outputs of their own."""
    import ovnative_amd as ov
    rng = np.random.default_rng(5)
    M, K, widths = 1090, 256, [1984, 64, 1920]
    w, _, _ = _weight(rng, sum(widths), K)
    aq, asc = ov.s8_nk_quantize(torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
                                .cuda())
    whole = ov.linear_q(aq, asc, w)
    at = 0
    for out, n in zip(ov.linear_q_sliced(aq, asc, w, widths), widths):
        assert same(out, whole[:, at:at + n].contiguous())
        at += n


def test_large_m_block_dots():
    """The per-block products of the large-M form's own kernel."""
    import ovnative_amd as ov
    rng = np.random.default_rng(6)
    M, N, K = 1030, 3841, 256
    w, q, _ = _weight(rng, N, K)
    aq = torch.from_numpy(rng.integers(-127, 128, (M, K)).astype(np.int8)).cuda()
    want = torch.stack([aq[:, b * 32:b * 32 + 32].double()
                        @ torch.from_numpy(q[:, b * 32:b * 32 + 32].T.copy()).cuda().double()
                        for b in range(K // 32)], dim=2).to(torch.int32)
    assert torch.equal(ov.block_dots(aq, w), want)
    assert torch.equal(ov.block_dots(ov.tile_major(aq), w, M=M, tiled=True), want)


def test_large_m_block_dots_long_k():
    """The same where K is in the large-M form's range: sampled rows and columns."""
    import ovnative_amd as ov
    rng = np.random.default_rng(8)
    M, N, K = 1030, 3841, 768
    w, q, _ = _weight(rng, N, K)
    aq = torch.from_numpy(rng.integers(-127, 128, (M, K)).astype(np.int8)).cuda()
    rows, cols = [0, 1, 63, 64, 127, 1024, 1029], [0, 31, 32, 127, 128, 3839, 3840]
    a = aq[rows].view(len(rows), K // 32, 32).int().cpu()
    b = torch.from_numpy(q[cols]).view(len(cols), K // 32, 32).int()
    want = (a[:, None] * b[None]).sum(dim=3).to(torch.int32).cuda()
    assert torch.equal(ov.block_dots(aq, w)[rows][:, cols], want)
    assert torch.equal(ov.block_dots(ov.tile_major(aq), w, M=M, tiled=True)[rows][:, cols], want)


# every SiLU tile: 1, 129, 513 rows, and both sides of the large-M form's switches
@pytest.mark.parametrize("M", [1, 129, 513, 639, 640, 705, 4095, 4097])
@pytest.mark.parametrize("special", [False, True], ids=["normal", "special"])
def test_silu_epilogue(M, special):
    import ovnative_amd as ov
    rng = np.random.default_rng(M)
    I, K = 192, 256
    (wg, _, _), (wu, _, _) = _weight(rng, I, K), _weight(rng, I, K)
    aq, asc = ov.s8_nk_quantize(torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
                                .cuda())
    if special:
        # row scales that put gate (and h) at zero, below and above every bound
        # of the short forms, and outside the finite values
        scale = torch.tensor([0.0, 1e-38, 1e-33, 1e-29, 1e-20, 1.0, 40.0, 300.0, 3e3, 1e17, 1e25,
                              3e38, float("inf"), float("nan")], device="cuda")
        asc *= scale[torch.arange(M, device="cuda") % len(scale)][:, None]
    gate, up = ov.linear_q(aq, asc, wg), ov.linear_q(aq, asc, wu)
    want_q, want_s = ov.silu_mul_quantize(gate, up)
    hq, hsc = ov.silu_gate_linear(aq, asc, ov.gate_up_weight(wg, wu))
    assert torch.equal(hq, want_q)
    assert same(hsc, want_s)


# Whole wavefronts inside the short forms' range, up to their bounds (the tiles of
# the test above all hold rows outside it): every row has the one scale, the gates
# reach -66 and 66, just below 2^60 (positive ones: 1 + e^-g must stay below 2^97), or
# just above 2^-100; `beyond` passes the first bound.  The up projection's own
# scales keep h in the quantiser's short range.
@pytest.mark.parametrize("M", [1, 129, 513, 640, 705, 4097])
@pytest.mark.parametrize("reach", ["span", "beyond", "large", "tiny"])
def test_silu_epilogue_bounds(M, reach):
    import ovnative_amd as ov
    rng = np.random.default_rng(M + 1)
    I, K = 192, 256
    A = rng.standard_normal((M, K)).astype(np.float32)
    qg, qu = (rng.integers(-127, 128, (I, K)).astype(np.int8) for _ in range(2))
    sg, su = (rng.uniform(1e-4, 1e-3, I).astype(np.float32) for _ in range(2))
    if reach in ("large", "tiny"):  # gates of one sign
        A, qg = np.abs(A), np.abs(qg)
    aq, asc = ov.s8_nk_quantize(torch.from_numpy(A).cuda())
    gate = ov.linear_q(aq, asc, ov.Weight.from_host(qg, sg))
    near, far = float(gate.abs().min()), float(gate.abs().max())
    factor = {"span": 65.9 / far, "beyond": 66.2 / -float(gate.min()),
              "large": 2.0 ** 60 * (1 - 1e-4) / far,
              "tiny": 2.0 ** -100 * (1 + 1e-4) / near}[reach]
    asc *= factor
    wg, wu = ov.Weight.from_host(qg, sg), ov.Weight.from_host(qu, (su / factor).astype(np.float32))
    gate, up = ov.linear_q(aq, asc, wg), ov.linear_q(aq, asc, wu)
    if reach == "span":
        assert 65 < float(gate.abs().max()) <= 66
    elif reach == "large":
        assert 2.0 ** 59.9 < float(gate.max()) <= 2.0 ** 60 and float(gate.min()) > 0
    elif reach == "tiny":
        assert 2.0 ** -100 <= float(gate.min()) < 2.0 ** -99.9
    want_q, want_s = ov.silu_mul_quantize(gate, up)
    hq, hsc = ov.silu_gate_linear(aq, asc, ov.gate_up_weight(wg, wu))
    assert torch.equal(hq, want_q)
    assert same(hsc, want_s)


# both sides of the 128-row tile's line (448 of them): 416, 448, 528 and 231
@pytest.mark.parametrize("M,I", [(4096, 832), (4096, 896), (4097, 1024), (4095, 448)])
def test_silu_tile_rows(M, I):
    import ovnative_amd as ov
    rng = np.random.default_rng(I)
    K = 256
    (wg, _, _), (wu, _, _) = _weight(rng, I, K), _weight(rng, I, K)
    aq, asc = ov.s8_nk_quantize(torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32))
                                .cuda())
    want_q, want_s = ov.silu_mul_quantize(ov.linear_q(aq, asc, wg), ov.linear_q(aq, asc, wu))
    hq, hsc = ov.silu_gate_linear(aq, asc, ov.gate_up_weight(wg, wu))
    assert torch.equal(hq, want_q)
    assert same(hsc, want_s)
