"""The fp32 attention operator on the bf16 matrix core: three-part operands at the
edges of its tiles and of fp32's range, additive biases and masks, and values that
are not finite (worked out with fp32 products).

Bars: the attention tolerance of tests/test_gpu_attention.py against float64 where
the values are finite; over the plain sizes also 1e-6 of the result's 2-norm, the
fp32 products' own error."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ATTN_TOL = 2e-5
NH, NKV, D = 4, 2, 128


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ovnative_amd
    ovnative_amd.load()
    torch.cuda.set_device(0)
    yield
    torch.cuda.synchronize()


def _reference(q, k, v, bias=None):
    out = torch.zeros_like(q, dtype=torch.float64)
    for h in range(NH):
        kv = h // (NH // NKV)
        s = (q[:, h * D:(h + 1) * D].double()
             @ k[:, kv * D:(kv + 1) * D].double().t().contiguous()) * D ** -0.5
        if bias is not None:
            s = s + bias.double()
        out[:, h * D:(h + 1) * D] = torch.softmax(s, dim=1) @ v[:, kv * D:(kv + 1) * D].double()
    return out


def _inputs(seed, rows):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn((rows, n * D), generator=g).cuda() for n in (NH, NKV, NKV)], g


@pytest.mark.parametrize("rows", [1, 2, 31, 32, 33, 127, 128, 129, 257, 700])
@pytest.mark.parametrize("biased", [False, True], ids=["plain", "bias"])
def test_sizes(rows, biased):
    import ovnative_amd as ov
    (q, k, v), g = _inputs(rows, rows)
    bias = torch.randn((rows, rows), generator=g).cuda() * 3 if biased else None
    got = ov.attention(q, k, v, [(bias, rows, 0, 0)], NH, NKV).double()
    want = _reference(q, k, v, bias)
    assert (got - want).abs().max() <= ATTN_TOL * max(1.0, float(want.abs().max()))
    assert (got - want).norm() <= 1e-6 * want.norm()


@pytest.mark.parametrize("scale", [1e-36, 1e-30, 1e-18, 1e18, 1e30, 1e36])
def test_range(scale):
    """Values far beyond f16 (which the split-f16 operator refuses); at 1e+-36 the
    low parts of Q or V are below bf16's range."""
    import ovnative_amd as ov
    (q, k, v), _ = _inputs(7, 100)
    got = ov.attention(q / scale, k * scale, v * scale, [(None, 100, 0, 0)], NH, NKV).double()
    want = _reference(q / scale, k * scale, v * scale)
    assert (got - want).norm() <= 2e-6 * want.norm()


def test_not_finite():
    import ovnative_amd as ov
    rows = 200
    (q, k, v), _ = _inputs(9, rows)
    segs = [(None, rows, 0, 0)]
    base = ov.attention(q, k, v, segs, NH, NKV)
    # an infinity in V: that column of its two heads, nothing else
    bad = v.clone()
    bad[17, 5] = float("inf")
    got = ov.attention(q, k, bad, segs, NH, NKV)
    cols = torch.zeros(NH * D, dtype=torch.bool)
    cols[5] = cols[D + 5] = True
    assert bool((got[:, cols] == float("inf")).all())
    assert bool(torch.isfinite(got[:, ~cols]).all())
    assert (got[:, ~cols] - base[:, ~cols]).abs().max() <= ATTN_TOL
    # a key whose every score is -inf has no weight
    qp, kb = q.clone(), k.clone()
    qp[:, ::D] = qp[:, ::D].abs() + 0.5
    kb[33, ::D] = float("-inf")
    got = ov.attention(qp, kb, v, segs, NH, NKV).double()
    keep = torch.arange(rows) != 33
    want = torch.zeros((rows, NH * D), dtype=torch.float64, device="cuda")
    for h in range(NH):
        kv = h // (NH // NKV)
        s = (qp[:, h * D:(h + 1) * D].double()
             @ k[keep][:, kv * D:(kv + 1) * D].double().t().contiguous()) * D ** -0.5
        want[:, h * D:(h + 1) * D] = (torch.softmax(s, dim=1)
                                      @ v[keep][:, kv * D:(kv + 1) * D].double())
    assert (got - want).abs().max() <= ATTN_TOL * max(1.0, float(want.abs().max()))
    # a NaN in one query row and head: it has no largest score, so zeros as for a
    # row without visible keys; nothing else changes
    qn = q.clone()
    qn[50, D + 3] = float("nan")
    got = ov.attention(qn, k, v, segs, NH, NKV)
    assert bool((got[50, D:2 * D] == 0).all())
    got[50, D:2 * D] = base[50, D:2 * D]
    assert (got - base).abs().max() <= ATTN_TOL


@pytest.mark.parametrize("low", [-1e30, torch.finfo(torch.float32).min, float("-inf")])
def test_masks(low):
    """Masks of the usual low values: whole blocks hidden, a row that sees one key,
    a row that sees none."""
    import ovnative_amd as ov
    rows = 300
    (q, k, v), g = _inputs(11, rows)
    vis = torch.rand((rows, rows), generator=g) < 0.5
    vis[:, 0] = True
    vis[:100, 160:] = False
    vis[7] = False
    vis[7, 250] = True
    vis[9] = False
    bias = torch.where(vis, 0.0, low).cuda()
    got = ov.attention(q, k, v, [(bias, rows, 0, 0)], NH, NKV).double()
    assert bool((got[9] == 0).all())
    seen = torch.arange(rows) != 9
    want = _reference(q, k, v, torch.where(vis.cuda(), 0.0, float("-inf")).double())
    assert (got - want)[seen].abs().max() <= ATTN_TOL * max(1.0, float(want[seen].abs().max()))


def test_bias_at_the_end_of_the_range():
    """A bias of 3e38: the keys that have it share the row's weight."""
    import ovnative_amd as ov
    rows = 70
    (q, k, v), _ = _inputs(13, rows)
    bias = torch.zeros((rows, rows))
    bias[:, 3] = bias[:, 40] = 3e38
    got = ov.attention(q, k, v, [(bias.cuda(), rows, 0, 0)], NH, NKV).double()
    for h in range(NH):
        kv = h // (NH // NKV)
        want = (v[3, kv * D:(kv + 1) * D].double() + v[40, kv * D:(kv + 1) * D].double()) / 2
        assert (got[:, h * D:(h + 1) * D] - want).abs().max() <= ATTN_TOL
