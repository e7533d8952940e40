"""What the fp32 attention operator's three-part operands and its exponentials must
not lose against fp32 products: no error of one sign, small probabilities beside
large values, small keys under a large scale, subnormal values.

Reference: float64 on the same device."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

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


def _reference(q, k, v, scale):
    out = torch.zeros_like(q, dtype=torch.float64)
    for h in range(NH):
        kv = h // (NH // NKV)
        s = (q[:, h * D:(h + 1) * D].double()
             @ k[:, kv * D:(kv + 1) * D].double().t().contiguous()) * scale
        out[:, h * D:(h + 1) * D] = torch.softmax(s, dim=1) @ v[:, kv * D:(kv + 1) * D].double()
    return out


def _inputs(seed, rows):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn((rows, n * D), generator=g).cuda() for n in (NH, NKV, NKV)]


def _run(q, k, v, scale=D ** -0.5):
    import ovnative_amd as ov
    rows = q.shape[0]
    got = ov.attention(q, k, v, [(None, rows, 0, 0)], NH, NKV, scale=scale).double()
    return got, _reference(q, k, v, scale)


@pytest.mark.parametrize("rows", [300, 600])
def test_no_error_of_one_sign(rows):
    """The mean error along the result's sign.  Rounding has none (150 000 outputs
    with 1e-7 of random error average to below 1e-9); the matrix core's sums leave
    up to 1e-8 of the root mean square.  Parts cut off instead of rounded: 4e-8."""
    q, k, v = _inputs(rows, rows)
    got, want = _run(q, k, v.abs())
    bias = ((got - want) * want.sign()).mean() / want.square().mean().sqrt()
    assert abs(float(bias)) <= 2.5e-8


def _two_keys(scores, values):
    """Row i and head h attend to key 0 with score 0 and to key 1 with score
    scores[i, h], both exact in fp32; `values` are those keys' rows of v."""
    rows = scores.shape[0]
    q = torch.zeros((rows, NH, D), device="cuda")
    q[:, :, 0], q[:, :, 1] = scores, 1.0
    k, v = torch.zeros((rows, NKV, D), device="cuda"), torch.zeros((rows, NKV, D), device="cuda")
    k[1, :, 0] = 1.0
    k[2:, :, 1] = -1000.0  # no weight
    v[0], v[1] = values
    return q.view(rows, -1), k.view(rows, -1), v.view(rows, -1)


def test_products():
    """Scores of one product each, of significands whose parts cut off lose most (7.8
    units of 2^-24) and of random ones: e^(-16 x y) within the product's error (the
    dropped parts' 2^-24 of it and its rounding's 2^-24, absolute in the exponent) and
    the exponential's."""
    g = torch.Generator().manual_seed(1)
    worst = torch.tensor([1 + 2.0 ** -7 - 2.0 ** -23, 1 + (2.0 ** 16 - 1) * 2.0 ** -23,
                          1 + 2.0 ** -7 - 2.0 ** -16, 1 + 2.0 ** -8 + 2.0 ** -16])
    x = torch.cat([worst, 1 + torch.rand((28,), generator=g)]).cuda()
    for y in x.tolist()[:8]:
        q, k, v = _two_keys(-16 * x[:, None].expand(-1, NH), (0.0, 1.0))
        k.view(-1, NKV, D)[1, :, 0] = y
        got, want = _run(q, k, v, scale=1.0)
        product = 16 * x[:, None].double() * y
        assert bool(((got - want).abs() / want <= 2.0 ** -23 * product + 3.6e-7).all()), y


@pytest.mark.parametrize("top", [0.0, -4.0, -10.0, -20.0, -40.0])
def test_probabilities(top):
    """e^x, x down to -60, to fp32's precision: the hardware's 2^y is good to one
    unit (2^-23), the quotient and the products round four times more by 2^-24; the
    argument's own rounding (up to 2^-24 |x|) must not come on top."""
    g = torch.Generator().manual_seed(int(-top))
    scores = (top - 20 * torch.rand((512, NH), generator=g)).cuda()
    got, want = _run(*_two_keys(scores, (0.0, 1.0)), scale=1.0)
    assert float(((got - want).abs() / want).max()) <= 3.6e-7


@pytest.mark.parametrize("below,e", [(60, 49), (60, 53), (60, 80), (80, 110), (83, 119), (86.5, 124),
                                     (88, 126)])
def test_small_probability_of_a_large_value(below, e):
    """A probability of e^-below beside a value of 2^e: their product counts.  Below
    2^-126 fp32 itself has only 2^-149 / p of the probability left."""
    g = torch.Generator().manual_seed(e)
    small, large = 1 + torch.rand((D,), generator=g), 2.0 ** e * (1 + 0.5 * torch.rand((D,), generator=g))
    scores = torch.full((64, NH), -float(below), device="cuda")
    got, want = _run(*_two_keys(scores, (small.cuda(), large.cuda())), scale=1.0)
    assert float(((got - want).abs() / want).max()) <= 3.6e-7 + 2.0 ** -149 / 2.71828 ** -below


@pytest.mark.parametrize("e", [30, 45, 49, 50, 51, 52, 53, 54, 55, 56, 57, 58, 60, 64])
def test_values_at_the_end_of_the_sums(e):
    """Values of 2^e on both sides of where the sums overflow (and the tile is worked
    out with fp32 products)."""
    q, k, v = _inputs(e, 200)
    got, want = _run(q, k, v.abs() * 2.0 ** e)
    assert (got - want).norm() <= 1e-6 * want.norm()


@pytest.mark.parametrize("e", [-120, -80, -31, -29, -20, 20, 60, 61, 80, 100, 120])
@pytest.mark.parametrize("where", ["q", "k"])
def test_scales(e, where):
    """A scale of 2^e with Q or K of 2^-e: the same scores, whichever parts that
    takes out of bf16's range."""
    q, k, v = _inputs(abs(e), 200)
    small = 2.0 ** -e
    got, want = _run(q * small if where == "q" else q, k * small if where == "k" else k, v,
                     scale=D ** -0.5 * 2.0 ** e)
    assert (got - want).norm() <= 1e-6 * want.norm()


@pytest.mark.parametrize("e", [-127, -130, -135, -140])
@pytest.mark.parametrize("rows", [32, 200])
def test_subnormal_values(rows, e):
    """V below fp32's normal range, where the matrix core reads zeros: within the
    rounding of the products and sums to multiples of 2^-149, one each a key at
    most, over four partial sums."""
    q, k, v = _inputs(rows, rows)
    got, want = _run(q, k, v.abs() * 2.0 ** e)
    assert float((got - want).abs().max()) <= rows * 2.0 ** -149
    assert (got - want).norm() <= 0.02 * want.norm()


def test_zero_columns():
    """Zeros in V (a head padded to its width) are zeros in the result."""
    q, k, v = _inputs(5, 300)
    v.view(-1, NKV, D)[:, :, 100:] = 0.0
    got, want = _run(q, k, v)
    assert bool((got.view(-1, NH, D)[:, :, 100:] == 0).all())
    assert (got - want).norm() <= 1e-6 * want.norm()


@pytest.mark.parametrize("rows,stride", [(3, (1 << 22) - 4), (3, 1 << 22), (1000, 1 << 20),
                                         (1023, 1 << 20), (1025, 1 << 20)])
def test_far_rows(rows, stride):
    """Rows of K and V far apart: both sides of the 24-bit row strides and 32-bit
    offsets of the tile's loads; the bits of the same rows close together, within
    one rounding where the fp32 products take over."""
    import ovnative_amd as ov
    q, k, v = _inputs(rows, rows)
    near = ov.attention(q, k, v, [(None, rows, 0, 0)], NH, NKV)
    far = []
    for t in (k, v):
        wide = torch.zeros((rows, stride), device="cuda")
        wide[:, :NKV * D] = t
        far.append(wide)
    got = ov.attention(q, *far, [(None, rows, 0, 0)], NH, NKV)
    assert (got - near).norm() <= 1e-6 * near.norm()
    assert bool(torch.isfinite(got).all())
