"""The split-f16 operator's biases: masks (0 / -1e30, attended as bit words),
other additive biases (attended as values), both kinds in one call, one bias
shared by several segments, in the short and the long kernel.

Bar: the attention tolerance of tests/test_gpu_attention.py against float64;
a mask gives the bits of the same mask that one harmless value (-0.5 on a
masked-out neighbour's fully masked row) sends through the value form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

ATTN_TOL = 2e-5
NH, NKV, D = 8, 4, 128


@pytest.fixture(scope="module", autouse=True)
def _device():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ovnative_amd
    ovnative_amd.load()
    torch.cuda.set_device(0)
    yield
    torch.cuda.synchronize()


def _reference(q, k, v, segs):
    out = torch.zeros_like(q, dtype=torch.float64)
    for bias, r, at, _ in segs:
        for h in range(NH):
            kv = h // (NH // NKV)
            s = (q[at:at + r, h * D:(h + 1) * D].double()
                 @ k[at:at + r, kv * D:(kv + 1) * D].double().t().contiguous()) * D ** -0.5
            if bias is not None:
                s = s + bias.double()
            o = torch.softmax(s, dim=1) @ v[at:at + r, kv * D:(kv + 1) * D].double()
            o[s.amax(dim=1) < -1e29] = 0.0
            out[at:at + r, h * D:(h + 1) * D] = o
    return out


def _mask(g, r):
    m = torch.where(torch.rand((r, r), generator=g) < 0.3, -1e30, 0.0)
    m[r // 2] = -1e30  # a fully masked row
    return m.cuda()


@pytest.mark.parametrize("long_min", [None, 0], ids=["by_size", "long"])
@pytest.mark.parametrize("rows", [1, 31, 64, 65, 129, 300])
def test_bias_kinds(rows, long_min):
    import ovnative_amd as ov
    g = torch.Generator().manual_seed(rows)
    mask, other = _mask(g, rows), torch.randn((rows, rows), generator=g).cuda()
    inf = torch.where(torch.rand((rows, rows), generator=g) < 0.2, float("-inf"), 0.0).cuda()
    inf.fill_diagonal_(0.0)
    kinds = [mask, None, other, mask, inf]
    segs = [(b, rows, i * rows, i * rows) for i, b in enumerate(kinds)]
    T = len(kinds) * rows
    q, k, v = (torch.randn((T, n * D), generator=g).cuda() for n in (NH, NKV, NKV))
    prev = ov.set_attention_long_min_tasks(long_min) if long_min is not None else None
    try:
        got = ov.attention(q, k, v, segs, NH, NKV, split=True)
        # the mask through the value form: a fully masked row (zeros whatever its
        # other values) holds one value that is neither 0 nor -1e30
        alt = mask.clone()
        alt[rows // 2] = -2e30
        again = ov.attention(q, k, v, [(alt if b is mask else b, *rest) for b, *rest in segs], NH,
                             NKV, split=True)
    finally:
        if prev is not None:
            ov.set_attention_long_min_tasks(prev)
    want = _reference(q, k, v, segs)
    assert (got - want).abs().max() <= ATTN_TOL * max(1.0, float(want.abs().max()))
    for i in (0, 3):
        assert (got[i * rows + rows // 2] == 0).all()
    assert torch.equal(got.view(torch.int32), again.view(torch.int32))


def test_threads_and_reports():
    """Calls from several threads on streams of their own, one of them with a
    value beyond f16: only that one is refused, every other result unchanged."""
    import threading
    import ovnative_amd as ov
    g = torch.Generator().manual_seed(1)
    rows = 96
    mask = _mask(g, rows)
    q, k, v = (torch.randn((rows, n * D), generator=g).cuda() for n in (NH, NKV, NKV))
    bad = v.clone()
    bad[3, 5] = 1e6
    segs = [(mask, rows, 0, 0)]
    want = ov.attention(q, k, v, segs, NH, NKV, split=True)
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    if i == 1:
                        with pytest.raises(ov.InvalidArgument):
                            ov.attention(q, k, bad, segs, NH, NKV, split=True)
                    else:
                        assert torch.equal(ov.attention(q, k, v, segs, NH, NKV, split=True), want)
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]


def test_value_biases_cost():
    """Biases of values cost reading them: 16 segments of 600 rows take at most
    twice the time of the same call without biases (1.4 times before the mask pass
    existed, 2.6 while every row of it reported through memory)."""
    import time
    import ovnative_amd as ov
    n, rows = 16, 600
    g = torch.Generator().manual_seed(2)
    q, k, v = (torch.randn((n * rows, w * D), generator=g).cuda() for w in (16, 8, 8))
    biases = [torch.randn((rows, rows), generator=g).cuda() for _ in range(n)]
    plain = [(None, rows, i * rows, i * rows) for i in range(n)]
    valued = [(b, rows, i * rows, i * rows) for i, b in enumerate(biases)]
    times = {}
    for _ in range(12):
        for name, segs in (("plain", plain), ("valued", valued)):
            t = time.perf_counter()
            for _ in range(5):
                ov.attention(q, k, v, segs, 16, 8, split=True)  # returns when done
            times.setdefault(name, []).append(time.perf_counter() - t)
    assert np.median(times["valued"]) <= 2.0 * np.median(times["plain"]), times


def test_refusal_cost():
    """A call whose every K is beyond f16 is refused in at most three times the time
    of the accepted call (20 times while every tile told the host), and the calls
    after it are accepted."""
    import time
    import ovnative_amd as ov
    n, rows = 16, 600
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn((n * rows, w * D), generator=g).cuda() for w in (16, 8, 8))
    far = k * 1e7
    segs = [(None, rows, i * rows, i * rows) for i in range(n)]
    want = ov.attention(q, k, v, segs, 16, 8, split=True)
    times = {"taken": [], "refused": []}
    for _ in range(12):
        t = time.perf_counter()
        got = ov.attention(q, k, v, segs, 16, 8, split=True)
        times["taken"].append(time.perf_counter() - t)
        assert torch.equal(got, want)
        t = time.perf_counter()
        with pytest.raises(ov.InvalidArgument):
            ov.attention(q, far, v, segs, 16, 8, split=True)
        times["refused"].append(time.perf_counter() - t)
    assert np.median(times["refused"]) <= 3 * np.median(times["taken"]), times


def test_more_calls_than_report_slots():
    """40 threads with a call in flight each (a call finds one of 32 report slots,
    or reports through its own workspace): masks, values and refusals as alone."""
    import threading
    import ovnative_amd as ov
    g = torch.Generator().manual_seed(4)
    rows = 300
    mask, other = _mask(g, rows), torch.randn((rows, rows), generator=g).cuda()
    q, k, v = (torch.randn((2 * rows, n * D), generator=g).cuda() for n in (NH, NKV, NKV))
    far = k.clone()
    far[rows + 7, 9] = 1e6
    segs = [(mask, rows, 0, 0), (other, rows, rows, rows)]
    want = ov.attention(q, k, v, segs, NH, NKV, split=True)
    torch.cuda.synchronize()
    errors, start = [], threading.Barrier(40)

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait(60)
                for _ in range(10):
                    if i % 5 == 1:
                        with pytest.raises(ov.InvalidArgument):
                            ov.attention(q, far, v, segs, NH, NKV, split=True)
                    else:
                        assert torch.equal(ov.attention(q, k, v, segs, NH, NKV, split=True), want)
        except BaseException as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(40)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]
