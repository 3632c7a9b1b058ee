"""Shapes of the ragged solve: one 256-thread workgroup per work item (per_cu 0),
and what the library reports of a call forced back.

Against the oracle per system, at the ragged tolerances (normwise 1e-12 FP64,
1e-5 FP32); a shape forced back gives the same bits.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from tests.test_gpu_ext import check_ragged, dev, ragged_case  # noqa: E402
from tridsolver_amd import _lib, api  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.set_device(0)


def _lengths(rng, longest, count):
    lens = np.round(np.exp(rng.uniform(0, np.log(longest), count))).astype(np.int64)
    edges = [0, 1, 2, longest // 2, longest // 2 + 1, longest - 1, longest, 0]
    lens[:len(edges)] = edges
    return lens


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("M,said,longest", [(4, 1024, 1024), (8, 2048, 2048), (16, 4096, 4096),
                                            (4, 1024, 4096), (8, 2048, 8192),
                                            (16, 4096, 8192)])
def test_forced_workgroup_per_item(M, said, longest, dtype):
    """per_cu 0 at each number of rows per lane, up to the rows 256 lanes hold and
    beyond (max_len understated), plain and Inc."""
    rng = np.random.default_rng(M + longest)
    off, a, b, c, d = ragged_case(rng, _lengths(rng, longest, 700), dtype)
    u = rng.uniform(-1, 1, len(d)).astype(dtype)
    with api.forced_ragged(M, per_cu=0):
        for inc in (False, True):
            td, tu = dev(d), dev(u) if inc else None
            api.ragged_batch(dev(a), dev(b), dev(c), td, dev(off), max_len=said, u=tu, sync=True)
            assert api.last_config() == (5, M, 0, 1, 0)
            if inc:
                assert np.array_equal(td.cpu().numpy(), d)
            check_ragged(off, a, b, c, d, (tu if inc else td).cpu().numpy(), dtype,
                         u if inc else None)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("max_len", [1000, 2048, 4096, 8192])
def test_reported_shape_can_be_forced(max_len, dtype):
    rng = np.random.default_rng(max_len)
    off, a, b, c, d = ragged_case(rng, _lengths(rng, max_len, 300), dtype)
    args = [dev(t) for t in (a, b, c)]
    x, y = dev(d), dev(d)
    api.ragged_batch(*args, x, dev(off), max_len=max_len, sync=True)
    cfg = api.last_config()
    with api.forced_ragged(cfg[1], per_cu=cfg[4], launches=cfg[3]):
        api.ragged_batch(*args, y, dev(off), max_len=max_len, sync=True)
        assert api.last_config() == cfg
    assert torch.equal(x, y)


def test_forced_shapes_refused():
    L = _lib.lib()
    for M, per_cu, launches in ((8, -1, 1), (8, 9, 1), (8, 0, 2), (16, 0, 4), (5, 0, 1)):
        assert L.tridHipForceRaggedConfig(M, per_cu, launches) == 3, (M, per_cu, launches)
    rng = np.random.default_rng(2)
    off, a, b, c, d = ragged_case(rng, [10, 300, 5], np.float64)
    f = [dev(t.astype(np.float32)) for t in (a, b, c, d)]
    with api.forced_ragged(16, per_cu=0):  # the mixed solves have a resident grid only
        with pytest.raises(_lib.TridError):
            api.ragged_batch_mixed(dev(a), dev(b), dev(c), dev(d), dev(off), max_len=300, sync=True)
        with pytest.raises(_lib.TridError):
            api.ragged_batch_mixed_f32(*f, dev(off), max_len=300, sync=True)


def _best_ms(call):
    """The shortest of eight timed calls."""
    times = []
    for _ in range(8):
        ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        ev[0].record()
        call()
        ev[1].record()
        torch.cuda.synchronize()
        times.append(ev[0].elapsed_time(ev[1]))
    return min(times)


def _operands(n, dtype):
    g = torch.Generator(device="cuda").manual_seed(5)
    a, c, d = (torch.rand(n, dtype=dtype, device="cuda", generator=g) - 0.5 for _ in range(3))
    return a, 2 + a.abs() + c.abs(), c, d


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_understated_max_len_is_not_slow(dtype):
    """Systems of twice the rows that max_len says are solved on the shape chosen for
    it; they read their arrays a second time, so three times the declared call's time
    is the bound (a solve of each lane's rows straight from memory took seven)."""
    n, count = 4096, 4000
    a, b, c, d = _operands(n * count, dtype)
    off = torch.arange(0, (n + 1) * count, n, device="cuda")[:count + 1].contiguous()
    best, x = {}, {}
    for said in (n // 2, n):
        x[said] = d.clone()
        api.ragged_batch(a, b, c, x[said], off, max_len=said)
        y = d.clone()
        best[said] = _best_ms(lambda: api.ragged_batch(a, b, c, y, off, max_len=said))
    print("understated %.3f ms, declared %.3f ms" % (best[n // 2], best[n]))
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    assert (x[n] - x[n // 2]).abs().max().item() <= tol * x[n].abs().max().item()
    assert best[n // 2] <= 3 * best[n]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_adding_to_u_costs_its_traffic(dtype):
    """The Inc form reads u besides: 6 / 5 of the plain solve's bytes, so 1.4 times its
    time is the bound (with every row's addition waiting for its own load it took 1.5)."""
    rng = np.random.default_rng(8)
    lens = np.exp(rng.uniform(np.log(237), np.log(6000), 16000)).astype(np.int64)
    off = dev(np.concatenate([[0], np.cumsum(lens)]))
    a, b, c, d = _operands(int(lens.sum()), dtype)
    u = torch.zeros_like(d)
    inc = _best_ms(lambda: api.ragged_batch(a, b, c, d, off, max_len=6000, u=u))
    plain = _best_ms(lambda: api.ragged_batch(a, b, c, d, off, max_len=6000))
    print("Inc %.3f ms, plain %.3f ms" % (inc, plain))
    assert inc <= 1.4 * plain
