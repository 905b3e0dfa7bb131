"""The sampler's call with its parameters and tokens in host memory: the same tokens as the kernels that read them from the device."""
import numpy as np
import pytest
import torch

from gpullama3_java_amd.csrc import lib
from gpullama3_java_amd.sampling import DeviceSampler, sample_host

pytestmark = pytest.mark.gpu


# one launch of parameters holds 256 rows
@pytest.mark.parametrize("rows", [1, 8, 255, 256, 257, 600])
def test_the_call_from_host_memory(rows):
    rng = np.random.default_rng(rows)
    V = 1031
    logits = torch.tensor(3 * rng.standard_normal((rows, V + 5)), dtype=torch.float32, device="cuda:0")[:, 2:2 + V]
    par = [rng.choice([0.0, 0.7, 1.3], rows), rng.choice([0.0, 0.5, 0.9, 1.0], rows), rng.random(rows)]
    par[0][0] = 0.7                                                     # (not every row greedy)
    par = [p.astype(np.float32).tolist() for p in par]
    sampler = DeviceSampler(torch.device("cuda:0"))
    got = sampler(logits, *par)
    on = [torch.tensor(p, dtype=torch.float32, device="cuda:0") for p in par]
    work = torch.empty(lib.sample_work_size(rows, V), device="cuda:0")
    out = torch.empty(rows, dtype=torch.int32, device="cuda:0")
    lib.sample(logits, work, *on, out)
    assert got == out.tolist() and got == sampler(logits, *par)          # (again: its scratch holds the first call's numbers)
    host = logits.cpu().numpy()
    assert sum(t != sample_host(host[r], *(p[r] for p in par)) for r, t in enumerate(got)) <= rows // 200    # (sums in another order)
    assert sampler(logits, [0.0] * rows, par[1], par[2]) == host.argmax(1).tolist()


@pytest.mark.parametrize("temperature", [0.8, 0.0])
def test_a_call_behind_longer_work_than_it_looks_for(temperature):
    """Some 10 ms of products are in front of it on the stream, where it looks for its tokens for half a millisecond and then waits for the stream."""
    rng = np.random.default_rng(4)
    logits = torch.tensor(3 * rng.standard_normal((8, 1031)), dtype=torch.float32, device="cuda:0")
    par = ([temperature] * 8, [0.9] * 8, rng.random(8).tolist())
    sampler = DeviceSampler(torch.device("cuda:0"))
    want = sampler(logits, *par)
    other = torch.randn(8192, 8192, device="cuda:0")
    torch.cuda.synchronize()
    for _ in range(3):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        late = torch.zeros_like(logits)
        begin.record()
        product = other @ other
        late.copy_(logits)                                              # (the logits themselves come late)
        end.record()
        got = sampler(late, *par)
        assert end.query() and begin.elapsed_time(end) > 1.0            # (all in front of it is done; it took longer than the look)
        assert got == want
        del product


@pytest.mark.parametrize("greedy", [False, True])
def test_tokens_of_an_earlier_call_are_not_taken_for_this_one_s(greedy):
    logits = torch.zeros(2, 3, 1031, device="cuda:0")
    places = torch.tensor([[5, 700, 1030], [6, 0, 44]])
    for call in range(2):
        logits[call, torch.arange(3), places[call]] = 60.0
    work = torch.empty(lib.sample_work_size(3, 1031) + 9, device="cuda:0")
    pinned = torch.empty(3, dtype=torch.int32, pin_memory=True)
    other = torch.randn(2048, 2048, device="cuda:0")
    for call in (0, 1, 0, 1):
        for _ in range(2):
            other @ other                                               # (so that the tokens are not there at the first look)
        lib.sample_host(logits[call], work, None if greedy else [[0.7] * 3, [0.9] * 3, [0.5] * 3], pinned)
        assert pinned.tolist() == places[call].tolist()


def test_the_call_from_host_memory_refuses():
    logits = torch.zeros(2, 50, device="cuda:0")
    work = torch.empty(lib.sample_work_size(2, 50) + 6, device="cuda:0")
    pinned = torch.empty(2, dtype=torch.int32, pin_memory=True)
    par = [[1.0, 1.0]] * 3
    for arguments in ((logits, work, par, torch.empty(2, dtype=torch.int32)), (logits, work, par, pinned[:1]), (logits, work[:-1], par, pinned),
                      (logits, work, [[1.0]] * 3, pinned), (logits.double(), work, par, pinned), (logits.T, work, None, pinned)):
        with pytest.raises(lib.KernelError):
            lib.sample_host(*arguments)
    with pytest.raises(ValueError):
        DeviceSampler(torch.device("cuda:0"))(logits, [1.0, 1.0], [1.0], [0.5, 0.5])


def test_the_call_where_tensors_are_made_on_the_gpu_by_default():
    logits = torch.zeros(2, 50, device="cuda:0")
    logits[0, 7] = logits[1, 31] = 40.0
    with torch.device("cuda:0"):
        assert DeviceSampler(torch.device("cuda:0"))(logits, [0.5] * 2, [0.9] * 2, [0.3] * 2) == [7, 31]


@pytest.mark.parametrize("own_streams", [False, True])
def test_calls_of_two_threads(own_streams):
    from concurrent.futures import ThreadPoolExecutor
    rng = np.random.default_rng(7)
    sampler = DeviceSampler(torch.device("cuda:0"))
    calls = []
    for rows, temperature in ((300, 0.7), (257, 1.3)):              # (two launches of parameters each; scratch of two sizes)
        logits = torch.tensor(3 * rng.standard_normal((rows, 1031)), dtype=torch.float32, device="cuda:0")
        par = ([temperature] * rows, [0.9] * rows, rng.random(rows).tolist())
        calls.append((logits, par, DeviceSampler(torch.device("cuda:0"))(logits, *par)))
    torch.cuda.synchronize()

    def calls_of(thread):
        logits, par, want = calls[thread]
        with torch.cuda.stream(torch.cuda.Stream() if own_streams else torch.cuda.default_stream()):
            return sum(sampler(logits, *par) != want for _ in range(100))
    with ThreadPoolExecutor(2) as threads:
        assert list(threads.map(calls_of, range(2))) == [0, 0]


def _flat(kind, rows, V, rng):
    if kind == "normal":                    # a nucleus of thousands, in many bins
        return rng.standard_normal((rows, V)) * 1.5
    if kind == "ties":                      # hundreds of equal values at every place
        return rng.integers(0, 40, (rows, V)) / 8.0
    if kind == "two values":                # the threshold and the drawn token in a bin with more values than the lists hold, or in the other
        return np.where(rng.random((rows, V)) < 0.5, 0.0, -0.5)
    if kind == "equal":                     # one value: no bin is short enough
        return np.zeros((rows, V))
    if kind == "fine":                      # no two values equal, all of a row in a bin or two
        return rng.standard_normal((rows, V)) * 1e-3
    if kind == "many equal":                # thousands of equal values in a list that holds them
        return np.where(rng.random((rows, V)) < min(1.0, 7000 / V), 3.0, rng.standard_normal((rows, V)) - 3.0)
    x = rng.standard_normal((rows, V))      # most of the row without any probability
    x[:, V // 2:] = -np.inf
    return x


# (short rows, the last slices empty; a vocabulary whose slices are two stretches; lists at, below and beyond their length)
@pytest.mark.parametrize("kind", ["normal", "ties", "two values", "equal", "fine", "many equal", "half"])
@pytest.mark.parametrize("V", [70, 8192, 16500, 128256, 140001])
def test_flat_rows(kind, V):
    """Rows whose nucleus reaches below the gathered candidates take the bins; the tokens are the definition's."""
    rng = np.random.default_rng(V)
    rows = 24
    x = _flat(kind, rows, V, rng).astype(np.float32)
    par = [[1.0] * rows, rng.choice([0.3, 0.7, 0.95, 0.999], rows).tolist(), rng.random(rows).astype(np.float32).tolist()]
    got = DeviceSampler(torch.device("cuda:0"))(torch.from_numpy(x).cuda(), *par)
    want = [sample_host(x[r], *(p[r] for p in par)) for r in range(rows)]
    order = [np.lexsort((np.arange(V), -x[r].astype(np.float64))) for r in range(rows)]
    place = [np.argsort(o) for o in order]
    # p is off by a few 2^-24 of itself, the running sum of the nucleus by as much of its mass, so a drawn token stands at most as many places
    # from the definition's as such an error spans: 2^-20 of the row's mass over the token's own probability, and one (where all values
    # are equal a third of the tokens are the neighbour). Tokens whose probabilities differ by less than the errors of two of them (2^-22 each: the
    # exponential, its argument and the division) may stand in either order, so as many places more.
    p = [np.exp(r.astype(np.float64) - r.max()) for r in x]
    for r in range(rows):
        span = 2.0 ** -20 * p[r].sum() / p[r][want[r]] + 1.0
        beside = np.abs(p[r] - p[r][want[r]])
        span += np.count_nonzero((beside > 0.0) & (beside <= 2.0 ** -21 * p[r][want[r]]))
        assert abs(int(place[r][got[r]]) - int(place[r][want[r]])) <= span, (r, got[r], want[r])


@pytest.mark.parametrize("kind, V, most", [("equal", 128256, 6.2), ("fine", 128256, 4.5), ("many equal", 128256, 4.0), ("ties", 128256, 6.0),
                                           ("two values", 8192, 4.0), ("ties", 8192, 3.0), ("equal", 8192, 4.0)])
def test_rows_of_few_values_take_no_longer_than_their_searches(kind, V, most):
    """Rows of equal values against rows of as many different ones, which take a third of the passes over the row: thousands of equal values
    are not compared with each other (that was 45 times the other's time), and a wave does not add to one counter lane by lane."""
    import time
    rng = np.random.default_rng(5)
    rows = 8
    sampler = DeviceSampler(torch.device("cuda:0"))
    par = [[1.0] * rows, [0.95] * rows, rng.random(rows).astype(np.float32).tolist()]

    def least(x):
        x = torch.from_numpy(x.astype(np.float32)).cuda()
        times = []
        for _ in range(12):
            t = time.perf_counter()
            sampler(x, *par)
            times.append(time.perf_counter() - t)
        return min(times)
    assert least(_flat(kind, rows, V, rng)) < most * least(_flat("normal", rows, V, rng))


def test_a_row_without_a_number():
    """Nothing to choose from (no finite maximum): a token of the vocabulary all the same, and the rows beside it are as alone."""
    x = torch.randn(3, 5000, generator=torch.Generator().manual_seed(2))
    alone = DeviceSampler(torch.device("cuda:0"))(x.cuda(), [0.9] * 3, [0.9] * 3, [0.3] * 3)
    for bad in (float("nan"), float("-inf")):
        y = x.clone()
        y[1] = bad
        got = DeviceSampler(torch.device("cuda:0"))(y.cuda(), [0.9] * 3, [0.9] * 3, [0.3] * 3)
        assert [got[0], got[2]] == [alone[0], alone[2]] and 0 <= got[1] < 5000
