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
