"""The host twin of the selection kernel against the plain implementation (no GPU)."""
import numpy as np
import pytest

import plain_llama as P
from gpullama3_java_amd.sampling import SamplingParams, sample_host, select_sampler, uniform


def test_uniform_is_a_function_of_its_counters():
    u = [uniform(3, r, s) for r in range(20) for s in range(50)]
    assert all(0 <= x < 1 for x in u) and len(set(u)) > 990
    assert uniform(3, 4, 5) == uniform(3, 4, 5) != uniform(4, 4, 5)
    assert all(np.float32(x) == x for x in u)                   # exact in float32
    assert abs(np.mean(u) - 0.5) < 0.03


@pytest.mark.parametrize("temperature, top_p", [(0.0, 0.95), (0.8, 0.95), (1.0, 1.0), (1.3, 0.0), (0.5, 0.3), (1.0, 1e-6)])
def test_twin_agrees_with_the_plain_rule(temperature, top_p):
    rng = np.random.default_rng(0)
    for n in (2, 17, 300):
        for _ in range(40):
            logits = (rng.standard_normal(n) * rng.uniform(0.5, 4)).astype(np.float32)
            u = float(np.float32(rng.random()))
            assert sample_host(logits, temperature, top_p, u) == P.sample(logits, temperature, top_p, u)


def test_ties_and_edges():
    assert sample_host(np.array([1, 3, 3, 2], np.float32), 0, 1, 0.5) == 1
    flat = np.zeros(8, np.float32)
    assert [sample_host(flat, 1.0, 1.0, u) for u in (0.0, 0.13, 0.99)] == [0, 1, 7]
    # equal probabilities under top-p: lower indices are kept first
    assert [sample_host(flat, 1.0, 0.3, u) for u in (0.0, 0.4, 0.99)] == [0, 1, 2]


def test_validation_as_the_reference_options():
    with pytest.raises(ValueError):
        SamplingParams(-0.1, 0.5)
    with pytest.raises(ValueError):
        SamplingParams(0.5, 1.5)
    assert select_sampler(100, 0.7, 0.9, 42) == SamplingParams(0.7, 0.9, 42)


def test_one_sampler_s_calls_of_several_threads_take_turns(monkeypatch):
    """A call's parameters and probabilities lie in scratch that the sampler's calls share, while the library runs without the
    interpreter's lock: the next call waits until this one has its tokens."""
    import time
    from concurrent.futures import ThreadPoolExecutor
    from types import SimpleNamespace

    import torch

    from gpullama3_java_amd.csrc import lib
    from gpullama3_java_amd.sampling import DeviceSampler
    monkeypatch.setattr(lib, "sample_work_size", lambda rows, vocab: rows * vocab)

    def sample_host(logits, work, parameters, out):
        work[:len(out)] = torch.tensor(parameters[2])
        time.sleep(0.002)
        out.copy_(work[:len(out)])
    monkeypatch.setattr(lib, "sample_host", sample_host)
    sampler = DeviceSampler(torch.device("cpu"))
    sampler._torch = SimpleNamespace(float32=torch.float32, int32=torch.int32,
                                     empty=lambda n, dtype, device, pin_memory=False: torch.empty(n, dtype=dtype, device=device))

    def calls(k):
        return all(sampler(torch.zeros(2 + k, 5), [1.0] * (2 + k), [0.9] * (2 + k), [k] * (2 + k)) == [k] * (2 + k) for _ in range(10))
    with ThreadPoolExecutor(4) as threads:
        assert all(threads.map(calls, range(4)))


# (arrays of other numbers than 32-bit floats are converted as lists are, not read as if they were)
@pytest.mark.parametrize("kinds", ["fff", "ddd", "fdl", "idd"])
def test_a_call_s_numbers_come_in_arrays_of_any_kind(monkeypatch, kinds):
    from array import array
    from types import SimpleNamespace

    import torch

    from gpullama3_java_amd.csrc import lib
    numbers = [[1] * 3 if kinds[0] == "i" else [0.8, 0.0, 1.3], [0.9, 1.0, 0.5], [0] * 3 if kinds[2] == "l" else [0.25, 0.1, 0.7]]
    given = []
    calls = SimpleNamespace(gl3_sample_work_floats=lambda rows, vocab: 0,
                            gl3_sample_host=lambda logits, ld, work, t, p, u, *rest: given.append([list(t), list(p), list(u)]) or 0)
    for name, stand_in in (("_dev", lambda *a, **kw: None), ("_ptr", lambda t: None), ("_stream", lambda: None), ("library", lambda: calls)):
        monkeypatch.setattr(lib, name, stand_in)
    out = SimpleNamespace(numel=lambda: 2, dtype=torch.int32, is_contiguous=lambda: True, is_pinned=lambda: True)
    for par in (numbers, [array(k, n) for k, n in zip(kinds, numbers)]):
        lib.sample_host(torch.zeros(2, 9), torch.zeros(300), par, out)
    want = [np.float32(n[:2]).tolist() for n in numbers]               # (a call of two rows takes two numbers each)
    assert given == [want, want]
