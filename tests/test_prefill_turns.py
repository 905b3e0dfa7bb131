"""The prefill attention whose two groups of waves take turns (heads of 128): its results against the plain reference and the kernel of
128 queries a block, whose bits they are."""
import numpy as np
import pytest
import torch

from gpullama3_java_amd.csrc import lib


def test_the_kernel_of_turns_asks_for_caches_at_16_byte_addresses():
    """Its loads into shared memory bring 16 bytes a lane. (A call that names it is refused before anything is launched; the library's own
    choice is another kernel.)"""
    import ctypes
    L = lib.library()
    memory = ctypes.create_string_buffer(4096)
    at = -(-ctypes.addressof(memory) // 16) * 16

    def call(k, v, splits=1):
        p = ctypes.c_void_p
        return L.gl3_attention_prefill(p(at), 256, p(at + k), p(at + v), p(at), p(at), p(at), None, 1, p(at), 256, 1, 1, 2, 1, 128, 64, 0, 0.1,
                                       lib.PREFILL_TURNS, None, 0, 0.0, 0, 0, 1, None, 0.0, 0.0, 0, None, 0, splits, 1, None, None, None)
    for k, v in ((2, 0), (0, 8)):
        assert call(k, v) != 0 and b"16-byte addresses" in L.gl3_last_error()
    assert call(0, 0, 2) != 0 and b"no splits" in L.gl3_last_error()
    choice = L.gl3_prefill_kernel
    assert choice(128, 64, 24, 8, 8, 1752, 5886, 1) == 2 and choice(128, 64, 24, 8, 8, 1752, 5886, 0) == 1          # (0: not plain)


def test_many_short_sequences_beside_a_long_one_take_the_kernel_of_128_queries():
    def choice(lengths, heads=24):
        return lib.library().gl3_prefill_kernel(128, 64, heads, 8, len(lengths), max(lengths), sum(lengths), 1)
    assert choice([1300] + [100] * 60) == 1 and choice([1300] + [100] * 60, 32) == 1 and choice([2048] + [300] * 31) == 1
    assert choice([8192], 32) == 2 and choice([4096]) == 2 and choice([8000] + [100] * 60) == 2 and choice([2048] + [20] * 60) == 2
    assert choice([1752, 96, 1390, 211, 803, 1101, 377, 156]) == 2 and choice([317, 1203, 701]) == 2 and choice([1024] * 2, 32) == 2
    assert choice([2000] * 8) == 2 and choice([1024] * 8) == 1 and choice([512] * 8) == 1
    assert choice([2048]) == 0 and choice([1024] * 2) == 0 and choice([100]) == 0           # (too few blocks for either)


def fn(before, new, wide_from, shuffled_rows=False):
    from test_gpu_kernels import dev

    def call(q, kc, vc, positions, seq_of, table, out, H, Kh, hs, page, window, scale):
        cu = dev(np.concatenate([[0], np.cumsum(new)]), torch.int32)
        seq_rows = None
        if shuffled_rows:                            # (sequence b's pages in row seq_rows[b] of a table with other rows between)
            order = np.random.default_rng(len(new)).permutation(2 * len(new))[:len(new)]
            seq_rows = dev(order, torch.int32)
            wide = torch.zeros((2 * len(new), table.shape[1]), dtype=torch.int32, device=table.device)
            wide[seq_rows.long()] = table
            table = wide
        lib.attention_prefill(q, kc, vc, cu, dev(before, torch.int32), table, out, max(new), H, Kh, hs, page, window, scale,
                              seq_rows=seq_rows, wide_from=wide_from)
    return call


def rounding(qs, sk, sv, ref, before, new):
    """What rounding may make of each output: a weight is rounded to bfloat16 (eight significant bits: half a unit of the last is at most
    2^-8 of it), so is the result; the sums are in 32 bits."""
    from test_gpu_kernels import P
    size = np.concatenate([P.attention(q, k, np.abs(v))[b:b + n] for q, k, v, b, n in zip(qs, sk, sv, before, new)])
    return (2.0 ** -8 + 1e-4) * (size + np.abs(ref))


# two, one and three heads a kv head and blocks of 128 and of 256 queries; waves, blocks and chunks with one row and all but one;
# sequences that start no block of the longest one's kind; more chunks than a register holds places of (64), twice as many
CASES = [(4, 2, 64, [0, 70, 0, 130, 5], [33, 1, 200, 17, 64]), (3, 1, 64, [0, 0, 0], [256, 257, 31]), (2, 2, 128, [63, 64, 65], [129, 128, 127]),
         (6, 2, 192, [4200, 0], [3, 300]), (2, 1, 64, [8200], [70]), (8, 8, 64, [1] * 64, list(range(1, 65)))]


@pytest.mark.gpu
@pytest.mark.parametrize("sharp", [1, 8])
@pytest.mark.parametrize("H, Kh, page, before, new", CASES)
def test_attention_of_turns(H, Kh, page, before, new, sharp):
    from test_gpu_kernels import attention_case, run_attention
    sk, sv, qs = attention_case(np.random.default_rng(H * page + sharp), H, Kh, 128, before, new, "bfloat16")
    qs = [q * sharp for q in qs]                     # (8: a few keys have all the weight, and maxima move in all chunks)
    run = lambda f: run_attention(f, sk, sv, qs, before, new, H, Kh, 128, "bfloat16", np.random.default_rng(1), page=page)
    got, ref = run(fn(before, new, lib.PREFILL_TURNS))
    # (by each output's own size: those behind thousands of keys are a tenth of those behind a few, and as large as a wrong chunk's)
    assert float((np.abs(got - ref) / rounding(qs, sk, sv, ref, before, new)).max()) <= 1
    np.testing.assert_array_equal(got, run(fn(before, new, 1))[0])      # (the same sums in the same order as the kernel of 128 queries a block)
    np.testing.assert_array_equal(got, run(fn(before, new, lib.PREFILL_TURNS, shuffled_rows=True))[0])


@pytest.mark.gpu
@pytest.mark.parametrize("at", [0, 31, 32, 63, 64, 95, 1000, 1037, 1038, 1055, 1060])
def test_values_that_are_not_finite_reach_as_far_as_in_the_kernel_beside_it(at):
    """A weight of zero does not make nothing of an infinite value: it spoils the queries in front of it whose keys share its 32, and
    what a page still holds behind the sequence's end (here from 1,038 on) likewise; no more than that on either kernel."""
    from test_gpu_kernels import attention_case, run_attention
    H, Kh, before, new = 4, 2, [700], [338]
    sk, sv, qs = attention_case(np.random.default_rng(at), H, Kh, 128, before, [400], "bfloat16")
    for value in (np.inf, np.nan):
        sv[0][at, 0, 77] = value
        run = lambda f: run_attention(f, sk, sv, qs, before, new, H, Kh, 128, "bfloat16", np.random.default_rng(1))[0]
        got = run(fn(before, new, lib.PREFILL_TURNS))
        np.testing.assert_array_equal(got, run(fn(before, new, 1)))
        waves = np.arange(700, 1038) - 700 >> 5      # (32 queries walk their keys together)
        last = np.minimum(waves * 32 + 731, 1037)
        assert np.isfinite(got[last // 32 < at // 32]).all() and np.isfinite(got[:, :, :77]).all() and np.isfinite(got[:, 2:]).all()
        assert not np.isfinite(got[np.arange(700, 1038) >= at, :2, 77]).any()


@pytest.mark.gpu
def test_attention_of_turns_with_one_key_that_counts_and_scores_that_are_not_numbers():
    from test_gpu_kernels import attention_case, run_attention
    H, Kh, before, new = 4, 2, [700], [300]
    sk, sv, qs = attention_case(np.random.default_rng(3), H, Kh, 128, before, new, "bfloat16")
    run = lambda k, q: run_attention(fn(before, new, lib.PREFILL_TURNS), k, sv, q, before, new, H, Kh, 128, "bfloat16", np.random.default_rng(1))
    for at in (0, 63, 64, 699):                      # the ends of chunks, a key of the first token's alone beside its own
        k, q = [s.copy() for s in sk], [s.copy() for s in qs]
        k[0][at] = 0
        k[0][at, :, 5] = 40.0
        q[0][700:, :, 5] = 8.0
        got, ref = run(k, q)
        np.testing.assert_allclose(got, ref, atol=1e-2 * np.abs(ref).max())
        np.testing.assert_allclose(got[:, 0], np.broadcast_to(sv[0][at, 0], got[:, 0].shape), atol=0.05)
    clean, _ = run(sk, qs)
    k = [s.copy() for s in sk]
    k[0][900:930, 1] = np.nan                        # seen by the tokens from position 900 on, through the second kv head
    got, _ = run(k, qs)
    assert np.isnan(got[200:, 2:]).all()
    np.testing.assert_array_equal(got[:200], clean[:200])
    np.testing.assert_array_equal(got[:, :2], clean[:, :2])


@pytest.mark.gpu
def test_thresholds_of_zero_and_below_are_the_library_s_choice():
    from test_gpu_kernels import attention_case, run_attention
    for hs in (64, 128):
        sk, sv, qs = attention_case(np.random.default_rng(hs), 4, 2, hs, [40], [70], "bfloat16")
        got = [run_attention(fn([40], [70], w), sk, sv, qs, [40], [70], 4, 2, hs, "bfloat16", np.random.default_rng(1))[0] for w in (0, -1, -64)]
        np.testing.assert_array_equal(got[1], got[0])
        np.testing.assert_array_equal(got[2], got[0])


@pytest.mark.gpu
def test_attention_of_turns_refuses_what_it_is_not_built_for():
    from test_gpu_kernels import attention_case, run_attention
    for hs, page, before, new, window in ((64, 64, [0], [70], 0), (128, 96, [0], [70], 0), (128, 64, [0], [70], 20), (128, 64, [0] * 65, [2] * 65, 0)):
        sk, sv, qs = attention_case(np.random.default_rng(4), 4, 2, hs, before, new, "bfloat16")
        with pytest.raises(lib.KernelError):
            run_attention(fn(before, new, lib.PREFILL_TURNS), sk, sv, qs, before, new, 4, 2, hs, "bfloat16", np.random.default_rng(1), page=page,
                          window=window)
