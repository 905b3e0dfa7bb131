"""The prefill attention whose two groups of waves take turns (heads of 128): the rule that takes it, and its results against the plain
reference and the kernels beside it."""
import numpy as np
import pytest
import torch

from gpullama3_java_amd.csrc import lib


def test_splits_on_the_kernel_of_turns():
    s = lib.prefill_turns_splits
    assert s(24, 8, 128, 64, 1, 512, 4512) == 5 and s(32, 8, 128, 64, 1, 512, 4512) == 4          # 48 and 64 blocks
    assert s(24, 8, 128, 64, 1, 64, 4064) == 8 and s(24, 8, 128, 64, 1, 1100, 7100) == 2 and s(32, 8, 128, 64, 1, 2048, 14048) == 1
    assert s(24, 8, 128, 64, 1, 300, 2047) == 0 and s(24, 8, 64, 64, 1, 512, 4512) == 0           # few keys; heads of 64
    assert s(24, 8, 128, 32, 1, 512, 4512) == 0 and s(24, 8, 128, 64, 65, 30, 4512) == 0          # pages of half a chunk; many sequences
    for heads, kv in ((24, 8), (32, 8), (8, 8), (128, 8), (1, 1)):
        for n_seqs in (1, 2, 7, 64):
            for T in (1, 128, 129, 257, 1000, 5000):
                n = s(heads, kv, 128, 64, n_seqs, T, 100000)
                assert 1 <= n <= 8 and (n == 1 or n * n_seqs * T * heads <= lib.PREFILL_SPLIT_ROWS)


def fn(before, new, wide_from, splits=1):
    from test_gpu_kernels import DEV, dev

    def call(q, kc, vc, positions, seq_of, table, out, H, Kh, hs, page, window, scale):
        cu = dev(np.concatenate([[0], np.cumsum(new)]), torch.int32)
        n = splits * len(positions) * H
        parts = dict(splits=splits, part_o=torch.full((n * hs,), float("nan"), device=DEV),
                     part_ml=torch.full((2 * n,), float("nan"), device=DEV)) if splits > 1 else {}
        lib.attention_prefill(q, kc, vc, cu, dev(before, torch.int32), table, out, max(new), H, Kh, hs, page, window, scale,
                              wide_from=wide_from, **parts)
    return call


# two, one and three heads a kv head and blocks of 128 and of 256 queries; waves, blocks and chunks with one row and all but one;
# sequences that start no block of the longest one's kind; more chunks than a register holds places of (64), twice as many
CASES = [(4, 2, 64, [0, 70, 0, 130, 5], [33, 1, 200, 17, 64]), (3, 1, 64, [0, 0, 0], [256, 257, 31]), (2, 2, 128, [63, 64, 65], [129, 128, 127]),
         (6, 2, 192, [4200, 0], [3, 300]), (2, 1, 64, [8200], [70]), (8, 8, 64, [1] * 64, list(range(1, 65)))]


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2, 8])
@pytest.mark.parametrize("H, Kh, page, before, new", CASES)
def test_attention_of_turns(H, Kh, page, before, new, splits):
    from test_gpu_kernels import attention_case, run_attention
    sk, sv, qs = attention_case(np.random.default_rng(H * page + splits), H, Kh, 128, before, new, "bfloat16")
    run = lambda f: run_attention(f, sk, sv, qs, before, new, H, Kh, 128, "bfloat16", np.random.default_rng(1), page=page)
    got, ref = run(fn(before, new, lib.PREFILL_TURNS, splits))
    np.testing.assert_allclose(got, ref, atol=1e-2 * np.abs(ref).max())
    other, _ = run(fn(before, new, 1, splits))
    # (weights are rounded to 16 bits around the running maximum of 64 keys here, of 32 there)
    np.testing.assert_allclose(got, other, atol=2.0 ** -7 * np.abs(ref).max())


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
def test_attention_of_turns_refuses_what_it_is_not_built_for():
    from test_gpu_kernels import attention_case, run_attention
    for hs, page, before, new, window in ((64, 64, [0], [70], 0), (128, 96, [0], [70], 0), (128, 64, [0], [70], 20), (128, 64, [0] * 65, [2] * 65, 0)):
        sk, sv, qs = attention_case(np.random.default_rng(4), 4, 2, hs, before, new, "bfloat16")
        with pytest.raises(lib.KernelError):
            run_attention(fn(before, new, lib.PREFILL_TURNS), sk, sv, qs, before, new, 4, 2, hs, "bfloat16", np.random.default_rng(1), page=page,
                          window=window)
