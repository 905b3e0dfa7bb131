"""The prefill attention with a block's keys shared out over several blocks: against the plain reference and the unsplit kernel."""
import numpy as np
import pytest
import torch

from test_gpu_kernels import DEV, K, attention_case, dev, run_attention

pytestmark = pytest.mark.gpu


def fn(lens_before, new, splits):
    lib = K()

    def call(q, kc, vc, positions, seq_of, table, out, H, Kh, hs, page, window, scale):
        cu = dev(np.concatenate([[0], np.cumsum(new)]), torch.int32)
        n = splits * len(positions) * H
        part_o, part_ml = torch.full((n * hs,), float("nan"), device=DEV), torch.full((2 * n,), float("nan"), device=DEV)
        lib.attention_prefill(q, kc, vc, cu, dev(lens_before, torch.int32), table, out, max(new), H, Kh, hs, page, window, scale,
                              wide_from=1, **(dict(splits=splits, part_o=part_o, part_ml=part_ml) if splits > 1 else {}))
    return call


# contexts of fewer chunks than splits, of one page, long ones; last blocks of one query and of 128
@pytest.mark.parametrize("splits", [2, 3, 8])
@pytest.mark.parametrize("H, Kh, hs, page", [(4, 2, 32, 64), (6, 2, 64, 64), (2, 1, 64, 96), (5, 5, 96, 32), (3, 1, 128, 64),
                                             (3, 1, 128, 32), (4, 2, 128, 96)])
def test_split_prefill_attention(H, Kh, hs, page, splits):
    rng = np.random.default_rng(H * hs + splits)
    before, new = [700, 0, 129, 1300, 31], [40, 3, 129, 1, 256]
    sk, sv, qs = attention_case(rng, H, Kh, hs, before, new, "bfloat16")
    got, ref = run_attention(fn(before, new, splits), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1), page=page)
    np.testing.assert_allclose(got, ref, atol=1e-2 * np.abs(ref).max())
    whole, _ = run_attention(fn(before, new, 1), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1), page=page)
    np.testing.assert_allclose(got, whole, atol=2.0 ** -7 * np.abs(ref).max())       # (weights are rounded to 16 bits around another maximum)


# pages of 64: as many splits as the second number says, two groups on the keys for 1, the kernel of 128 queries for 0; of 96, and caches between 16-byte addresses: as the first says
@pytest.mark.parametrize("hs, page, shift, taken", [(64, 64, 0, True), (128, 64, 0, True), (128, 96, 0, False), (64, 64, 4, False)])
@pytest.mark.parametrize("eight", [0, 1, 2, 5])
def test_a_number_of_splits_for_the_kernel_of_eight_waves(hs, page, shift, taken, eight):
    H, Kh, before, new = 4, 2, [1300], [200]
    sk, sv, qs = attention_case(np.random.default_rng(hs + eight), H, Kh, hs, before, new, "bfloat16")

    def run(**kw):
        def call(q, kc, vc, positions, seq_of, table, out, *rest):
            moved = [torch.empty(c.numel() + 8, dtype=c.dtype, device=DEV)[shift:shift + c.numel()].view(c.shape).copy_(c) for c in (kc, vc)]
            n = 5 * 200 * H
            part_o, part_ml = torch.full((n * hs,), float("nan"), device=DEV), torch.full((2 * n,), float("nan"), device=DEV)
            K().attention_prefill(q, *moved, dev([0, 200], torch.int32), dev(before, torch.int32), table, out, 200, *rest, part_o=part_o, part_ml=part_ml, **kw)
        return run_attention(call, sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1), page=page)
    got, ref = run(splits=4, eight_splits=eight)
    np.testing.assert_allclose(got, ref, atol=1e-2 * np.abs(ref).max())
    alone = dict(splits=1, wide_from=K().PREFILL_KEYS) if eight == 1 else dict(splits=4, wide_from=1) if eight == 0 else dict(splits=eight)
    np.testing.assert_array_equal(got, run(**alone)[0] if taken else run(splits=4)[0])
    assert not np.array_equal(got, run(splits=4 if taken else 3)[0])


def test_split_prefill_attention_with_one_key_that_counts_and_a_window():
    rng = np.random.default_rng(3)
    H, Kh, hs, before, new = 4, 2, 64, [1500], [70]
    sk, sv, qs = attention_case(rng, H, Kh, hs, before, new, "bfloat16")
    for at in (3, 777, 1499):                        # in the first, a middle and the last split
        k = [s.copy() for s in sk]
        k[0][at] = 0
        k[0][at, :, 5] = 40.0
        q = [s.copy() for s in qs]
        q[0][1500:, :, 5] = 8.0
        got, ref = run_attention(fn(before, new, 4), k, sv, q, before, new, H, Kh, hs, "bfloat16", rng)
        np.testing.assert_allclose(got, ref, atol=1e-2 * np.abs(ref).max())
        np.testing.assert_allclose(got[:, 0], np.broadcast_to(sv[0][at, 0], got[:, 0].shape), atol=0.05)
    got, ref = run_attention(fn(before, new, 4), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", rng, window=100)
    np.testing.assert_allclose(got, ref, atol=1e-2 * np.abs(ref).max())


# 1,570 keys are 25 chunks of 64 in 4 splits: all of the second split's, part of it, the last two splits' keys that a row sees
@pytest.mark.parametrize("lo, hi", [(384, 768), (400, 402), (768, 1500)])
def test_split_prefill_attention_keeps_nan_scores(lo, hi):
    """Scores that are not numbers are in the result of every row that sees them, also where all of a split's scores are."""
    rng = np.random.default_rng(6)
    H, Kh, hs, before, new = 4, 2, 64, [1500], [70]
    sk, sv, qs = attention_case(rng, H, Kh, hs, before, new, "bfloat16")
    clean, _ = run_attention(fn(before, new, 4), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1))
    sk[0][lo:hi, 1] = np.nan
    got, _ = run_attention(fn(before, new, 4), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1))
    assert np.isnan(got[:, 2:]).all()
    np.testing.assert_array_equal(got[:, :2], clean[:, :2])


def test_split_prefill_attention_refuses_what_it_is_not_built_for():
    lib = K()
    rng = np.random.default_rng(4)
    H, Kh, hs, before, new = 4, 2, 64, [300], [70]
    sk, sv, qs = attention_case(rng, H, Kh, hs, before, new, "bfloat16")

    def bad(**kw):
        def call(q, kc, vc, positions, seq_of, table, out, *rest):
            cu = dev([0, 70], torch.int32)
            n = 70 * H
            arguments = dict(splits=2, part_o=torch.zeros(2 * n * hs, device=DEV), part_ml=torch.zeros(4 * n, device=DEV))
            arguments.update(kw)
            lib.attention_prefill(q, kc, vc, cu, dev(before, torch.int32), table, out, 70, *rest, **arguments)
        return call
    for kw in (dict(sink=0.5), dict(slopes=torch.zeros(H, device=DEV)), dict(splits=9), dict(part_o=torch.zeros(8, device=DEV)), dict(part_ml=None)):
        with pytest.raises((lib.KernelError, AttributeError)):
            run_attention(bad(**kw), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", rng)
