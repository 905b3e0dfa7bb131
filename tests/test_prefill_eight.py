"""The prefill attention of eight waves (heads of 64 and 128): its results against the plain reference and the kernel of 128 queries a block."""
import numpy as np
import pytest

from gpullama3_java_amd.csrc import lib
from test_prefill_turns import fn, rounding


def test_which_calls_take_it():
    def choice(lengths, heads=32, n_kv=8, hs=64, page=64, plain=1):
        return lib.library().gl3_prefill_eight(hs, page, heads, n_kv, len(lengths), max(lengths), sum(lengths), plain)
    assert choice([2048]) == 3 and choice([37]) == 3 and choice([317, 1203, 701]) == 3 and choice([4096]) == 3 and choice([8192]) == 4
    assert choice([512] * 8) == 4 and choice([83] * 64) == 4 and choice([8192], 16, 16) == 3 and choice([200] * 16, 24) == 0
    assert choice([32]) == 0 and choice([2048], page=96) == 0 and choice([2048], plain=0) == 0 and choice([2048], hs=96) == 0
    large = dict(heads=24, hs=128)
    assert choice([2048], **large) == 3 and choice([333], **large) == 3 and choice([256], **large) == 0 and choice([3000], **large) == 0
    assert choice([1203, 317, 701], **large) == 3 and choice([512] * 8, **large) == 0 and choice([2048], hs=128) == 0
    assert choice([512] * 8, hs=128) == 4 and choice([1000] * 4, hs=128) == 4 and choice([256] * 32, hs=128) == 0 and choice([8192], hs=128) == 0


def test_sequences_of_unequal_lengths_and_last_blocks_that_are_partly_empty():
    """Not the form that takes longer than the kernel beside it: two heads a block where one sequence's way is what the step waits for, rounds of few blocks."""
    def choice(lengths, heads=32, n_kv=8, hs=64):
        return lib.library().gl3_prefill_eight(hs, 64, heads, n_kv, len(lengths), max(lengths), sum(lengths), 1)
    # two heads a block where the step is several times its longest sequence
    assert choice([1300] + [100] * 20) == 3 and choice([2000] + [800] * 5) == 3 and choice([1000] * 8) == 4 and choice([300] * 6) == 4 and choice([40] * 32) == 4
    assert choice([1000] * 4) == 3 and choice([600] + [200] * 40) == 4 and choice([300] * 10 + [80] * 10, 16) == 0
    # no pairs of heads
    assert choice([300] * 8, 24) == 0 and choice([300] * 12, 16, 16) == 0 and choice([384] * 12, 24) == 0 and choice([1000] * 6, 24) == 3
    assert choice([1300] + [100] * 20, 24) == 3 and choice([1469] * 8, 24) == 3
    large = dict(hs=128)
    assert choice([2000], **large) == choice([2048], **large) == 0 and choice([1900], **large) == 3 and choice([650], 64, **large) == 0 and choice([640], 64, **large) == 3
    assert choice([3502, 20, 20, 20], 16, **large) == 3 and choice([700, 200, 200, 200], **large) == 3 and choice([512] * 16, **large) == 0
    assert choice([840, 808, 583, 140, 802, 45, 398, 400], **large) == 0 and choice([1641] + [500] * 23, **large) == 0
    assert choice([427] * 8, **large) == 0 and choice([822, 600, 300, 202], **large) == 4 and choice([427] * 8, 64, **large) == 4


def test_splits_on_the_faster_of_two_kernels():
    def s(heads, n_seqs, T, before, hs=128):
        return lib.eight_splits(lib.prefill_splits(heads, n_seqs, T, [before] * n_seqs, T + before), heads, n_seqs, T, T + before, hs)
    assert s(24, 1, 1300, 1500) == 0 and s(24, 1, 900, 1024) == 0 and s(24, 1, 300, 1500) == 0 and s(24, 1, 1300, 12000) == 3
    assert s(24, 1, 512, 512) == 2 and s(24, 1, 512, 3584) == 5 and s(24, 1, 447, 4096) == 5 and s(32, 1, 64, 4000) == 8 and s(32, 1, 1000, 3000) == 1
    assert s(24, 1, 1300, 1500, 64) == lib.prefill_splits(24, 1, 1300, [1500], 2800, eight=64) > 0


def test_splits_of_its_blocks():
    def s(heads, n_seqs, T, before, hs=64):
        return lib.prefill_splits(heads, n_seqs, T, [before] * n_seqs, T + before, eight=hs)
    assert s(32, 1, 64, 4000) == 8 and s(32, 1, 150, 3000) == 4 and s(32, 1, 512, 1024) == 2 and s(32, 1, 512, 4096) == 2
    assert s(32, 1, 1000, 6000) == 1 and s(32, 3, 300, 1000) == 1 and s(32, 1, 512, 500) == 1 and s(16, 4, 100, 2000) == 4
    assert s(24, 1, 512, 2048, 128) == 5 and s(24, 1, 512, 512, 128) == 2
    for heads in (1, 2, 24, 32, 128, 511):
        for n_seqs in (1, 2, 7):
            for T in (1, 128, 129, 1000, 5000):
                for hs in (64, 128):
                    n = s(heads, n_seqs, T, 100000, hs)
                    assert 1 <= n <= 8 and (n == 1 or n * n_seqs * T * heads <= lib.PREFILL_SPLIT_ROWS)
                    assert 2 * n >= lib.prefill_splits(heads, n_seqs, T, [100000] * n_seqs, T + 100000)      # (a maximum a group: no fewer than on the other kernel)


@pytest.mark.parametrize("more, taken", [({}, True), (dict(head_dim=64), True), (dict(page_size=192), True), (dict(page_size=96), False), (dict(head_dim=96), False),
                                         (dict(window=100), False), (dict(chunk=64), False), (dict(sink=0.5), False), (dict(n_v_heads=1), False), (dict(at=4), False)])
def test_its_splits_are_for_its_calls_alone(monkeypatch, more, taken):
    """``eight_splits`` stands in for ``splits`` where the kernel of eight waves can run: not with another mask, other sizes, or caches between 16-byte addresses."""
    from types import SimpleNamespace

    import torch
    given = []
    calls = SimpleNamespace(gl3_attention_prefill=lambda *a: given.append((a[-5], a[19])) or 0)
    for name, stand_in in (("_dev", lambda *a, **kw: None), ("_ptr", lambda t: None), ("_stream", lambda: None), ("library", lambda: calls)):
        monkeypatch.setattr(lib, name, stand_in)
    kw = dict(head_dim=128, page_size=64, window=None, at=0) | more
    hs, page, window, at = (kw.pop(name) for name in ("head_dim", "page_size", "window", "at"))

    def cache(heads, *tile):
        return torch.empty(heads * hs * page + 8, dtype=torch.bfloat16)[at:at + heads * hs * page].view(1, heads, *tile)
    q, out = torch.zeros(3, 2 * hs), torch.zeros(3, 2 * hs)
    i32 = torch.zeros(2, dtype=torch.int32)
    for n, call in ((0, (3, 1)), (1, (1, lib.PREFILL_KEYS)), (2, (2, 0))):
        lib.attention_prefill(q, cache(2, page, hs), cache(kw.get("n_v_heads", 2), hs, page), i32, i32[:1], i32.view(2, 1), out, 3, 2, 2, hs, page, window, 0.1,
                              splits=3, part_o=torch.zeros(18 * hs), part_ml=torch.zeros(36), eight_splits=n, **kw)
        assert given.pop() == (call if taken else (3, 0))


# (no splits at all, where the other kernel has two; fewer; the other kernel's; not its sizes: none of its own)
@pytest.mark.parametrize("heads, hs, page, T, before, eight", [(32, 64, 64, 1000, 6000, 1), (24, 128, 128, 512, 3584, 5), (32, 64, 64, 150, 3000, 4), (24, 128, 64, 1300, 1500, 0), (32, 64, 96, 512, 512, None),
                                                               (32, 96, 64, 512, 512, None)])
def test_a_layer_asks_for_its_splits(monkeypatch, heads, hs, page, T, before, eight):
    from types import SimpleNamespace

    import torch

    from gpullama3_java_amd.parts import ops
    walks = []

    class Contexts(list):
        def __iter__(self):
            walks.append(1)
            return super().__iter__()
    ctx = SimpleNamespace(n_seqs=1, max_q_len=T, max_kv_len=T + before, kv_before_host=Contexts([before]), cu_seqlens=None, kv_before=None,
                          buffer_if_room=lambda name, shape, dtype: torch.empty(shape, dtype=dtype, device="meta"))
    calls = []
    monkeypatch.setattr(ops, "attention_kernel", lambda *a: "prefill")
    monkeypatch.setattr(lib, "attention_prefill", lambda *a, **kw: calls.append((kw["splits"], kw.get("eight_splits"))))
    ops.attention(ctx, torch.zeros(1), torch.zeros(1, 8, page, hs), None, None, None, heads, 8, hs, None, 0.1)
    assert calls == [(lib.prefill_splits(heads, 1, T, [before], T + before), eight)] and len(walks) == 1
    assert eight in (0, None, lib.prefill_splits(heads, 1, T, [before], T + before, eight=hs))


# one, two, three and four heads a kv head; waves, blocks and chunks with one row and all but one, one chunk (none for the second group); sequences that start no
# block of the longest one's kind; more chunks than a register holds places of (64), twice as many
CASES = [(4, 2, 64, [0, 70, 0, 130, 5], [33, 1, 200, 17, 64]), (3, 1, 64, [0, 0, 0], [256, 257, 31]), (8, 2, 128, [63, 64, 65], [129, 128, 127]),
         (6, 2, 192, [4200, 0], [3, 300]), (2, 1, 64, [8200], [70]), (8, 8, 64, [1] * 64, list(range(1, 65))), (32, 8, 64, [0], [700])]


@pytest.mark.gpu
@pytest.mark.parametrize("sharp", [1, 8])
@pytest.mark.parametrize("hs", [64, 128])
@pytest.mark.parametrize("H, Kh, page, before, new", CASES)
def test_attention_of_eight_waves(H, Kh, page, before, new, hs, sharp):
    from test_gpu_kernels import attention_case, run_attention
    sk, sv, qs = attention_case(np.random.default_rng(H * page + sharp), H, Kh, hs, before, new, "bfloat16")
    qs = [q * sharp for q in qs]                     # (8: a few keys have all the weight, and maxima move in all chunks)
    run = lambda f: run_attention(f, sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1), page=page)
    got, ref = run(fn(before, new, lib.PREFILL_KEYS))
    assert float((np.abs(got - ref) / rounding(qs, sk, sv, ref, before, new)).max()) <= 1
    np.testing.assert_array_equal(got, run(fn(before, new, lib.PREFILL_KEYS, shuffled_rows=True))[0])
    if H // Kh % 2 == 0:
        got, _ = run(fn(before, new, lib.PREFILL_HEADS))
        np.testing.assert_array_equal(got, run(fn(before, new, 1))[0])      # (the same sums in the same order as the kernel of 128 queries a block)
        np.testing.assert_array_equal(got, run(fn(before, new, lib.PREFILL_HEADS, shuffled_rows=True))[0])


@pytest.mark.gpu
@pytest.mark.parametrize("hs", [64, 128])
def test_scores_that_are_not_numbers_are_in_the_rows_that_see_them(hs):
    from test_gpu_kernels import attention_case, run_attention
    H, Kh, before, new = 4, 2, [700], [300]
    sk, sv, qs = attention_case(np.random.default_rng(3), H, Kh, hs, before, new, "bfloat16")
    for mode in (lib.PREFILL_KEYS, lib.PREFILL_HEADS):
        run = lambda k: run_attention(fn(before, new, mode), k, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1))[0]
        clean = run(sk)
        for lo, hi in ((900, 930), (768, 832), (0, 64)):      # (a part of a chunk, all of an even one, all of the first)
            k = [s.copy() for s in sk]
            k[0][lo:hi, 1] = np.nan
            got = run(k)
            first = max(0, lo - 700)
            assert np.isnan(got[first:, 2:]).all()
            np.testing.assert_array_equal(got[:first], clean[:first])
            np.testing.assert_array_equal(got[:, :2], clean[:, :2])


@pytest.mark.gpu
@pytest.mark.parametrize("hs", [64, 128])
@pytest.mark.parametrize("at", [0, 31, 32, 63, 64, 95, 127, 1000, 1023, 1024, 1037, 1038, 1055, 1060])
def test_values_that_are_not_finite_reach_as_far_as_in_the_kernel_of_128_queries(at, hs):
    """An infinite value or a NaN spoils the queries that share their 64 keys with it (heads of 64; of 128: 32 keys), in front of it or behind the sequence's end
    (here from 1,038 on), and no others; on two groups of keys both that hold it and that do not."""
    from test_gpu_kernels import attention_case, run_attention
    H, Kh, before, new = 4, 2, [700], [338]
    sk, sv, qs = attention_case(np.random.default_rng(at), H, Kh, hs, before, [400], "bfloat16")
    keys = 64 if hs == 64 else 32
    positions = np.arange(700, 1038)
    last = np.minimum((positions - 700 >> 5) * 32 + 731, 1037)       # (32 queries walk their keys together)
    for value in (np.inf, np.nan):
        sv[0][at, 0, 57] = value
        run = lambda f: run_attention(f, sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1))[0]
        by_heads, by_keys = run(fn(before, new, lib.PREFILL_HEADS)), run(fn(before, new, lib.PREFILL_KEYS))
        np.testing.assert_array_equal(by_heads, run(fn(before, new, 1)))
        for got in (by_heads, by_keys):
            assert np.isfinite(got[last // keys < at // keys]).all() and np.isfinite(got[:, :, :57]).all() and np.isfinite(got[:, 2:]).all()
            assert not np.isfinite(got[positions >= at, :2, 57]).any()


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [lib.PREFILL_KEYS, lib.PREFILL_HEADS])
@pytest.mark.parametrize("beside", [1, 3])
def test_short_sequences_beside_a_long_one_do_not_make_it_longer(beside, mode):
    """Blocks that leave at once, of sequences that are over, do not send the others to half of the chip (with three short ones that was 1.5 and 2.0 times the
    time of the long one alone, whose blocks are paired otherwise: 1.0 and less since)."""
    import torch
    H, Kh, hs, long = 16, 8, 128, 3502

    def least(new):
        T, pages = sum(new), [-(-n // 64) for n in new]
        q, out = torch.randn(T, H * hs, device="cuda").bfloat16(), torch.empty(T, H * hs, dtype=torch.bfloat16, device="cuda")
        kc, vc = (torch.randn(sum(pages), Kh, *size, device="cuda").bfloat16() for size in ((64, hs), (hs, 64)))
        table = torch.zeros(len(new), max(pages), dtype=torch.int32)
        for b, n in enumerate(pages):
            table[b, :n] = torch.arange(n) + sum(pages[:b])
        i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
        cu, held, table = i32([sum(new[:b]) for b in range(len(new) + 1)]), i32([0] * len(new)), table.cuda()
        times = []
        for _ in range(12):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(8):
                lib.attention_prefill(q, kc, vc, cu, held, table, out, max(new), H, Kh, hs, 64, None, 0.1, wide_from=mode)
            end.record()
            torch.cuda.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)
    assert least([long] + [17] * beside) < 1.25 * least([long])


@pytest.mark.gpu
def test_it_refuses_what_it_is_not_built_for():
    from test_gpu_kernels import K, attention_case, run_attention
    before, new = [0], [40]
    for H, Kh, hs, page, mode in ((3, 1, 64, 64, lib.PREFILL_HEADS), (2, 1, 32, 64, lib.PREFILL_KEYS), (2, 1, 64, 96, lib.PREFILL_KEYS)):
        sk, sv, qs = attention_case(np.random.default_rng(3), H, Kh, hs, before, new, "bfloat16")
        with pytest.raises(K().KernelError, match="eight waves"):
            run_attention(fn(before, new, mode), sk, sv, qs, before, new, H, Kh, hs, "bfloat16", np.random.default_rng(1), page=page)
