"""Rules that choose a prompt step's kernels (the plan of the tiled products into the residual rows, the splits of its attention):
plain arithmetic on the host, at sizes they were measured at."""
import pytest
import torch

from gpullama3_java_amd.csrc import lib


def test_plans_of_products_into_the_residual_rows_keep_their_slices(monkeypatch):
    """Which kernel a product runs on has no say in its sums: K in the slices of ``mfma_plan``, no chain of 32-bit sums is longer.
    The tile is that kernel's choice, for narrow products too (-tile: ``mfma_plan``'s, which is for two blocks a CU, on the kernel
    without turns only)."""
    from types import SimpleNamespace

    from gpullama3_java_amd.parts import ops
    got = []
    monkeypatch.setattr(lib, "gemm_mfma_fits", lambda *a: True)
    for rule in ("gemm_skinny_wide_fits", "gemm_skinny_fits"):
        monkeypatch.setattr(lib, rule, lambda *a: False)
    monkeypatch.setattr(lib, "gemm_mfma", lambda a, w, out, epilogue, more_slices=None, shape=0, **kw:
                        got.append((shape, 1 if more_slices is None else more_slices.shape[0] + 1)))
    for M in (65, 100, 150, 300, 512, 700, 1000, 2048, 3000, 4096, 5886, 8192):
        for N, Kd in ((2048, 2048), (2048, 8192), (3072, 3072), (3072, 8192), (4096, 4096), (4096, 14336), (2048, 8200), (512, 4096), (1024, 8192), (1536, 8960)):
            a, w = (torch.empty((n, Kd), dtype=torch.bfloat16, device="meta") for n in (M, N))
            ctx = SimpleNamespace(fuse=True, pending=None, ssq=None, normed=None, replayed=False, disabled=frozenset(),
                                  buffer=lambda name, shape, dtype: torch.empty(shape, dtype=dtype, device="meta"))
            ops.linear(a, w, torch.empty((M, N), device="meta"), lib.EPI_ADD, ctx)
            shape, slices = lib.mfma_plan(M, N, Kd)
            assert got.pop() == (-shape, slices)


def test_splits_of_a_prompt_step_s_attention():
    s = lib.prefill_splits
    assert s(32, 1, 512, [4000], 4512) == 4 and s(24, 1, 512, [4000], 4512) == 6 and s(32, 1, 64, [4000], 4064) == 8
    assert s(24, 1, 2048, [12000], 14048) == 2 and s(32, 1, 2048, [12000], 14048) == 1          # 384 and 512 blocks
    assert s(32, 1, 512, [512], 1024) == 4 and s(32, 1, 40, [2000], 2040) == 7                 # 256 keys a split
    assert s(24, 1, 1024, [0], 1024) == 1 and s(24, 1, 1024, [1000], 2024) == 1 and s(32, 1, 64, [500], 564) == 1
    assert s(32, 3, 100, [2000, 0, 3000], 3100) == 1 and s(32, 3, 100, [2000, 100, 3000], 3100) == 6 and s(32, 1, 64, None, 4064) == 1
    for heads in (1, 24, 32, 128, 511):
        for n_seqs in (1, 2, 7):
            for T in (1, 128, 129, 1000, 5000):
                n = s(heads, n_seqs, T, [T] * n_seqs, 100000)
                assert 1 <= n <= 8 and (n == 1 or n * n_seqs * T * heads <= lib.PREFILL_SPLIT_ROWS)


@pytest.mark.parametrize("head_dim", [16, 128])
def test_a_prompt_step_runs_without_splits_where_their_buffers_have_no_room(monkeypatch, head_dim):
    """A portion behind a long context asks for buffers that it can do without: on a full device it runs as it would without them."""
    from types import SimpleNamespace

    from gpullama3_java_amd.engine.context import StepContext, Workspace
    from gpullama3_java_amd.parts import ops

    engine = SimpleNamespace(cache=None, dtype=torch.bfloat16, device=torch.device("cpu"), workspace=Workspace("cpu"))
    ctx = StepContext(engine, 300, 1, [300], [4000], [0], False, 300, 4300)
    calls, asked, room = [], [], [0]
    empty = torch.empty

    def small_device(n, **kw):
        asked.append(n)
        if n > room[0]:
            raise torch.cuda.OutOfMemoryError("no room")
        room[0] -= n
        return empty(n, **kw)
    monkeypatch.setattr(ops, "attention_kernel", lambda *a: "prefill")
    monkeypatch.setattr(lib, "attention_prefill", lambda *a, **kw: calls.append(kw.get("splits", 1) if "wide_from" not in kw else None))
    q, cache = torch.zeros(300, 64), torch.zeros(1, 1, 64, head_dim)

    def steps():
        with monkeypatch.context() as m:
            m.setattr(torch, "empty", small_device)
            for _ in range(2):
                ops.attention(ctx, q, cache, cache, None, q, 32, 8, head_dim, None, 0.25)
    small, large = lib.PREFILL_SPLIT_ROWS * 2, lib.PREFILL_SPLIT_ROWS * head_dim
    for total, held in ((0, 0), (small, small), (large, small), (large + small - 1, small), (large + small, large + small)):
        room[0] = total
        engine.workspace = Workspace("cpu")
        calls.clear(), asked.clear()
        steps()
        splits = lib.prefill_splits(32, 1, 300, [4000], 4300) if held > small else 1
        assert calls == [splits] * 2 and (splits > 1) == (held > small)
        assert len(asked) == len(set(asked))                                                   # (each buffer asked for once)
        assert sum(t.numel() for t in engine.workspace._flat.values()) == held                 # (what is of no use is not kept)


def test_two_tiles_of_a_32_bit_product_over_very_many_rows_of_weights():
    """No single row of large tiles there: the weights are read twice, and the smaller tile alone takes less time."""
    def rows_of_large_tiles(M, N, gated=0):
        return lib.library().gl3_f32_stream_two(M, N, gated) // 64
    assert [rows_of_large_tiles(M, 128256) for M in (70, 82, 96)] == [0] * 3 and rows_of_large_tiles(73, 65536) == rows_of_large_tiles(77, 65536, 1) == 0
    assert rows_of_large_tiles(210, 128256) == 3 and rows_of_large_tiles(288, 65536) == 2
    assert rows_of_large_tiles(67, 32768) == 1 and rows_of_large_tiles(77, 14336, 1) == 1 and rows_of_large_tiles(513, 2048) == 8


def test_two_tiles_of_a_product_over_very_many_rows_of_weights():
    """Few rows of the operand: one tile, whose blocks read the weights once; many, or fewer rows of weights: two where the last round is mostly empty."""
    def two(M, N, K, gated=0):
        return lib.library().gl3_turns_shape(M, N, K, 1, gated) > 8
    for N, K, gated in ((128256, 2048, 0), (128256, 4096, 0), (65536, 2048, 0), (32768, 4096, 1), (256000, 1024, 0)):
        assert not any(two(M, N, K, gated) for M in range(66, 1025))
    assert two(1030, 151936, 1024) and two(600, 32768, 4096) and two(2221, 8192, 2048, 1) and two(5886, 3072, 3072)
