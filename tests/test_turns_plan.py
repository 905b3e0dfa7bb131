"""Rules that choose a prompt step's kernels (the plan of the tiled products over whole steps of 64 columns, the splits of its attention):
plain arithmetic on the host, at sizes they were measured at."""
from gpullama3_java_amd.csrc import lib


def test_plans_of_products_into_the_residual_rows():
    plan = lib.turns_plan
    # the large tile where its blocks fill the chip; K in slices where they do not
    assert plan(8192, 4096, 14336) == (2, 1) and plan(8192, 2048, 2048) == (2, 1)
    assert plan(2048, 4096, 14336) == (2, 2) and plan(2221, 2048, 8192) == (2, 3)
    # 128 rows x 256: one round where the large tile leaves half of the chip idle
    assert plan(2048, 3072, 3072) == (5, 1) and plan(4096, 2048, 2048) == (5, 1) and plan(2048, 4096, 4096) == (5, 1)
    # 128 x 128 where those would, whole or, for few rows, in slices
    assert plan(2048, 2048, 8192) in ((1, 1), (5, 2)) and plan(2048, 2048, 2048) == (1, 1) and plan(512, 3072, 8192) == (1, 2)
    assert plan(100, 2048, 8192) == (1, 8) and plan(150, 4096, 14336) == (1, 4)
    assert lib.turns_planned(2048, 8192) and not lib.turns_planned(2048, 8200) and not lib.turns_planned(1024, 8192)
    for M in range(65, 9000, 433):
        for N, K in ((2048, 8192), (3072, 3072), (4096, 14336), (1000, 576), (3072, 256), (16, 64)):
            shape, slices = plan(M, N, K)
            assert shape in (1, 2, 5) and 1 <= slices <= 8 and (slices == 1 or K // slices >= 512)


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
