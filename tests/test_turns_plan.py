"""The plan of the tiled products over whole steps of 64 columns: plain arithmetic on the host, at sizes it was measured at."""
from gpullama3_java_amd.csrc import lib


def test_plans_of_products_into_the_residual_rows():
    plan = lib.turns_plan
    # the large tile where its blocks fill the chip; K in slices where they do not
    assert plan(8192, 4096, 14336) == (2, 1) and plan(8192, 2048, 2048) == (2, 1)
    assert plan(2048, 4096, 14336) == (2, 2) and plan(2221, 2048, 8192) == (2, 3)
    # 128 rows a tile: one round where the large tile leaves half of the chip idle, and few rows in slices
    assert plan(2048, 3072, 3072) == (5, 1) and plan(4096, 2048, 2048) == (5, 1)
    assert plan(2048, 2048, 8192) == (5, 2) and plan(512, 3072, 8192) in ((5, 4), (5, 5)) and plan(300, 2048, 8192) == (5, 8)
    assert lib.turns_planned(2048, 8192) and not lib.turns_planned(2048, 8200) and not lib.turns_planned(1024, 8192)
    for M in range(65, 9000, 433):
        for N, K in ((2048, 8192), (3072, 3072), (4096, 14336), (1000, 576), (3072, 256), (16, 64)):
            shape, slices = plan(M, N, K)
            assert shape in (2, 5) and 1 <= slices <= 8 and (slices == 1 or K // slices >= 512)
