"""Products of 49 to 64 rows over a weight in one of its copies' orders, whose rows of ``a`` go from memory straight into shared memory, the weight's two pairs of
k-steps ahead: the sums of the kernel for stored rows, and nothing but the call's own rows and columns read."""
import numpy as np
import pytest
import torch

from gpullama3_java_amd.csrc import lib

pytestmark = pytest.mark.gpu


def rows_among_nans(M, Kd, gen):
    whole = torch.full((M + 2, Kd + 64), float("nan"), dtype=torch.bfloat16, device="cuda")
    a = whole[1:M + 1, 32:Kd + 32]
    a.copy_(torch.randn(M, Kd, generator=gen, device="cuda"))
    return a


# one pair of k-steps for one wave of eight; a pair for all but one and for one more than eight; an odd number for each; slices that share them unevenly, the last with none
@pytest.mark.parametrize("Kd, slices", [(64, 1), (448, 1), (576, 1), (576, 4), (1088, 7), (1536, 1), (2048, 4), (8192, 4)])
@pytest.mark.parametrize("M", [49, 57, 64])
def test_rows_two_pairs_ahead(M, Kd, slices):
    gen = torch.Generator(device="cuda").manual_seed(M * Kd + slices)
    a = rows_among_nans(M, Kd, gen)
    for N in (48, 2048, 6160):
        w = torch.randn(N, Kd, generator=gen, device="cuda").bfloat16()
        w16, w8 = w.clone(), w.clone()
        w16.tiled, w8.tiled8 = lib.tile_weight(w16), lib.tile_weight8(w8)
        exact, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
        was = torch.randn(M, N, generator=gen, device="cuda")
        for strips in (2, 4):
            def run(weight, epilogue, dtype):
                # (a wider matrix, in front of a further row)
                out = torch.full((slices, M + 1, N + 4), -7.0, dtype=dtype, device="cuda")
                got = out[:, :M, :N] if slices > 1 else out[0, :M, :N]
                if epilogue == lib.EPI_ADD:
                    got.copy_(was)
                lib.gemm_skinny_wide(a, weight, got, epilogue, strips=strips)
                assert torch.all(out[:, M:] == -7.0) and torch.all(out[:, :, N:] == -7.0)
                return got
            calls = [(lib.EPI_STORE, torch.float32)] + [(lib.EPI_STORE, torch.bfloat16), (lib.EPI_ADD, torch.float32)] * (slices == 1)
            for epilogue, dtype in calls:
                got = run(lib.hold_once(w16), epilogue, dtype)
                assert torch.equal(got, run(w, epilogue, dtype)), (N, strips, epilogue, dtype)
                # (strips of 8: the pairs are other waves', so sums in another order: each of Kd + 8 + slices additions rounds by half a unit)
                total = (run(lib.hold_once(w8), epilogue, dtype).double().sum(0) if slices > 1 else run(lib.hold_once(w8), epilogue, dtype).double())
                want = exact + was.double() if epilogue == lib.EPI_ADD else exact
                bound = (Kd + 8 + slices) * 2.0 ** -24 * (size + was.double().abs()) + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
                assert bool(((total - want).abs() <= bound).all()), (N, strips, epilogue, dtype)


@pytest.mark.parametrize("H, Kh, hs, Kd", [(32, 8, 64, 2048), (24, 8, 128, 320), (4, 2, 16, 64)])
def test_queries_keys_and_values_two_pairs_ahead(H, Kh, hs, Kd):
    M, page = 61, 64
    gen = torch.Generator(device="cuda").manual_seed(H * Kd)
    a = rows_among_nans(M, Kd, gen)
    w = torch.randn((H + 2 * Kh) * hs, Kd, generator=gen, device="cuda").bfloat16() / Kd ** 0.5
    copy = w.clone()
    copy.tiled = lib.tile_weight(copy, qkv=(H, Kh, hs, True, False))
    positions = torch.arange(M, dtype=torch.int32, device="cuda") * 3 % 128
    rows = torch.arange(M, dtype=torch.int32, device="cuda")
    table = torch.randperm(2 * M, generator=torch.Generator().manual_seed(1)).view(M, 2).int().cuda()
    angle = torch.rand(128, hs // 2, generator=gen, device="cuda") * 6.3
    got = []
    for weight in (w, lib.hold_once(copy)):
        q = torch.zeros(M, H * hs, dtype=torch.bfloat16, device="cuda")
        k, v = (torch.zeros(2 * M, Kh, *size, dtype=torch.bfloat16, device="cuda") for size in ((page, hs), (hs, page)))
        lib.qkv_rope_cache(a, None, 0, 0.0, weight, q, positions, rows, table, angle.cos(), angle.sin(), k, v, H, Kh, hs, False, page)
        got.append((q, k, v))
    for one, other in zip(*got):
        assert torch.equal(one, other) and not torch.isnan(one).any() and one.any()
