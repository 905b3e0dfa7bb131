"""The 32-bit products and attention on the matrix cores at the edges of their tiles: against a plain reference, against the kernels for any sizes,
and a row alone against the same row in company."""
import numpy as np
import pytest
import torch

from test_gpu_kernels import K, attention_case, dev, run_attention

pytestmark = pytest.mark.gpu


def bound(a, w, K_):
    """What 32-bit sums may be off by: each sum is a chain of at most 256 products behind one of K / 256 partial sums, and
    every link rounds to 2^-24 of at most the sum of magnitudes."""
    return (256 + K_ / 256 + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T)


# rows of one tile and one more (16, 32, 64, 128), columns likewise, K in one piece of 4, up to a chunk of 256 and beyond it, pairs
# of chunks with and without a last one of its own
@pytest.mark.parametrize("M, N, Kd", [(1, 16, 4), (1, 2048, 8192), (8, 44, 4100), (7, 33, 4608), (3, 130, 72), (16, 33, 256), (17, 48, 260), (32, 257, 1028), (33, 77, 96), (48, 2048, 8192),
                                      (64, 129, 516), (65, 200, 300), (130, 513, 2052), (513, 1024, 1024), (1030, 2500, 64)])
def test_float32_products(M, N, Kd):
    lib = K()
    rng = np.random.default_rng(M * N + Kd)
    a, w = rng.standard_normal((M, Kd)).astype(np.float32), rng.standard_normal((2 * N, Kd)).astype(np.float32)
    bias, factor = rng.standard_normal(2 * N).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    A, W, B, F = dev(a), dev(w), dev(bias), dev(factor)
    both = a.astype(np.float64) @ w.astype(np.float64).T
    off = bound(a, w, Kd)
    out = torch.full((M, N + 3), -7.0, device=A.device)
    lib.gemm_generic(A, W[:N], out[:, 1:N + 1])                                    # rows of the output apart
    assert (np.abs(out[:, 1:N + 1].double().cpu().numpy() - both[:, :N]) <= off[:, :N]).all()
    assert torch.all(out[:, 0] == -7.0) and torch.all(out[:, N + 1:] == -7.0)
    res = rng.standard_normal((M, N)).astype(np.float32)
    x = dev(res)
    lib.gemm_generic(A, W[:N], x, lib.EPI_ADD, bias=B[:N], col_scale=F)
    want = res + (both[:, :N] + bias[:N]) * factor.astype(np.float64)
    slack = 4 * 2.0 ** -24 * (np.abs(res) + (np.abs(both[:, :N]) + np.abs(bias[:N])) * np.abs(factor))
    assert (np.abs(x.double().cpu().numpy() - want) <= off[:, :N] * np.abs(factor) + slack).all()
    gated = torch.empty(M, N, device=A.device)
    lib.gemm_generic(A, W, gated, lib.EPI_GATED, bias=B)
    gate, up = both[:, :N] + bias[:N], both[:, N:] + bias[N:]
    sig = 1.0 / (1.0 + np.exp(-gate))
    # (|silu'| <= 1.1; the exponential and the division are within 4 units of the last place)
    slack = (1.1 * (off[:, :N] + 2.0 ** -23 * np.abs(gate)) * (np.abs(up) + off[:, N:])
             + np.abs(gate * sig) * (off[:, N:] + 2.0 ** -23 * np.abs(up)) + 8 * 2.0 ** -24 * np.abs(gate * sig * up))
    assert (np.abs(gated.double().cpu().numpy() - gate * sig * up) <= slack + 1e-30).all()
    # a row alone, and rows that begin at any float, give the same bits
    one, shifted = torch.empty(1, N, device=A.device), torch.empty(M, Kd + 1, device=A.device)[:, 1:]
    shifted.copy_(A)
    for r in {0, M // 2, M - 1}:
        lib.gemm_generic(A[r:r + 1], W[:N], one)
        assert torch.equal(one[0], out[r, 1:N + 1])
        lib.gemm_generic(shifted[r:r + 1], W, one, lib.EPI_GATED, bias=B)
        assert torch.equal(one[0], gated[r])
    # W at an odd float: the kernel for any sizes
    odd = torch.empty(N * Kd + 1, device=A.device)[1:].view(N, Kd)
    odd.copy_(W[:N])
    general = torch.empty(M, N, device=A.device)
    lib.gemm_generic(A, odd, general)
    one_chain = (Kd + 2) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(w[:N]).astype(np.float64).T)
    assert (np.abs((general - out[:, 1:N + 1]).double().cpu().numpy()) <= off[:, :N] + one_chain).all()


# every tile that products of many rows take (2: 128 x 128, 3: 128 x 64, 4: 64 x 64, 5: 64 x 32), one row and one column beyond whole
# tiles; K of a chunk and a tail, of four chunks and a tail, of eight
@pytest.mark.parametrize("Kd", [260, 1028, 2052])
@pytest.mark.parametrize("tile, gated, M, N", [(2, False, 2049, 3585), (3, False, 1025, 3073), (4, False, 513, 3073), (5, False, 129, 257),
                                               (2, True, 1281, 4097), (3, True, 513, 3073), (4, True, 193, 3585), (5, True, 97, 65)])
def test_float32_products_in_every_tile(tile, gated, M, N, Kd):
    lib = K()
    assert lib.library().gl3_f32_shape(M, N, int(gated)) == tile
    gen = torch.Generator(device="cuda").manual_seed(M + Kd)
    A, W = (torch.randn(n, Kd, generator=gen, device="cuda") for n in (M, 2 * N if gated else N))
    res = torch.randn(M, N, generator=gen, device="cuda")
    both = A.double() @ W.double().T
    off = (256 + Kd / 256 + 2) * 2.0 ** -24 * (A.double().abs() @ W.double().abs().T)        # (as in ``bound``)
    one = torch.empty(1, N, device="cuda")
    if gated:
        out = torch.full((M, N + 1), -7.0, device="cuda")
        lib.gemm_generic(A, W, out[:, :N], lib.EPI_GATED)
        gate, up = both[:, :N], both[:, N:]
        sig = torch.sigmoid(gate)
        # (|silu'| <= 1.1; the exponential and the division are within 4 units of the last place)
        slack = (1.1 * (off[:, :N] + 2.0 ** -23 * gate.abs()) * (up.abs() + off[:, N:]) + (gate * sig).abs() * (off[:, N:] + 2.0 ** -23 * up.abs())
                 + 8 * 2.0 ** -24 * (gate * sig * up).abs())
        assert ((out[:, :N] - gate * sig * up).abs() <= slack + 1e-30).all() and torch.all(out[:, N] == -7.0)
    else:
        out, x = torch.full((M, N + 1), -7.0, device="cuda"), res.clone()
        lib.gemm_generic(A, W, out[:, :N])
        lib.gemm_generic(A, W, x, lib.EPI_ADD)
        assert ((out[:, :N] - both).abs() <= off).all() and torch.all(out[:, N] == -7.0)
        assert torch.equal(x, res + out[:, :N])
    # a row alone gives the same bits (the kernel for few rows: the same order of sums)
    for r in (0, 63, 64, M // 2, M - 2, M - 1):
        lib.gemm_generic(A[r:r + 1], W, one, lib.EPI_GATED if gated else lib.EPI_STORE)
        assert torch.equal(one[0], out[r, :N])


# every tile over whole steps of 32 k (1: 128 rows of W x 128 tokens, 2: 128 x 64, 3: 64 x 64, 4: 64 x 32, 5: 32 x 32), one row and one column
# beyond whole tiles; K of a step (fewer than are asked for ahead), of a chunk and a step, of eight chunks
@pytest.mark.parametrize("Kd", [32, 288, 2048])
@pytest.mark.parametrize("tile, gated, M, N", [(1, False, 2049, 3585), (2, False, 1025, 3585), (3, False, 513, 3073), (4, False, 513, 2049), (5, False, 65, 257),
                                               (1, True, 1153, 3073), (2, True, 513, 8193), (3, True, 769, 1025), (4, True, 17, 65), (4, True, 97, 130)])
def test_float32_products_in_every_tile_of_whole_steps(tile, gated, M, N, Kd):
    lib = K()
    assert lib.library().gl3_f32_stream_shape(M, N, int(gated)) == tile
    gen = torch.Generator(device="cuda").manual_seed(M + Kd)
    A, W = (torch.randn(n, Kd, generator=gen, device="cuda") for n in (M, 2 * N if gated else N))
    wide = torch.zeros(M + 1, Kd + 4, device="cuda")           # rows of A apart; the same rows at an odd float: the other kernel
    wide[:M, :Kd] = A
    odd = torch.empty(M * (Kd + 1) + 1, device="cuda")[1:].view(M, Kd + 1)[:, :Kd]
    odd.copy_(A)
    out, other = torch.full((M, N + 1), -7.0, device="cuda"), torch.empty(M, N, device="cuda")
    epilogue = lib.EPI_GATED if gated else lib.EPI_STORE
    lib.gemm_generic(wide[:M, :Kd], W, out[:, :N], epilogue)
    lib.gemm_generic(odd, W, other, epilogue)
    assert torch.all(out[:, N] == -7.0) and torch.equal(out[:, :N], other)       # the same sums in the same order
    if not gated:
        off = (256 + Kd / 256 + 2) * 2.0 ** -24 * (A.double().abs() @ W.double().abs().T)        # (as in ``bound``)
        assert ((out[:, :N] - A.double() @ W.double().T).abs() <= off).all()
        x = torch.randn(M, N, generator=gen, device="cuda")
        want = x + out[:, :N]
        lib.gemm_generic(A, W, x, lib.EPI_ADD)
        assert torch.equal(x, want)
    one = torch.empty(1, N, device="cuda")
    for r in (0, 15, M // 2, M - 2, M - 1):
        lib.gemm_generic(A[r:r + 1], W, one, epilogue)
        assert torch.equal(one[0], out[r, :N])


# (large and small tile, rows of large tiles) each pair of tiles that there is: one row, all but one and several tiles of them behind the large ones,
# columns beyond whole tiles; one step of K, a chunk and a step
@pytest.mark.parametrize("Kd", [32, 288])
@pytest.mark.parametrize("large, small, rows, gated, M, N", [(1, 4, 19, False, 2478, 5120), (1, 5, 19, False, 2440, 5120), (2, 4, 12, False, 816, 5120), (2, 5, 21, False, 1406, 3070),
                                                             (3, 5, 8, False, 513, 2048), (3, 5, 5, False, 333, 3071),
                                                             (1, 4, 18, True, 2305, 3584), (2, 4, 2, True, 130, 8190), (2, 4, 10, True, 671, 8192), (2, 4, 10, True, 705, 1490)])
def test_float32_products_in_two_tiles(large, small, rows, gated, M, N, Kd):
    """The same bits as the rows in smaller companies, which go by one tile each, or by none."""
    lib = K()
    code = lib.library().gl3_f32_stream_two(M, N, int(gated))
    assert (code // 8 % 8, code % 8, code // 64) == (large, small, rows)
    gen = torch.Generator(device="cuda").manual_seed(M + Kd)
    A, W = torch.randn(M, Kd + 4, generator=gen, device="cuda")[:, :Kd], torch.randn(2 * N if gated else N, Kd, generator=gen, device="cuda")
    bias = torch.randn(W.shape[0], generator=gen, device="cuda")
    for epilogue in (lib.EPI_GATED,) if gated else (lib.EPI_STORE, lib.EPI_ADD):
        out = torch.full((M, N + 1), -7.0, device="cuda")
        was = out[:, :N].clone()
        lib.gemm_generic(A, W, out[:, :N], epilogue, bias=bias)
        assert torch.all(out[:, N] == -7.0)
        for lo in range(0, M, 60):                       # (60 rows: no two tiles)
            assert lib.library().gl3_f32_stream_two(min(60, M - lo), N, int(gated)) == 0
            part = was[lo:lo + 60].clone()
            lib.gemm_generic(A[lo:lo + 60], W, part, epilogue, bias=bias)
            assert torch.equal(part, out[lo:lo + 60, :N]), (epilogue, lo)


def test_float32_products_keep_small_numbers_and_infinities():
    lib = K()
    a, w = np.zeros((20, 64), np.float32), np.zeros((32, 64), np.float32)
    a[0, 3], w[5, 3] = 2e-39, 0.5                        # below the smallest normal number
    a[1, 7], w[6, 7] = 1e-20, 3e-20
    a[2, 9], w[:, 9] = np.inf, 1.0
    out = torch.empty(20, 32, device="cuda:0")
    lib.gemm_generic(dev(a), dev(w), out)
    out = out.cpu().numpy()
    assert out[0, 5] == np.float32(1e-39) and out[1, 6] == np.float32(np.float32(1e-20) * np.float32(3e-20))
    assert np.isinf(out[2]).all() and np.isfinite(np.delete(out, 2, 0)).all()


# ------------------------------------------------------------------ attention
# heads alone and in groups (3: rows of a tile that are no whole tokens; 17: a group in two tiles), contexts of one key, of the
# edges of a step of 64 and of a wave's turn (8 steps), several sequences in a tile's tokens; enough tokens for whole tiles in the last
@pytest.mark.parametrize("H, Kh, hs, before, new", [(4, 2, 32, [0, 70, 130, 5], [33, 1, 2, 1]), (8, 2, 64, [0, 511, 0], [1, 2, 130]),
                                                    (3, 1, 96, [62, 0], [4, 63]), (2, 2, 128, [0, 600], [65, 1]), (17, 1, 64, [0, 9], [20, 3]),
                                                    (32, 8, 64, [100, 0], [200, 150])])
def test_float32_attention(H, Kh, hs, before, new):
    lib = K()
    rng = np.random.default_rng(H * hs)
    sk, sv, qs = attention_case(rng, H, Kh, hs, before, new, "float32")
    got, ref = run_attention(lib.attention_generic, sk, sv, qs, before, new, H, Kh, hs, "float32", np.random.default_rng(5))
    np.testing.assert_allclose(got, ref, atol=2e-5 * np.abs(ref).max())
    # a window that hides nothing takes the kernel for any rule
    general, _ = run_attention(lib.attention_generic, sk, sv, qs, before, new, H, Kh, hs, "float32", np.random.default_rng(5), window=1 << 20)
    np.testing.assert_allclose(got, general, atol=4e-6 * np.abs(ref).max())
    # so does a cache that does not begin at 16 bytes: the same numbers as that kernel's, bit for bit
    def shifted(q, kc, vc, *rest, **more):
        caches = [torch.empty(c.numel() + 1, device=c.device)[1:].view(c.shape).copy_(c) for c in (kc, vc)]
        lib.attention_generic(q, *caches, *rest, **more)
    apart, _ = run_attention(shifted, sk, sv, qs, before, new, H, Kh, hs, "float32", np.random.default_rng(5))
    np.testing.assert_array_equal(apart, general)
    # every token alone: the same bits
    first = 0
    for b, (n0, n) in enumerate(zip(before, new)):
        for p in sorted({0, 1, n // 2, n - 1} & set(range(n))):
            cut = [[s[b][:n0 + p + 1]] for s in (sk, sv, qs)]
            one, _ = run_attention(lib.attention_generic, *cut, [n0 + p], [1], H, Kh, hs, "float32", rng)
            np.testing.assert_array_equal(one[0], got[first + p])
        first += n


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_float32_attention_leaves_values_out_that_a_row_does_not_see(bad):
    lib = K()
    rng = np.random.default_rng(2)
    H, Kh, hs, n, at = 4, 2, 64, 150, 101
    sk, sv, qs = attention_case(rng, H, Kh, hs, [0], [n], "float32")
    clean, _ = run_attention(lib.attention_generic, sk, sv, qs, [0], [n], H, Kh, hs, "float32", np.random.default_rng(5))
    sv[0][at, 1, 7] = bad
    got, _ = run_attention(lib.attention_generic, sk, sv, qs, [0], [n], H, Kh, hs, "float32", np.random.default_rng(5))
    np.testing.assert_array_equal(got[:at], clean[:at])
    assert not np.isfinite(got[at:, 2:, 7]).any()
    got[at:, 2:, 7] = clean[at:, 2:, 7] = 0
    np.testing.assert_array_equal(got, clean)


# keys of one wave's whole turn, of part of one, of two turns (a row's other waves have finite scores)
@pytest.mark.parametrize("lo, hi", [(64, 128), (70, 72), (128, 256)])
def test_float32_attention_keeps_nan_scores(lo, hi):
    """Scores that are not numbers are in the result of every row that sees them, also where all of a wave's scores are, and in no other."""
    lib = K()
    rng = np.random.default_rng(8)
    H, Kh, hs, n = 4, 2, 64, 300
    sk, sv, qs = attention_case(rng, H, Kh, hs, [0], [n], "float32")
    clean, _ = run_attention(lib.attention_generic, sk, sv, qs, [0], [n], H, Kh, hs, "float32", np.random.default_rng(5))
    sk[0][lo:hi, 1] = np.nan
    got, _ = run_attention(lib.attention_generic, sk, sv, qs, [0], [n], H, Kh, hs, "float32", np.random.default_rng(5))
    assert np.isnan(got[lo:, 2:]).all()
    np.testing.assert_array_equal(got[:lo], clean[:lo])
    np.testing.assert_array_equal(got[:, :2], clean[:, :2])
    general, _ = run_attention(lib.attention_generic, sk, sv, qs, [0], [n], H, Kh, hs, "float32", np.random.default_rng(5), window=1 << 20)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(general))


# one block a CU (the loads of a step in registers at once) and more: contexts of one step and of several rounds of the eight waves, pages
# of half a step, of a step and of one and a half, tables no wider than the context
@pytest.mark.parametrize("page", [32, 64, 96])
@pytest.mark.parametrize("H, Kh, hs", [(8, 8, 32), (16, 8, 64), (8, 8, 96), (16, 8, 128)])
def test_float32_attention_is_the_same_with_a_step_s_loads_at_once(H, Kh, hs, page):
    lib, rng = K(), np.random.default_rng(H + hs + page)
    before, new = [0, 1100, 31, 500], [520, 3, 33, 17]
    sk, sv, qs = attention_case(rng, H, Kh, hs, before, new, "float32")
    sv[1][1101, 0, 0] = np.inf                       # a value that the first of its three tokens does not see
    calls = []

    def call(q, kc, vc, positions, seq_of, table, out, *rest):
        lib.attention_generic(q, kc, vc, positions, seq_of, table, out, *rest)
        calls.append(out.clone())
        for t in (0, 63, 64, 519, 520, 521, 522, 523, 555, 572):      # (eight blocks; all tokens are hundreds)
            one = torch.empty_like(out[:1])
            lib.attention_generic(q[t:t + 1], kc, vc, positions[t:t + 1], seq_of[t:t + 1], table, one, *rest)
            assert torch.equal(one[0].isnan(), out[t].isnan()) and torch.equal(one[0].nan_to_num(), out[t].nan_to_num()), t
    got, ref = run_attention(call, sk, sv, qs, before, new, H, Kh, hs, "float32", np.random.default_rng(1), page=page)
    fine = np.isfinite(ref)
    assert not fine.all() and np.array_equal(np.isfinite(got), fine)
    np.testing.assert_allclose(got[fine], ref[fine], atol=2e-5 * np.abs(ref[fine]).max())


# (the widths at which the norm's threads and their pieces change, one chunk and sixteen)
@pytest.mark.parametrize("hs, adjacent, rotated", [(16, False, True), (64, False, True), (64, True, True), (128, False, True), (96, True, True), (64, False, False)])
@pytest.mark.parametrize("M, Kd", [(1, 256), (2, 1024), (4, 1280), (3, 2048), (4, 3072), (3, 4096)])
def test_query_key_value_rows_with_norm_rotation_and_cache_in_one_kernel(hs, adjacent, rotated, M, Kd):
    """Against norm, product and rotation one after the other: the same queries and the same cache, bit for bit, everywhere."""
    lib = K()
    H, G, page, pages = 6, 2, 32, 9
    gen = torch.Generator(device="cuda").manual_seed(hs + M)
    x = torch.randn(M, Kd, generator=gen, device="cuda") * torch.tensor([1.0, 1e-3, 30.0, 5.0], device="cuda")[:M, None]
    nw = 1.0 + 0.1 * torch.randn(Kd, generator=gen, device="cuda")
    w = torch.randn((H + 2 * G) * hs, Kd, generator=gen, device="cuda") * 0.05
    cos = sin = None
    if rotated:
        cos, sin = (torch.randn(pages * page, hs // 2, generator=gen, device="cuda") for _ in range(2))
    table = torch.tensor([[3, 1, 7], [0, 8, 2], [5, 4, 6]], dtype=torch.int32, device="cuda")
    rows = torch.tensor([2, 0, 1, 0], dtype=torch.int32, device="cuda")[:M].contiguous()
    positions = torch.tensor([70, 31, 32, 0], dtype=torch.int32, device="cuda")[:M].contiguous()
    caches = [[torch.full((pages, G, page, hs), -7.0, device="cuda"), torch.full((pages, G, hs, page), -7.0, device="cuda")] for _ in range(2)]
    normed, qkv, q = torch.empty_like(x), torch.empty(M, (H + 2 * G) * hs, device="cuda"), torch.empty(M, H * hs, device="cuda")
    lib.rmsnorm(x, nw, normed, 1e-5)
    lib.gemm_generic(normed, w, qkv)
    lib.rope_cache_write(qkv, positions, rows, table, cos, sin, *caches[0], H, G, hs, hs if rotated else 0, adjacent, page)
    lib.qkv_f32_normed(x, nw, 1e-5, w, q, positions, rows, table, cos, sin, *caches[1], H, G, hs, adjacent, page)
    assert torch.equal(q, qkv[:, :H * hs])
    assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])


@pytest.mark.parametrize("M, Kd", [(5, 256), (1, 320), (1, 4352), (4, 4096)])
def test_rows_that_the_one_kernel_does_not_take(M, Kd):
    """More rows, other widths, more than a block keeps: said so beforehand and refused."""
    lib = K()
    x, nw, w = torch.zeros(M, Kd, device="cuda"), torch.zeros(Kd, device="cuda"), torch.zeros(48, Kd, device="cuda")
    k, v = torch.zeros(1, 1, 32, 16, device="cuda"), torch.zeros(1, 1, 16, 32, device="cuda")
    zero = torch.zeros(M, dtype=torch.int32, device="cuda")
    assert not lib.qkv_f32_normed_fits(x, nw, w, 16, 0)
    with pytest.raises(lib.KernelError):
        lib.qkv_f32_normed(x, nw, 1e-5, w, torch.empty(M, 16, device="cuda"), zero, zero, zero[:1, None].contiguous(), None, None, k, v, 1, 1, 16, False, 32)
