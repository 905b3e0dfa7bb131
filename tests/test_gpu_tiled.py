"""The tiled products at the edges of their tiles and of their pipelines, over every order that a weight may lie in."""
import numpy as np
import pytest
import torch

from test_gpu_kernels import DEV, K, dev, rounded

pytestmark = pytest.mark.gpu


def held(lib, w, order):
    if order == "stored":
        return w
    v = w.clone()
    if order == "strips of 16":
        v.tiled = lib.tile_weight(v)
    else:
        v.tiled8 = lib.tile_weight8(v)
    return lib.hold_once(v)


def off_by(a, w, out_bits):
    """32-bit sums of K products: at most K roundings of the sum of magnitudes; the output rounded to ``out_bits``."""
    s = np.abs(a).astype(np.float64) @ np.abs(w).astype(np.float64).T
    return a.shape[1] * 2.0 ** -24 * s, 2.0 ** -out_bits


# (rows and columns of one tile of 128 or 256, one more, one less and many; K of one, two, three and an odd number of steps;
# 2,304 columns are nine tiles of 256 over the XCDs)
@pytest.mark.parametrize("shape", [1, 2, 5])
@pytest.mark.parametrize("order", ["stored", "strips of 16", "strips of 8"])
@pytest.mark.parametrize("M, N, Kd", [(1, 16, 64), (255, 256, 128), (257, 272, 192), (300, 2304, 320), (513, 128, 1088), (1100, 528, 2048)])
def test_tiled_products(shape, order, M, N, Kd):
    lib = K()
    rng = np.random.default_rng(M + N + Kd)
    a, w = rounded(rng.standard_normal((M, Kd)), "bfloat16"), rounded(rng.standard_normal((N, Kd)) / np.sqrt(Kd), "bfloat16")
    A = torch.zeros(M, Kd + 8, device=DEV, dtype=torch.bfloat16)[:, :Kd]              # (rows apart)
    A.copy_(dev(a))
    W = held(lib, dev(w, torch.bfloat16), order)
    ref = a.astype(np.float64) @ w.astype(np.float64).T
    sums, _ = off_by(a, w, 24)
    factor, bias = rng.standard_normal(N).astype(np.float32), rng.standard_normal(N).astype(np.float32)
    for pad in (0, 3):                                                                # (3: no four columns of a row at once)
        out = torch.full((M, N + pad), -7.0, device=DEV)
        for again in range(2):
            lib.gemm_mfma(A, W, out[:, :N], shape=shape)
            assert (np.abs(out[:, :N].double().cpu().numpy() - ref) <= sums + 1e-30).all(), again
        assert torch.all(out[:, N:] == -7.0)
    half = torch.zeros(M, N, device=DEV, dtype=torch.bfloat16)
    lib.gemm_mfma(A, W, half, shape=shape, bias=dev(bias))
    want = ref + bias
    assert (np.abs(half.double().cpu().numpy() - want) <= 2.0 ** -8 * np.abs(want) + 2 * sums + 1e-6).all()
    res = rng.standard_normal((M, N)).astype(np.float32)
    for more in (0, 1, 3, 4, 7):                                                     # (K of five steps: the last of four slices has none)
        if (more + 1) * 64 > Kd:
            continue
        x = dev(res)
        part = torch.full((more, M, N), -7.0, device=DEV) if more else None
        lib.gemm_mfma(A, W, x, lib.EPI_ADD, more_slices=part, shape=shape, col_scale=dev(factor))
        got = x.double().cpu().numpy() + (part.double().sum(0).cpu().numpy() if more else 0.0)
        assert (np.abs(got - (res + ref * factor)) <= sums * np.abs(factor) + 2.0 ** -21 * (np.abs(res) + np.abs(ref * factor)) + 1e-6).all(), more


@pytest.mark.parametrize("shape", [1, 2, 5])
@pytest.mark.parametrize("order", ["stored", "strips of 16"])
@pytest.mark.parametrize("M, N, Kd", [(3, 16, 64), (256, 128, 192), (258, 144, 128), (700, 1040, 576)])
def test_tiled_gated_products(shape, order, M, N, Kd):
    lib = K()
    rng = np.random.default_rng(M * 3 + N)
    a, w = rounded(rng.standard_normal((M, Kd)), "bfloat16"), rounded(rng.standard_normal((2 * N, Kd)) / np.sqrt(Kd), "bfloat16")
    W = held(lib, dev(w, torch.bfloat16), order)
    ref = a.astype(np.float64) @ w.astype(np.float64).T
    want = ref[:, :N] / (1 + np.exp(-ref[:, :N])) * ref[:, N:]
    out, wide = torch.zeros(M, N, device=DEV), torch.full((M, N + 1), -7.0, device=DEV, dtype=torch.bfloat16)
    lib.gemm_mfma(dev(a, torch.bfloat16), W, out, lib.EPI_GATED, shape=shape)
    assert np.abs(out.cpu().numpy() - want).max() <= 2e-5 * np.abs(want).max()         # (the fast exponential: 2^-20)
    lib.gemm_mfma(dev(a, torch.bfloat16), W, wide[:, :N], lib.EPI_GATED, shape=shape)
    assert torch.equal(wide[:, :N], out.to(torch.bfloat16)) and torch.all(wide[:, N:] == -7.0)


# (rows and columns in no whole tiles, slices of unequal length; the plans: 8, 2, 4, 3, 2 and 1 slices)
@pytest.mark.parametrize("M, N, Kd", [(150, 2064, 4672), (2048, 2048, 8192), (513, 2048, 2048), (1000, 2304, 2240), (2047, 2048, 2112), (2050, 3072, 1024)])
def test_products_into_the_residual_rows_keep_their_sums(M, N, Kd):
    """The plan of a product into the residual rows on the kernel whose waves take turns: the same sums, bit for bit, as tiles on the
    kernel without turns in the slices of ``mfma_plan``."""
    lib = K()
    rng = np.random.default_rng(M)
    A, W = dev(rounded(rng.standard_normal((M, Kd)), "bfloat16"), torch.bfloat16), dev(rounded(rng.standard_normal((N, Kd)), "bfloat16"), torch.bfloat16)
    res = dev(rng.standard_normal((M, N)))

    def rows(shape, slices):
        x, part = res.clone(), torch.full((slices - 1, M, N), -7.0, device=DEV) if slices > 1 else None
        lib.gemm_mfma(A, W, x, lib.EPI_ADD, more_slices=part, shape=shape)
        if part is not None:
            lib.add_slices_rmsnorm(x, part)
        return x
    tile, slices = lib.mfma_plan(M, N, Kd)
    assert torch.equal(rows(-tile, slices), rows(3, slices))


# slices of equal and unequal length, a last one without a step
@pytest.mark.parametrize("M, N, Kd, slices", [(257, 272, 192, 1), (300, 256, 320, 4), (513, 528, 1088, 3), (130, 1024, 4160, 8), (1100, 2048, 8192, 2)])
def test_a_tile_and_its_kernel_have_no_say_in_the_sums(M, N, Kd, slices):
    """Tiles on the kernel whose waves take turns (1, 2, 5) and on the one without (3, 4): bit for bit the same sums for the same slices of K."""
    lib = K()
    gen = torch.Generator(device="cuda").manual_seed(M)
    A, W = (torch.randn(n, Kd, generator=gen, device="cuda").to(torch.bfloat16) for n in (M, N))
    res = torch.randn(M, N, generator=gen, device="cuda")
    got = []
    for shape in (3, 4, 1, 2, 5):
        x, part = res.clone(), torch.full((slices - 1, M, N), -7.0, device=DEV) if slices > 1 else None
        lib.gemm_mfma(A, W, x, lib.EPI_ADD, more_slices=part, shape=shape)
        got.append(torch.cat([x[None], part]) if part is not None else x[None])
        assert torch.equal(got[-1], got[0]), shape


# (one row, a part of a small tile and more than one of them behind the large ones; rows of output apart and not; K in slices of which the last has no step)
@pytest.mark.parametrize("order", ["stored", "strips of 16", "strips of 8"])
@pytest.mark.parametrize("shape, M, N, Kd", [(9, 257, 272, 192), (13, 300, 2304, 320), (9, 513, 128, 1088), (17, 770, 528, 320), (13, 1100, 528, 192)])
def test_two_tiles_of_a_product_give_the_sums_of_one(order, shape, M, N, Kd):
    """256 x 256 for the first 256 * (shape / 8) rows, shape % 8 behind them: bit for bit what tiles of 128 x 128 alone give."""
    lib = K()
    gen = torch.Generator(device="cuda").manual_seed(M)
    A = torch.randn(M, Kd + 8, generator=gen, device="cuda").to(torch.bfloat16)[:, :Kd]
    w = torch.randn(2 * N, Kd, generator=gen, device="cuda").to(torch.bfloat16)
    W, G = held(lib, w[:N], order), None if order == "strips of 8" else held(lib, w, order)
    bias, factor, res = (torch.randn(n, generator=gen, device="cuda") for n in ((N,), (N,), (M, N)))

    def both(dtype, weight, epilogue, pad=0, slices=1, **kw):
        got = []
        for tile in (1, shape):
            x = torch.full((M, N + pad), -7.0, device=DEV, dtype=dtype)
            x[:, :N] = res
            part = torch.full((slices - 1, M, N), -7.0, device=DEV) if slices > 1 else None
            lib.gemm_mfma(A, weight, x[:, :N], epilogue, more_slices=part, shape=tile, **kw)
            assert torch.all(x[:, N:] == -7.0)
            got.append(torch.cat([x[None, :, :N], part]) if slices > 1 else x)
        assert torch.equal(*got), (dtype, epilogue, pad, slices)
    for pad in (0, 3):
        both(torch.float32, W, lib.EPI_STORE, pad, bias=bias)
        both(torch.bfloat16, W, lib.EPI_STORE, pad, bias=bias, col_scale=factor)
        both(torch.float32, W, lib.EPI_ADD, pad)
        if G is not None:
            both(torch.bfloat16, G, lib.EPI_GATED, pad)
    for slices in (2, 3) + ((4,) if Kd == 320 else ()):
        both(torch.float32, W, lib.EPI_ADD, slices=slices, col_scale=factor)


def test_two_tiles_are_refused_where_they_do_not_fit():
    """No rows behind the large tiles, a K of no whole steps, gated values of 32 bits: nothing is launched."""
    lib = K()
    a, w = torch.zeros(512, 200, device=DEV, dtype=torch.bfloat16), torch.zeros(256, 200, device=DEV, dtype=torch.bfloat16)
    x = torch.zeros(512, 256, device=DEV)
    for rows, k, shape, epilogue in ((256, 128, 9, lib.EPI_STORE), (512, 128, 17, lib.EPI_STORE), (512, 200, 9, lib.EPI_STORE), (512, 128, 9, lib.EPI_GATED),
                                     (512, 128, 10, lib.EPI_STORE)):
        with pytest.raises(lib.KernelError, match="tile"):
            lib.gemm_mfma(a[:rows, :k], w[:, :k].contiguous(), x[:rows, :128 if epilogue == lib.EPI_GATED else 256], epilogue, shape=shape)


@pytest.mark.parametrize("shape", [-6, -4, -3, 6])
def test_unknown_tiles_are_refused(shape):
    """A plan names one of the library's own tiles (1, 2, 5); nothing is launched for another."""
    lib = K()
    a, w, x = (torch.zeros(128, 128, device=DEV, dtype=d) for d in (torch.bfloat16, torch.bfloat16, torch.float32))
    with pytest.raises(lib.KernelError, match="unknown tile shape"):
        lib.gemm_mfma(a, w, x, shape=shape)


# (columns in whole eights, in fours and in neither; one row, whole tiles, one row more than a tile)
@pytest.mark.parametrize("shape", [1, 2, 5])
@pytest.mark.parametrize("M, N", [(1, 8), (2, 3), (129, 136), (256, 256), (257, 260), (300, 523)])
def test_epilogues_of_the_tiled_products(shape, M, N):
    """An output that may be stored sixteen bytes at a time against one that begins at an odd place and is stored element by element:
    the same bits, whatever the epilogue applies, and nothing beside the output is written."""
    lib = K()
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    Kd = 192
    A, W = (torch.randn(n, Kd, generator=gen, device="cuda").to(torch.bfloat16) for n in (M, 2 * N))
    bias, factor = torch.randn(2 * N, generator=gen, device="cuda"), torch.randn(N, generator=gen, device="cuda")
    res = torch.randn(M, N, generator=gen, device="cuda")

    def both(dtype, epilogue, add=False, **kw):
        w = W if epilogue == lib.EPI_GATED else W[:N]
        outs = []
        for pad, first in ((8 - N % 8, 0), (3, 1)):
            whole = torch.full((M, N + pad + first), -7.0, device=DEV, dtype=dtype)
            out = whole[:, first:first + N]
            if add:
                out.copy_(res)
            lib.gemm_mfma(A, w, out, epilogue, shape=shape, **kw)
            assert torch.all(whole[:, :first] == -7.0) and torch.all(whole[:, first + N:] == -7.0)
            outs.append(out.clone())
        assert torch.equal(outs[0], outs[1]), (dtype, epilogue, kw)
        return outs[0].double()
    sums = A.double() @ W.double().T
    size = A.double().abs() @ W.double().abs().T                                      # (a sum of 192 products: 192 roundings of it at most)
    for dtype, bits in ((torch.bfloat16, 8), (torch.float32, 23)):
        for kw, want in (({}, sums[:, :N]), ({"bias": bias[:N].contiguous()}, sums[:, :N] + bias[:N].double()),
                         ({"col_scale": factor}, sums[:, :N] * factor.double())):
            off = (both(dtype, lib.EPI_STORE, **kw) - want).abs()
            assert (off <= 2.0 ** -bits * want.abs() + Kd * 2.0 ** -23 * size[:, :N] * max(1.0, factor.abs().max().item())).all()
        for kw in ({}, {"bias": bias}, {"act": "gelu_tanh"}, {"act_limit": 3.0, "act_shift": 1.0}):
            gate, up = (sums + (bias.double() if "bias" in kw else 0.0)).split(N, 1)
            if "act_limit" in kw:
                gate, up = gate.clamp(max=3.0), up.clamp(-3.0, 3.0) + 1.0
            want = (torch.nn.functional.gelu(gate, approximate="tanh") if "act" in kw else gate / (1.0 + torch.exp(-gate))) * up
            off = (both(dtype, lib.EPI_GATED, **kw) - want).abs()
            # (a sum's error goes through a rule whose slope is at most 1.1 times the other factor; the exponential: 2^-20)
            slack = 1.2 * Kd * 2.0 ** -23 * (size[:, :N] * (up.abs() + 1.0) + size[:, N:] * (gate.abs() + 1.0))
            assert (off <= (2.0 ** -bits + 2.0 ** -17) * want.abs() + slack + 1e-6).all(), (dtype, kw)
    want = sums[:, :N] + res.double()
    assert ((both(torch.float32, lib.EPI_ADD, add=True) - want).abs() <= 2.0 ** -23 * want.abs() + Kd * 2.0 ** -23 * size[:, :N]).all()


@pytest.mark.parametrize("shape", [1, 2, 5])
@pytest.mark.parametrize("M, N", [(1, 3), (129, 130), (300, 523)])
def test_slices_whose_columns_are_no_whole_fours(shape, M, N):
    """The sums of later slices of K in rows of any width, at any place: those of rows of whole fours, and nothing beside them is written."""
    lib = K()
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    wide = -(-N // 4) * 4
    A, W, factor = (torch.randn(n, generator=gen, device="cuda") for n in ((M, 192), (wide, 192), (wide,)))
    A, W = A.to(torch.bfloat16), W.to(torch.bfloat16)
    for scale in (None, factor):
        x, want = torch.zeros(M, wide, device=DEV), torch.empty(2, M, wide, device=DEV)
        lib.gemm_mfma(A, W, x, lib.EPI_ADD, more_slices=want, shape=shape, col_scale=scale)
        for first, ld in ((0, N), (0, wide + 4), (1, N + 1)):
            y, whole = torch.zeros(M, N, device=DEV), torch.full((2, M, ld), -7.0, device=DEV)
            part = whole[:, :, first:first + N]
            lib.gemm_mfma(A, W[:N], y, lib.EPI_ADD, more_slices=part, shape=shape, col_scale=None if scale is None else factor[:N])
            assert torch.equal(part, want[:, :, :N]) and torch.equal(y, x[:, :N])
            assert torch.all(whole[:, :, :first] == -7.0) and torch.all(whole[:, :, first + N:] == -7.0)


@pytest.mark.parametrize("M, N, Kd, dtype", [(512, 50257, 1024, torch.float32), (2048, 32001, 2048, torch.float32), (2048, 32001, 2048, torch.bfloat16)])
def test_columns_that_are_no_whole_fours_take_little_longer(M, N, Kd, dtype):
    """Rows of an odd number of columns against rows of whole eights: stored one element at a time from the registers they took 1.3 to 1.6 times as long."""
    lib = K()
    wide = -(-N // 8) * 8
    A, W = (torch.randn(n, Kd, device=DEV).to(torch.bfloat16) for n in (M, wide))
    outs = [torch.empty(M, n, device=DEV, dtype=dtype) for n in (N, wide)]
    times = [[], []]
    for _ in range(8):
        for i, out in enumerate(outs):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(5):
                lib.gemm_mfma(A, W[:out.shape[1]], out)
            b.record()
            b.synchronize()
            times[i].append(a.elapsed_time(b))
    assert min(times[0]) < 1.25 * min(times[1])


@pytest.mark.parametrize("M, N, Kd", [(66, 1000, 1024), (400, 2048, 2048)])
def test_a_bias_costs_little(M, N, Kd):
    """32-bit sums with a bias against the same without: read behind the steps, between the stores, the bias took a fifth to a third of the product's time."""
    lib = K()
    A, W = (torch.randn(n, Kd, device=DEV).to(torch.bfloat16) for n in (M, N))
    out, bias = torch.empty(M, N, device=DEV), torch.randn(N, device=DEV)
    graphs = []
    for b in (None, bias):
        lib.gemm_mfma(A, W, out, bias=b)
        torch.cuda.synchronize()
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            for _ in range(20):
                lib.gemm_mfma(A, W, out, bias=b)
    least = [float("inf")] * 2
    for _ in range(10):
        for i, graph in enumerate(graphs):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            graph.replay()
            b.record()
            b.synchronize()
            least[i] = min(least[i], a.elapsed_time(b))
    assert least[1] < 1.15 * least[0], least


# (rows of whole fours, whose bias is read in front of the steps, and others; columns beyond the last tile's)
@pytest.mark.parametrize("shape", [1, 2, 5])
@pytest.mark.parametrize("M, N", [(3, 4), (130, 260), (66, 1000), (129, 131), (2, 3)])
def test_every_column_gets_its_own_bias(shape, M, N):
    """Products of nothing leave the bias alone, in every row."""
    lib = K()
    A, W = (torch.zeros(n, 192, device=DEV, dtype=torch.bfloat16) for n in (M, N))
    bias = torch.arange(1, N + 1, device=DEV, dtype=torch.float32)
    for first in (0, 1):                        # (at sixteen bytes and at an odd place)
        whole = torch.full((M, N + 5), -7.0, device=DEV)
        out = whole[:, first:first + N] if first else torch.full((M, N), -7.0, device=DEV)
        lib.gemm_mfma(A, W, out, bias=torch.cat([bias[:1], bias])[1:] if first else bias, shape=shape)
        assert torch.equal(out, bias.expand(M, N))
        assert torch.all(whole[:, N + first:] == -7.0) and torch.all(whole[:, :first] == -7.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_the_gated_rule_over_the_range_of_its_gate(dtype):
    """v / (1 + e^-v) for gates that a bias alone makes: every magnitude, the ends where e^-v leaves the floats, and what is no number."""
    lib = K()
    ends = [0.0, -0.0, 1e-30, -1e-30, 1e-38, -1e-38, -80.0, -87.0, -88.5, -88.7, -89.0, -100.0, -1e30, 1e30, 3e38, -3e38, float("inf"), float("-inf"), float("nan")]
    gen = torch.Generator(device="cuda").manual_seed(4)
    N = 1 << 17
    v = torch.empty(N, device=DEV).uniform_(-88.0, 88.0, generator=gen)
    v[::2] = torch.exp2(torch.empty(N // 2, device=DEV).uniform_(-120.0, 6.4, generator=gen)) * torch.where(v[1::2] < 0, -1.0, 1.0)
    v[:len(ends)] = torch.tensor(ends, device=DEV)
    out = torch.empty(1, N, device=DEV, dtype=dtype)
    zeros = [torch.zeros(n, 64, device=DEV, dtype=torch.bfloat16) for n in (1, 2 * N)]
    lib.gemm_mfma(*zeros, out, lib.EPI_GATED, bias=torch.cat([v, torch.ones_like(v)]))
    got, x = out[0].double(), v.double()
    e = torch.exp(-x)
    want = x / (1.0 + e)
    # a rounding of the sum and one of the quotient; the exponential counts by its share e / (1 + e): its argument, |v| log2(e), is rounded and
    # so is the factor (three halves of 2^-24 of |v|), its own result is a unit off; then the output's rounding (16 bits: 2^-9, or half of the smallest step, 2^-133, below 2^-126)
    share = torch.where(torch.isinf(e), 1.0, e / (1.0 + e))
    bound = want.abs() * (2.0 ** -24 * (2.0 + share * (1.5 * x.abs() + 2.0)) * 1.001 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0)) + (2.0 ** -134 if dtype == torch.bfloat16 else 0.0) + 2.0 ** -147
    inside = (x > -88.0) & (x < 1e31)
    assert ((got - want).abs() <= bound)[inside].all()
    below = (x <= -88.0) & torch.isfinite(x)              # (e^-v is an infinity from -88.73 down: minus nothing)
    assert ((got <= 0) & (got >= want * 1.01 - 1e-45))[below].all()
    by_end = dict(zip(map(str, ends), got[:len(ends)].tolist()))
    assert by_end["inf"] == float("inf") and by_end["-inf"] != by_end["-inf"] and by_end["nan"] != by_end["nan"]
    assert by_end["3e+38"] == pytest.approx(3e38, rel=2.0 ** -8) and by_end["0.0"] == by_end["-0.0"] == 0.0
