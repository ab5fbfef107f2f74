"""The product of many rows in bfloat16 against float64, at the edges of its tiles."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from macllm_infer_amd.kernels import build, ops as module
    build.ensure_modules(["common", "rows_gemm", "decode"])
    return module


def rand(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed))


def bound(x, weight, want):
    """Float32 sums of K products in any order (2^-24 of the sum of magnitudes for each) and one rounding to bfloat16."""
    sums = x.double().abs() @ weight.double().abs().T
    return x.shape[1] * 2.0 ** -24 * sums + 2.0 ** -8 * want.abs() + 1e-30


@pytest.mark.parametrize("M, N, K", [(1, 1, 64), (17, 17, 64), (63, 64, 128), (64, 65, 192), (65, 130, 256), (127, 16, 320),
                                     (129, 257, 64), (130, 2100, 384), (1030, 70, 448), (300, 1000, 1024)])
def test_every_tile_gives_the_rounded_product(M, N, K):
    x, w, b = rand(M, K, seed=1).to(torch.bfloat16), (rand(N, K, seed=2) / math.sqrt(K)).to(torch.bfloat16), rand(N, seed=3)
    plain = x.double() @ w.double().T
    first = None
    for tile in (0, 1, 2, 3, -1):
        got = ops().rows_gemm(x.to(DEV), w.to(DEV), tile=tile)
        with_bias = ops().rows_gemm(x.to(DEV), w.to(DEV), b.to(DEV), tile=tile)
        sums = ops().rows_gemm(x.to(DEV), w.to(DEV), keep_float32=True, tile=tile)
        assert bool(((got.cpu().double() - plain).abs() <= bound(x, w, plain)).all())
        want = plain + b.double()
        assert bool(((with_bias.cpu().double() - want).abs() <= bound(x, w, want) + 2.0 ** -23 * b.abs()).all())
        assert sums.dtype == torch.float32 and bool(((sums.cpu().double() - plain).abs() <= bound(x, w, plain * 0.0)).all())
        first = got if first is None else first
        assert torch.equal(got, first), tile                    # a row is summed in the order of k, whatever the tile


@pytest.mark.parametrize("M, inner, K", [(1, 8, 64), (65, 40, 128), (64, 64, 192), (130, 72, 320), (257, 1032, 256), (2050, 24, 64)])
def test_the_gated_activation_in_the_product(M, inner, K):
    x, b = rand(M, K, seed=4).to(torch.bfloat16), rand(2 * inner, seed=6)
    w = (rand(2 * inner, K, seed=5) * 2.0 / math.sqrt(K)).to(torch.bfloat16)
    for bias in (None, b):
        sums = x.double() @ w.double().T + (0.0 if bias is None else bias.double())
        gate, up = sums.view(M, inner // 8, 2, 8).unbind(2)
        want = (gate * torch.sigmoid(gate) * up).reshape(M, inner)
        # the sums' error e and their rounding (2^-8 of either) reach the result by at most 1.1 |up| of the gate's and |silu(gate)| of the
        # up half's, the activation adds four ulps
        e = float((x.double().abs() @ w.double().abs().T).max() * K * 2.0 ** -24 + 1e-6)
        most = float((1.1 * up.abs() + gate.abs()).max())
        for tile in (0, 1, 2, 3, -1):
            got = ops().rows_gemm(x.to(DEV), w.to(DEV), None if bias is None else bias.to(DEV), swiglu=True, tile=tile)
            assert got.shape == (M, inner)
            rounded = 2.0 ** -8 * (1.1 * up.abs() * gate.abs() + (gate * torch.sigmoid(gate)).abs() * up.abs()).reshape(M, inner)
            assert bool(((got.cpu().double() - want).abs() <= 2.0 ** -8 * want.abs() + rounded * 1.01 + most * e).all()), tile


@pytest.mark.parametrize("M, N, K", [(32, 128, 64), (33, 4096, 1024), (65, 80, 192), (130, 1040, 512), (515, 4096, 1024), (2048, 4096, 1024),
                                     (600, 512, 2048)])
def test_the_gated_activation_in_the_product_has_the_bits_of_a_launch_behind_it(M, N, K):
    """Of this package's product, and of the library's, where that sums in k order too (64 features and more, K up to 1,024)."""
    module = ops()
    x, b = rand(M, K, seed=4).to(torch.bfloat16).to(DEV), rand(N, seed=6).to(DEV)
    w = (rand(N, K, seed=5) * 2.0 / math.sqrt(K)).to(torch.bfloat16).to(DEV)
    for bias in (None, b):
        products = [module.rows_gemm(x, w, bias)]
        if bias is None and K <= 1024:
            products.append(torch.mm(x, w.t()))
        got = [module.rows_gemm(x, w, bias, swiglu=True, tile=tile) for tile in (0, 1, 2, 3)] + [module.linear_swiglu(x, w, bias)]
        for product in products:
            behind = torch.empty(M, N // 2, dtype=torch.bfloat16, device=DEV)
            module.swiglu(product, behind, 8)
            assert all(torch.equal(one, behind) for one in got)


def test_rows_of_a_wider_matrix_infinities_and_what_is_refused():
    module = ops()
    wide = rand(70, 200, seed=7).to(torch.bfloat16).to(DEV)
    w = rand(33, 128, seed=8).to(torch.bfloat16).to(DEV)
    x = wide[:, 16:144]
    assert torch.equal(module.rows_gemm(x, w), module.rows_gemm(x.contiguous(), w))
    x = x.clone()
    x[3, 5], x[9, 0] = math.inf, math.nan
    got = module.rows_gemm(x, w).cpu()
    others = [row for row in range(70) if row not in (3, 9)]
    assert bool(torch.isfinite(got[others]).all()) and bool(got[3].isinf().all()) and bool(got[9].isnan().all())
    assert not module.rows_gemm_supported(wide[:, 1:129], w)              # rows that start between 16-byte pieces
    with pytest.raises(module.KernelError):
        module.rows_gemm(rand(4, 96).to(torch.bfloat16).to(DEV), rand(4, 96).to(torch.bfloat16).to(DEV))     # K no multiple of 64


@pytest.mark.parametrize("M, N, K", [(32, 48, 64), (40, 1024, 1024), (300, 260, 512), (600, 1024, 2048)])
def test_linear_takes_it_where_it_pays_and_gives_the_librarys_numbers(M, N, K):
    module = ops()
    assert module.rows_gemm_pays(M, N, K) and module.rows_gemm_pays(M, N, K, keep_float32=True) == (K == 64)
    assert not module.rows_gemm_pays(31, N, K)
    x, w, b = rand(M, K, seed=9).to(torch.bfloat16).to(DEV), (rand(N, K, seed=10) / math.sqrt(K)).to(torch.bfloat16).to(DEV), rand(N, seed=11).to(DEV)
    # two roundings to bfloat16 of sums that differ by float32 rounding: a neighbouring value at most
    for bias in (None, b):
        got = module.linear(x, w, bias)
        library = torch.mm(x.float(), w.float().T) + (0.0 if bias is None else bias)
        assert bool(((got.float() - library).abs() <= 2.0 ** -8 * library.abs() + K * 2.0 ** -22).all())
    sums = module.linear(x, w, None, keep_float32=True)
    assert sums.dtype == torch.float32 and float((sums - torch.mm(x.float(), w.float().T)).abs().max()) < K * 2.0 ** -22


def test_linear_takes_rows_that_overlap_and_operands_without_elements():
    """Expanded rows and rows of a sliding window are the library's, as they are where no product of this package pays; so is a
    product with no features or of nothing."""
    module = ops()
    x, w = rand(70, 128, seed=12).to(torch.bfloat16).to(DEV), rand(48, 128, seed=13).to(torch.bfloat16).to(DEV)
    assert module.rows_gemm_pays(70, 48, 128) and module.rows_gemm_supported(x, w)
    row, window = x[5:6].expand(70, 128), x.view(-1).as_strided((70, 128), (64, 1))
    for rows in (row, window):
        assert not module.rows_gemm_supported(rows, w)
        assert torch.equal(module.linear(rows, w, None), torch.mm(rows.contiguous(), w.t()))
        # (W [70, 128] against x's first rows: the same numbers the other way round)
        assert torch.equal(module.linear(x[:48], rows, None), torch.mm(x[:48], rows.contiguous().t()))
    assert module.linear(x, w[:0], None).shape == (70, 0)
    empty = module.linear(x[:, :0], w[:, :0], None)
    assert empty.shape == (70, 48) and not bool(empty.any())
