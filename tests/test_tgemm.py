"""Prompt-sized bf16 GEMM with a tile for every size (csrc/ops/tgemm.hip) against the fp32 product of the same operands."""
import pytest
import torch

from llmd_amd import ops

TILES = [(2, 2), (3, 2), (3, 3), (3, 4), (4, 3), (4, 4), (4, 6), (4, 8), (5, 4), (5, 6), (5, 8), (6, 4), (6, 6), (6, 8),
         (8, 5), (8, 6), (8, 7)]


def _operands(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed + M * 31 + N * 7 + K)
    return (torch.randn(M, K, generator=g, device="cuda").bfloat16(),
            (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16())


def _close(y, ref):
    # one rounding to bf16 (2^-9 of the value), and fp32 sums of K products of order 1 / sqrt(K)
    assert (y.float() - ref).abs().le(ref.abs() * 2.0 ** -8 + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("mi,ni", TILES)
def test_tiles_edges(mi, ni):
    """One row and column group, a tile less one row, whole tiles and the first row of the next one; one K-step up to
    more than the stages hold; rows further apart than K."""
    for M, N, K in ((1, 8, 64), (32 * mi - 1, 32 * ni - 8, 128), (32 * mi, 32 * ni, 320), (64 * mi + 1, 96 * ni + 8, 448)):
        x, w = _operands(M, N, K)
        wide = torch.zeros(M, K + 8, device="cuda", dtype=torch.bfloat16)
        wide[:, :K] = x
        bias = torch.linspace(-2, 2, N, device="cuda").bfloat16()
        ref = x.float() @ w.float().t()
        y = ops.native().tgemm(x, w, None, 0, mi * 100 + ni * 10 + 1)
        _close(y, ref)
        assert torch.equal(ops.native().tgemm(wide[:, :K], w, None, 0, mi * 100 + ni * 10 + 1), y)
        _close(ops.native().tgemm(x, w, bias, False, mi * 100 + ni * 10 + 1), ref + bias.float())
        w2 = torch.cat([w, w.flip(0)])
        _close(ops.native().tgemm(x, w2, None, 1, mi * 100 + ni * 10 + 1), torch.nn.functional.silu(ref) * ref.flip(1))
        z = ops.native().tgemm(x, w2, None, 0, mi * 100 + ni * 10 + 1)
        assert torch.equal(ops.native().tgemm(x, w2, None, 2, mi * 100 + ni * 10 + 1), ops.gated_act(z, ops.ACT_SILU))


@pytest.mark.gpu
@pytest.mark.parametrize("mi,ni,ranges", [(2, 2, 8), (4, 4, 2), (4, 8, 4), (6, 8, 3), (8, 8, 2), (8, 8, 3)])
def test_ranges_of_k(mi, ni, ranges):
    """The ranges' sums are added in order and rounded once; the last range may be the shorter one."""
    for M, N, K in ((1, 8, 64 * 22), (32 * mi + 1, 64 * ni + 8, 64 * 23)):
        x, w = _operands(M, N, K)
        bias = torch.linspace(-2, 2, N, device="cuda").bfloat16()
        ref = x.float() @ w.float().t()
        code = mi * 100 + ni * 10 + ranges
        _close(ops.native().tgemm(x, w, None, 0, code), ref)
        _close(ops.native().tgemm(x, w, bias, False, code), ref + bias.float())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 2048, 2048), (300, 5120, 2048), (700, 2176, 1536), (1429, 4096, 4096)])
def test_linear_takes_it(M, N, K):
    """ops.linear on an unlisted shape: the same bits as the tile's own call, in a row's result whatever M."""
    code = ops.native().tgemm_plan(M, N, K, 0)
    assert code and code % 10 == 1
    x, w = _operands(M, N, K)
    y = ops.linear(x, w)
    _close(y, x.float() @ w.float().t())
    assert torch.equal(y, ops.native().tgemm(x, w, None, 0, code))
    assert torch.equal(y[:65], ops.native().tgemm(x[:65], w, None, 0, 221))


def test_gated_forms_where_the_product_is_whole():
    """In place of a product and the activation's pass only where that product has one range of K: its bits, and no slower."""
    plan = ops.native().tgemm_plan
    assert plan(1429, 11264, 2048, 2) and plan(300, 1024, 8192, 0) % 10 > 1
    for M in (257, 300, 385, 512, 1000, 2048, 4500):
        for N in (256, 512, 1024, 2048, 11264):
            for K in (512, 2048, 4096, 8192, 16384):
                assert plan(M, N, K, 0) % 10 <= 1 or plan(M, N, K, 2) == 0, (M, N, K)


@pytest.mark.parametrize("M,N,K,left", [(128, 15168, 6400, True), (113, 15168, 6400, True), (112, 15168, 6400, False), (128, 15168, 2048, False),
                                        (128, 18944, 6400, False), (1920, 28928, 576, True), (1920, 28944, 576, False), (1920, 28928, 1088, False),
                                        (1429, 4096, 4096, False), (2600, 3072, 2048, False)])
def test_sizes_left_to_the_library(M, N, K, left):
    """128 rows on tiles for two thirds of the CUs that wait for their weights; columns in whole tiles of 256, short K, that fill the rounds
    of 256 x 256 tiles; and sizes on the other side of each line."""
    assert (ops.native().tgemm_plan(M, N, K, 0) == 0) == left


@pytest.mark.gpu
def test_refused_or_left():
    """Operands that the kernel does not read stay with the library; one of its tiles for another shape raises."""
    x, w = _operands(130, 256, 128)
    nat = ops.native()
    for a, b in ((x.float(), w.float()), (x[None], w), (x, w[:255]), (x[:, ::2], w[:, ::2]), (x[:64], w),
                 (torch.cat([x, x], 1)[:, 4:132], w)):
        assert nat.tgemm(a, b) is None
    assert ops.tgemm(x.clone().requires_grad_(), w) is None
    g = ops.linear(x.clone().requires_grad_(), w)
    assert g.requires_grad
    assert nat.tgemm(x[:, :120].contiguous(), w[:, :120].contiguous()) is None  # K of no whole step
    with pytest.raises(RuntimeError):
        nat.tgemm(x, w, None, 0, 991)
    with pytest.raises(RuntimeError):
        nat.tgemm(x, w, None, 0, 443)  # two steps of K in three ranges


def test_cpu_tensors_stay_with_the_library():
    x, w = torch.randn(130, 64).bfloat16(), torch.randn(16, 64).bfloat16()
    assert ops.tgemm(x, w) is None
    assert torch.equal(ops.linear(x, w), torch.nn.functional.linear(x, w))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 5632, 2048), (9, 2048, 1024), (16, 1024, 8192), (17, 5632, 2048), (64, 768, 4096), (65, 5632, 2048),
                                   (700, 2048, 5632), (256, 1024, 16384)])
def test_squared_relu_in_the_epilogue(M, N, K):
    """Every kernel that ops.linear takes for these sizes, with one range of K and several: the bits of the two passes."""
    from llmd_amd.ops import seqmix as sm

    x, w = _operands(M, N, K)
    y = ops.linear_relu2(x, w)
    assert y is not None and torch.equal(y, sm.relu2(ops.linear(x, w)))
