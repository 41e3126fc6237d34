"""Prompt-sized fp32 GEMM on the bf16 matrix units (csrc/ops/fgemm.hip) against the 64-bit product of the same operands."""
import pytest
import torch

from llmd_amd import ops

pytestmark = pytest.mark.gpu


def _operands(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N * 7 + K)
    x = torch.randn(M, K, generator=g, device="cuda")
    return x * torch.exp(2 * torch.randn(M, K, generator=g, device="cuda")), torch.randn(N, K, generator=g, device="cuda")


def _close(y, x, w, bias=None, least=0.0):
    ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    if bias is not None:
        ref, size = ref + bias.double(), size + bias.double().abs()
    # per 32 products a rounding of the sum to the nearest (the six kinds of products of parts apart: a sixteenth of that), the parts
    # left out at most 2^-24 of a product, and the roundings of ranges and bias
    K = x.shape[1]
    assert ((y.double() - ref).abs() <= size * (K / 32 * 1.1 + 8) * 2.0 ** -24 + least).all()


@pytest.mark.parametrize("mi,ni", [(4, 4), (3, 3), (4, 2), (2, 2)])
def test_tiles_edges(mi, ni):
    """One row and column, a tile less one, whole tiles and the first row of the next; a single step, an odd number of steps, a rest of
    K; rows further apart than K."""
    for M, N, K in ((1, 1, 32), (32 * mi - 1, 32 * ni - 1, 64), (32 * mi, 32 * ni, 96 + 4), (64 * mi + 1, 96 * ni + 3, 160 + 28)):
        x, w = _operands(M, N, K)
        bias = torch.linspace(-2, 2, N, device="cuda")
        code = mi * 100 + ni * 10 + 1
        y = ops.native().fgemm(x, w, None, code)
        _close(y, x, w)
        _close(ops.native().fgemm(x, w, bias, code), x, w, bias)
        wide = torch.zeros(M, K + 4, device="cuda")
        wide[:, :K] = x
        assert torch.equal(ops.native().fgemm(wide[:, :K], w, None, code), y)


@pytest.mark.parametrize("M,N,K,code", [(130, 260, 32 * 7, 442), (65, 100, 32 * 9 + 4, 333), (200, 64, 32 * 8, 223)])
def test_ranges_of_k(M, N, K, code):
    x, w = _operands(M, N, K)
    bias = torch.linspace(-2, 2, N, device="cuda")
    _close(ops.native().fgemm(x, w, None, code), x, w)
    _close(ops.native().fgemm(x, w, bias, code), x, w, bias)


@pytest.mark.parametrize("code", [441, 332, 421, 221])
@pytest.mark.parametrize("ex,ew", [(-104, 0), (-112, 0), (0, -116), (-124, 100), (60, -132), (-140, 120), (-60, -56), (90, -100), (50, 40)])
def test_small_and_large_numbers(ex, ew, code):
    """Numbers all of whose parts or some of them are below bf16's normal range, among them fp32's own denormals; numbers and sums that
    overflow when scaled. The same relative bound, but for the last bit of a denormal sum."""
    x, w = _operands(140, 100, 32 * 9 + 4)
    x, w = (x.double() * 2.0 ** ex).float(), (w.double() * 2.0 ** ew).float()
    y = ops.native().fgemm(x, w, None, code)
    assert y.abs().max() > 0
    _close(y, x, w, least=2.0 ** -149)


@pytest.mark.parametrize("code", [441, 331, 421, 221, 222])
def test_infinities_and_nans_stay_in_their_rows(code):
    """Numbers that the parts cannot hold: their rows as fp32 has them, the others' bits unchanged."""
    x, w = _operands(140, 152, 128)
    y = ops.native().fgemm(x, w, None, code)
    bad, rows = x.clone(), [3, 64, 100, 139]
    for r, v in zip(rows, (float("inf"), float("nan"), -float("inf"), 3.4e38)):
        bad[r, 77] = v
    z = ops.native().fgemm(bad, w, None, code)
    rest = torch.ones(140, dtype=torch.bool)
    rest[rows] = False
    assert torch.equal(z[rest], y[rest])
    full = bad.double() @ w.double().t()
    full = torch.where(full.abs() > 3.4028235e38, full.sign() * float("inf"), full)  # (none is within rounding of the border)
    assert torch.equal(z.isnan(), full.isnan()) and torch.equal(z.isinf(), full.isinf())
    assert torch.equal(z[z.isinf()], full[full.isinf()].float())


def test_linear_takes_it_and_leaves_the_rest():
    M, N, K = 700, 3072, 1024
    code = ops.native().fgemm_plan(M, N, K)
    assert code
    x, w = _operands(M, N, K)
    y = ops.linear(x, w)
    assert torch.equal(y, ops.native().fgemm(x, w, None, code))
    _close(y, x, w)
    nat = ops.native()
    assert nat.fgemm_plan(64, N, K) == 0 and nat.fgemm_plan(700, 132, K) == 0
    for a, b in ((x.bfloat16(), w.bfloat16()), (x[None], w), (x[:, 1:1021], w[:, 1:1021]), (x[:, ::2], w[:, ::2])):
        assert nat.fgemm(a, b) is None
    assert ops.fgemm(x.clone().requires_grad_(), w) is None
    with pytest.raises(RuntimeError):
        nat.fgemm(x, w, None, 991)
