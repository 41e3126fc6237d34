"""A router's product on its own kernel: sums of exact products in fp32, in an order that does not depend on the sizes."""
import pytest
import torch

from llmd_amd import ops

pytestmark = pytest.mark.gpu


def _rand(*shape, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to("cuda", torch.bfloat16)


# rows around the 16 and 32 of a workgroup, columns around 16, 32 and 48, fewer steps of 64 k than waves, as many, with a remainder;
# the sizes of models with the next form at 1025 rows
@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (15, 16, 128), (16, 17, 192), (17, 15, 256), (31, 33, 320), (33, 48, 576), (47, 49, 1088), (64, 132, 2048),
                                   (1025, 132, 2048), (2551, 132, 2048), (300, 256, 7168)])
def test_router_product(M, N, K):
    x, w, b = _rand(M, K + 64)[:, :K], _rand(N, K + 8, seed=1)[:, :K], _rand(N, seed=2)
    want = x.double() @ w.double().t()
    # a number passes through K / 4 additions of a wave and three more, each off by 2^-24 of sum |x w|
    bound = x.double().abs() @ w.double().abs().t() * (K // 4 + 64 + 3) * 2 ** -24
    C = ops.native()
    first = None
    for form in range(3):
        y = C.router_product(x, w, None, True, form)
        assert y.dtype == torch.float32 and ((y.double() - want).abs() <= bound).all()
        first = y if first is None else first
        assert torch.equal(y, first)  # one order of the sums in every form
        z = C.router_product(x, w, b, False, form)
        assert torch.equal(z, (y + b.float()).bfloat16())
    assert torch.equal(ops.router_product(x, w), first)
    assert torch.equal(ops.router_product(x[M // 2:], w), first[M // 2:])


def test_router_product_leaves_the_rest():
    x, w = _rand(9, 256), _rand(16, 256, seed=1)
    assert ops.router_product(x, w) is not None
    assert ops.router_product(x[:, :96], w[:, :96].contiguous()) is None             # K in steps of 64
    assert ops.router_product(x.float(), w.float()) is None
    assert ops.router_product(_rand(9, 257)[:, 1:], w) is None                       # off 16 bytes
    assert ops.router_product(x.t().contiguous().t(), w) is None
    assert ops.router_product(x[:0], w) is None
    with torch.enable_grad():
        assert ops.router_product(x, w.clone().requires_grad_()) is None
    y = ops.router_linear(_rand(8192, 2048), _rand(128, 2048, seed=1))               # on the larger tiles
    want = _rand(8192, 2048).double() @ _rand(128, 2048, seed=1).double().t()
    assert (y.double() - want).abs().max() <= 2 ** -8 * want.abs().max()             # rounded once to bf16


def test_router_linear_takes_other_calls_as_before():
    x, w, b = _rand(2, 3, 256), _rand(16, 256, seed=1), _rand(16, seed=2)
    assert torch.equal(ops.router_linear(x, w, b), torch.nn.functional.linear(x, w, b))
    xc, wc = x.cpu(), w.cpu()
    assert torch.equal(ops.router_linear(xc, wc), torch.nn.functional.linear(xc, wc))


@pytest.mark.parametrize("rows,dtype", [(9, torch.bfloat16), (1000, torch.bfloat16), (8192, torch.bfloat16), (300, torch.float32)])
def test_a_bias_that_is_differentiated(rows, dtype):
    """The library's product, which has a backward, whatever the rows: a router's, and a dense one's on the tiles."""
    N = 128 if dtype == torch.bfloat16 else 4096
    x, w, b = _rand(rows, 2048).to(dtype), _rand(N, 2048, seed=1).to(dtype), _rand(N, seed=2).to(dtype).requires_grad_()
    for f in (ops.router_linear, lambda x, w, b: ops.fgemm(x, w, b) if dtype == torch.float32 else ops.tgemm(x, w, b)):
        with torch.enable_grad():
            y = f(x, w, b)
            if y is None:  # left to the library
                continue
            y.sum().backward()
        assert torch.equal(b.grad, torch.full_like(b, float(rows)).to(dtype))
        b.grad = None
        with torch.no_grad():
            assert not f(x, w, b).requires_grad


def test_capture():
    x, w = _rand(64, 2048), _rand(132, 2048, seed=1)
    want = ops.router_product(x, w)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = ops.router_product(x, w)
    for seed in (3, 4):
        x.copy_(_rand(64, 2048, seed=seed))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, ops.router_product(x, w)) and not torch.equal(y, want)
