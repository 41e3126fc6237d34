"""Projections handed on as sums over ranges of K, and the residual's passes that read them (csrc/seqmix/sm_elementwise.hip, sm_hyper.hip)."""
from types import SimpleNamespace

import pytest
import torch

from llmd_amd import ops
from llmd_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


def _rand(*shape, dtype=torch.bfloat16, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed + sum(shape))
    return (torch.randn(*shape, device="cuda", generator=g) * scale).to(dtype)


@pytest.mark.parametrize("M,N,K", [(1, 2048, 2048), (9, 2048, 5632), (16, 1024, 8192), (5, 520, 1280), (16, 2048, 1024), (17, 2048, 2048),
                                   (64, 2048, 5632), (33, 1000, 1024), (9, 4096, 4096)])
def test_parts_are_the_product(M, N, K):
    x, w = _rand(M, K), _rand(N, K, seed=1, scale=K ** -0.5)
    p = ops.linear_parts(x, w)
    if p is None:
        assert (M, N) == (9, 4096)
        return
    assert p.shape[1:] == (M, N) and p.shape[0] >= 2
    want = x.double() @ w.double().t()
    assert (p.double().sum(0) - want).abs().max() < 2e-5  # K / ranges products of about 1 / sqrt(K) each, summed in fp32
    if M > 16:
        assert torch.equal(p[0] if p.shape[0] == 1 else _added(p), ops.linear(x, w))


def _added(p):
    s = p[0]
    for k in range(1, p.shape[0]):
        s = s + p[k]
    return s.bfloat16()


@pytest.mark.parametrize("T,d,n", [(1, 2048, 2), (9, 2048, 8), (64, 1000, 3), (3, 8192, 2), (5, 8200, 2), (4, 2052, 2)])
@pytest.mark.parametrize("S", [1, 2, 4, 5])
def test_readers_of_parts(T, d, n, S):
    """The bits of the pass over the sums and the reader behind it; rows off the 16-byte forms are added up first."""
    p, w, wn = _rand(n, T, d, dtype=torch.float32), _rand(d, seed=1), _rand(d, seed=2)
    y = _added(p)
    if S == 1:
        x0, x1 = (_rand(T, d, dtype=torch.float32, seed=3) for _ in range(2))
        for nxt in (wn, None):
            a, b = (sm.post_norm_add(v, w, x, 1e-5, torch.bfloat16, nxt) for v, x in ((y, x0), (p, x1)))
            assert torch.equal(a, b) and torch.equal(x0, x1)
    X0, X1 = (_rand(S, T, d, dtype=torch.float32, seed=4) for _ in range(2))
    mix, out, nin = _rand(S, S, dtype=torch.float32), _rand(S, dtype=torch.float32), _rand(S, dtype=torch.float32, seed=5)
    a, b = (sm.hyper_update_norm(X, v, mix, out, nin, wn, 1e-5, torch.bfloat16, True) for v, X in ((y, X0), (p, X1)))
    assert torch.equal(a, b) and torch.equal(X0, X1)


@pytest.mark.parametrize("T,d,taps", [(1, 2048, 4), (9, 2048, 4), (64, 1000, 3), (3, 8192, 2), (2, 4104, 4)])
def test_convolution_in_the_norm(T, d, taps):
    """post_norm_add with the next reader's convolution: the bits of the two passes, states rolled and only those of the step."""
    y, w, wn, cw = _rand(T, d), _rand(d, seed=1), _rand(d, seed=2), _rand(d, taps, seed=3, scale=0.2)
    x0, x1 = (_rand(T, d, dtype=torch.float32, seed=4) for _ in range(2))
    s0, s1 = (_rand(T + 3, taps - 1, d, seed=5) for _ in range(2))
    i32 = dict(dtype=torch.int32, device="cuda")
    seq = SimpleNamespace(row_seq=torch.arange(T, **i32), seq_start=torch.arange(T + 1, **i32), seq_slot=torch.randperm(T + 3)[:T].to(**i32),
                          seq_init=(torch.arange(T, **i32) % 3 != 1).int(), max_q=1)
    assert sm.row_conv(x0, cw, seq, torch.bfloat16)
    for _ in range(2):
        a = sm.input_conv(sm.post_norm_add(y, w, x0, 1e-5, torch.bfloat16, wn), cw, s0, seq)
        b = sm.post_norm_add(y, w, x1, 1e-5, torch.bfloat16, wn, conv=(cw, s1, seq))
        assert torch.equal(a, b) and torch.equal(x0, x1) and torch.equal(s0, s1)
    odd = torch.empty(T * d + 8, device="cuda", dtype=torch.bfloat16)[1:T * d + 1].view(T, d).copy_(y)  # off 16 bytes: one pass after the other
    b = sm.post_norm_add(odd, w, x1, 1e-5, torch.bfloat16, wn, conv=(cw, s1, seq))
    a = sm.input_conv(sm.post_norm_add(odd, w, x0, 1e-5, torch.bfloat16, wn), cw, s0, seq)
    assert torch.equal(a, b) and torch.equal(s0, s1)


@pytest.mark.parametrize("T,F,n", [(1, 2560, 2), (64, 512, 8), (9, 1004, 3), (5, 36, 2)])
@pytest.mark.parametrize("kind", ["gelu_tanh", "silu", "swish_limit"])
def test_gated_units_of_parts(T, F, n, kind):
    p = _rand(n, T, 2 * F, dtype=torch.float32, scale=3.0)
    assert torch.equal(sm.gated_act(p, F, kind, 7.0), sm.gated_act(_added(p), F, kind, 7.0))


@pytest.mark.parametrize("M,F,K", [(257, 512, 2048), (901, 2560, 2048), (300, 264, 1024), (2722, 1024, 2048)])
def test_clamped_units_in_the_epilogue(M, F, K):
    """The bits of the product and the units' pass, infinities and numbers beyond the limit among the sums."""
    x, w = _rand(M, K), _rand(2 * F, K, seed=1, scale=3 * K ** -0.5)
    w[3], w[F + 5] = float("inf"), float("-inf")
    y = ops.linear_clamped(x, w, 2.5)
    assert y is not None
    want = sm.gated_act(ops.linear(x, w), F, "swish_limit", 2.5)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize("T,H,K,N", [(1, 16, 512, 128), (9, 16, 128, 512), (17, 3, 256, 16), (33, 5, 128, 48), (64, 32, 512, 128), (16, 128, 128, 64)])
def test_head_product(T, H, K, N):
    x, w = _rand(T, H, K + 64)[:, :, :K], _rand(H, N, K, seed=1, scale=K ** -0.5)
    buf = torch.full((T, H, N + 64), 7.0, device="cuda", dtype=torch.bfloat16)
    assert sm.head_product(x, w, buf[:, :, :N])
    want = torch.einsum("thk,hnk->thn", x.double().cpu(), w.double().cpu())
    assert (buf[:, :, :N].double().cpu() - want).abs().max() <= 2 ** -8 * want.abs().max()  # rounded once to bf16
    assert (buf[:, :, N:] == 7).all()


def test_head_product_leaves_the_rest():
    x, w = _rand(4, 8, 128), _rand(8, 64, 128)
    out = torch.empty(4, 8, 64, device="cuda", dtype=torch.bfloat16)
    assert not sm.head_product(x[:, :, :64], w[:, :, :64].contiguous(), out)                          # k in quarters of 32
    assert not sm.head_product(_rand(65, 8, 128), w, torch.empty(65, 8, 64, device="cuda", dtype=torch.bfloat16))
    assert not sm.head_product(_rand(33, 64, 128), _rand(64, 64, 128), torch.empty(33, 64, 64, device="cuda", dtype=torch.bfloat16))
    assert not sm.head_product(_rand(4, 8, 129)[:, :, 1:], w, out)                                    # off 16 bytes


@pytest.mark.parametrize("M,N,K", [(1, 132, 2048), (16, 16, 128), (17, 15, 256), (64, 132, 2048), (300, 8, 384), (800, 132, 2048), (33, 256, 1024)])
def test_router_logits(M, N, K):
    """fp32 sums of exact products: each of the four partial sums adds up to 512 times, off by 2^-24 of sum |x w| each."""
    x, w = _rand(M, K + 64)[:, :K], _rand(N, K, seed=1)
    y = sm.router_logits(x, w)
    want = x.double() @ w.double().t()
    bound = x.double().abs() @ w.double().abs().t() * (min(K // 4, 512) + 3) * 2 ** -24
    assert y.dtype == torch.float32 and ((y.double() - want).abs() <= bound).all()
    if (N, K) == (132, 2048):  # the order of the float product in its place
        assert torch.equal(y, torch.nn.functional.linear(x.float(), w.float()))
    assert sm.router_logits(x[:, :96], w[:, :96].contiguous()) is None
    if N >= 16:  # 512 blocks of 16 x 16 and more
        assert sm.router_logits(_rand(8192, K), w) is None


def test_router_logits_of_longer_rows_stay_with_the_library():
    """Beyond K 2048 the order of the sums is not the float product's."""
    assert sm.router_logits(_rand(9, 2048), _rand(132, 2048)) is not None and sm.router_logits(_rand(9, 2176), _rand(132, 2176)) is None


@pytest.mark.parametrize("T,d,S", [(1, 2048, 2), (64, 2048, 1), (5, 1000, 3), (3, 4096, 4), (2, 4104, 2), (7, 17, 16)])
@pytest.mark.parametrize("rms", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_embedding_and_first_norm(T, d, S, rms, dtype):
    """The bits of the two passes; ids outside the table give zeros."""
    table, w, w_in = _rand(50, d, dtype=dtype), _rand(d, seed=1, dtype=dtype), _rand(S, dtype=torch.float32)
    ids = torch.arange(T, device="cuda") * 7 % 50
    ids[-1] = 50 if T > 1 else 3
    X0, X1 = (torch.full((S, T, d), float("nan"), device="cuda") for _ in range(2))
    sm.hyper_embed(ids, table, X0)
    a = sm.hyper_norm(X0, w_in, w, 1e-5, dtype, rms)
    b = sm.hyper_embed_norm(ids, table, X1, w_in, w, 1e-5, dtype, rms)
    assert torch.equal(X0, X1) and torch.equal(a, b)
