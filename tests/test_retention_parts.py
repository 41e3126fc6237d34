"""Retention of bf16 portions on the bf16 matrix units: numbers in three parts, beside the same rows in float32 on the fp32 units."""
import pytest
import torch

from llmd_amd.ops import seqmix as sm
from tests.test_koduzen import _seq, rope_table

pytestmark = pytest.mark.gpu


def _run(p, lens, H, dk, dv, gate, rot, decay, state, init):
    nd = len(lens)
    powers = (torch.tensor(decay, dtype=torch.float64)[:, None] ** torch.arange(sm.RETENTION_CHUNK + 1)).float().cuda()
    seq = _seq("cuda", list(lens), list(range(nd)), init, lens=[n + 7 for n in lens])
    pos = torch.cat([torch.arange(7, 7 + n) for n in lens]).cuda()
    s = state.clone()
    out = sm.retention(p, H, dk, dv, gate, pos, rope_table(rot, 300.0, 2048, "cuda") if rot else None, rot, powers, 1e-6, s, seq)
    return out, s


def _rows(T, H, dk, dv, gate, seed=0):
    n = 2 * H * dk + (2 if gate else 1) * H * dv
    return torch.randn(T, -(-n // 8) * 8, generator=torch.Generator().manual_seed(seed)).bfloat16().cuda()


def _exact_state(p, lens, H, dk, dv, decay, state, init):
    """64 bits, no rotation."""
    x, want, a = p.double(), [], 0
    for i, n in enumerate(lens):
        k = x[a:a + n, H * dk:2 * H * dk].view(n, H, dk) * dk ** -0.5
        v = x[a:a + n, 2 * H * dk:2 * H * dk + H * dv].view(n, H, dv)
        d = torch.tensor(decay, dtype=torch.float64, device="cuda")
        w = d[None] ** torch.arange(n - 1, -1, -1, device="cuda")[:, None]
        s = ((k * w[:, :, None]).permute(1, 2, 0).contiguous() @ v.permute(1, 0, 2).contiguous())
        want.append(s + (d[:, None, None] ** n * state[i].double() if init[i] else 0))
        a += n
    return torch.stack(want)


# all heads that the kernels take, rotated in full, in part (halves of 4 and 28) and not; runs that end a piece of 32, a chunk of 64, and
# one token before and behind
@pytest.mark.parametrize("H,dk,dv,rot,gate,lens", [(2, 64, 128, 64, True, (2, 31, 33)), (1, 64, 256, 56, False, (32, 63, 130)),
                                                   (3, 128, 256, 128, True, (65, 64, 901)), (2, 128, 128, 0, False, (97, 300)),
                                                   (1, 64, 256, 0, False, (1, 129, 16, 17)), (2, 128, 256, 8, True, (1, 1, 47, 49)),
                                                   (16, 128, 256, 0, False, (1024,))])
def test_retention_parts(H, dk, dv, rot, gate, lens):
    decay = [1.0 - 2.0 ** (-5.0 - i) for i in range(H)]
    p = _rows(sum(lens), H, dk, dv, gate)
    state = torch.randn(len(lens), H, dk, dv, generator=torch.Generator().manual_seed(1)).cuda()
    init = [i % 2 for i in range(len(lens))]
    got, s = _run(p, lens, H, dk, dv, gate, rot, decay, state, init)
    want, f = _run(p.float(), lens, H, dk, dv, gate, rot, decay, state, init)
    # sums of up to 64 + dk products of numbers around 1, each fp32 product and sum 2^-24 off; then one rounding to bf16 (gates: two)
    tol = 2 ** -8 * (2.0 if gate else 1.0)
    assert ((got.float() - want).abs() <= tol * want.abs() + 1e-4 * want.abs().max()).all()
    assert (s - f).abs().max() <= (64 + dk) * 2 ** -24 * f.abs().max()
    if not rot:
        exact = _exact_state(p, lens, H, dk, dv, decay, state, init)
        assert (s - exact).norm() <= 1.05 * (f - exact).norm()


@pytest.mark.parametrize("at,value", [("q", float("inf")), ("k", float("nan")), ("k", float("-inf")), ("v", float("inf")), ("v", 3e38), ("k", 1e35),
                                      ("state", float("inf")), ("state", 1e36), ("state", float("nan"))])
def test_numbers_that_are_not_finite_or_overflow(at, value):
    """They spoil what they belong to and nothing else: the sums that hold them, as on the fp32 units."""
    H, dk, dv, lens = 2, 64, 128, (70, 20)
    p = _rows(90, H, dk, dv, False)
    state = torch.randn(2, H, dk, dv, generator=torch.Generator().manual_seed(1)).cuda()
    if at == "state":
        state[0, 0, 3, 5] = value
    else:
        p[30, {"q": 5, "k": H * dk + 5, "v": 2 * H * dk + 5}[at]] = value
    got, s = _run(p, lens, H, dk, dv, False, 0, [0.97, 0.9], state, [1, 1])
    want, f = _run(p.float(), lens, H, dk, dv, False, 0, [0.97, 0.9], state, [1, 1])
    assert torch.allclose(s, f, rtol=1e-5, atol=1e-5 * f[torch.isfinite(f) & (f.abs() < 1e6)].abs().max().item(), equal_nan=True)
    got, want = got.float().view(90, H, dv), want.view(90, H, dv)
    clean = torch.ones(90, H, dtype=torch.bool, device="cuda")
    clean[:70, 0] = False
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 1e-4)[clean].all()
    # rows ahead of the number do not know it; those behind it are what the fp32 units make of them
    ahead = slice(0, 0 if at == "state" else 30)
    assert torch.isfinite(got[ahead]).all()
    behind = slice(30, 70)
    assert torch.equal(torch.isnan(got[behind, 0]), torch.isnan(want[behind, 0]))


@pytest.mark.parametrize("scale", [2.0 ** -60, 2.0 ** 40])
def test_small_and_large_numbers(scale):
    H, dk, dv, lens = 1, 128, 128, (100,)
    p = _rows(100, H, dk, dv, False)
    p[:, H * dk:] *= scale  # k and v: sums of 2^-120 and 2^80
    state = torch.zeros(1, H, dk, dv, device="cuda")
    _, s = _run(p, lens, H, dk, dv, False, 0, [0.97], state, [0])
    exact = _exact_state(p, lens, H, dk, dv, [0.97], state, [0])
    assert (s.double() - exact).norm() <= 4e-7 * exact.norm()


def test_capture():
    H, dk, dv, lens = 4, 128, 256, (200, 64)
    p = _rows(264, H, dk, dv, True)
    decay = [0.99, 0.97, 0.9, 0.5]
    powers = (torch.tensor(decay, dtype=torch.float64)[:, None] ** torch.arange(sm.RETENTION_CHUNK + 1)).float().cuda()
    seq = _seq("cuda", list(lens), [0, 1], [1, 0], lens=list(lens))
    pos = torch.cat([torch.arange(n) for n in lens]).cuda()
    cs = rope_table(dk, 300.0, 2048, "cuda")
    old = torch.randn(2, H, dk, dv, generator=torch.Generator().manual_seed(1)).cuda()
    state = old.clone()
    go = lambda: sm.retention(p, H, dk, dv, True, pos, cs, dk, powers, 1e-6, state, seq)  # noqa: E731
    go()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = go()
    for seed in (3, 4, 5):
        p.copy_(_rows(264, H, dk, dv, True, seed))
        state.copy_(old)
        want = go()
        after = state.clone()
        state.copy_(old)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(state, after)
