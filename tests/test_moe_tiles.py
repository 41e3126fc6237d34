"""Grouped expert GEMMs at the edges of their tiles: rows per expert around the 16-row blocks, the 32-row border between the
two bodies and the 128-row tile, more than one tile, empty experts; K with and without a rest, N with and without whole
blocks; both types, the streaming form where it applies, and the FMA form for sizes without 16-byte pieces."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 16, 17, 0, 32, 33, 48, 64, 65, 127, 128, 129, 257]


def _counts_to_ids(counts, identity):
    """One choice per token: counts[e] tokens for expert e, ``identity`` for the entry past them, shuffled."""
    ids = [e for e, n in enumerate(counts) for _ in range(n)] + [len(counts)] * identity
    g = torch.Generator().manual_seed(1)
    return torch.tensor(ids, dtype=torch.int32)[torch.randperm(len(ids), generator=g)].view(-1, 1)


@pytest.mark.parametrize("stream_from", [0, 1 << 20], ids=["stream", "tile"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,F", [(256, 256), (384, 192), (264, 72), (64, 40), (37, 50)])
def test_gated_experts_tile_edges(d, F, dtype, stream_from, monkeypatch):
    from llmd_amd.ops import seqmix as sm

    monkeypatch.setattr(sm, "MOE_STREAM_FROM", stream_from)
    g = torch.Generator().manual_seed(d)
    E = len(ROWS)
    ids = _counts_to_ids(ROWS, 5)
    T = ids.shape[0]
    h = torch.randn(T, d, generator=g).to(dtype)
    w = torch.rand(T, 1, generator=g) + 0.5
    w1 = (torch.randn(E, 2 * F, d, generator=g) / d ** 0.5).to(dtype)
    w2 = (torch.randn(E, d, F, generator=g) / F ** 0.5).to(dtype)
    got = sm.moe_gated_ffn(h.cuda(), ids.cuda(), w.cuda(), w1.cuda(), w2.cuda(), "silu").cpu().double()
    want = torch.empty(T, d, dtype=torch.float64)
    size = torch.zeros(T, d, dtype=torch.float64)  # sums of the magnitudes behind every result
    for e in range(E + 1):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        x = h[rows].double()
        if e == E:
            want[rows], size[rows] = x, x.abs()
            continue
        a = x @ w1[e, :F].double().T
        a = a * torch.sigmoid(a) * (x @ w1[e, F:].double().T)
        want[rows], size[rows] = a @ w2[e].double().T, a.abs() @ w2[e].abs().double().T
    want, size = want * w, size * w
    # bf16: the activation, the expert's row and the result are each rounded once (2^-9); the activation's own inputs are fp32
    # sums. fp32: sums of d and F products, activation in fp32. Roundings add up over ``size`` at worst.
    eps = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -23 * 8
    assert ((got - want).abs() <= 3 * eps * (size + want.abs()) + eps).all()


@pytest.mark.parametrize("act", ["gelu", "relu2"])
@pytest.mark.parametrize("stream_from", [0, 1 << 20], ids=["stream", "tile"])
def test_ungated_experts_two_blocks_of_columns(act, stream_from, monkeypatch):
    from llmd_amd.ops import seqmix as sm
    from llmd_amd.ops import seqmix_ref as ref

    monkeypatch.setattr(sm, "MOE_STREAM_FROM", stream_from)
    g = torch.Generator().manual_seed(3)
    E, d, F, T, k = 4, 256, 384, 300, 2
    h = torch.randn(T, d, generator=g).bfloat16()
    ids = torch.rand(T, E, generator=g).topk(k, -1).indices.int()
    w = torch.rand(T, k, generator=g)
    w1 = (torch.randn(E, F, d, generator=g) / d ** 0.5).bfloat16()
    w2 = (torch.randn(E, d, F, generator=g) / F ** 0.5).bfloat16()
    got = sm.moe_ffn(h.cuda(), ids.cuda(), w.cuda(), w1.cuda(), w2.cuda(), act).cpu().float()
    want = ref.moe_ffn(h.float(), ids, w, w1.float(), w2.float(), act)
    # three roundings to bf16 (activation, rows, sum): far below 1 % of the result's size
    assert (got - want).norm() <= 0.01 * want.norm()


@pytest.mark.parametrize("d,F", [(256, 256), (264, 72), (64, 40)])
def test_interleaved_experts_few_rows(d, F):
    """ops.moe_experts of decode-sized steps (gate and up rows interleaved): every tile size, pairs of other ranks (-1)."""
    from llmd_amd import ops

    g = torch.Generator().manual_seed(d)
    E = len(ROWS)
    ids = _counts_to_ids(ROWS, 5)
    ids[ids == E] = -1
    T = ids.shape[0]
    assert T < ops.MOE_V3_MIN_ROWS * E * 2
    h = torch.randn(T, d, generator=g).bfloat16()
    w = torch.rand(T, 1, generator=g) + 0.5
    w1 = (torch.randn(E, 2 * F, d, generator=g) / d ** 0.5).bfloat16()
    w2 = (torch.randn(E, d, F, generator=g) / F ** 0.5).bfloat16()
    was, ops.MOE_V3 = ops.MOE_V3, False
    try:
        got = ops.moe_experts(h.cuda(), ids.cuda(), w.cuda(), w1.cuda(), w2.cuda(), ops.ACT_SILU).cpu().double()
    finally:
        ops.MOE_V3 = was
    for e in range(-1, E):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        if e < 0:
            assert (got[rows] == 0).all()
            continue
        x = h[rows].double()
        a = x @ w1[e, 0::2].double().T
        a = a * torch.sigmoid(a) * (x @ w1[e, 1::2].double().T)
        want, size = a @ w2[e].double().T * w[rows], a.abs() @ w2[e].abs().double().T * w[rows]
        # the activation, the expert's row and the result are each rounded to bf16 once
        assert ((got[rows] - want).abs() <= 3 * 2.0 ** -9 * (size + want.abs()) + 2.0 ** -9).all()


@pytest.mark.parametrize("d,F", [(256, 96), (100, 72)])
def test_float32_rows_alone_and_together(d, F):
    """fp32 experts form their products from three bf16 parts of every number: within the bound of fp32 sums for every tile
    height, a row's bits whatever its tile, and rows with infinities, NaNs or numbers that a part cannot hold as fp32 has them
    without a trace in the others."""
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(d)
    E = 8
    ids = _counts_to_ids([9, 30, 40, 60, 75, 90, 110, 128], 0)
    T = ids.shape[0]
    h = torch.randn(T, d, generator=g) * torch.exp(2 * torch.randn(T, d, generator=g))
    w1 = torch.randn(E, F, d, generator=g) / d ** 0.5
    w2 = torch.randn(E, d, F, generator=g) / F ** 0.5

    def run(h, ids):
        n = len(h)
        return sm.moe_ffn(h.cuda(), ids.cuda(), torch.ones(n, 1, device="cuda"), w1.cuda(), w2.cuda(), "relu2").cpu()

    got = run(h, ids)
    x, e = h.double(), ids[:, 0].long()
    a = torch.einsum("td,tfd->tf", x, w1.double()[e])
    ea = torch.einsum("td,tfd->tf", x.abs(), w1.double()[e].abs()) * (d + 8) * 2.0 ** -24  # of the first sums
    a, ea = a.clamp(min=0) ** 2, 2 * (a.abs() + ea) * ea + a * a * 2.0 ** -23
    want = torch.einsum("tf,tdf->td", a, w2.double()[e])
    bound = torch.einsum("tf,tdf->td", ea + a * (F + 8) * 2.0 ** -24, w2.double()[e].abs())
    assert ((got - want).abs() <= bound).all()
    few = torch.arange(0, T, 7)
    assert torch.equal(run(h[few], ids[few]), got[few])
    bad = h.clone()
    rows = [int((e == i).nonzero()[3]) for i in range(E)]
    values = [float("inf"), -float("inf"), float("nan"), 3.4e38] * 2
    for r, v in zip(rows, values):
        bad[r, 5] = v
    out = run(bad, ids)
    rest = torch.ones(T, dtype=torch.bool)
    rest[rows] = False
    assert torch.equal(out[rest], got[rest])
    for r, v in zip(rows, values):
        z = w1[e[r]].double() @ bad[r].double()  # +-inf, NaN or large: squares that overflow
        full = torch.where(z.isnan(), 0.0, z.clamp(min=0) ** 2).float()
        want = torch.where(full[None] * w2[e[r]] == 0, torch.zeros(()), full[None] * w2[e[r]])
        assert torch.equal(out[r].isfinite(), torch.isfinite(want.sum(1)))


@pytest.mark.parametrize("ex,ew", [(-112, 0), (-124, 60), (0, -116), (60, -132), (-135, 70)])
def test_float32_small_numbers(ex, ew):
    """Rows and weights whose bf16 parts reach below bf16's normal range, fp32's own denormals among them: within the relative bound of
    ordinary numbers, through both products. The clamped units of sums z this small are z / 2, and the second weights pick them."""
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(7)
    d, F, E = 100, 72, 4
    ids = _counts_to_ids([9, 30, 60, 110], 0)
    T = ids.shape[0]
    up = lambda t, e: (t.double() * 2.0 ** e).float()  # noqa: E731
    h, w1 = up(torch.randn(T, d, generator=g), ex), up(torch.randn(E, F, d, generator=g) / d ** 0.5, ew)
    w2 = torch.eye(d, F).expand(E, d, F).contiguous()
    got = sm.moe_gated_ffn(h.cuda(), ids.cuda(), torch.ones(T, 1, device="cuda"), torch.cat([w1, w1], 1).cuda(), w2.cuda(),
                           "swish_limit", limit=1e30).cpu().double()
    e = ids[:, 0].long()
    z = torch.einsum("td,tfd->tf", h.double(), w1.double()[e])
    size = torch.einsum("td,tfd->tf", h.double().abs(), w1.double()[e].abs())
    # d fp32 additions at worst, the units' reciprocal and products, the last bit of denormal results
    bound = size / 2 * (d + 8) * 2.0 ** -24 + z.abs() * 2.0 ** -20 + 2.0 ** -148
    assert ((got[:, :F] - z / 2).abs() <= bound).all() and got[:, :F].abs().max() > 0 and (got[:, F:] == 0).all()
