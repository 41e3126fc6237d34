"""The streamed expert GEMM (csrc/include/moe_ring.h) at the edges of its tiles: rows per expert around the pairs of 16-row
blocks and the tile of 120, several tiles, more items than workgroups and fewer, a last block of weight rows that is half empty,
only one of the two products with sizes for it."""
import pytest
import torch

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 32, 33, 64, 65, 96, 97, 0, 119, 120, 121, 240, 241, 375]


@pytest.mark.parametrize("act", ["swish_limit", "relu2"])
@pytest.mark.parametrize("d,F,counts", [(320, 256, EDGES), (1024, 512, EDGES), (256, 256, [3]), (256, 1024, [70] * 64),
                                        (320, 200, EDGES), (264, 320, EDGES), (512, 8, [121]), (320, 320, [3])])
def test_streamed_experts(d, F, counts, act, monkeypatch):
    from llmd_amd.ops import seqmix as sm

    monkeypatch.setattr(sm, "MOE_STREAM_FROM", 0)
    g = torch.Generator(device="cuda").manual_seed(d + F)
    E, gated = len(counts), act != "relu2"
    ids = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(len(ids), generator=g, device="cuda")].int()[:, None]
    T = len(ids)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()  # noqa: E731
    h, w1, w2 = rand(T, d), rand(E, F * (2 if gated else 1), d) * d ** -0.5, rand(E, d, F) * F ** -0.5
    w = torch.ones(T, 1, device="cuda")
    assert sm._moe_tables(sm.native(), ids, E, h, w1, w2, gated)[3] == 120
    got = sm.moe_gated_ffn(h, ids, w, w1, w2, act, limit=3.0) if gated else sm.moe_ffn(h, ids, w, w1, w2, act)
    for e in range(E):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        z = h[rows].double() @ w1[e].double().T
        if gated:
            a, u = z[:, :F].clamp(max=3.0), z[:, F:].clamp(-3.0, 3.0)
            z = a * torch.sigmoid(1.702 * a) * (u + 1.0)
        else:
            z = torch.relu(z) ** 2
        want, size = z @ w2[e].double().T, z.abs() @ w2[e].abs().double().T
        # activation, row and result are each rounded once to bf16 (2^-9): at worst that adds up over ``size``
        assert ((got[rows].double() - want).abs() <= 3 * 2.0 ** -9 * (size + want.abs()) + 2.0 ** -9).all(), e


@pytest.mark.parametrize("kind", ["silu", "swish_limit"])
@pytest.mark.parametrize("d,F,rows", [(320, 256, 70), (1024, 512, 130), (256, 264, 31)])
def test_weights_on_the_input(d, F, rows, kind, monkeypatch):
    """Several choices per token whose weights scale the expert's input (both sums, before the activation)."""
    from llmd_amd.ops import seqmix as sm

    monkeypatch.setattr(sm, "MOE_STREAM_FROM", 0)
    g = torch.Generator(device="cuda").manual_seed(d + rows)
    E, k = 10, 3
    T = rows * E // k + 1
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    ids = (rand(T, E) + rand(E)).topk(k, -1).indices.int()
    h, w1, w2 = rand(T, d).bfloat16(), (rand(E, 2 * F, d) * d ** -0.5).bfloat16(), (rand(E, d, F) * F ** -0.5).bfloat16()
    w = torch.rand(T, k, generator=g, device="cuda") * 1.5 + 0.1
    assert sm._moe_tables(sm.native(), ids, E, h, w1, w2, True)[3] == 120
    got = sm.moe_gated_ffn(h, ids, w, w1, w2, kind, scale_input=True, limit=2.0)
    want, size, rounded = (torch.zeros(T, d, dtype=torch.float64, device="cuda") for _ in range(3))
    for e in range(E):
        t, j = (ids == e).nonzero(as_tuple=True)
        z = w[t, j].double()[:, None] * (h[t].double() @ w1[e].double().T)
        a, u = z[:, :F], z[:, F:]
        if kind == "silu":
            z = a * torch.sigmoid(a) * u
        else:
            a, u = a.clamp(max=2.0), u.clamp(-2.0, 2.0)
            z = a * torch.sigmoid(1.702 * a) * (u + 1.0)
        y = z @ w2[e].double().T
        want.index_add_(0, t, y)
        size.index_add_(0, t, z.abs() @ w2[e].abs().double().T)
        rounded.index_add_(0, t, y.abs())
    # activation, every expert's row and the result are each rounded once to bf16 (2^-9)
    assert ((got.double() - want).abs() <= 3 * 2.0 ** -9 * (size + rounded) + 2.0 ** -9).all()
