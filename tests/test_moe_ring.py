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
