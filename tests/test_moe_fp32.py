"""fp32 experts on the matrix cores (csrc/include/moe_tile.h): tiles of every number of 16-row blocks and their edges, several
tiles of an expert, rows and columns that do not fill their last step or block, tiles taken by expert and by size, how by size the
work lies on the XCDs."""
import pytest
import torch

FEW = [0, 1, 15, 16, 17, 20, 3, 31]
MANY = [1, 16, 17, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 127, 128, 129, 240, 385]


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["swish_limit", "relu2"])
@pytest.mark.parametrize("d,F", [(64, 64), (36, 20), (320, 200)])
@pytest.mark.parametrize("counts", [FEW, MANY, [3], [40], [129] * 40, [17] * 63, [17] * 64])
def test_experts(d, F, counts, act):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator(device="cuda").manual_seed(d + len(counts))
    E, gated = len(counts), act != "relu2"
    ids = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda"))
    ids = ids[torch.randperm(len(ids), generator=g, device="cuda")].int()[:, None]
    T = len(ids)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    h, w1, w2 = rand(T, d), rand(E, F * (2 if gated else 1), d) * d ** -0.5, rand(E, d, F) * F ** -0.5
    w = torch.ones(T, 1, device="cuda")
    slot_row, tiles, _, tm = sm._moe_tables(sm.native(), ids, E, h, w1, w2, gated)
    assert tm == 128 and (tiles.numel() == 1 + 4 * (slot_row.numel() // tm)) == (T > 16 * E)
    got = sm.moe_gated_ffn(h, ids, w, w1, w2, act, limit=3.0) if gated else sm.moe_ffn(h, ids, w, w1, w2, act)
    for e in range(E):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        x, b = h[rows].double(), w1[e].double()
        z, dz = x @ b.T, (d + 4) * 2.0 ** -24 * (x.abs() @ b.abs().T)  # a sum of d products, each rounded once
        if gated:  # slopes: of a sigmoid(1.702 a) below 1.2, times u + 1 <= 4; of u + 1 below 3
            a, u = z[:, :F].clamp(max=3.0), z[:, F:].clamp(-3.0, 3.0)
            z, dz = a * torch.sigmoid(1.702 * a) * (u + 1.0), 5 * dz[:, :F] + 3 * dz[:, F:]
        else:
            z, dz = torch.relu(z) ** 2, (2 * z.abs() + dz) * dz
        dz = dz + 2.0 ** -19 * z.abs()  # the activation itself
        c = w2[e].double()
        bound = dz @ c.abs().T + (F + 4) * 2.0 ** -24 * (z.abs() @ c.abs().T)
        assert ((got[rows].double() - z @ c.T).abs() <= bound + 1e-30).all(), e


@pytest.mark.gpu
@pytest.mark.parametrize("spread", [1, 5, 300])
@pytest.mark.parametrize("n", [0, 100, 4000, 9000])
def test_tiles_by_size(n, spread):
    from llmd_amd.ops import seqmix as sm

    E, tm = 300, 128
    ids = (torch.rand(n, generator=torch.Generator().manual_seed(n)) ** 2 * spread).int()
    cnt = torch.bincount(ids.long(), minlength=E)
    mt = max(1, (n + min(E, n) * (tm - 1)) // tm)
    t = lambda m: torch.full((m,), 7, dtype=torch.int32, device="cuda")  # noqa: E731
    row, tiles, slot = t(mt * tm), t(1 + 4 * mt), t(n)
    sm.native().moe_group(ids.cuda(), E, tm, row, tiles, slot)
    tiles = tiles.cpu().long()
    total = int(tiles[0])
    assert total == int(((cnt + tm - 1) // tm).sum())
    order = tiles[1 + 3 * mt:1 + 3 * mt + total]
    assert sorted(order.tolist()) == list(range(total))
    blocks = ((tiles[1:1 + 3 * total:3] >> 16) + 15) // 16
    assert (blocks[order].diff() <= 0).all()


@pytest.mark.parametrize("NB", [1, 3, 8, 11, 44, 88])
def test_work_by_size_over_the_xcds(NB):
    """Workgroups go to the eight XCDs in turn: every block of every tile is some workgroup's, no XCD has more than its share by
    an eighth (or one block)."""
    sm = pytest.importorskip("llmd_amd._C_seqmix")
    for total in [*range(0, 20), 23, 24, 25, 31, 33, 62, 63, 64, 65, 71, 72, 73, 128, 129, 203]:
        for max_tiles in (total, total + 37):
            work = [sm.moe_deal(total, NB, b) for b in range((max_tiles + 7) // 8 * 8 * NB)]
            at = [(b & 7, w) for b, w in enumerate(work) if w[0] < total]
            assert sorted(w for _, w in at) == [(r, nb) for r in range(total) for nb in range(NB)]
            most = max(sum(x == xcd for x, _ in at) for xcd in range(8))
            assert most <= max(-(-total * NB // 8), total * NB / 8 * 1.125), (total, most)
