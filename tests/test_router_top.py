"""Expert choice on the GPU at the edges of its forms (64, 128, 256, 512 outputs), with many equal scores, infinities and bf16
logits, against the plain references: ties go to the lower index, the order of the chosen ones is falling."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _logits(T, E, seed):
    g = torch.Generator().manual_seed(seed)
    z = torch.randn(T, E, generator=g)
    z[1] = torch.randint(0, 3, (E,), generator=g).float()      # ties
    z[2] = 0.0                                                 # all equal
    z[3, ::2] = -float("inf")
    z[4] = torch.randint(-1, 2, (E,), generator=g).float() * 0.5
    return z


@pytest.mark.parametrize("E,k", [(8, 8), (63, 4), (64, 1), (65, 7), (128, 8), (132, 8), (257, 16), (512, 6)])
@pytest.mark.parametrize("sigmoid", [False, True])
def test_route(E, k, sigmoid):
    from llmd_amd.ops import seqmix as sm

    z = _logits(37, E, E)
    ids, w = sm.moe_route(z.cuda(), k, sigmoid)
    top = torch.sort(z, descending=True, stable=True)  # ties: the lower index first
    rids, rw = top.indices[:, :k], torch.sigmoid(top.values[:, :k]) if sigmoid else torch.softmax(top.values[:, :k], -1)
    rows = [t for t in range(37) if k <= int(torch.isfinite(z[t]).sum())]
    assert torch.equal(ids.cpu()[rows], rids[rows].int())
    assert torch.allclose(w.cpu()[rows], rw[rows], rtol=1e-5, atol=1e-7)


@pytest.mark.parametrize("E,k,groups,keep", [(64, 8, 1, 1), (132, 8, 4, 2), (130, 5, 13, 3), (512, 16, 64, 8), (12, 3, 4, 1)])
def test_route_scores(E, k, groups, keep):
    from llmd_amd.ops import seqmix as sm
    from llmd_amd.ops import seqmix_ref as ref

    z = _logits(37, E, E + 1)
    corr = torch.randint(-2, 3, (E,), generator=torch.Generator().manual_seed(E)).float() * 2.0 ** -6
    ids, w = sm.moe_route_scores(z.cuda(), corr.cuda(), k, groups, keep, 1.5)
    rids, rw = ref.moe_route_scores(z, corr, k, groups, keep, 1.5)
    # rows of equal scores differ in nothing but rounding: there the reference's own order is the one of exact ties only
    rows = [t for t in range(37) if t not in (1, 2, 3, 4)]
    assert torch.equal(ids.cpu()[rows], rids[rows].int())
    assert torch.allclose(w.cpu()[rows], rw[rows], rtol=1e-5, atol=1e-7)
    for t in (1, 2, 4):  # chosen sets with the same choice scores
        s = torch.softmax(z[t], -1) + corr
        assert torch.allclose(s[ids.cpu()[t].long()], s[rids[t].long()], atol=1e-6)


@pytest.mark.parametrize("E,k", [(16, 2), (64, 6), (128, 8), (256, 8), (384, 16)])
@pytest.mark.parametrize("scoring", [0, 1, 2])
def test_topk_bf16_logits(E, k, scoring):
    from llmd_amd import ops
    from llmd_amd.ops import reference as ref

    z = _logits(37, E, E + 2)[5:].bfloat16()
    a, wa = ops.moe_topk(z.cuda(), k, scoring=scoring, renorm=True)
    b, wb = ops.moe_topk(z.float().cuda(), k, scoring=scoring, renorm=True)
    assert torch.equal(a, b) and torch.equal(wa, wb)  # the same numbers, widened in the kernel
    r, wr = ref.moe_topk(z.float(), k, scoring, None, 1, 1, True, 1.0)
    assert torch.allclose(torch.sort(wa.cpu(), -1).values, torch.sort(wr, -1).values, rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("bm", [64, 192, 256])
def test_align_tables(bm):
    from llmd_amd import ops

    E, g = 70, torch.Generator().manual_seed(bm)
    n = 9001
    ids = torch.randint(-1, E, (n,), generator=g).int()
    ids[ids == 3] = 4                                          # an expert without rows
    max_p = (n + E * (bm - 1) + bm - 1) // bm * bm
    t = lambda m: torch.full((m,), 7, dtype=torch.int32, device="cuda")  # noqa: E731
    srt, tile_e, offs, total, inv = t(max_p), t(max_p // bm), t(E + 1), t(1), t(n)
    ops.native().moe_align(ids.cuda(), E, srt, tile_e, offs, total, inv, bm)
    srt, tile_e, offs, inv = (x.cpu().long() for x in (srt, tile_e, offs, inv))
    cnt = torch.bincount(ids[ids >= 0].long(), minlength=E)
    seg = (cnt + bm - 1) // bm * bm
    assert torch.equal(offs, torch.cat([torch.zeros(1, dtype=torch.long), seg.cumsum(0)])) and int(total) == int(seg.sum())
    assert torch.equal(tile_e[:int(total) // bm], torch.repeat_interleave(torch.arange(E), seg // bm))
    assert (tile_e[int(total) // bm:] == -1).all() and torch.equal(inv < 0, ids < 0)
    ok = (ids >= 0).nonzero()[:, 0]
    assert torch.equal(srt[inv[ok]], ok) and int((srt >= 0).sum()) == len(ok)
    first = offs[ids[ok].long()]
    assert (inv[ok] >= first).all() and (inv[ok] < first + cnt[ids[ok].long()]).all()


@pytest.mark.parametrize("n,E", [(100, 1025), (4097, 1025), (100, 4096), (4097, 4096), (1, 4096)])
def test_align_tables_of_many_experts(n, E):
    """More experts than a workgroup has threads, on both sides of the line to many workgroups."""
    from llmd_amd import ops

    bm = 64
    ids = torch.randint(-1, E, (n,), generator=torch.Generator().manual_seed(n + E)).int()
    max_p = (n + E * (bm - 1) + bm - 1) // bm * bm
    t = lambda m: torch.full((m,), 7, dtype=torch.int32, device="cuda")  # noqa: E731
    srt, tile_e, offs, total, inv = t(max_p), t(max_p // bm), t(E + 1), t(1), t(n)
    ops.native().moe_align(ids.cuda(), E, srt, tile_e, offs, total, inv, bm)
    srt, tile_e, offs, inv = (x.cpu().long() for x in (srt, tile_e, offs, inv))
    cnt = torch.bincount(ids[ids >= 0].long(), minlength=E)
    seg = (cnt + bm - 1) // bm * bm
    assert torch.equal(offs, torch.cat([torch.zeros(1, dtype=torch.long), seg.cumsum(0)])) and int(total) == int(seg.sum())
    assert torch.equal(tile_e[:int(total) // bm], torch.repeat_interleave(torch.arange(E), seg // bm))
    assert (tile_e[int(total) // bm:] == -1).all() and torch.equal(inv < 0, ids < 0)
    ok = (ids >= 0).nonzero()[:, 0]
    assert torch.equal(srt[inv[ok]], ok) and int((srt >= 0).sum()) == len(ok)
