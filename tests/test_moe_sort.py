"""Pairs sorted by expert over many workgroups: at the line to the single-workgroup form and at the edges of their blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4096, 4097, 6144, 20256])
@pytest.mark.parametrize("E", [1, 70, 300])
def test_group_tables(n, E):
    from llmd_amd import ops
    from llmd_amd.ops import seqmix as sm

    ids = torch.randint(-1, E + 1, (n,), generator=torch.Generator().manual_seed(n + E)).int()
    if E > 3:
        ids[ids == 3] = 4                                      # an expert without rows
    here = (ids >= 0) & (ids < E)
    cnt = torch.bincount(ids[here].long(), minlength=E)
    for tm, call in ((64, lambda *a: sm.native().moe_group(a[0], E, 64, *a[1:])), (128, lambda *a: ops.native().moe_group(a[0], E, *a[1:]))):
        mt = (n + E * (tm - 1) + tm - 1) // tm
        t = lambda m: torch.full((m,), 7, dtype=torch.int32, device="cuda")  # noqa: E731
        row, tiles, slot = t(mt * tm), t(1 + 3 * mt), t(n)
        call(ids.cuda(), row, tiles, slot)
        row, tiles, slot = row.cpu().long(), tiles.cpu().long(), slot.cpu().long()
        nt = (cnt + tm - 1) // tm
        first = nt.cumsum(0) - nt
        assert int(tiles[0]) == int(nt.sum())
        want = [[e | min(tm, int(cnt[e]) - tm * i) << 16, int(first[e]), int(nt[e])] for e in range(E) for i in range(int(nt[e]))]
        assert tiles[1:1 + 3 * len(want)].view(-1, 3).tolist() == want
        ok = here.nonzero()[:, 0]
        assert (slot[~here] == -1).all() and torch.equal(row[slot[ok]], ok)
        rank = slot[ok] - first[ids[ok].long()] * tm
        assert (rank >= 0).all() and (rank < cnt[ids[ok].long()]).all()


@pytest.mark.parametrize("n,E", [(0, 5), (1, 1), (8, 128), (100, 1025), (4097, 1025), (100, 4096), (4097, 4096), (100, 4097), (4097, 4097),
                                 (130, 8192), (4224, 33)])
@pytest.mark.parametrize("spread", [1, 4, 1000])
def test_tables_of_the_least_size(n, E, spread):
    """Tables with no tile to spare, pairs on one, four or many experts; more experts than a workgroup has threads, on both
    sides of the line to many workgroups (above 4096 experts one workgroup sorts all)."""
    from llmd_amd import ops
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(n + E)
    some = torch.randperm(E, generator=g)[:spread]
    ids = some[torch.arange(n) % len(some)].int()
    cnt = torch.bincount(ids.long(), minlength=E)
    calls = [(64, lambda *a: sm.native().moe_group(a[0], E, 64, *a[1:])), (128, lambda *a: sm.native().moe_group(a[0], E, 128, *a[1:]))]
    if E <= 4096:
        calls.append((128, lambda *a: ops.native().moe_group(a[0], E, *a[1:])))
    for tm, call in calls:
        mt = max(1, (n + min(E, n) * (tm - 1)) // tm)
        t = lambda m: torch.full((m,), 7, dtype=torch.int32, device="cuda")  # noqa: E731
        row, tiles, slot = t(mt * tm), t(1 + 3 * mt), t(n)
        call(ids.cuda(), row, tiles, slot)
        row, tiles, slot = row.cpu().long(), tiles.cpu().long(), slot.cpu().long()
        nt = (cnt + tm - 1) // tm
        first = nt.cumsum(0) - nt
        assert int(tiles[0]) == int(nt.sum()) <= mt
        want = [[e | min(tm, int(cnt[e]) - tm * i) << 16, int(first[e]), int(nt[e])] for e in range(E) for i in range(int(nt[e]))]
        assert tiles[1:1 + 3 * len(want)].view(-1, 3).tolist() == want
        assert torch.equal(row[slot], torch.arange(n))
        rank = slot - first[ids.long()] * tm
        assert (rank >= 0).all() and (rank < cnt[ids.long()]).all()


@pytest.mark.parametrize("gated", ["ops", "seqmix", "seqmix float32"])
def test_workspace_of_small_steps(gated):
    """One token with eight choices among 128 experts: eight tiles, not one for each expert."""
    from llmd_amd import ops
    from llmd_amd.ops import seqmix as sm

    E, d, F, k = 128, 256, 64, 8
    dt = torch.float32 if "32" in gated else torch.bfloat16
    g = torch.Generator(device="cuda").manual_seed(0)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dt)  # noqa: E731
    x, w1, w2 = rand(1, d), rand(E, 2 * F, d) * d ** -0.5, rand(E, d, F) * F ** -0.5
    ids, w = torch.arange(3, 3 + k, dtype=torch.int32, device="cuda")[None], torch.full((1, k), 1 / k, device="cuda")

    def call():
        if gated == "ops":
            return ops.moe_experts(x, ids, w, w1, w2, ops.ACT_SILU)
        return sm.moe_gated_ffn(x, ids, w, w1, w2, "silu")

    call()
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    call()
    # rows of h or a (F) and y (d) of eight tiles of 128 slots, tables, and 512 bytes of rounding for each of about ten tensors
    assert torch.cuda.max_memory_allocated() - before <= 8 * 128 * (F + d) * dt.itemsize + 16384
