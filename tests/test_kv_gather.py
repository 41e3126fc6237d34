"""The gather of an 8-bit cache's blocks (ops.kv_dequant_gather) on the GPU: blocks of less and more than a workgroup's part, tables
with and without contexts, contexts around the last block that has to be copied."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hkv,bs,D", [(1, 16, 64), (8, 64, 128), (3, 32, 128), (2, 64, 64)])
@pytest.mark.parametrize("known", [False, True])
def test_gather(Hkv, bs, D, known):
    from llmd_amd import ops

    g = torch.Generator().manual_seed(Hkv + bs)
    S, mb, n = 4, 23, 40
    k, v = ((torch.randn(n, Hkv, bs, D, generator=g) * 3).to(ops.FP8) for _ in range(2))
    bt = torch.randint(0, n, (S, mb), generator=g, dtype=torch.int32)
    bt[2, 5:] = -1
    ctx = torch.tensor([1, bs * mb, 5 * bs, 6 * bs + 1], dtype=torch.int32)
    kw, vw, tw = ops.kv_dequant_gather(k, v, bt)
    kd, vd, t = ops.kv_dequant_gather(k.cuda(), v.cuda(), bt.cuda(), ctx.cuda() if known else None)
    assert torch.equal(t.cpu(), tw)
    for s in range(S):
        # the last tile of 64 keys that an item meets is whole
        m = mb if not known else min(mb, -(-(-(-int(ctx[s]) // 64) * 64) // bs))
        at = slice(s * mb, s * mb + m)
        assert torch.equal(kd[at].cpu().float(), kw[at].float()) and torch.equal(vd[at].cpu().float(), vw[at].float())


@pytest.mark.parametrize("rows,lens", [(3, 3), (5, 3), (3, 6)])
def test_prefill_with_other_numbers_of_contexts(rows, lens):
    """A table may have more rows than the step has sequences, and the contexts' buffer more entries."""
    from llmd_amd import ops

    g = torch.Generator().manual_seed(rows + lens)
    Hq, Hkv, D, bs, n, mb = 8, 2, 128, 64, 30, 6
    k, v = (torch.randn(n, Hkv, bs, D, generator=g).to(ops.FP8).cuda() for _ in range(2))
    bt = torch.randperm(n, generator=g)[:rows * mb].view(rows, mb).int().cuda()
    ql, cl = [40, 1, 100], [40, 130, 380]
    q = torch.randn(sum(ql), Hq * D, generator=g).bfloat16().cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    items = i32(ops.build_prefill_items(ql, cl, ops.prefill_tokens_per_item(Hq, Hkv, D, bs, False)))
    run = lambda bt, c: ops.paged_prefill(q, k, v, bt, i32([0, 40, 41]), i32(ql), c, Hq, Hkv, D, D ** -0.5, items=items)  # noqa: E731
    want = run(bt[:3].contiguous(), i32(cl))
    got = run(bt, i32(cl + [7] * (lens - 3)))
    assert torch.isfinite(want).all() and torch.equal(got, want)


@pytest.mark.parametrize("D,bs,G", [(128, 64, 4), (64, 16, 1), (128, 32, 2)])
def test_prefill_does_not_read_what_is_not_copied(D, bs, G):
    """Long tables, short contexts, copies in memory that held NaNs."""
    from llmd_amd import ops

    g = torch.Generator().manual_seed(D + bs)
    Hkv, n, mb = 2, 70, 64
    Hq = Hkv * G
    k, v = (torch.randn(n, Hkv, bs, D, generator=g).to(ops.FP8).cuda() for _ in range(2))
    ql, cl = [1, 33, 64, 200, 5], [1, 33, 65, 257, 6 * 64 - 1]
    S = len(ql)
    bt = torch.randint(0, n, (S, mb), generator=g, dtype=torch.int32).cuda()
    q = torch.randn(sum(ql), Hq * D, generator=g).bfloat16().cuda()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    start = i32([sum(ql[:i]) for i in range(S)])
    items = i32(ops.build_prefill_items(ql, cl, ops.prefill_tokens_per_item(Hq, Hkv, D, bs, False)))
    run = lambda k, v, bt: ops.paged_prefill(q, k, v, bt, start, i32(ql), i32(cl), Hq, Hkv, D, D ** -0.5, items=items)  # noqa: E731
    # the same blocks, widened by torch, in the kernel that takes them as they are
    want = run(k.bfloat16(), v.bfloat16(), bt)
    for turn in range(2):
        held = [torch.full((S * mb, Hkv, bs, D), -1, dtype=torch.int16, device="cuda") for _ in range(4)]
        del held
        got = run(k, v, bt)
        assert torch.isfinite(got).all() and torch.equal(got, want), turn
