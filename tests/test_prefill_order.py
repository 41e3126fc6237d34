"""Prompt attention over the paged cache: the order in which workgroups take (item, head group) pairs, at grids of one round and more,
head groups in multiples of 8 and not, numbers that 8 does and does not divide: every pair is taken, and has its bits in the plain order."""
import pytest
import torch

from llmd_amd import ops
from llmd_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


# (heads, kv heads, [(earlier, tokens)]) -> workgroups
@pytest.mark.parametrize("Hq,Hkv,runs,wgs", [
    (32, 4, [(0, 1025)], 264), (32, 4, [(0, 2048)], 512), (32, 4, [(0, 2049)], 520), (64, 8, [(70, 31), (0, 530)], 288),
    (24, 3, [(0, 1381)], 264), (20, 4, [(0, 1700)], 280), (40, 8, [(5, 1700)], 560), (8, 1, [(0, 8200)], 514), (18, 3, [(0, 1800), (0, 1)], 270)])
def test_every_item_is_taken(Hq, Hkv, runs, wgs):
    D, bs = 64, 64
    g = torch.Generator().manual_seed(Hq)
    pages = [-(-(e + n) // bs) for e, n in runs]
    kc, vc = (torch.randn(sum(pages), Hkv, bs, D, generator=g).bfloat16().cuda() for _ in range(2))
    bt = torch.zeros(len(runs), max(pages), dtype=torch.int32)
    for i, n in enumerate(pages):
        bt[i, :n] = torch.arange(sum(pages[:i]), sum(pages[:i]) + n)
    ql, ctx = [n for _, n in runs], [e + n for e, n in runs]
    qs = [sum(ql[:i]) for i in range(len(ql))]
    q = torch.randn(sum(ql), Hq * D, generator=g).bfloat16().cuda()
    groups = Hkv * (Hq // Hkv // {0: 4, 2: 2}.get(Hq // Hkv % 4, 1))
    items = ops.build_prefill_items(ql, ctx, ops.prefill_tokens_per_item(Hq, Hkv, D, bs, False))
    assert len(items) * groups == wgs
    items = torch.tensor(items, dtype=torch.int32).cuda()
    args = [torch.tensor(x, dtype=torch.int32).cuda() for x in (qs, ql, ctx)]

    def run(part):
        return ops.paged_prefill(q, kc, vc, bt.cuda(), *args, Hq, Hkv, D, D ** -0.5, items=part, out=out)

    out = torch.full((sum(ql), Hq * D), float("nan"), dtype=torch.bfloat16, device="cuda")
    got = run(items).clone()
    out.fill_(float("nan"))
    for a in range(0, len(items), 256 // groups):  # grids of at most 256: the plain order
        run(items[a:a + 256 // groups])
    assert torch.equal(got, out)
    n = min(ql[0], 300)  # and the oracle's numbers, over the first rows
    want = ref.paged_prefill(q[:n].float(), kc.float(), vc.float(), bt[:1].cuda(), torch.tensor([0]), torch.tensor([n]),
                             torch.tensor([runs[0][0] + n]), Hq, Hkv, D, D ** -0.5)
    # bf16 results: 2^-9 of each. A weight is rounded to bf16 (2^-9) and so are the scaled queries: a score is off by 64 roundings of 2^-9 of
    # products of about 1, times 64^-0.5: 2^-9, four times that for the largest of many. Of values up to about 5
    assert ((got[:n].float() - want).abs() <= 2 ** -8 * want.abs() + 5 * (2 ** -7 + 2 ** -9)).all()
