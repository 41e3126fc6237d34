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
