"""Values of a step's tokens in the transposed pages: eight neighbouring places at a time, wherever in the step and in a page they begin."""
import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [64, 8, 12])  # (12: no groups of eight)
@pytest.mark.parametrize("vdim,form", [(128, "wide"), (128, "plain"), (40, "plain"), (128, "v_from_k")])
@pytest.mark.parametrize("runs", [[(0, 256)], [(5, 1), (70, 1), (333, 101), (7, 90), (64, 80)], [(3, 259), (0, 7), (1, 8)]],
                         ids=["aligned", "portions", "ends"])
def test_value_groups(runs, vdim, form, bs):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(vdim)
    meta, pages = _meta(runs, bs, "cpu")
    T, Hq, Hkv, dim = sum(n for _, n in runs), 6, 2, 128
    pos = torch.cat([torch.arange(e, e + n) for e, n in runs])
    slots = torch.cat([meta.tables[i].long()[torch.arange(e, e + n) // bs] * bs + torch.arange(e, e + n) % bs for i, (e, n) in enumerate(runs)])
    slots[T // 2] = -1  # one that is not written
    nv = 0 if form == "v_from_k" else Hkv * vdim
    p = torch.randn(T, (Hq + Hkv) * dim + nv, generator=g).bfloat16()
    cs, qk_w = torch.randn(1024, 64, generator=g), torch.rand((Hq + Hkv) * dim if form == "wide" else 2 * dim, generator=g)
    args = dict(qk_w=qk_w if form == "wide" else qk_w.view(2, dim), wide_norm=form == "wide", v_from_k=form == "v_from_k")
    caches = []
    for dev in ("cpu", "cuda"):
        cache = torch.full((pages, Hkv, bs, dim + vdim), 7.0).bfloat16().to(dev)
        q = torch.empty(T, Hq, dim, dtype=torch.bfloat16, device=dev)
        sm.qkv_rope_cache(p.to(dev), None, pos.to(dev), cs.to(dev), Hq, Hkv, dim, vdim, 64, False, 1e-6, None, 0, 0.0, slots.to(dev), cache, q,
                          **{k: v.to(dev) if torch.is_tensor(v) else v for k, v in args.items()})
        caches.append((cache.cpu(), q.cpu()))
    (c0, q0), (c1, q1) = caches
    v0, v1 = (c.view(pages, Hkv, -1)[:, :, bs * dim:] for c in (c0, c1))
    assert torch.equal(v0, v1)  # values are copies
    # keys and queries: fp32 throughout, one rounding to bf16 on both sides
    assert ((c1.float() - c0.float()).abs() <= 2 ** -7 * c0.float().abs() + 1e-5).all()
    assert ((q1.float() - q0.float()).abs() <= 2 ** -7 * q0.float().abs() + 1e-5).all()


@pytest.mark.parametrize("Hkv,vdim", [(1, 8), (1, 72), (3, 24), (1, 264)])
@pytest.mark.parametrize("wide", [True, False])
def test_waves_with_few_columns(Hkv, vdim, wide):
    """A workgroup's last wave has eight columns: its other lanes hold the tokens' places all the same."""
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(vdim)
    runs, bs, Hq, dim = [(5, 1), (333, 101), (7, 90), (64, 80)], 64, 6, 128
    meta, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    pos = torch.cat([torch.arange(e, e + n) for e, n in runs])
    slots = torch.cat([meta.tables[i].long()[torch.arange(e, e + n) // bs] * bs + torch.arange(e, e + n) % bs for i, (e, n) in enumerate(runs)])
    p = torch.randn(T, (Hq + Hkv) * dim + Hkv * vdim, generator=g).bfloat16()
    cs, qk_w = torch.randn(1024, 64, generator=g), torch.rand((Hq + Hkv) * dim if wide else 2 * dim, generator=g)
    got = []
    for dev in ("cpu", "cuda"):
        cache = torch.full((pages, Hkv, bs, dim + vdim), 7.0).bfloat16().to(dev)
        q = torch.empty(T, Hq, dim, dtype=torch.bfloat16, device=dev)
        sm.qkv_rope_cache(p.to(dev), None, pos.to(dev), cs.to(dev), Hq, Hkv, dim, vdim, 64, False, 1e-6, None, 0, 0.0, slots.to(dev), cache, q,
                          qk_w=(qk_w if wide else qk_w.view(2, dim)).to(dev), wide_norm=wide)
        got.append(cache.cpu().view(pages, Hkv, -1)[:, :, bs * dim:])
    assert torch.equal(got[0], got[1])
