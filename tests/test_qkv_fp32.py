"""The 16-byte form of the fp32 rotation and cache writes: values of eight tokens stored at once and one by one, page borders,
the forms of norm, rotation and values, against the operator on the CPU."""
import pytest
import torch

from llmd_amd.models.mixers import rope_table
from llmd_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,first", [(300, 48), (259, 50), (5, 63)])
@pytest.mark.parametrize("form", ["plain", "unit", "first", "wide", "keys", "mixed", "bias"])
@pytest.mark.parametrize("Hq,Hkv,dim,rot,inter", [(6, 3, 128, 64, False), (4, 1, 32, 32, True), (8, 8, 16, 0, False)])
def test_against_cpu(T, first, form, Hq, Hkv, dim, rot, inter):
    if form == "wide" and inter:
        pytest.skip("norms over whole projections turn half-split pairs")
    g = torch.Generator().manual_seed(T + Hq)
    r = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    n = (Hq + Hkv) * dim + (0 if form == "keys" else Hkv * dim)
    qkv, bias, cache = r(T, n), r(n) if form == "bias" else None, r(9, Hkv, 64, 2 * dim)
    pos = torch.arange(first, first + T)
    slots = torch.randperm(9, generator=g)[pos // 64] * 64 + pos % 64
    slots[3] = -1
    w = None if form in ("plain", "keys", "mixed", "bias") else 1 + 0.3 * r(*(((Hq + Hkv) * dim,) if form == "wide" else (2, dim)))
    cs = rope_table(rot, 300.0, 512, "cpu", None) if rot else None
    out = []
    for dev in ("cpu", "cuda"):
        to = lambda t: None if t is None else t.to(dev).clone()  # noqa: E731
        q, c = torch.empty(T, Hq, dim, device=dev), to(cache)
        sm.qkv_rope_cache(to(qkv), to(bias), to(pos), to(cs), Hq, Hkv, dim, dim, rot, inter, None if w is None else 1e-5,
                          to(qkv[:, -Hkv * dim:].contiguous()) if form == "mixed" else None, 2 if form == "mixed" else 0, 0.3,
                          to(slots), c, q, to(w), form == "first", form == "keys", wide_norm=form == "wide")
        out.append((q.cpu(), c.cpu()))
    for want, got in zip(*out):
        # a mean of up to Hq dim squares, weights, rotation: each step rounded once, in two orders
        assert (got - want).abs().max() <= (Hq * dim + 40) * 2.0 ** -23 * want.abs().max()
