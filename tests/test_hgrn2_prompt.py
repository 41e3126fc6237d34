"""HGRN2 over prompts, bf16: the matrix-core form at its edges (blocks of 16, chunks of 64, the compiled head sizes) against the
plain recurrence, with decays from none to total."""
import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[64], [65, 1, 16], [1, 1, 1, 17, 128, 63], [2, 79]], ids=str)
@pytest.mark.parametrize("H,dk,dv,lower,shift", [(2, 64, 64, None, 0.0), (3, 33, 65, 0.0, -12.0), (1, 128, 128, 0.999, 0.0),
                                                 (2, 1, 1, None, 0.0), (2, 30, 7, 0.5, 0.0), (1, 65, 16, 1.0, 0.0)])
def test_hgrn2_prompts(H, dk, dv, lower, shift, lens, monkeypatch):
    from llmd_amd.ops import seqmix as sm

    monkeypatch.setattr(sm, "HGRN2_CHUNK_FROM", 2)

    g = torch.Generator().manual_seed(dk + sum(lens))
    T, n = sum(lens), len(lens)
    p = torch.randn(T, 2 * H * dk + H * dv + 3, generator=g).bfloat16()
    fb = torch.randn(H * dk, generator=g) + shift
    low = torch.rand(H * dk, generator=g) if lower is None else torch.full((H * dk,), lower)
    nw, state = torch.rand(dv, generator=g).bfloat16() + 0.5, torch.randn(n + 1, H, dk, dv, generator=g)
    got = {}
    for dev, x in (("cpu", p.float()), ("cuda", p)):
        m, _ = _meta([(0, k) for k in lens], 64, dev)
        m.seq_slot = torch.arange(n, 0, -1, dtype=torch.int32).to(dev)
        m.seq_init = torch.tensor([i % 2 for i in range(n)], dtype=torch.int32).to(dev)
        st = state.clone().to(dev)
        w = nw.float() if dev == "cpu" else nw
        o = sm.hgrn2_scan(x.to(dev), H, dk, dv, fb.to(dev), low.to(dev), w.to(dev), 1e-5, st, m)
        got[dev] = (o.float().cpu(), st.cpu())
    (want, ws), (o, st) = got["cpu"], got["cuda"]
    # a result's bf16 rounding; before it fp32 values of the size of the head's largest: sums of up to 128 products (1e-5) of write
    # strengths 1 - sigmoid(x), which hold 2^-24 / e^-x of themselves: 1e-5 at x = 5
    scale = want.view(T, H, dv).abs().amax(-1, keepdim=True).expand(T, H, dv).reshape(T, H * dv)
    assert ((o - want).abs() <= 2 ** -8 * want.abs() + 2e-5 * (1 + scale)).all()
    assert (st - ws).abs().max() <= 2e-5 * ws.abs().max()  # up to 128 steps of one rounding each, hardware exponentials


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("at", [0, 7, 15, 16, 70, 98])
def test_later_values_do_not_reach_earlier_tokens(at, bad):
    """An infinite or undefined value changes its own token and those after it, in its head, and nothing else."""
    from llmd_amd.ops import seqmix as sm

    T, H, dk, dv = 99, 2, 64, 40
    g = torch.Generator().manual_seed(at)
    p = torch.randn(T, H * (2 * dk + dv), generator=g).bfloat16().cuda()
    fb, low, nw = torch.randn(H * dk, generator=g).cuda(), torch.rand(H * dk, generator=g).cuda(), torch.ones(dv).bfloat16().cuda()
    out = []
    for v in (0.5, bad):
        p[at, 2 * H * dk + dv + 3] = v  # head 1, column 3
        m, _ = _meta([(0, T)], 64, "cuda")
        st = torch.zeros(1, H, dk, dv, device="cuda")
        out.append((sm.hgrn2_scan(p, H, dk, dv, fb, low, nw, 1e-5, st, m).view(T, H, dv), st))
    (want, ws), (got, gs) = out
    assert torch.equal(got[:at], want[:at]) and torch.equal(got[:, 0], want[:, 0]) and torch.equal(gs[:, 0], ws[:, 0])
    assert not got[at:, 1, 3].isfinite().any() and not gs[0, 1, :, 3].isfinite().any()
    other = torch.arange(dv) != 3
    assert torch.equal(gs[0, 1][:, other], ws[0, 1][:, other])


@pytest.mark.parametrize("dtype,dk", [(torch.float32, 32), (torch.bfloat16, 32), (torch.bfloat16, 130)], ids=str)
def test_chunk_length_option(dtype, dk):
    """Chunks above 64 tokens (LLMD_HGRN2_CHUNK_LEN, read at import) for the scanned form; the matrix-core form keeps its 64."""
    import os
    import subprocess
    import sys

    code = f"""
import torch
from test_grouped_f32 import _meta
from llmd_amd.ops import seqmix as sm
T, H, dk, dv, dt = 300, 2, {dk}, 16, {dtype}
g = torch.Generator().manual_seed(1)
p = torch.randn(T, H * (2 * dk + dv), generator=g).to(dt)
fb, low, nw = torch.randn(H * dk, generator=g), torch.rand(H * dk, generator=g), torch.ones(dv).to(dt)
out = []
for dev in ("cpu", "cuda"):
    m, _ = _meta([(0, T)], 64, dev)
    w = (lambda x: x.float()) if dev == "cpu" else (lambda x: x.cuda())
    out.append(sm.hgrn2_scan(w(p), H, dk, dv, w(fb), w(low), w(nw), 1e-5, torch.zeros(1, H, dk, dv, device=dev), m).float().cpu())
assert list(m._chunks) == [{100 if dtype == torch.float32 or dk > 128 else 64}], list(m._chunks)
# bf16 results: 2^-9 of each; fp32 sums of up to 130 products of values of the size of the head's largest
scale = out[0].abs().max()
assert ((out[1] - out[0]).abs() <= ({2 ** -8 if dtype == torch.bfloat16 else 0.0}) * out[0].abs() + 2e-5 * (1 + scale)).all()
"""
    env = dict(os.environ, LLMD_HGRN2_CHUNK_LEN="100", PYTHONPATH=os.pathsep.join(sys.path))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
