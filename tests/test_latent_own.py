"""Latent attention of prompts over keys and values of their own against 64 bits, as an op and in a layer beside single tokens."""
import copy

import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu


def _exact(q, q_rot, cache, uk, uv, scale, meta, gate):
    """In 64 bits: q [T, H, 128], q_rot [T, H, 64], cache [blocks, bs, R + 64], uk, uv [H, 128, R]."""
    T, H, _ = q.shape
    R, bs = uk.shape[2], cache.shape[1]
    out = torch.empty(T, H, 128, dtype=torch.float64)
    for t in range(T):
        s, n = int(meta.row_seq[t]), int(meta.row_len[t])
        rows = torch.cat([cache[int(b)] for b in meta.tables[s, :-(-n // bs)]])[:n]
        k, v = rows[:, :R] @ uk.transpose(1, 2), rows[:, :R] @ uv.transpose(1, 2)  # [H, n, 128]
        z = ((k @ q[t, :, :, None])[..., 0] + q_rot[t] @ rows[:, R:].T) * scale
        out[t] = (torch.softmax(z, -1)[:, None] @ v)[:, 0]
    return out if gate is None else out * torch.sigmoid(gate)[:, :, None]


@pytest.mark.parametrize("runs", [[(0, 2)], [(0, 31), (0, 32), (0, 33)], [(40, 1), (7, 1), (0, 65), (64, 64), (95, 3)], [(129, 130)]],
                         ids=["smallest", "tiles", "singles", "items"])
@pytest.mark.parametrize("H,R,bs,gated", [(16, 512, 64, True), (1, 64, 16, False), (5, 192, 24, True)])
def test_latent_own(H, R, bs, gated, runs):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(H + R)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    meta, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    q, q_abs, cache, gate = rand(T, H * 192), rand(T, H, R + 64), rand(pages, bs, R + 64), rand(T, H)
    uk, uv = rand(H, 128, R) * R ** -0.5, rand(H, 128, R) * R ** -0.5
    want = _exact(q.double().view(T, H, 192)[:, :, :128], q_abs.double()[:, :, R:], cache.double(), uk.double(), uv.double(), 0.07, meta,
                  gate.double() if gated else None)
    for i, (e, n) in enumerate(runs):  # what lies past a sequence's end must not matter
        cache[int(meta.tables[i, (e + n - 1) // bs]), (e + n - 1) % bs + 1:] = float("nan")
    m, _ = _meta(runs, bs, "cuda")
    m.ctx_lens, m.q_lens = [e + n for e, n in runs], [n for _, n in runs]
    first = m.singles()
    out = torch.full((T, H, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    w_kv = torch.cat([uk, uv], 1).reshape(-1, R).cuda()
    sm.latent_own(q.cuda(), q_abs.cuda(), cache.cuda(), w_kv, 0.07, R, m, first, gate.cuda() if gated else None, out)
    got, want = out.cpu()[first:], want[first:]
    assert out[:first].isnan().all()  # left to the other form
    # keys, values and results rounded to bf16, 2^-9 each at most: the first move scores by 2^-9 of their spread
    assert (got.double() - want).norm() <= 3 * 2 ** -9 * want.norm() and ((got - want).abs() <= 2 ** -5 * want.abs().clamp(min=1)).all()


@pytest.mark.parametrize("runs,own", [([(150, 1), (90, 1), (40, 150), (0, 77)], 2), ([(0, 300)], 0), ([(300, 1), (17, 1)], None), ([(3, 40)], None)])
def test_layer(runs, own):
    """A layer takes either form or both in one step, and its single tokens the kernel of steps that hold nothing else."""
    from llmd_amd.engine.attn_meta import AttnMeta
    from llmd_amd.models.mixers import LatentAttention
    from llmd_amd.ops import seqmix as sm

    torch.manual_seed(1)
    layer = LatentAttention(256, 16, 128, 64, 128, 512, 192 ** -0.5, 64, 10000.0, 1e-6, 1024, "cpu", torch.bfloat16, q_rank=128, gate=True)
    for p in layer.parameters():
        p.data.normal_(0, 0.05) if p.dim() > 1 else p.data.uniform_(0.8, 1.2)
    T = sum(n for _, n in runs)
    h = torch.randn(T, 256).bfloat16()
    outs = []
    for dev, dt in (("cpu", torch.float32), ("cuda", torch.bfloat16)):
        m, pages = _meta(runs, 64, dev)
        m.ctx_lens, m.q_lens = [e + n for e, n in runs], [n for _, n in runs]
        pos = torch.cat([torch.arange(e, e + n) for e, n in runs])
        slots = torch.cat([m.tables[i].cpu()[torch.arange(e, e + n) // 64] * 64 + torch.arange(e, e + n) % 64 for i, (e, n) in enumerate(runs)])
        l = copy.deepcopy(layer).to(dev, dt)
        l.cos_sin = layer.cos_sin.to(dev)  # stays fp32
        l.finalize()
        cache = torch.randn(pages, 1, 1, 64, 576, generator=torch.Generator().manual_seed(2)).bfloat16()
        l.bind_cache(cache.to(dev, dt))
        if dev == "cuda":
            assert sm.latent_own_from(m, 16, 128, 64, 128, 512, dt) == own
        outs.append(l(h.to(dev, dt), AttnMeta(num_tokens=T, positions=pos.to(dev), slot_mapping=slots.long().to(dev), seq=m)).float().cpu())
    # bf16 throughout: about ten roundings of 2^-9 in a row
    assert (outs[1] - outs[0]).norm() <= 10 * 2 ** -9 * outs[0].norm()


@pytest.mark.parametrize("H,at_once", [(5, 2), (64, 24), (64, 64), (3, 1), (128, 128)])
def test_heads_in_groups(H, at_once, monkeypatch):
    """Keys and values of some heads at a time, where those of all would take too much memory."""
    from llmd_amd.ops import seqmix as sm

    runs, R, bs = [(40, 1), (3, 70), (0, 33)], 128, 64
    g = torch.Generator().manual_seed(H)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    meta, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    q, q_abs, cache, gate = rand(T, H * 192), rand(T, H, R + 64), rand(pages, bs, R + 64), rand(T, H)
    uk, uv = rand(H, 128, R) * R ** -0.5, rand(H, 128, R) * R ** -0.5
    want = _exact(q.double().view(T, H, 192)[:, :, :128], q_abs.double()[:, :, R:], cache.double(), uk.double(), uv.double(), 0.07, meta, gate.double())
    m, _ = _meta(runs, bs, "cuda")
    monkeypatch.setattr(sm, "LATENT_OWN_BYTES", 106 * 512 * at_once + 511)
    out = torch.full((T, H, 128), float("nan"), dtype=torch.bfloat16, device="cuda")
    sm.latent_own(q.cuda(), q_abs.cuda(), cache.cuda(), torch.cat([uk, uv], 1).reshape(-1, R).cuda(), 0.07, R, m, 1, gate.cuda(), out)
    got, want = out.cpu()[1:], want[1:]
    assert out[:1].isnan().all()
    assert (got.double() - want).norm() <= 3 * 2 ** -9 * want.norm() and ((got - want).abs() <= 2 ** -5 * want.abs().clamp(min=1)).all()


@pytest.mark.parametrize("H,R,runs,own", [(16, 512, [(0, 128)], 0), (1, 512, [(4000, 64)], 0), (64, 64, [(0, 2048)], 0), (64, 512, [(4000, 9)], 0),
                                          (16, 512, [(9, 1), (0, 20)], None), (128, 512, [(9, 1), (500, 16)], 1), (128, 512, [(9, 1)], None),
                                          (16, 96, [(0, 128)], None)])
def test_form(H, R, runs, own):
    from llmd_amd.ops import seqmix as sm

    assert sm.latent_own_from(_meta(runs, 64, "cuda")[0], H, 128, 64, 128, R, torch.bfloat16) == own


def test_layer_with_anothers_cache():
    """A layer that reads an earlier layer's latents makes keys and values of them with its own weights."""
    from llmd_amd.engine.attn_meta import AttnMeta
    from llmd_amd.models.mixers import LatentAttention
    from llmd_amd.ops import seqmix as sm

    torch.manual_seed(1)
    runs, T = [(70, 1), (40, 150), (0, 77)], 228
    args = (256, 16, 128, 64, 128, 512, 192 ** -0.5, 64, 10000.0, 1e-6, 1024, "cpu", torch.bfloat16)
    first = LatentAttention(*args, q_rank=128)
    second = LatentAttention(*args, q_rank=128, gate=True, kv_source=first)
    both = torch.nn.ModuleList([first, second])
    for p in both.parameters():
        p.data.normal_(0, 0.05) if p.dim() > 1 else p.data.uniform_(0.8, 1.2)
    h, outs = torch.randn(T, 256).bfloat16(), []
    for dev, dt in (("cpu", torch.float32), ("cuda", torch.bfloat16)):
        m, pages = _meta(runs, 64, dev)
        pos = torch.cat([torch.arange(e, e + n) for e, n in runs])
        slots = torch.cat([m.tables[i].cpu()[torch.arange(e, e + n) // 64] * 64 + torch.arange(e, e + n) % 64 for i, (e, n) in enumerate(runs)])
        a, b = copy.deepcopy(both).to(dev, dt)
        for layer in (a, b):
            layer.cos_sin = first.cos_sin.to(dev)  # stays fp32
            layer.finalize()
        assert b._src[0] is a
        a.bind_cache(torch.randn(pages, 1, 1, 64, 576, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev, dt))
        if dev == "cuda":
            assert sm.latent_own_from(m, 16, 128, 64, 128, 512, dt) == 1
        meta = AttnMeta(num_tokens=T, positions=pos.to(dev), slot_mapping=slots.long().to(dev), seq=m)
        x = h.to(dev, dt)
        outs.append([y.float().cpu() for y in (a(x, meta), b(x, meta))])
    for got, want in zip(outs[1], outs[0]):  # (as in test_layer)
        assert (got - want).norm() <= 10 * 2 ** -9 * want.norm()
