"""float32 grouped attention on the matrix cores against the plain reference: sizes around the compiled forms, portions and
single tokens (with cut key ranges), every score option."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _meta(runs, bs, dev):
    from llmd_amd.engine.attn_meta import SeqMeta

    ql = [n for _, n in runs]
    ctx = [e + n for e, n in runs]
    W = max(-(-c // bs) for c in ctx) + 1
    tables = np.zeros((len(runs), W), np.int32)
    order, at = np.random.default_rng(0).permutation(sum(-(-c // bs) for c in ctx)).astype(np.int32), 0
    for i, c in enumerate(ctx):
        n = -(-c // bs)
        tables[i, :n] = order[at:at + n]
        at += n
    t = lambda x: torch.tensor(x, dtype=torch.int32).to(dev)  # noqa: E731
    return SeqMeta(num_seqs=len(runs), seq_start=t(np.cumsum([0] + ql)), seq_slot=t([0] * len(runs)),
                   seq_init=t([int(e > 0) for e, _ in runs]), row_seq=t(np.repeat(np.arange(len(runs)), ql)),
                   row_len=t(np.concatenate([np.arange(e, e + n) + 1 for e, n in runs])),
                   tables=torch.from_numpy(tables).to(dev), max_len=max(ctx), max_q=max(ql), q_lens=ql, ctx_lens=ctx), at


@pytest.mark.parametrize("runs", [[(0, 37), (5, 1), (100, 64)], [(700, 1), (31, 1), (32, 1)], [(0, 1)]],
                         ids=["portions", "single", "first"])
@pytest.mark.parametrize("opts", [{}, {"window": 40, "keep_first": 3, "sinks": True}, {"chunk": 50, "slopes": True}, {"gate": True}],
                         ids=["causal", "window", "chunk", "gate"])
@pytest.mark.parametrize("Hq,Hkv,dim,vdim,bs", [(8, 2, 128, 128, 64), (6, 2, 40, 24, 32), (4, 4, 96, 256, 64), (3, 1, 30, 17, 16)])
def test_grouped_attention_f32(Hq, Hkv, dim, vdim, bs, opts, runs):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(dim)
    got = {}
    rand = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    meta, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    q, cache, gate = rand(T, Hq, dim), rand(pages, Hkv, bs, dim + vdim), rand(T, Hq * vdim)
    slopes, sinks = torch.rand(Hq, generator=g) * 0.05, rand(Hq)
    for dev in ("cpu", "cuda"):
        m, _ = _meta(runs, bs, dev)
        kw = dict(opts)
        kw = {k: {"sinks": sinks, "slopes": slopes, "gate": gate}[k].to(dev) if v is True else v for k, v in kw.items()}
        c = cache.to(dev)
        if dev == "cuda":  # what lies past a sequence's end must not matter
            for i, (e, n) in enumerate(runs):
                last, used = (e + n - 1) // bs, (e + n - 1) % bs + 1
                p = int(m.tables[i, last])
                c[p].view(Hkv, -1)[:, :bs * dim].view(Hkv, bs, dim)[:, used:] = float("nan")
                c[p].view(Hkv, -1)[:, bs * dim:].view(Hkv, vdim, bs)[:, :, used:] = float("nan")
        got[dev] = sm.grouped_attention(q.to(dev), c, dim, vdim, dim ** -0.5, m, **kw).cpu()
    # scores are sums of ``dim`` products of order 1, outputs weighted means of values of order 1: a few hundred fp32 roundings
    assert (got["cuda"] - got["cpu"]).abs().max() <= 2e-5


@pytest.mark.parametrize("opts", [{}, {"window": 300, "keep_first": 3, "sinks": True}, {"window": 40, "keep_first": 290},
                                  {"chunk": 270, "slopes": True}, {"gate": True, "window": 700}],
                         ids=["causal", "window", "kept", "chunk", "gate"])
@pytest.mark.parametrize("Hq,Hkv,dim,bs", [(8, 2, 128, 64), (3, 1, 30, 16), (6, 6, 200, 32)])
def test_rows_do_not_depend_on_the_step(Hq, Hkv, dim, bs, opts, monkeypatch):
    """A token's result has the same bits in a whole prompt, in portions of it, alone, in a batch of single tokens whose key
    ranges run as workgroups of their own, and in one where they do not."""
    from llmd_amd.ops import seqmix as sm

    n, at = 900, [0, 30, 255, 256, 257, 511, 600, 899]
    g = torch.Generator().manual_seed(dim)
    whole, pages = _meta([(0, n)], bs, "cuda")
    q = torch.randn(n, Hq, dim, generator=g) * 2.0 ** torch.randint(-1, 4, (n, Hq, 1), generator=g)
    cache, gate = torch.randn(pages, Hkv, bs, 2 * dim, generator=g), torch.randn(n, Hq * dim, generator=g)
    vals = {"sinks": torch.randn(Hq, generator=g), "slopes": torch.rand(Hq, generator=g) * 0.05}

    def run(runs, rows, dev="cuda"):
        m, _ = _meta(runs, bs, dev)
        m.tables = whole.tables[:, :].expand(len(runs), -1).contiguous().to(dev)
        kw = {k: (gate[rows] if k == "gate" else vals[k]).to(dev) if v is True else v for k, v in opts.items()}
        return sm.grouped_attention(q[rows].to(dev), cache.to(dev), dim, dim, dim ** -0.5, m, **kw).cpu()

    want = run([(0, n)], list(range(n)))
    plain = run([(0, n)], list(range(n)), "cpu")
    # scores are sums of ``dim`` products, up to 8 times their usual size, outputs weighted means of values of order 1
    assert (want - plain).abs().max() <= 1e-4
    cuts = (0, 250, 251, 519, n)
    for a, b in zip(cuts, cuts[1:]):
        assert torch.equal(run([(a, b - a)], list(range(a, b))), want[a:b])
    singles = [(p, 1) for p in at]
    for wgs in (512, 1):
        monkeypatch.setattr(sm, "GQA_DECODE_WGS", wgs)
        assert torch.equal(run(singles, at), want[at])
        for p in at:
            assert torch.equal(run([(p, 1)], [p]), want[p:p + 1])


def test_rows_do_not_depend_on_the_plan():
    """Ranges planned for contexts far longer than the step's (a captured step), more of them than workgroups."""
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(1)
    for B, n in ((1, 3000), (40, 700)):
        m, pages = _meta([(n - 1 - i, 1) for i in range(B)], 64, "cuda")
        q, cache = torch.randn(B, 8, 64, generator=g).cuda(), torch.randn(pages, 4, 64, 128, generator=g).cuda()
        out = []
        for m.max_len in (n, 9000, 131072):
            for kw in ({}, {"window": 500, "keep_first": 200}):
                out.append(sm.grouped_attention(q, cache, 64, 64, 0.125, m, **kw))
        assert all(torch.equal(a, b) for a, b in zip(out, out[2:]))
