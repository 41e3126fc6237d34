"""Grouped attention over prompts, bf16: the form for whole sizes at its edges against the plain reference: every score option,
portions that end inside a tile, with unwritten keys after them, pages of one and of several tiles."""
import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("runs", [[(0, 1), (0, 2)], [(0, 37), (5, 1), (100, 64)], [(31, 2), (32, 33), (250, 6)]],
                         ids=["smallest", "portions", "edges"])
@pytest.mark.parametrize("opts", [{}, {"window": 40, "keep_first": 3, "sinks": True}, {"chunk": 50, "slopes": True},
                                  {"gate": True, "window": 33}], ids=["causal", "window", "chunk", "gate"])
@pytest.mark.parametrize("Hq,Hkv,dim,bs", [(8, 2, 128, 64), (4, 4, 64, 32), (6, 2, 64, 160), (3, 1, 256, 96), (64, 1, 128, 64)])
def test_grouped_prompt(Hq, Hkv, dim, bs, opts, runs):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(dim + Hq)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    meta, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    q, cache, gate = rand(T, Hq, dim), rand(pages, Hkv, bs, 2 * dim), rand(T, Hq * dim)
    slopes, sinks = torch.rand(Hq, generator=g) * 0.05, torch.randn(Hq, generator=g)
    kw = lambda dev, f: {k: {"sinks": sinks, "slopes": slopes, "gate": f(gate)}[k].to(dev) if v is True else v  # noqa: E731
                         for k, v in opts.items()}
    want = sm.grouped_attention(q.float(), cache.float(), dim, dim, dim ** -0.5, meta, **kw("cpu", torch.Tensor.float))
    for i, (e, n) in enumerate(runs):  # what lies past a sequence's end must not matter
        c = cache[int(meta.tables[i, (e + n - 1) // bs])].view(Hkv, -1)
        used = (e + n - 1) % bs + 1
        c[:, :bs * dim].view(Hkv, bs, dim)[:, used:] = float("nan")
        c[:, bs * dim:].view(Hkv, dim, bs)[:, :, used:] = float("nan")
    m, _ = _meta(runs, bs, "cuda")
    got = sm.grouped_attention(q.cuda(), cache.cuda(), dim, dim, dim ** -0.5, m, **kw("cuda", lambda x: x)).float().cpu()
    # bf16 results: 2^-9 of each; weights in two bf16 parts: 2^-16 of a mean of values up to about 5, and fp32 sums of dim products
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-4).all()


@pytest.mark.parametrize("bs,dim", [(64, 128), (64, 64), (64, 256), (16, 128), (16, 40)])  # whole sizes, general form
@pytest.mark.parametrize("opts", [{}, {"window": 70, "keep_first": 3, "sinks": True}], ids=["causal", "window"])
def test_rows_do_not_depend_on_the_cut(bs, dim, opts):
    """A token's output has the same bits wherever its prompt is cut into portions, whatever its neighbours' scores are."""
    from llmd_amd.ops import seqmix as sm

    n, Hq, Hkv = 300, 6, 2
    g = torch.Generator().manual_seed(dim)
    whole, pages = _meta([(0, n)], bs, "cuda")
    q = torch.randn(n, Hq, dim, generator=g) * 2.0 ** torch.randint(0, 6, (n, Hq, 1), generator=g)  # some rows' maxima jump
    q, cache = q.bfloat16().cuda(), torch.randn(pages, Hkv, bs, 2 * dim, generator=g).bfloat16().cuda()
    sinks = torch.randn(Hq, generator=g).cuda()
    kw = {k: sinks if v is True else v for k, v in opts.items()}
    out = []
    for cuts in ((0, n), (0, 77, n), (0, 3, 130, 131, n)):
        rows = []
        for a, b in zip(cuts, cuts[1:]):
            m, _ = _meta([(a, b - a)], bs, "cuda")
            m.tables = whole.tables
            if b - a == 1:
                m.max_q = 2   # beside a portion: not a step of single tokens
            rows.append(sm.grouped_attention(q[a:b], cache, dim, dim, dim ** -0.5, m, **kw))
        out.append(torch.cat(rows))
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("opts", [{}, {"window": 70, "keep_first": 3, "sinks": True}, {"chunk": 50, "slopes": True}, {"gate": True}],
                         ids=["causal", "window", "chunk", "gate"])
def test_bits_do_not_depend_on_the_form(dim, opts):
    """Pages of whole tiles and smaller ones (the general form) give the same bits."""
    from llmd_amd.ops import seqmix as sm

    runs, Hq, Hkv = [(0, 300), (45, 1), (100, 77)], 6, 2
    g = torch.Generator().manual_seed(dim)
    T = sum(n for _, n in runs)
    q = (torch.randn(T, Hq, dim, generator=g) * 2.0 ** torch.randint(0, 4, (T, Hq, 1), generator=g)).bfloat16().cuda()
    vals = {"sinks": torch.randn(Hq, generator=g), "slopes": torch.rand(Hq, generator=g) * 0.05,
            "gate": torch.randn(T, Hq * dim, generator=g).bfloat16()}
    kw = {k: vals[k].cuda() if v is True else v for k, v in opts.items()}
    keys, values = (torch.randn(len(runs), Hkv, 512, dim, generator=g).bfloat16() for _ in range(2))  # [sequence, head, key]
    out = []
    for bs in (64, 32, 16, 8):
        m, pages = _meta(runs, bs, "cuda")
        cache = torch.zeros(pages, Hkv, bs, 2 * dim).bfloat16()
        for i, (e, n) in enumerate(runs):
            for p in range(-(-(e + n) // bs)):
                c = cache[int(m.tables[i, p])].view(Hkv, -1)
                c[:, :bs * dim] = keys[i, :, p * bs:(p + 1) * bs].reshape(Hkv, -1)
                c[:, bs * dim:] = values[i, :, p * bs:(p + 1) * bs].transpose(1, 2).reshape(Hkv, -1)
        out.append(sm.grouped_attention(q, cache.cuda(), dim, dim, dim ** -0.5, m, **kw))
    assert all(torch.equal(out[0], o) for o in out[1:])


@pytest.mark.parametrize("bs", [64, 16])  # whole sizes, general form
@pytest.mark.parametrize("opts", [{}, {"sinks": 1}, {"slopes": True}], ids=["plain", "sink", "slopes"])
def test_scores_that_climb(bs, opts):
    """Scores that rise along the keys by less and by more than the weights' reference lets stand, that lie far below and far above zero
    from the first key on, and sinks far above and below all of them."""
    from llmd_amd.ops import seqmix as sm

    n, Hq, Hkv, dim = 230, 8, 2, 128
    g = torch.Generator().manual_seed(3)
    m, pages = _meta([(0, n)], bs, "cpu")
    # every key: a first coordinate that climbs with its position; every head: how much of it its queries take, in units of log2
    climb = torch.tensor([0.0, 0.02, 0.3, 3.0, -0.3, -3.0, 0.05, 0.0])
    base = torch.tensor([0.0, -900.0, 40.0, -200.0, 700.0, 0.0, -30.0, 300.0])
    q = torch.randn(n, Hq, dim, generator=g).bfloat16()
    q[:, :, 0], q[:, :, 1] = (climb * dim ** 0.5).bfloat16(), (base * dim ** 0.5 / 256).bfloat16()
    keys, values = (torch.randn(Hkv, pages * bs, dim, generator=g).bfloat16() for _ in range(2))
    cache = torch.zeros(pages, Hkv, bs, 2 * dim).bfloat16()
    for p in range(-(-n // bs)):
        k = keys[:, p * bs:(p + 1) * bs].clone()
        k[..., 0], k[..., 1] = torch.arange(p * bs, (p + 1) * bs).bfloat16(), 256.0
        c = cache[int(m.tables[0, p])].view(Hkv, -1)
        c[:, :bs * dim] = k.reshape(Hkv, -1)
        c[:, bs * dim:] = values[:, p * bs:(p + 1) * bs].transpose(1, 2).reshape(Hkv, -1)
    vals = {"sinks": torch.tensor([5.0, -800.0, -1000.0, 400.0, 2000.0, 3.0, 0.0, -50.0]), "slopes": torch.rand(Hq, generator=g) * 0.05}
    kw = {k: vals[k] for k in opts}
    want = sm.grouped_attention(q.double(), cache.double(), dim, dim, dim ** -0.5, m, **kw)
    md, _ = _meta([(0, n)], bs, "cuda")
    got = sm.grouped_attention(q.cuda(), cache.cuda(), dim, dim, dim ** -0.5, md, **{k: v.cuda() for k, v in kw.items()})
    # scores of up to about 1000 in fp32 (their products' sums are 2^-24 of that off, a few times): weights off by 2^-11; values up to about 5
    assert ((got.double().cpu() - want).abs() <= 2 ** -8 * want.abs() + 5e-3).all()


# portions in whole sizes and in the general form, one and two blocks of rows per wave, key ranges apart (single tokens, pages of 16), and
# the kernel of single tokens
@pytest.mark.parametrize("runs,bs,dim", [([(0, 230)], 64, 128), ([(0, 230)], 16, 128), ([(50, 90), (700, 1)], 16, 40), ([(900, 1), (40, 1)], 16, 128),
                                         ([(900, 1), (40, 1)], 64, 128)])
def test_sinks_far_below_all_scores(runs, bs, dim):
    """A sink of minus infinity, or so low that its multiple by log2(e) is, counts nothing, and no sink spoils the scores above it,
    however far above they are."""
    from llmd_amd.ops import seqmix as sm

    Hq, Hkv = 8, 2
    g = torch.Generator().manual_seed(dim)
    m, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    q, cache = torch.randn(T, Hq, dim, generator=g).bfloat16(), torch.randn(pages, Hkv, bs, 2 * dim, generator=g).bfloat16()
    # scores of about +-150 in odd heads: in base 2 beyond what an fp32 weight relative to zero can be
    q[:, 1::2] *= 40
    low, inf = torch.finfo, float("inf")
    sinks = torch.tensor([-inf, -inf, low(torch.bfloat16).min, low(torch.float32).min, -1e30, -1e30, -1e10, -1e10])
    args = (dim, dim, dim ** -0.5)
    md, _ = _meta(runs, bs, "cuda")
    for sk in (sinks, sinks.flip(0), torch.tensor([-1e4, 0.0, -inf, 1e10, 300.0, -1e6, 1e4, -3e7])):
        want = sm.grouped_attention(q.double(), cache.double(), *args, m, sinks=sk)
        got = sm.grouped_attention(q.cuda(), cache.cuda(), *args, md, sinks=sk.cuda()).double().cpu()
        # as in test_scores_that_climb: scores of up to about 1000 in fp32
        assert ((got - want).abs() <= 2 ** -8 * want.abs() + 5e-3).all()


@pytest.mark.parametrize("runs,bs", [([(0, 100)], 64), ([(0, 100)], 16), ([(900, 1), (40, 1)], 16)])
def test_low_sinks_among_low_scores(runs, bs):
    """Sinks that are counted behind the keys, below, among and above scores of about -2^20."""
    from llmd_amd.ops import seqmix as sm

    Hq, Hkv, dim, base = 8, 2, 64, -2.0 ** 20
    g = torch.Generator().manual_seed(bs)
    m, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    # sums of whole numbers, exact in fp32, times 1/8
    q = torch.randint(-1, 2, (T, Hq, dim), generator=g).bfloat16()
    q[:, :, 0] = 1024
    cache = torch.randn(pages, Hkv, bs, 2 * dim, generator=g).bfloat16()
    k = cache.view(pages, Hkv, -1)[:, :, :bs * dim].view(pages, Hkv, bs, dim)
    k.copy_(torch.randint(-1, 2, k.shape, generator=g))
    k[..., 0] = -8192
    sinks = torch.tensor([base + d for d in (-300.0, -30.0, -2.0, 0.0, 3.0, 6.0, 30.0, 300.0)])
    md, _ = _meta(runs, bs, "cuda")
    want = sm.grouped_attention(q.double(), cache.double(), dim, dim, dim ** -0.5, m, sinks=sinks)
    got = sm.grouped_attention(q.cuda(), cache.cuda(), dim, dim, dim ** -0.5, md, sinks=sinks.cuda()).double().cpu()
    # log2(e) and the sink's multiple by it, 1.5e6, rounded to fp32: the sink's weight is 2^0.15 off
    assert ((got - want).abs() <= 0.12 * want.abs() + 2e-3).all()
