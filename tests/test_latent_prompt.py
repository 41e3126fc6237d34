"""Latent attention over prompts, bf16: the wide form (latent rows of 512 or 576) at its edges against the plain reference."""
import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("runs", [[(0, 1), (0, 2)], [(0, 37), (5, 1), (100, 64)], [(31, 2), (32, 33), (250, 6)]],
                         ids=["smallest", "portions", "edges"])
@pytest.mark.parametrize("H,R,dr,bs,window,gated", [(16, 512, 64, 64, 0, False), (16, 512, 0, 32, 0, True), (3, 448, 64, 96, 40, False),
                                                    (64, 510, 66, 64, 33, True), (1, 17, 495, 32, 1, False),
                                                    (16, 512, 64, 16, 0, False)])
def test_latent_prompt(H, R, dr, bs, window, gated, runs):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(H + R)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16()  # noqa: E731
    meta, pages = _meta(runs, bs, "cpu")
    T = sum(n for _, n in runs)
    q, cache, gate = rand(T, H, R + dr), rand(pages, bs, R + dr), rand(T, H)
    want = sm.latent_attention(q.float(), cache.float(), meta.tables, meta.row_seq, meta.row_len, 0.05, R,
                               gate=gate.float() if gated else None, window=window)
    for i, (e, n) in enumerate(runs):  # what lies past a sequence's end must not matter
        cache[int(meta.tables[i, (e + n - 1) // bs]), (e + n - 1) % bs + 1:] = float("nan")
    m, _ = _meta(runs, bs, "cuda")
    got = sm.latent_attention(q.cuda(), cache.cuda(), m.tables, m.row_seq, m.row_len, 0.05, R, 4, seq=m,
                              gate=gate.cuda() if gated else None, window=window).float().cpu()
    # bf16 results: 2^-9 of each; weights in two bf16 parts: 2^-16 of a mean of values up to about 5, and fp32 sums of 576 products
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-4).all()


@pytest.mark.parametrize("R,dr,bs,window", [(512, 64, 64, 0), (512, 0, 64, 50), (512, 64, 16, 0), (256, 64, 64, 0)])
def test_rows_do_not_depend_on_the_cut(R, dr, bs, window):
    """A token's output has the same bits wherever its prompt is cut into portions, whatever its neighbours' scores are."""
    from llmd_amd.ops import seqmix as sm

    n, H = 300, 6
    g = torch.Generator().manual_seed(R + dr)
    whole, pages = _meta([(0, n)], bs, "cuda")
    q = torch.randn(n, H, R + dr, generator=g) * 2.0 ** torch.randint(0, 6, (n, H, 1), generator=g)  # some rows' maxima jump
    q, cache = q.bfloat16().cuda(), torch.randn(pages, bs, R + dr, generator=g).bfloat16().cuda()
    out = []
    for cuts in ((0, n), (0, 77, n), (0, 3, 130, 131, n)):
        rows = []
        for a, b in zip(cuts, cuts[1:]):
            m, _ = _meta([(a, b - a)], bs, "cuda")
            if b - a == 1:
                m.max_q = 2   # beside a portion: not a step of single tokens
            rows.append(sm.latent_attention(q[a:b], cache, whole.tables, m.row_seq, m.row_len, 0.05, R, 4, seq=m, window=window))
        out.append(torch.cat(rows))
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
