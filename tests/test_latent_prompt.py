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


@pytest.mark.gpu
@pytest.mark.parametrize("longest", [1, 63, 64, 65, 130, 2047, 2048, 2049, 3000])
def test_decode_ranges_follow_the_longest_context(longest):
    """Ranges planned for 4096 keys, of one tile up to 2048 and two behind: every key is met once, whatever the replay's lengths."""
    from llmd_amd.ops import seqmix as sm

    H, R, dr, bs, n = 16, 512, 64, 64, 3
    g = torch.Generator(device="cuda").manual_seed(longest)
    lens = [longest, max(1, longest - 64), max(1, longest // 2)]
    W = 64
    cache = torch.randn(n * W, bs, R + dr, device="cuda", generator=g).bfloat16()
    q = torch.randn(n, H, R + dr, device="cuda", generator=g).bfloat16()
    i32 = dict(dtype=torch.int32, device="cuda")
    tables = torch.randperm(n * W, device="cuda", generator=g).to(torch.int32).view(n, W)
    items = torch.tensor([[i, i, 1] for i in range(n)], **i32)
    rows = torch.tensor(lens, **i32)
    for ns, split in ((32, 128), (16, 256), (64, 64)):
        out = torch.empty(n, H, R, dtype=torch.bfloat16, device="cuda")
        po, pm = torch.full((n * ns * 64 * R,), float("nan"), device="cuda"), torch.full((n * ns * 128,), float("nan"), device="cuda")
        assert sm.native().latent_attention_mfma(q, cache, tables, items, rows, 0.05, R, out, ns, split, po, pm, None, 0, H,
                                                 torch.tensor([longest], **i32))
        for i, L in enumerate(lens):
            kv = cache[tables[i].long()].view(-1, R + dr)[:L].double()
            want = torch.softmax(q[i].double() @ kv.t() * 0.05, -1) @ kv[:, :R]
            assert (out[i].double() - want).norm() / want.norm() < 4e-3  # bf16 results, 2^-9 each
