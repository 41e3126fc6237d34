"""Latent attention in fp32 on the matrix cores against 64 bits, and its bits in different steps."""
import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu


def _exact(q, cache, meta, scale, R, gate, window):
    out = torch.empty(q.shape[0], q.shape[1], R, dtype=torch.float64)
    for t in range(q.shape[0]):
        s, n = int(meta.row_seq[t]), int(meta.row_len[t])
        rows = torch.cat([cache[int(b)] for b in meta.tables[s, :-(-n // cache.shape[1])]])[max(0, n - window) if window else 0:n].double()
        out[t] = torch.softmax(q[t].double() @ rows.T * scale, -1) @ rows[:, :R]
    return out if gate is None else out * torch.sigmoid(gate.double())[:, :, None]


@pytest.mark.parametrize("runs", [[(0, 1), (0, 2)], [(0, 37), (5, 1), (100, 40)], [(127, 1), (128, 1), (31, 1), (600, 1)], [(250, 10), (0, 33)]],
                         ids=["smallest", "portions", "singles", "ranges"])
@pytest.mark.parametrize("H,dr,bs,window,gated", [(16, 64, 64, 0, True), (3, 0, 32, 0, False), (8, 64, 96, 50, False), (20, 64, 64, 0, True),
                                                  (64, 0, 64, 130, False), (1, 64, 64, 1, True)])
def test_latent_f32(H, dr, bs, window, gated, runs):
    from llmd_amd.ops import seqmix as sm

    g = torch.Generator().manual_seed(H + dr)
    meta, pages = _meta(runs, bs, "cpu")
    T, R, Dk = sum(n for _, n in runs), 512, 512 + dr
    q, cache, gate = torch.randn(T, H, Dk, generator=g), torch.randn(pages, bs, Dk, generator=g), torch.randn(T, H, generator=g)
    want = _exact(q, cache, meta, 0.05, R, gate if gated else None, window)
    for i, (e, n) in enumerate(runs):  # what lies past a sequence's end must not matter
        cache[int(meta.tables[i, (e + n - 1) // bs]), (e + n - 1) % bs + 1:] = float("nan")
    m, _ = _meta(runs, bs, "cuda")
    got = sm.latent_attention(q.cuda(), cache.cuda(), m.tables, m.row_seq, m.row_len, 0.05, R, 4, seq=m, gate=gate.cuda() if gated else None,
                              window=window).double().cpu()
    # scores of about 1.2 from sums of 576 products, each rounded to 2^-24 of them; means of values up to about 5 with such weights
    assert ((got - want).abs() <= 2e-5 * want.abs().clamp(min=1)).all()


@pytest.mark.parametrize("H,window", [(16, 0), (20, 70), (8, 0)])
def test_rows_are_the_same_in_every_step(H, window):
    """A token's bits: ranges apart or in one workgroup, alone or beside others, wherever the prompt is cut."""
    from llmd_amd.ops import seqmix as sm

    n, Dk = 400, 576
    g = torch.Generator().manual_seed(H)
    whole, pages = _meta([(0, n)], 64, "cuda")
    q, cache = torch.randn(n, H, Dk, generator=g).cuda(), torch.randn(pages, 64, Dk, generator=g).cuda()

    def run(a, b):
        m, _ = _meta([(a, b - a)], 64, "cuda")
        return sm.latent_attention(q[a:b], cache, whole.tables, m.row_seq, m.row_len, 0.05, 512, 4, seq=m, window=window)

    out = run(0, n)
    assert torch.equal(out, torch.cat([run(0, 77), run(77, 200), run(200, n)]))
    for t in (0, 31, 127, 128, 129, 300, 399):
        assert torch.equal(out[t:t + 1], run(t, t + 1))  # a step of one token: ranges apart


def test_more_ranges_than_workgroups():
    """Ranges apart, more of them than a token's workgroups: each walks several. 30 tokens, 40 ranges: 34 workgroups a token."""
    from llmd_amd.ops import seqmix as sm

    runs, H, Dk = [(5000, 1), (4500, 1)] + [(40 * i, 1) for i in range(28)], 16, 576
    g = torch.Generator().manual_seed(0)
    m, pages = _meta(runs, 64, "cuda")
    q, cache = torch.randn(len(runs), H, Dk, generator=g), torch.randn(pages, 64, Dk, generator=g)
    got = sm.latent_attention(q.cuda(), cache.cuda(), m.tables, m.row_seq, m.row_len, 0.05, 512, 1, seq=m)
    m.max_q = 2  # one workgroup for all ranges, joined in the same order
    assert torch.equal(got, sm.latent_attention(q.cuda(), cache.cuda(), m.tables, m.row_seq, m.row_len, 0.05, 512, 1, seq=m))
    want = _exact(q, cache, _meta(runs, 64, "cpu")[0], 0.05, 512, None, 0)
    assert ((got.double().cpu() - want).abs() <= 2e-5 * want.abs().clamp(min=1)).all()  # (as above)


def test_captured_step():
    """Ranges planned for the longest context, lengths that change between the replays."""
    from llmd_amd.ops import seqmix as sm

    H, Dk, n = 16, 576, 5
    g = torch.Generator().manual_seed(0)
    m, pages = _meta([(999, 1)] * n, 64, "cuda")
    q, cache, gate = torch.randn(n, H, Dk, generator=g).cuda(), torch.randn(pages, 64, Dk, generator=g).cuda(), torch.randn(n, H, generator=g).cuda()
    go = lambda: sm.latent_attention(q, cache, m.tables, m.row_seq, m.row_len, 0.05, 512, 1, seq=m, gate=gate)  # noqa: E731
    go()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = go()
    for lens in ([1, 1, 1, 1, 1], [1000, 128, 129, 1, 700], [31, 32, 33, 640, 127]):
        m.row_len.copy_(torch.tensor(lens, dtype=torch.int32))
        q.copy_(torch.randn(n, H, Dk, generator=g))
        short, _ = _meta([(k - 1, 1) for k in lens], 64, "cuda")
        short.tables = m.tables
        want = sm.latent_attention(q, cache, m.tables, short.row_seq, short.row_len, 0.05, 512, 1, seq=short, gate=gate)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
