"""Attention of captured single-token steps: key ranges planned for the longest context a replay may have, used as far as the
replay's own longest one reaches (``SeqMeta.longest``). Scratch and results hold NaN before the call."""
import pytest
import torch
from test_grouped_f32 import _meta

pytestmark = pytest.mark.gpu

MAX_LEN = 5000


@pytest.fixture
def planned(monkeypatch):
    """Numbers of key ranges that the matrix-core calls plan; torch.empty gives NaN."""
    from llmd_amd.ops import seqmix as sm

    empty, native, seen = torch.empty, sm.native(), []

    def poisoned(*a, **k):
        t = empty(*a, **k)
        return t.fill_(float("nan")) if t.is_floating_point() else t

    class Spy:
        def __getattr__(self, name):
            f = getattr(native, name)
            if not name.endswith("attention_mfma"):
                return f

            def call(*a):
                seen.append(next(a[i] for i in ((10,) if name.startswith("grouped") else (8,))))
                return f(*a)

            return call

    spy = Spy()
    monkeypatch.setattr(sm, "native", lambda: spy)
    monkeypatch.setattr(torch, "empty", poisoned)
    return seen


def _step(longest, B, bs):
    ctx = [longest] + [max(1, longest * (i + 1) // (B + 1)) for i in range(B - 1)]
    runs = [(c - 1, 1) for c in ctx]
    host, pages = _meta(runs, bs, "cpu")
    dev, _ = _meta(runs, bs, "cuda")
    dev.max_len = MAX_LEN
    dev.longest = torch.tensor([longest], dtype=torch.int32, device="cuda")
    return host, dev, pages


def _ranges_used(longest, nsplit, split):
    keys = min(split, max(128, -(-min(longest, nsplit * split) // (nsplit * 64)) * 64))
    return max(1, -(-min(longest, nsplit * split) // keys))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
@pytest.mark.parametrize("opts", [{}, {"window": 1500, "keep_first": 70, "sinks": True}, {"chunk": 1100, "slopes": True, "gate": True}],
                         ids=["causal", "window", "chunk"])
@pytest.mark.parametrize("B", [1, 3, 40])
@pytest.mark.parametrize("longest", [1, 128, 129, 700, 1001, 2600, MAX_LEN])
def test_grouped(longest, B, opts, dtype, planned):
    from llmd_amd.ops import seqmix as sm

    Hq, Hkv, dim, bs = 8, 2, 64, 64
    g = torch.Generator().manual_seed(longest + B)
    host, dev, pages = _step(longest, B, bs)
    q, cache = torch.randn(B, Hq, dim, generator=g).to(dtype), torch.randn(pages, Hkv, bs, 2 * dim, generator=g).to(dtype)
    vals = {"sinks": torch.randn(Hq, generator=g), "slopes": torch.rand(Hq, generator=g) * 0.01,
            "gate": torch.randn(B, Hq * dim, generator=g).to(dtype)}
    kw = lambda d, f: {k: f(vals[k].to(d)) if v is True else v for k, v in opts.items()}  # noqa: E731
    want = sm.grouped_attention(q.float(), cache.float(), dim, dim, dim ** -0.5, host, **kw("cpu", torch.Tensor.float))
    got = sm.grouped_attention(q.cuda(), cache.cuda(), dim, dim, dim ** -0.5, dev, **kw("cuda", lambda x: x)).float().cpu()
    # bf16: 2^-9 of each result, weights in two bf16 parts (2^-16 of a mean of values up to about 5); fp32: a few hundred roundings
    rel, tol = (2 ** -8, 2e-4) if dtype == torch.bfloat16 else (0.0, 2e-5)
    assert ((got - want).abs() <= rel * want.abs() + tol).all()
    if B == 1 and not opts:  # cut finely; at most four ranges and more of them are merged by different code
        assert planned == [32 if dtype == torch.bfloat16 else 40]  # of 160 and 128 keys
        assert (_ranges_used(longest, 32, 160) > 4) == (longest > 512)


@pytest.mark.parametrize("window", [0, 1500])
@pytest.mark.parametrize("R,dr", [(512, 64), (130, 30)])
@pytest.mark.parametrize("B", [1, 3, 40])
@pytest.mark.parametrize("longest", [1, 128, 129, 700, 1001, 2600, MAX_LEN])
def test_latent(longest, B, R, dr, window, planned):
    from llmd_amd.ops import seqmix as sm

    H, bs = 6, 64
    g = torch.Generator().manual_seed(longest + B)
    host, dev, pages = _step(longest, B, bs)
    q = torch.randn(B, H, R + dr, generator=g).bfloat16()
    cache, gate = torch.randn(pages, bs, R + dr, generator=g).bfloat16(), torch.randn(B, H, generator=g).bfloat16()
    want = sm.latent_attention(q.float(), cache.float(), host.tables, host.row_seq, host.row_len, 0.05, R, gate=gate.float(),
                               window=window)
    got = sm.latent_attention(q.cuda(), cache.cuda(), dev.tables, dev.row_seq, dev.row_len, 0.05, R, seq=dev, gate=gate.cuda(),
                              window=window).float().cpu()
    # as above; fp32 sums of up to 576 products
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2e-4).all()
    if B == 1 and not window:
        assert planned == [-(-MAX_LEN // (-(-MAX_LEN // (39 * 64)) * 64))]
