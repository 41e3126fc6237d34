"""Input convolution of steps with longer runs, four tokens per workgroup, beside the same tokens one step each."""
import dataclasses

import pytest
import torch
from test_grouped_f32 import _meta

from llmd_amd.ops import seqmix as sm

pytestmark = pytest.mark.gpu


# runs that end before, at and behind four tokens and shorter than the filter, with and without an old state; channels of one and of several
# workgroups; the longest filter taken here and one beyond
@pytest.mark.parametrize("taps", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("C", [8, 2048, 2056])
@pytest.mark.parametrize("pair", [False, True])
def test_runs_are_their_tokens(taps, C, pair):
    runs = [(5, 1), (0, 2), (3, 2), (9, 3), (0, 4), (7, 5), (6, 7), (0, 8), (2, 9), (0, 70)]  # (tokens before, tokens)
    g = torch.Generator().manual_seed(taps * C)
    rand = lambda *s: torch.randn(*s, generator=g).bfloat16().cuda()  # noqa: E731
    T = sum(n for _, n in runs)
    h, w, w2, old = rand(T, C), rand(C, taps), rand(C, taps) if pair else None, rand(len(runs), taps - 1, C)
    state = old.clone()
    seq = dataclasses.replace(_meta(runs, 64, "cuda")[0], seq_slot=torch.arange(len(runs), dtype=torch.int32, device="cuda"))
    got = sm.input_conv(h, w, state, seq, w2)
    one = old.clone()
    want = [torch.empty_like(h) for _ in range(2)]
    at = 0
    for i, (e, n) in enumerate(runs):
        for k in range(n):
            first, _ = _meta([(e + k, 1)], 64, "cuda")
            y = sm.input_conv(h[at:at + 1], w, one[i:i + 1], first, w2)
            for o, v in zip(want, y if pair else (y,)):
                o[at] = v[0]
            at += 1
    assert torch.equal(state, one)
    for o, v in zip(want, got if pair else (got,)):
        assert torch.equal(o, v)
