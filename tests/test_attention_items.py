"""The work items of the matrix-core attention kernels, built with numpy, against the plain listing."""
import random

import numpy as np
import pytest
import torch

from llmd_amd.engine.attn_meta import SeqMeta


@pytest.mark.parametrize("per", [1, 4, 16])
@pytest.mark.parametrize("balance", [0, 3, 64])
@pytest.mark.parametrize("runs", [[], [1], [0, 5], [1] * 7, [1, 1, 33, 16, 17], [300]])
def test_items(runs, balance, per):
    rng = random.Random(len(runs))
    ctx = [n + rng.randrange(100) for n in runs]
    z = torch.zeros(1, dtype=torch.int32)
    seq = SeqMeta(len(runs), z, z, z, z, z, z, q_lens=runs, ctx_lens=ctx)
    rows, keys, t0 = [], [], 0
    for s, n in enumerate(runs):
        for a in range(0, n, per):
            rows.append([s, t0 + a, min(per, n - a)])
            keys.append(ctx[s] - n + a + rows[-1][2])
        t0 += n
    if balance:
        order = sorted(range(len(rows)), key=lambda i: -keys[i])
        rows = [rows[i] for b in range(0, len(order), balance)
                for i in (order[b:b + balance] if (b // balance) % 2 == 0 else order[b:b + balance][::-1])]
    got = seq.attention_items(per, balance)
    assert got.dtype == torch.int32 and got.shape == (len(rows), 3) and np.array_equal(got.numpy(), np.array(rows).reshape(-1, 3))
