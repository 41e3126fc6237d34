"""Keys and values that a prompt's latent attention makes: never more at a time than the cache's budget leaves room for."""
import pytest
import torch
from test_grouped_f32 import _meta


@pytest.mark.parametrize("H", [1, 16, 17, 64, 128])
@pytest.mark.parametrize("keys", [100, 16384, 65536])
def test_bytes_at_a_time(H, keys, monkeypatch):
    from llmd_amd import ops
    from llmd_amd.ops import seqmix as sm

    made, taken = [], []

    class Native:
        def latent_gather(self, *a):
            pass

        def latent_own(self, q, q_abs, R, kv, rot, bounds, items, row_len, scale, out, gate, h0):
            taken.extend(range(h0, h0 + kv.shape[1] // 256))

    def linear(x, w):
        made.append(x.shape[0] * w.shape[0] * 2)
        return torch.empty(x.shape[0], w.shape[0], dtype=x.dtype, device="meta")

    monkeypatch.setattr(sm, "native", lambda: Native())
    monkeypatch.setattr(ops, "linear", linear)
    m, _ = _meta([(keys - 2, 2)], 64, "cpu")
    meta = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device="meta")  # noqa: E731
    sm.latent_own(meta(2, H * 192), meta(2, H, 192), meta(1, 64, 192), meta(H * 256, 128), 0.1, 128, m, 0, None, meta(2, H, 128))
    assert taken == list(range(H)) and max(made) <= 1 << 29
    assert len(made) == 1 or min(made) >= (1 << 29) // 3  # and not in more pieces than that asks for
