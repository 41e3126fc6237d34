"""Decode-sized projections of unlisted shapes: the rule's plans on both kernels at the edges of their tiles."""
import pytest
import torch

from llmd_amd import ops


def test_rule_bounds():
    assert ops.decode_rule(8, 2046, 2048) is None and ops.decode_rule(8, 2048, 2080) is None and ops.decode_rule(65, 2048, 2048) is None
    assert ops.decode_rule(16, 2560, 8192) is None                                            # long rows of x
    assert ops.decode_rule(17, 2048, 2048) == (ops.mgemm, (1, 4, 4)) and ops.decode_rule(64, 32000, 2048) == (ops.mgemm, (1, 1, 4))
    assert ops.decode_rule(3, 32000, 2048) == (ops.mgemm, (1, 1, 4))                           # more weights than 32 MB


def test_rule_by_rounds_of_tiles():
    """A round of the chip that is full and one that is not: hipBLASLt from 17 rows on. Tiles for little more than half of the
    CUs: three K ranges, where K is long and the rows are few."""
    one, three = (ops.mgemm, (1, 1, 4)), (ops.mgemm, (1, 3, 4))
    for N in (16385 + 3, 18432, 24576, 26560):
        assert ops.decode_rule(17, N, 3072) is None and ops.decode_rule(64, N, 1536) is None and ops.decode_rule(16, N, 3072) == one
    assert ops.decode_rule(17, 16384, 3072) == one and ops.decode_rule(64, 26624, 3072) == one
    for N in (8196, 9216, 10880):
        assert ops.decode_rule(32, N, 3072) == three and ops.decode_rule(1, N, 4096) == three
        assert ops.decode_rule(33, N, 3072) == one and ops.decode_rule(32, N, 3008) == one
    assert ops.decode_rule(17, 10884, 3072) == one and ops.decode_rule(17, 8192, 3072) == (ops.mgemm, (1, 2, 4))


@pytest.mark.parametrize("model,streams,reads", [("tiny-koduzen", 4, True), ("tiny-koduzen", 5, False), ("tiny-negunex", 2, True),
                                                 ("tiny-negunex", 16, False)])
def test_sums_over_ranges_only_for_streams_that_read_them(model, streams, reads):
    """hyper_update_norm reads them for up to four streams; the products before more of them add up their ranges themselves."""
    import dataclasses

    from llmd_amd.engine.config import EngineConfig
    from llmd_amd.models import build_model
    from llmd_amd.models.layers import ColumnLinear

    mc = dataclasses.replace(EngineConfig.create(model).model_config, hyper_streams=streams)
    last = [getattr(m, "o", None) or getattr(m, "down", None) for l in build_model(mc, device="cpu", max_pos=64).layers
            for m in (l.mix, l.mlp)]
    last = [m for m in last if isinstance(m, ColumnLinear)]
    assert last and all(m.parts == reads for m in last)


def test_sums_over_ranges_only_for_rows_that_read_them():
    from llmd_amd.models.mixers import GatedMLP, SquaredReluMLP, reads_parts
    from llmd_amd.ops import seqmix as sm

    mlp = lambda ff: GatedMLP(64, ff, "silu", "cpu", torch.bfloat16)  # noqa: E731
    assert mlp(96).gate_up.parts and not mlp(100).gate_up.parts
    for d, reads in ((8192, True), (8200, False), (2052, False)):
        m = SquaredReluMLP(8, 8, "cpu", torch.bfloat16)
        reads_parts(sm.norm_reads_parts(d), m)
        assert m.down.parts == reads
    assert sm.streams_read_parts(4, 2052) and not sm.streams_read_parts(4, 2050)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("N,K", [(4, 768), (132, 2048), (2128, 2048), (4100, 768), (16380, 1024), (1024, 8192), (2048, 4096),
                                 (32772, 832), (3072, 1536)])
def test_rule_against_float32(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K + 8, device="cuda", generator=g).bfloat16()[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    got = ops.linear(x, w).float()
    want = (x.double() @ w.double().T).float()
    # bf16 rounding of the result, fp32 rounding of K products of order 1 (partial sums up to about 4 sqrt(K))
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2 ** -22 * 4 * K ** 0.5 * K ** 0.5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(M, N, K) for M in (1, 16) for N, K in ((12288, 1024), (20480, 768), (21844, 768))] +
                         [(M, N, K) for M in (1, 17, 32) for N, K in ((8196, 3072), (10880, 3136))] + [(17, 16388, 768), (64, 26560, 768)])
def test_rule_against_float32_wide(M, N, K):
    """Three, five and six blocks of weight rows per workgroup; three K ranges, even and not; a sparse second round of tiles."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K + 8, device="cuda", generator=g).bfloat16()[:, :K]
    w = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    rule = ops.decode_rule(M, N, K)
    assert (rule is None) == (M > 16 and N > 16384)
    got = ops.linear(x, w).float()
    want = (x.double() @ w.double().T).float()
    # bf16 rounding of the result, fp32 rounding of K products of order 1 (partial sums up to about 4 sqrt(K))
    assert ((got - want).abs() <= 2 ** -8 * want.abs() + 2 ** -22 * 4 * K).all()


def _same_silu(got, want):
    """Tiles of gate and up rows begin their sweeps of K elsewhere than tiles of either: sums in another order, a few of which fall on
    the next number in bf16, 2^-7 away at most. |g| < 6 here, so silu(g) u moves by up to (1 + |g|) + 1 times that, and its own
    rounding. Sums near zero: a wave adds up to 64 times, each time off by 2^-24 of at most sum |x w| < 64, and |u| < 4."""
    assert ((got - want).abs() <= 2 ** -7 * 9 * want.abs() + 1e-3).all() and (got != want).float().mean() < 0.02


def _normed(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, r = (torch.randn(M, K, device="cuda", dtype=torch.bfloat16, generator=g) for _ in range(2))
    w = torch.randn(N, K, device="cuda", dtype=torch.bfloat16, generator=g) * K ** -0.5
    gamma = torch.randn(K, device="cuda", dtype=torch.bfloat16, generator=g)
    x1, r1 = x.clone(), r.clone()
    ops.fused_add_rms_norm(x1, r1, gamma, 1e-5)
    return x, r, w, gamma, x1, r1


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1, 6144, 4096), (1, 28672, 4096), (1, 2048, 2048), (1, 528, 1024), (1, 4096, 768), (2, 6144, 4096),
                                   (1, 10240, 8192), (1, 8192, 8192)])
def test_norm_and_silu_in_the_stream_kernel(M, N, K):
    """The bits of fused_add_rms_norm and linear, or skinny_gemm's SiLU, and a residual that stays."""
    x, r, w, gamma, x1, r1 = _normed(M, N, K)
    r0, plan = r.clone(), ops.skinny_whole(x, w)
    assert plan is not None
    y = ops.linear(x1, w)
    act = ops.skinny_gemm(x1, w, plan, 2)
    _same_silu(act, ops.gated_act(y, ops.ACT_SILU))
    for silu, want in ((False, y), (True, act)):
        out, res = ops.norm_linear(x, r, gamma, 1e-5, w, silu)
        assert torch.equal(out, want) and torch.equal(res, r1) and torch.equal(r, r0)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2])
@pytest.mark.parametrize("rb,occ", [(1, 2), (3, 2), (8, 1)])
@pytest.mark.parametrize("N,K", [(144, 256), (1040, 2048), (400, 4352), (272, 8192)])
def test_norm_in_the_stream_kernel_of_any_plan(M, rb, occ, N, K):
    """Rows of one 16-byte piece per thread up to four, with and without a rest; row blocks that N does not fill."""
    x, r, w, gamma, x1, r1 = _normed(M, N, K)
    res = torch.empty_like(r)
    for silu in (False, True):
        y = torch.empty(M, N // 2 if silu else N, device="cuda", dtype=torch.bfloat16)
        ops.native().skinny_norm(y, x, r, gamma, 1e-5, res, w, rb, occ, silu)
        assert torch.equal(y, ops.skinny_gemm(x1, w, (rb, 1, occ), 2 if silu else 0)) and torch.equal(res, r1)


@pytest.mark.gpu
def test_norm_in_the_stream_kernel_of_two_rows_at_most():
    x, r, w, gamma, _, _ = _normed(3, 1040, 2048)
    assert ops.norm_linear(x, r, gamma, 1e-5, w) is None
    with pytest.raises(RuntimeError):
        ops.native().skinny_norm(torch.empty(3, 1040, device="cuda", dtype=torch.bfloat16), x, r, gamma, 1e-5, torch.empty_like(r), w, 1, 2, False)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [7, 16, 17, 33, 64])
def test_silu_in_the_stream_kernel_of_more_rows(M):
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn(M, 1024, device="cuda", dtype=torch.bfloat16, generator=g)
    w = torch.randn(1040, 1024, device="cuda", dtype=torch.bfloat16, generator=g) / 32
    for rb in (1, 2, 3):
        want = ops.gated_act(ops.skinny_gemm(x, w, (rb, 1, 1)), ops.ACT_SILU)
        _same_silu(ops.skinny_gemm(x, w, (rb, 1, 1), 2), want)
