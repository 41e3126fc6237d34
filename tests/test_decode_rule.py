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
