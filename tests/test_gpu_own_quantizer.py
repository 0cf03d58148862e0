"""Batched decode whose workgroups quantize the activations themselves (few rows, short k): against the oracle,
and bit for bit against the same call on activation records, whose quantizer is a launch of its own."""
import pytest

from np_ref import random_q6_k_blocks
from test_gpu_parity import DECODE_TOL, make_weight, qa, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


# k: one unit, three units, ragged panels, a half-filled last block run, four- and eight-unit rows; rows: the fewest, one tile, a
# last tile of one row, 64; n: one row tile, a half-filled one, more row tiles than one workgroup takes
@pytest.mark.parametrize("dtype,n,k,m", [
    (8, 16, 256, 5), (8, 3000, 1024, 16), (8, 40, 1056, 17), (8, 200, 96, 64), (8, 1024, 1024, 33), (8, 72, 2048, 8),
    (12, 24, 768, 5), (12, 500, 1024, 64), (12, 72, 1280, 33), (12, 4100, 1024, 15), (12, 40, 4096, 3), (12, 4096, 4096, 6),
    (14, 33, 512, 7), (14, 1000, 1024, 49), (14, 40, 4096, 3),
    (8, 3072, 1024, 64), (8, 2050, 992, 49), (12, 6000, 1024, 40), (14, 3072, 768, 64),  # taller workgroups, alone and in the group
    (12, 3244, 1024, 48), (8, 6144, 768, 60),  # as tall as it takes for one per compute unit (of each XCD, too); more than that
])
def test_own_quantizer_equals_records(qa, oracle, dtype, n, k, m):  # noqa: F811
    import torch
    blocks = random_q6_k_blocks(91 + k, n, k).reshape(-1) if dtype == 14 else make_weight(oracle, dtype, n, k, 91 + k)
    x = oracle.randn(92 + m, (m, k))
    x[m // 2, : min(k, 256)] = 0.0
    mm = qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType(dtype), blocks, (n, k)))
    rows = torch.full((m + 20, k), float("nan"), device="cuda")  # what lies behind the last row is not used
    rows[:m] = torch.from_numpy(x)
    xd = rows[:m]
    y = mm.forward(xd)
    assert rel_err(y.cpu().numpy(), oracle.qmatmul(dtype, x, blocks, n)) < DECODE_TOL
    res = torch.from_numpy(oracle.randn(93, (m, n))).cuda()
    assert torch.equal(mm.forward_fused(xd, residual=res), y + res)
    for part in qa.forward_group((mm, mm, mm), xd):
        assert torch.equal(part, y)
    for part in qa.ActivationRecords.quantize(qa.GgmlDType(dtype), xd).forward_group((mm, mm)):
        assert torch.equal(part, y)


@pytest.mark.parametrize("m", [5, 16, 33])
def test_output_over_the_activations(qa, oracle, m):  # noqa: F811
    """y and x the same memory: the rows are read whole before a sum is stored."""
    import torch
    n = k = 1024
    blocks = make_weight(oracle, 8, n, k, 7)
    x = oracle.randn(8 + m, (m, k))
    mm = qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType.Q8_0, blocks, (n, k)))
    xd = torch.from_numpy(x).cuda()
    want = mm.forward(xd)
    mm.forward_fused(xd, out=xd)
    assert torch.equal(xd, want)
