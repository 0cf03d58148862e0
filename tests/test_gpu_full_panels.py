"""Batched decode (5 .. 64 rows) of Q8_0 and Q6_K matrices: panels that all hold four units run straight-line,
others with a branch per unit; one LDS window or several, one tile of rows or several."""
import numpy as np
import pytest

from np_ref import random_q6_k_blocks
from test_gpu_parity import DECODE_TOL, make_weight, qa, rel_err  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [8, 14])
@pytest.mark.parametrize("n,k,m", [
    (40, 1024, 5), (16, 1024, 16), (72, 2048, 17), (24, 3072, 64),  # whole panels, one window
    (33, 9216, 16), (33, 9216, 33),                                 # whole panels, two windows
    (40, 768, 8), (40, 1280, 16), (56, 1536, 17),                   # three-unit, ragged and three-unit panels
])
def test_whole_and_partial_panels(qa, oracle, dtype, n, k, m):  # noqa: F811
    import torch
    blocks = random_q6_k_blocks(77 + k, n, k).reshape(-1) if dtype == 14 else make_weight(oracle, dtype, n, k, 77 + k)
    x = oracle.randn(78 + m, (m, k))
    x[0, :256] = 0.0  # a unit without a scale
    mm = qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType(dtype), blocks, (n, k)))
    xd = torch.from_numpy(x).cuda()
    y = mm.forward(xd)
    res = torch.from_numpy(oracle.randn(79, (m, n))).cuda()
    want = oracle.qmatmul(dtype, x, blocks, n)
    assert rel_err(y.cpu().numpy(), want) < DECODE_TOL
    fused = mm.forward_fused(xd, residual=res)  # the kernel with the epilogue
    assert torch.equal(fused, y + res)
    for part in qa.forward_group((mm, mm), xd):  # the launch of a group
        assert rel_err(part.cpu().numpy(), want) < DECODE_TOL
    assert np.isfinite(want).all()
