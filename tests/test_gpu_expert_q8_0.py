"""Q8_0 expert stacks on the expert form (many pairs per expert): panels of four and of three units run
straight-line, ragged ones with a branch per unit; against the oracle and against the one-shot form."""
import numpy as np
import pytest

from test_gpu_parity import make_weight, qa  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,hidden,inter,t", [
    (4, 1024, 768, 70),    # four- and three-unit panels, up to four tiles at a time and a second pass
    (3, 1536, 1024, 24),   # three and four
    (3, 1280, 320, 33),    # ragged panels
    (2, 4096, 512, 40),    # 16 units: two tiles at a time; two-unit panels
])
def test_q8_0_experts(qa, oracle, E, hidden, inter, t):  # noqa: F811
    import torch
    from izwi_amd import capi
    dt, top_k = qa.GgmlDType.Q8_0, 2
    gate, up, down = (make_weight(oracle, 8, E * n, k, 500 + n + i) for i, (n, k) in enumerate([(inter, hidden), (inter, hidden), (hidden, inter)]))
    experts = qa.MoeExperts(qa.QTensor.from_blocks(dt, gate, (E, inter, hidden)), qa.QTensor.from_blocks(dt, up, (E, inter, hidden)),
                            qa.QTensor.from_blocks(dt, down, (E, hidden, inter)))
    x, logits = oracle.randn(510, (t, hidden)), oracle.randn(511, (t, E))
    run = lambda: experts.layer(torch.from_numpy(logits).cuda(), torch.from_numpy(x).cuda(), top_k)  # noqa: E731
    got = run()
    ids, wts = oracle.moe_route(logits, top_k)
    want = oracle.moe_forward(8, x, ids, wts, gate, up, down, E, inter)
    # a last-bit difference of silu(gate) * up may move an 8-bit quant of the second product by one step
    assert np.linalg.norm(got.cpu().numpy() - want) <= 1e-3 * np.linalg.norm(want)
    assert torch.equal(run(), got)
    try:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(0))
        other = run()
    finally:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(-1))
    assert torch.linalg.norm(got - other) <= 1e-3 * torch.linalg.norm(other)
