"""Which kernels a call is made of, where both sides of a rule give the same bits or the same values up to rounding:
kernel names of a child process under torch's profiler (a child, because the switches are read once per process)."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = """
import json, sys
import numpy as np, torch
import izwi_amd as qa
from izwi_amd import capi
from oracle import oracle

def matrix(n, k, dtype=12):
    return qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType(dtype), oracle.quantize(dtype, oracle.randn(n, (n, k), std=0.02)), (n, k)))

def experts(E, hidden, inter):
    one = {n * k: oracle.quantize(12, oracle.randn(n, (n, k), std=0.02)).reshape(-1) for n, k in ((inter, hidden), (hidden, inter))}
    stack = lambda n, k: qa.QTensor.from_blocks(qa.GgmlDType.Q4K, np.tile(one[n * k], E), (E, n, k))
    return qa.MoeExperts(stack(inter, hidden), stack(inter, hidden), stack(hidden, inter))

def call(kind, *sizes):
    if kind == "moe":
        E, hidden, inter, top_k, t = sizes
        layer, x, logits = experts(E, hidden, inter), torch.randn(t, hidden, device="cuda"), torch.randn(t, E, device="cuda")
        return lambda: layer.layer(logits, x, top_k)
    if kind == "attention":
        heads, kv_heads, d, positions = sizes
        q, cache = torch.randn(1, heads, 1, d, device="cuda"), torch.randn(1, kv_heads, positions, d, device="cuda")
        return lambda: qa.try_fused_decode_gqa_attention(q, cache, cache, heads, kv_heads, d, d ** -0.5)
    if kind == "attention in place":
        heads, kv_heads, d, positions, at = sizes  # out begins `at` values into q
        q, cache = torch.randn((heads + 1) * d, device="cuda"), torch.randn(1, kv_heads, positions, d, device="cuda")
        return lambda: capi.check(capi.lib().izwi_decode_gqa_attention_f32(
            q.data_ptr(), cache.data_ptr(), cache.data_ptr(), heads, kv_heads, d, positions, positions, d ** -0.5,
            q.data_ptr() + 4 * at, capi.DEVICE, None))
    if kind == "group":
        dtype, ns, k, m = sizes
        parts, x = [matrix(n, k, dtype) for n in ns], torch.randn(m, k, device="cuda")
        return lambda: qa.forward_group(parts, x)
    if kind == "sort":
        E, pairs = sizes
        ids = torch.randint(0, E, (pairs, 1), device="cuda", dtype=torch.int32)
        return lambda: qa.moe_sort(ids, E)
    n, k, m = sizes
    mm, x = matrix(n, k), torch.randn(m, k, device="cuda")
    return lambda: mm.forward(x)

out = []
for case in json.loads(sys.argv[1]):
    run = call(*case)
    run()
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
        run()
        torch.cuda.synchronize()
    out.append([e.key for e in prof.key_averages()])
print("NAMES " + json.dumps(out))
"""


def kernels(cases, **env):
    """Kernel names of one call of each case, in a process with these environment variables."""
    run = subprocess.run([sys.executable, "-c", CHILD, json.dumps(cases)], cwd=ROOT, env={**os.environ, "PYTHONPATH": ROOT, **env},
                         capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr[-2000:]
    names = json.loads(next(line for line in run.stdout.splitlines() if line.startswith("NAMES "))[6:])
    if not any("kernel" in name for call in names for name in call):
        pytest.skip("this torch's profiler reports no kernels")
    return [" ".join(call) for call in names]


def test_expert_layers_of_few_experts():
    """From nine pairs per expert the expert products, from fourteen where experts are few and k is long."""
    cases = [["moe", 4, 2048, 2048, 2, 18], ["moe", 4, 2048, 2048, 2, 28], ["moe", 16, 2048, 1536, 4, 52], ["moe", 16, 2048, 1536, 4, 56],
             ["moe", 4, 2048, 1024, 2, 18], ["moe", 4, 2048, 1024, 2, 17], ["moe", 64, 512, 512, 8, 72]]
    taken = ["moe_gemm_q4k_kernel" in names for names in kernels(cases)]
    assert taken == [False, True, False, True, True, False, True]


def test_expert_layers_of_sixteen_experts_and_more():
    """Above eight pairs per expert the expert products."""
    cases = [["moe", 64, 512, 512, 8, 64], ["moe", 64, 512, 512, 8, 65], ["moe", 16, 512, 512, 2, 64], ["moe", 16, 512, 512, 1, 129],
             ["moe", 15, 512, 512, 1, 128]]
    taken = ["moe_gemm_q4k_kernel" in names for names in kernels(cases)]
    assert taken == [False, True, False, True, False]


def test_expert_layers_above_eight_pairs_where_uneven_counts_cost():
    """Fewer than 48 experts with more than four units of k wait for nine pairs per expert."""
    cases = [["moe", 32, 1024, 1024, 4, 69], ["moe", 32, 1024, 1024, 4, 72], ["moe", 16, 2048, 768, 2, 70], ["moe", 47, 512, 768, 1, 420],
             ["moe", 48, 512, 768, 1, 420], ["moe", 64, 2048, 2048, 8, 69]]
    taken = ["moe_gemm_q4k_kernel" in names for names in kernels(cases)]
    assert taken == [False, True, False, False, True, True]


def test_expert_threshold_of_the_environment():
    """IZWI_QMM_MOE_MFMA_MIN_ROWS: below that many pairs per expert no matrix-core kernel, the products included."""
    case = ["moe", 8, 512, 512, 2, 80]  # 20 pairs per expert
    assert "moe_gemm_q4k_kernel" in kernels([case])[0]
    raised, = kernels([case], IZWI_QMM_MOE_MFMA_MIN_ROWS="21")
    assert "moe_gemm" not in raised and "mfma" not in raised
    assert "moe_gemm_q4k_kernel" in kernels([case], IZWI_QMM_MOE_MFMA_MIN_ROWS="20")[0]


def test_expert_products_with_long_items_first():
    """Gate | up alone, around 22 to 32 and 61 to 72 pairs per expert."""
    cases = [["moe", 16, 512, 512, 4, 4 * per] for per in (21, 22, 32, 33, 60, 61, 72, 73)]
    names = kernels(cases)
    assert ["moe_gemm_q4k_kernel<true, true>" in n for n in names] == [False, True, True, False, False, True, True, False]
    assert all("moe_gemm_q4k_kernel<false, false>" in n and "moe_gemm_q4k_kernel<false, true>" not in n for n in names)


def test_prefill_kernels_by_size_and_by_the_environment():
    """The few-row kernel up to 128 rows and one tile per compute unit, the 256-row tiles beyond and wherever
    IZWI_QMM_GEMM_TILE asks for them."""
    cases = [["product", 512, 1024, 65], ["product", 512, 256, 300], ["product", 33024, 256, 129]]
    for names, few_row in zip(kernels(cases), (True, True, False)):
        assert ("gemm_regb_kernel" in names, "gemm_pipe_kernel" in names) == (few_row, not few_row)
    forced = kernels(cases, IZWI_QMM_GEMM_TILE="256,128,2")
    assert all("gemm_regb_kernel" not in names and "gemm_pipe_kernel" in names for names in forced)
    assert ["splitk_reduce_kernel" in names for names in forced] == [True, False, False]  # (k = 256 is one unit)


def test_prefill_splits_where_they_pay():
    """A split along k costs a launch per member and its sums both ways: one where few tiles meet a long k, none for a
    product that 128-column tiles cover in one round."""
    split = ["splitk_reduce_kernel" in names for names in kernels([["product", 11000, 1536, 300], ["group", 12, [6144, 6144], 2048, 400],
                                                                   ["product", 2200, 6144, 2000]])]
    assert split == [False, False, True]


def test_attention_launches_by_length_and_heads():
    """One launch up to 320 positions (256 where a workgroup of the splits would hold one query head of 128 elements)."""
    cases = [["attention", 16, 8, 128, 320], ["attention", 16, 8, 128, 321], ["attention", 32, 8, 128, 320], ["attention", 8, 8, 64, 320],
             ["attention", 40, 8, 128, 256], ["attention", 40, 8, 128, 257], ["attention", 4, 2, 256, 33]]
    assert ["attn_one_kernel" in names for names in kernels(cases)] == [True, False, True, True, True, False, False]


def test_attention_in_place_keeps_a_head_in_one_workgroup():
    """Several workgroups per head (the last template argument) only where none reads what another writes."""
    cases = [["attention", 16, 8, 128, 40], ["attention", 100, 10, 128, 300], ["attention", 16, 8, 64, 300]]
    assert [any(f", 2, {wgs}>" in names for wgs in (4, 2)) for names in kernels(cases)] == [True] * 3
    for at in (0, 4, 64):
        placed = kernels([["attention in place", *sizes, at] for _, *sizes in cases])
        assert ["8, 2, 1>" in names or "16, 1, 1>" in names for names in placed] == [True] * 3
    beside, = kernels([["attention in place", 1, 1, 128, 40, 128]])  # right behind q
    assert "8, 2, 4>" in beside


def test_attention_splits_of_the_environment():
    """IZWI_ATTN_WGS_PER_CU and IZWI_ATTN_MIN_CHUNK size the splits at every length of the cache, the short ones
    that otherwise take one launch included."""
    cases = [["attention", 16, 8, 128, 300], ["attention", 8, 2, 64, 40]]
    assert all("attn_one_kernel" in names for names in kernels(cases))
    for env in ({"IZWI_ATTN_MIN_CHUNK": "32"}, {"IZWI_ATTN_WGS_PER_CU": "1"}):
        for names in kernels(cases, **env):
            assert "attn_partial_kernel" in names and "attn_merge" in names and "attn_one_kernel" not in names
    whole = kernels(cases, IZWI_ATTN_MIN_CHUNK="300")  # one split: no merge
    assert all("attn_partial_kernel" in names and "attn_merge" not in names for names in whole)


def test_sort_launches():
    """One workgroup up to 2048 pairs, two launches of many beyond; with more experts than those count (512) one
    workgroup as far as its LDS reaches, and only then the three launches with a serial scan."""
    cases = [["sort", 128, 2048], ["sort", 128, 2049], ["sort", 512, 2049], ["sort", 513, 2049], ["sort", 513, 2688], ["sort", 589, 2049],
             ["sort", 513, 2689]]
    forms = [tuple(f in names for f in ("sort_block_kernel", "sort_wide_kernel", "sort_scan_kernel")) for names in kernels(cases)]
    block, wide, scan = (True, False, False), (False, True, False), (False, False, True)
    assert forms == [block, wide, wide, block, block, block, scan]


def test_taller_workgroups_of_the_batched_decode():
    """Workgroups grow until they may quantize their rows themselves only where every compute unit then has one, or
    they take fewer rounds; elsewhere the quantizer is a launch of its own."""
    cases = [["group", 8, [3072, 3072], 1024, 64], ["group", 12, [9728, 1024, 1024], 1024, 48], ["group", 8, [8960, 8960], 768, 56],
             ["group", 8, [8960, 8960], 256, 56], ["group", 8, [12288, 1024, 1024], 1024, 64], ["group", 8, [12288, 1024, 1024], 768, 64]]
    assert ["quantize_ws_kernel" in names for names in kernels(cases)] == [False, False, False, False, True, True]
