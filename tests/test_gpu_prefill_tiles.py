"""GPU tests (pytest -m gpu) of the 256-row tiles of the prefill product (gemm_pipe_kernel): ragged rows, columns
and k, splits along k, strips of 256 columns with a narrower rest, groups, and the residual read in front of the
stores, in place as well.  Products that would take the few-row kernel come here through the in-LDS form.

Reference: float64 products of the bf16 activations with the dequantized weights rounded to bf16; bounds as in
test_gpu_prefill_regb.py.  With a residual the result is the plain call's f32 sum plus the residual, rounded once:
the same bits."""
import json
import os
import subprocess
import sys

import pytest
import torch

from test_gpu_prefill_regb import BF16_TOL, F32_TOL, Q4_K, Q6_K, Q8_0, dense, off, qa, weight  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture
def tiles(qa):  # noqa: F811
    before = qa.get_prefill_form()
    qa.set_prefill_form(0)
    yield
    qa.set_prefill_form(before)


def check(qa, oracle, dtype, m, n, k):  # noqa: F811
    print(f"tiles dtype={dtype} m={m} n={n} k={k}", flush=True)
    mm = weight(qa, oracle, dtype, n, k, 700 + n)
    x = torch.from_numpy(oracle.randn(701 + m, (m, k))).cuda().to(torch.bfloat16)
    want = x.double() @ dense(mm).t()
    y = mm.forward_bf16_to_f32(x)
    assert off(y, want) < F32_TOL
    assert off(mm.forward(x), want) < BF16_TOL
    assert torch.equal(mm.forward(x.float()), y)
    res = torch.from_numpy(oracle.randn(702 + m, (m, n))).cuda()
    for r in (res, res.to(torch.bfloat16)):
        total = (y + r.float()).to(r.dtype)
        assert torch.equal(mm.forward_fused(x, residual=r, out_dtype=r.dtype), total)
        inout = r.clone()
        mm.forward_fused(x, residual=inout, out=inout, out_dtype=r.dtype)
        assert torch.equal(inout, total)


@pytest.mark.parametrize("dtype,m,n,k", [
    (Q4_K, 129, 300, 256), (Q4_K, 256, 256, 768), (Q4_K, 300, 1000, 4096), (Q4_K, 513, 130, 2048),
    (Q8_0, 129, 257, 288), (Q8_0, 260, 384, 1056), (Q8_0, 511, 1025, 3072),
    (Q6_K, 129, 255, 512), (Q6_K, 300, 513, 4096), (Q6_K, 700, 1000, 12288), (Q6_K, 257, 128, 2560)])
def test_small_products(qa, oracle, tiles, dtype, m, n, k):  # noqa: F811
    check(qa, oracle, dtype, m, n, k)


# 256 x 192 tiles (one round of these, more than one of 128 columns, too few k steps for a split): whole and ragged last
# column tiles, rest of a tile of 16 to 191 columns, k that ends inside a unit and inside a step
@pytest.mark.parametrize("dtype,m,n,k", [(Q4_K, 300, 16512, 512), (Q4_K, 257, 16600, 256), (Q4_K, 700, 12016, 768), (Q8_0, 500, 17000, 288),
                                         (Q8_0, 512, 16896, 256), (Q8_0, 270, 16533, 800)])
def test_tiles_of_192_columns(qa, oracle, tiles, dtype, m, n, k):  # noqa: F811
    check(qa, oracle, dtype, m, n, k)


# more 128 x 128 tiles than compute units: taken by size.  Q6_K at 65900 columns: whole rounds of 256-column strips, then
# half-size tiles; the others have a rest in both directions
@pytest.mark.parametrize("dtype,m,n,k", [(Q4_K, 2100, 2100, 256), (Q8_0, 190, 17000, 320), (Q6_K, 1000, 5000, 1024), (Q4_K, 150, 65900, 256),
                                         (Q6_K, 150, 65900, 256)])
def test_large_products(qa, oracle, dtype, m, n, k):  # noqa: F811
    check(qa, oracle, dtype, m, n, k)


# results and residuals that start on 2, 4 or 16 bytes, rows of a multiple of eight values and not, sums of whole pieces and of
# single values, as the plan has them (below: every form).  The same sums, so the same bits
@pytest.mark.parametrize("dtype,m,n,k", [(Q4_K, 300, 520, 4096), (Q4_K, 301, 515, 4096), (Q4_K, 1100, 4096, 4096), (Q8_0, 700, 12024, 768),
                                         (Q4_K, 2050, 2056, 512), (Q8_0, 300, 66000, 256)])
def test_results_and_residuals_by_alignment(qa, oracle, tiles, dtype, m, n, k):  # noqa: F811
    alignments(qa, oracle, dtype, m, n, k)


def alignments(qa, oracle, dtype, m, n, k):  # noqa: F811
    print(f"alignments dtype={dtype} m={m} n={n} k={k}", flush=True)
    mm = weight(qa, oracle, dtype, n, k, 730)
    x = torch.from_numpy(oracle.randn(731, (m, k))).cuda().to(torch.bfloat16)
    y = mm.forward_bf16_to_f32(x)
    assert off(y, x.double() @ dense(mm).t()) < F32_TOL
    for out_dtype in (torch.float32, torch.bfloat16):
        res = torch.from_numpy(oracle.randn(732, (m, n))).cuda().to(out_dtype)
        total = (y + res.float()).to(out_dtype)

        def at(skip):
            return torch.zeros(m * n + 32, dtype=out_dtype, device="cuda")[skip:skip + m * n].view(m, n)

        for to, of in ((0, 0), (1, 0), (0, 2), (8, 8), (1, 1)):
            out, r = at(to), at(of).copy_(res)
            assert torch.equal(mm.forward_fused(x, out=out, out_dtype=out_dtype), y.to(out_dtype))
            assert torch.equal(mm.forward_fused(x, residual=r, out=out, out_dtype=out_dtype), total), (out_dtype, to, of)
            assert torch.equal(r, res)


@pytest.mark.parametrize("dtype,m,ns,k", [(Q6_K, 300, (513, 128, 200), 4096), (Q4_K, 129, (1000, 256), 2048), (Q8_0, 400, (257, 257), 1056),
                                          (Q4_K, 300, (9000, 8000), 256), (Q8_0, 400, (8200, 130, 8300), 544)])  # 192-column tiles
def test_groups(qa, oracle, tiles, dtype, m, ns, k):  # noqa: F811
    parts = [weight(qa, oracle, dtype, n, k, 720 + i) for i, n in enumerate(ns)]
    x = torch.from_numpy(oracle.randn(721, (m, k))).cuda().to(torch.bfloat16)
    for got_f, got_b, mm in zip(qa.forward_group(parts, x.float()), qa.forward_group(parts, x), parts):
        want = x.double() @ dense(mm).t()
        assert off(got_f, want) < F32_TOL
        assert off(got_b, want) < BF16_TOL


FORCED = """
import json, sys
sys.path[:0] = sys.argv[1:3]
import izwi_amd as qa
from oracle import oracle
import test_gpu_prefill_tiles as t
for case in json.loads(sys.argv[3]):
    t.check(qa, oracle, *case)
    t.alignments(qa, oracle, *case)
print("PASSED")
"""


# Every form of tile, whole along k and in slices (up to one per unit of k, the last ones shorter), and strips of whole tiles in
# front of narrower ones, asked for by name: whole and ragged last tiles in both directions, n a multiple of eight and not.  In a
# process of its own, because the switch is read once
@pytest.mark.parametrize("form", ["256,256,1", "256,256,2", "256,256,4", "256,192,1", "256,192,2", "256,192,3", "256,128,1", "256,128,2",
                                  "256,128,1,2", "256,192,1,1", "256,128,2,1"])
def test_forms_by_name(qa, form):  # noqa: F811
    cases = [(Q4_K, 129, 520, 1024), (Q4_K, 300, 777, 1280), (Q8_0, 257, 1000, 1120), (Q8_0, 256, 515, 1024), (Q6_K, 300, 1040, 1024),
             (Q6_K, 515, 769, 2048)]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, "-c", FORCED, root, os.path.join(root, "tests"), json.dumps(cases)], cwd=root,
                         env={**os.environ, "IZWI_QMM_GEMM_TILE": form}, capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and "PASSED" in run.stdout, run.stdout[-1000:] + run.stderr[-2000:]
