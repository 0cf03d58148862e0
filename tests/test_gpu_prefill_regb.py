"""GPU tests (pytest -m gpu) of the register form of the prefill product (few rows, small products):
weights unpacked straight into matrix operands, k split over two wave groups and over workgroups.

Reference: float64 products of the bf16 activations with the dequantized weights rounded to bf16.
The kernel's fused multiply-add rounds once where the codec rounds twice, which moves the bf16
rounding of about one weight in 2^14 by one step (2^-8): 2^-8 * 2^-7 = 3e-5 of the result's norm;
f32 sums add about 1e-6.  Bound: 2e-4 (f32 results); a bf16 result is off by at most half of its last
place, 2^-8 of each value and so of the norm."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K = 8, 12, 14
F32_TOL = 2e-4
BF16_TOL = 2.0 ** -8 + F32_TOL


@pytest.fixture(scope="module")
def qa():
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible: the HIP path cannot run (there is no fallback)")
    import izwi_amd
    izwi_amd.lib()
    torch.cuda.set_device(0)
    return izwi_amd


def weight(qa, oracle, dtype, n, k, seed):
    if dtype == Q6_K:
        rng = np.random.default_rng(seed)
        blocks = rng.integers(0, 256, size=(n * k // 256, 210), dtype=np.uint8)
        blocks[:, 208:] = (1e-3 * rng.uniform(0.5, 2.0, size=blocks.shape[0])).astype(np.float16).view(np.uint8).reshape(-1, 2)
        blocks = blocks.reshape(-1)
    else:
        blocks = oracle.quantize(dtype, oracle.randn(seed, (n, k), std=0.02))
    return qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType(dtype), blocks, (n, k)))


def dense(mm):
    return mm.qtensor.dequantize().to(torch.bfloat16).double()


def off(y, want):
    return float((y.double() - want).norm() / want.norm())


@pytest.mark.parametrize("dtype,m,n,k", [
    (Q4_K, 1, 16, 256), (Q4_K, 33, 100, 768), (Q4_K, 65, 128, 256), (Q4_K, 96, 129, 1280), (Q4_K, 97, 300, 512),
    (Q4_K, 128, 1024, 4096), (Q4_K, 129, 272, 3072), (Q4_K, 192, 1000, 2048), (Q4_K, 500, 384, 1024),
    (Q8_0, 65, 130, 288), (Q8_0, 100, 64, 32), (Q8_0, 128, 1024, 1056), (Q8_0, 70, 96, 3072), (Q8_0, 193, 200, 800),
    (Q6_K, 65, 128, 256), (Q6_K, 96, 130, 768), (Q6_K, 127, 257, 2560), (Q6_K, 300, 1024, 4096)])
def test_product_and_its_epilogues(qa, oracle, dtype, m, n, k):
    product_and_its_epilogues(qa, oracle, dtype, m, n, k)


# row tiles of 64, 96 and 128 rows (narrow products take the lowest ones): whole and ragged last tiles in both directions,
# one row tile and two, k that ends inside a unit
@pytest.mark.parametrize("m,n", [(64, 16500), (101, 9000), (65, 16500), (96, 16512), (97, 16500), (128, 16500), (150, 16000), (250, 15900)])
@pytest.mark.parametrize("dtype,k", [(Q4_K, 512), (Q8_0, 288), (Q6_K, 256)])
def test_row_tile_heights(qa, oracle, dtype, m, n, k):
    product_and_its_epilogues(qa, oracle, dtype, m, n, k)


# units of 256 k per workgroup around the depth of the kernel's loads (four or six units of weights, two or three of
# activations): one to five without a split, then eight slices of 4 .. 14 units, the last one a unit shorter
@pytest.mark.parametrize("units", [1, 2, 3, 4, 5] + [8 * j - 1 for j in (4, 5, 6, 7, 8, 9, 10, 12, 13, 14)])
@pytest.mark.parametrize("dtype,m", [(Q4_K, 33), (Q8_0, 64), (Q6_K, 96), (Q4_K, 101), (Q8_0, 128)])
def test_units_of_a_workgroup(qa, oracle, dtype, m, units):
    k = 256 * units - (64 if dtype == Q8_0 else 0)  # k of Q8_0 may end inside a unit
    print(f"regb dtype={dtype} m={m} units={units}", flush=True)
    mm = weight(qa, oracle, dtype, 200, k, 310 + units)
    x = torch.from_numpy(oracle.randn(311 + m, (m, k))).cuda().to(torch.bfloat16)
    assert off(mm.forward_bf16_to_f32(x), x.double() @ dense(mm).t()) < F32_TOL


def product_and_its_epilogues(qa, oracle, dtype, m, n, k):
    print(f"regb dtype={dtype} m={m} n={n} k={k}", flush=True)
    mm = weight(qa, oracle, dtype, n, k, 300 + n)
    x = torch.from_numpy(oracle.randn(301 + m, (m, k))).cuda().to(torch.bfloat16)
    want = x.double() @ dense(mm).t()
    assert off(mm.forward_bf16_to_f32(x), want) < F32_TOL
    assert off(mm.forward(x), want) < BF16_TOL
    if m > 64:  # (fewer rows run the integer arithmetic in these calls)
        res = torch.from_numpy(oracle.randn(302 + m, (m, n))).cuda()
        assert off(mm.forward(x.float()), want) < F32_TOL
        assert off(mm.forward_fused(x, residual=res, out_dtype=torch.float32), want + res.double()) < F32_TOL
        resb = res.to(torch.bfloat16)
        y = resb.clone()
        mm.forward_fused(x, residual=y, out=y)  # in place
        assert off(y, want + resb.double()) < BF16_TOL


# one member and several of it would be split along k differently if the group were planned as one matrix
@pytest.mark.parametrize("types,m,ns,k", [
    ((Q4_K, Q4_K, Q4_K), 65, (256, 128, 100), 512), ((Q4_K, Q4_K, Q6_K), 101, (512, 130, 130), 2048),
    ((Q4_K, Q4_K, Q4_K), 101, (4096, 1024, 1024), 4096), ((Q4_K, Q4_K, Q6_K), 65, (4096, 1024, 1024), 4096),
    ((Q4_K, Q4_K), 128, (12288, 12288), 4096), ((Q8_0, Q8_0), 70, (6144, 6144), 2048), ((Q4_K, Q4_K), 128, (128, 1024), 1024),
    ((Q8_0, Q8_0, Q8_0), 96, (1024, 64, 300), 3072), ((Q6_K, Q6_K), 80, (300, 2048), 6144),
    ((Q8_0, Q8_0), 128, (384, 640), 1056), ((Q6_K, Q4_K, Q6_K, Q4_K), 300, (16, 257, 128, 48), 768)])
def test_groups_equal_their_members(qa, oracle, types, m, ns, k):
    """Bit for bit up to 128 rows; beyond, where the group is planned as one matrix, up to the order of the f32
    sums: k / 16 additions of the matrix instruction, each off by at most half of 2^-23 of a partial sum, which is
    below 1e-5 of the norm for the k here."""
    parts = [weight(qa, oracle, t, n, k, 400 + 7 * i) for i, (t, n) in enumerate(zip(types, ns))]
    x = torch.from_numpy(oracle.randn(401, (m, k))).cuda().to(torch.bfloat16)
    for got_f, got_b, mm in zip(qa.forward_group(parts, x.float()), qa.forward_group(parts, x), parts):
        alone = mm.forward(x.float())
        if m <= 128:
            assert torch.equal(got_f, alone) and torch.equal(got_b, mm.forward(x))
        assert off(got_f, alone.double()) < 1e-5
        want = x.double() @ dense(mm).t()
        assert off(got_f, want) < F32_TOL
        assert off(got_b, want) < BF16_TOL


def test_group_entry_of_few_rows_equals_its_members(qa, oracle):
    """izwi_qmm_forward_group_bf16 is the bf16 product at any number of rows, a single one included."""
    import ctypes as C
    from izwi_amd import capi
    parts = [weight(qa, oracle, Q4_K, n, 4096, 450 + n) for n in (1024, 200, 4096)]
    for m in (1, 33, 64):
        x = torch.from_numpy(oracle.randn(451 + m, (m, 4096))).cuda().to(torch.bfloat16)
        ys = [torch.empty(m, p.qtensor.dims2()[0], device="cuda", dtype=torch.bfloat16) for p in parts]
        pointers = C.c_void_p * len(parts)
        capi.check(capi.lib().izwi_qmm_forward_group_bf16(pointers(*[p.qtensor._h for p in parts]), len(parts), x.data_ptr(), m,
                                                          pointers(*[y.data_ptr() for y in ys]), capi.OUT_BF16, capi.DEVICE,
                                                          torch.cuda.current_stream().cuda_stream))
        for y, p in zip(ys, parts):
            assert torch.equal(y, p.forward(x))


@pytest.mark.parametrize("m", [65, 101, 128])
def test_gate_up_sums_equal_the_projections(qa, oracle, m):
    """The two sums under silu(gate) * up are those of the projections alone: with `up` (or `gate`) replaced the
    other factor is unchanged, so h is silu(g) * u of the separate results in the same f32 operations."""
    gate, up = (weight(qa, oracle, Q4_K, 3072, 4096, 460 + i) for i in range(2))
    x = torch.from_numpy(oracle.randn(461 + m, (m, 4096))).cuda()
    g, u = gate.forward(x), up.forward(x)
    pair = qa.forward_group((gate, up), x)
    assert torch.equal(pair[0], g) and torch.equal(pair[1], u)
    h = qa.Qwen3GateUpProjection.new_separate(gate, up).forward_silu_mul(x)
    want = g.double() / (1.0 + torch.exp(-g.double())) * u.double()
    # silu in f32: expf (1 ulp), one addition, one division and one product of 2^-24 each
    assert bool(((h.double() - want).abs() <= 6 * 2.0 ** -24 * want.abs() + 1e-30).all())


# silu(gate) * up in the products' own launch (k not split): one to four blocks of 32 rows per row tile, the last 64 columns
# of gate and up whole and ragged, one column tile, k that ends inside a unit
@pytest.mark.parametrize("dtype,m,n,k", [(Q4_K, 65, 64, 256), (Q4_K, 101, 200, 768), (Q8_0, 128, 100, 288), (Q6_K, 97, 1000, 512), (Q4_K, 70, 16400, 256),
                                         (Q8_0, 96, 16400, 512), (Q4_K, 128, 8200, 512), (Q6_K, 129, 6000, 256), (Q8_0, 300, 3000, 768),
                                         (Q6_K, 97, 1024, 512), (Q4_K, 101, 8192, 256), (Q8_0, 300, 3072, 768), (Q8_0, 65, 256, 288)])
def test_gated_products(qa, oracle, dtype, m, n, k):
    print(f"gated dtype={dtype} m={m} n={n} k={k}", flush=True)
    gate, up, down = (weight(qa, oracle, dtype, *shape, 480 + i) for i, shape in enumerate([(n, k), (n, k), (256, n // 256 * 256 or 256)]))
    x = torch.from_numpy(oracle.randn(481 + m, (m, k))).cuda()
    g, u = qa.forward_group((gate, up), x)
    gate_up = qa.Qwen3GateUpProjection.new_separate(gate, up)
    h = gate_up.forward_silu_mul(x)
    want = g.double() / (1.0 + torch.exp(-g.double())) * u.double()
    # silu in f32: expf (1 ulp), one addition, one division and one product of 2^-24 each
    assert bool(((h.double() - want).abs() <= 6 * 2.0 ** -24 * want.abs() + 1e-30).all())
    if n % 256 == 0:
        assert torch.equal(qa.Qwen3Mlp(gate_up, down).forward(x), down.forward(h))


def test_gated_products_reserve_no_room_for_the_separate_ones(qa, oracle):
    """The scratch memory of a stream's first call: bf16 x (64 KB, and at least 1 MiB) and not two f32 products (2 x 32 MiB,
    and half as much again) that the one launch does not write."""
    from izwi_amd import capi
    m, n, k = 128, 65536, 256
    gate, up = (weight(qa, oracle, Q4_K, n, k, 490 + i) for i in range(2))
    x, h = torch.randn(m, k, device="cuda"), torch.empty(m, n, device="cuda")

    def call(stream):
        capi.check(capi.lib().izwi_qmm_forward_gate_up_silu_f32(gate.qtensor._h, up.qtensor._h, x.data_ptr(), m, h.data_ptr(), capi.DEVICE,
                                                                stream.cuda_stream))
        torch.cuda.synchronize()

    call(torch.cuda.current_stream())
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    call(stream)
    assert free - torch.cuda.mem_get_info()[0] <= 32 << 20


@pytest.mark.parametrize("dtype", [Q8_0, Q4_K])
@pytest.mark.parametrize("m", [65, 129, 150, 179, 192])
def test_mlp_of_a_small_model_at_prefill_rows(qa, oracle, dtype, m):
    """gate | up split along k leave their partial sums in scratch memory beside their results."""
    gate, up, down = (weight(qa, oracle, dtype, n, k, 500 + i) for i, (n, k) in enumerate([(3072, 1024), (3072, 1024), (1024, 3072)]))
    x = torch.from_numpy(oracle.randn(501 + m, (m, 1024))).cuda()
    xd = x.to(torch.bfloat16).double()
    h = torch.nn.functional.silu(xd @ dense(gate).t()) * (xd @ dense(up).t())
    gate_up = qa.Qwen3GateUpProjection.new_separate(gate, up)
    got = gate_up.forward_silu_mul(x)
    assert off(got, h) < 2 * F32_TOL  # two products
    y = qa.Qwen3Mlp(gate_up, down).forward(x)
    assert torch.equal(y, down.forward(got))
    assert off(y, got.to(torch.bfloat16).double() @ dense(down).t()) < F32_TOL


@pytest.mark.parametrize("dtype,m,n,k", [(Q4_K, 1, 64, 256), (Q4_K, 65, 200, 768), (Q8_0, 100, 130, 288), (Q6_K, 140, 96, 512), (Q4_K, 300, 300, 256)])
@pytest.mark.parametrize("skip", [1, 2, 5])  # values in front of the rows: they start on 2, 4 and 10 bytes
def test_rows_that_do_not_start_on_sixteen_bytes(qa, oracle, dtype, m, n, k, skip):
    parts = [weight(qa, oracle, dtype, n, k, 600 + i) for i in range(2)]
    x = torch.from_numpy(oracle.randn(601 + m, (m, k))).cuda().to(torch.bfloat16)
    rows = torch.empty(skip + m * k, dtype=torch.bfloat16, device="cuda")[skip:].view(m, k)
    rows.copy_(x)
    assert rows.data_ptr() % 16
    assert torch.equal(parts[0].forward(rows), parts[0].forward(x))
    assert torch.equal(parts[0].forward_bf16_to_f32(rows), parts[0].forward_bf16_to_f32(x))
    if m > 64:
        res = torch.from_numpy(oracle.randn(602, (m, n))).cuda().to(torch.bfloat16)
        assert torch.equal(parts[0].forward_fused(rows, residual=res), parts[0].forward_fused(x, residual=res))
        for a, b in zip(qa.forward_group(parts, rows), qa.forward_group(parts, x)):
            assert torch.equal(a, b)


# results and residuals that start on 2, 4 or 16 bytes, rows of a multiple of eight values and not, k whole and in slices: the
# same sums, so the same bits
@pytest.mark.parametrize("dtype,m,n,k", [(Q4_K, 97, 520, 256), (Q8_0, 70, 515, 288), (Q6_K, 129, 100, 512), (Q4_K, 300, 1032, 1024), (Q4_K, 101, 516, 4096),
                                         (Q8_0, 65, 131, 4096)])
def test_results_and_residuals_by_alignment(qa, oracle, dtype, m, n, k):
    mm = weight(qa, oracle, dtype, n, k, 93)
    x = torch.from_numpy(oracle.randn(94, (m, k))).cuda().to(torch.bfloat16)
    y = mm.forward_bf16_to_f32(x)
    assert off(y, x.double() @ dense(mm).t()) < F32_TOL
    for out_dtype in (torch.float32, torch.bfloat16):
        res = torch.from_numpy(oracle.randn(95, (m, n))).cuda().to(out_dtype)
        total = (y + res.float()).to(out_dtype)

        def at(skip):
            return torch.zeros(m * n + 32, dtype=out_dtype, device="cuda")[skip:skip + m * n].view(m, n)

        for to, of in ((0, 0), (1, 0), (0, 2), (8, 8), (1, 1)):
            out, r = at(to), at(of).copy_(res)
            assert torch.equal(mm.forward_fused(x, out=out, out_dtype=out_dtype), y.to(out_dtype))
            assert torch.equal(mm.forward_fused(x, residual=r, out=out, out_dtype=out_dtype), total), (out_dtype, to, of)
            assert torch.equal(r, res)


def test_copied_rows_in_a_captured_graph(qa, oracle):
    """The copy of rows that do not start on 16 bytes is part of the graph: every replay reads the rows of its time."""
    m, n, k = 100, 300, 512
    mm = weight(qa, oracle, Q4_K, n, k, 650)
    rows = torch.empty(1 + m * k, dtype=torch.bfloat16, device="cuda")[1:].view(m, k)
    xs = [torch.from_numpy(oracle.randn(651 + i, (m, k))).cuda().to(torch.bfloat16) for i in range(4)]
    rows.copy_(xs[0])
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        mm.forward(rows)  # the stream's scratch grows before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = mm.forward(rows)
    for x in xs:
        rows.copy_(x)
        want = mm.forward(x)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
