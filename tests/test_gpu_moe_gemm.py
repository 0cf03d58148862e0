"""The expert products over 64-pair chunks (Q4_K stacks, many pairs per expert): the same integers and the
same f32 operations as the 16-row-tile kernels, so the same bits; and the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qa():
    import izwi_amd
    return izwi_amd


def _stacks(qa, oracle, E, hidden, inter, seed):
    dt = qa.GgmlDType.Q4K
    raw = [oracle.quantize(int(dt), oracle.randn(seed + i, (E * n, k), std=0.05))
           for i, (n, k) in enumerate([(inter, hidden), (inter, hidden), (hidden, inter)])]
    shapes = [(E, inter, hidden), (E, inter, hidden), (E, hidden, inter)]
    return raw, qa.MoeExperts(*(qa.QTensor.from_blocks(dt, b, s) for b, s in zip(raw, shapes)))


# panels of one to four units and a ragged one (1280 = 5 units in panels of four), one to three parts of the
# down projection's 512 rows with a half-filled one, experts with no, one, 32, 33, 64 and 65 pairs
@pytest.mark.parametrize("E,hidden,inter,counts", [
    (6, 256, 256, [0, 1, 32, 33, 64, 65]),
    (5, 1280, 512, [3, 31, 130, 0, 96]),
    (4, 2048, 768, [63, 64, 17, 200]),
    (3, 768, 1792, [40, 20, 1]),
    (9, 512, 2048, [0, 0, 70, 0, 0, 128, 0, 0, 5]),
])
def test_chunks_equal_the_tile_kernels(qa, oracle, E, hidden, inter, counts):
    import torch
    from izwi_amd import capi
    raw, experts = _stacks(qa, oracle, E, hidden, inter, 4100 + hidden)
    t = sum(counts)
    assert t >= 9 * E  # the sizes these kernels are taken for
    rng = np.random.default_rng(5)
    ids_np = rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(t, 1)
    x_np = oracle.randn(4200, (t, hidden))
    x_np[t // 2, 256:] = 0.0  # units without a scale
    x = torch.from_numpy(x_np).cuda()
    ids = torch.from_numpy(ids_np).cuda()
    wts_np = rng.uniform(0.1, 1.0, (t, 1)).astype(np.float32)
    wts = torch.from_numpy(wts_np).cuda()
    perm, offsets = qa.moe_sort(ids, E)
    got = experts.forward(x, ids, wts, perm, offsets)
    try:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(1))
        tiles = experts.forward(x, ids, wts, perm, offsets)
    finally:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(-1))
    assert torch.equal(got.view(torch.int32), tiles.view(torch.int32))
    want = oracle.moe_forward(12, x_np, ids_np, wts_np, *raw, E, inter)
    g = got.cpu().numpy()
    # a last-bit difference of silu(gate) * up may move an 8-bit quant of the second product by one step
    assert np.linalg.norm(g - want) <= 1e-3 * np.linalg.norm(want)


# long work items before short ones (22 to 32 and 61 to 72 pairs per expert, several items per compute unit): even and
# skewed counts, experts with none, too few short ones for the last round, a run of an XCD's items (items of gate | up) longer than
# what is put in order
@pytest.mark.parametrize("per_expert,skew,inter,items", [
    (21, 0, 768, 384), (22, 0, 768, 384), (27, 9, 768, None), (32, 20, 768, None), (30, 60, 768, None), (33, 5, 768, None), (61, 0, 768, 384),
    (64, 30, 768, None), (68, 60, 768, None), (69, 3, 768, None), (72, 0, 768, 768), (73, 3, 768, None),
    (68, 0, 1280, 8 * 160), (28, 9, 2304, 125 * 9)])
def test_long_items_first(qa, per_expert, skew, inter, items):
    import torch
    from izwi_amd import capi
    E, hidden = 128, 1280
    rng = np.random.default_rng(4700 + per_expert)

    def stack(n, k):
        blocks = rng.integers(0, 256, size=(E * n * k // 256, 144), dtype=np.uint8)
        blocks[:, :4] = (1e-3 * rng.uniform(0.5, 2.0, size=(blocks.shape[0], 2))).astype(np.float16).view(np.uint8)
        return qa.QTensor.from_blocks(qa.GgmlDType.Q4K, blocks.reshape(-1), (E, n, k))

    experts = qa.MoeExperts(stack(inter, hidden), stack(inter, hidden), stack(hidden, inter))
    counts = np.full(E, per_expert)
    for i in range(skew):  # from one expert to another, some until nothing is left
        take = min(int(counts[2 * i]), int(rng.integers(1, per_expert + 1)) if i % 3 else per_expert)
        counts[2 * i] -= take
        counts[2 * i + 1] += take
    assert items is None or items == ((counts + 63) // 64).sum() * (inter // 256)
    t = int(counts.sum())
    ids = torch.from_numpy(rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(t, 1)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(4701)
    x = torch.randn(t, hidden, device="cuda", generator=gen)
    wts = torch.rand(t, 1, device="cuda", generator=gen)
    perm, offsets = qa.moe_sort(ids, E)
    got = experts.forward(x, ids, wts, perm, offsets)
    try:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(1))
        tiles = experts.forward(x, ids, wts, perm, offsets)
    finally:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(-1))
    assert torch.equal(got.view(torch.int32), tiles.view(torch.int32))


# runs of an XCD's items around one, two and three rounds of 32 workgroups, of two the second items given out by length: all short, all
# long, and both in every order; one, two and five units of k, of which a second item's are requested from the start
@pytest.mark.parametrize("hidden", [256, 512, 1280])
@pytest.mark.parametrize("per_xcd", [32, 33, 47, 63, 64, 65, 97])
def test_second_items_by_length(qa, per_xcd, hidden):
    import torch
    from izwi_amd import capi
    E, inter, rng = 8 * per_xcd // 2, 512, np.random.default_rng(4900 + per_xcd)  # two items per expert and chunk

    def stack(n, k):
        blocks = rng.integers(0, 256, size=(E * n * k // 256, 144), dtype=np.uint8)
        blocks[:, :4] = (1e-3 * rng.uniform(0.5, 2.0, size=(blocks.shape[0], 2))).astype(np.float16).view(np.uint8)
        return qa.QTensor.from_blocks(qa.GgmlDType.Q4K, blocks.reshape(-1), (E, n, k))

    experts = qa.MoeExperts(stack(inter, hidden), stack(inter, hidden), stack(hidden, inter))
    for counts in (np.full(E, 11), np.full(E, 34), np.where(rng.random(E) < 0.4, 40, 12), np.where(np.arange(E) < E // 3, 12, 50)):
        t = int(counts.sum())
        ids = torch.from_numpy(rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(t, 1)).cuda()
        gen = torch.Generator(device="cuda").manual_seed(4901)
        x, wts = torch.randn(t, hidden, device="cuda", generator=gen), torch.rand(t, 1, device="cuda", generator=gen)
        perm, offsets = qa.moe_sort(ids, E)
        got = experts.forward(x, ids, wts, perm, offsets)
        try:
            capi.check(capi.lib().izwi_qmm_set_moe_expert_form(1))
            tiles = experts.forward(x, ids, wts, perm, offsets)
        finally:
            capi.check(capi.lib().izwi_qmm_set_moe_expert_form(-1))
        assert torch.equal(got.view(torch.int32), tiles.view(torch.int32))


# a workgroup's items in turn, eight of them and, of gate | up and of down with one unit of k, past the tables' sixteen: one, two, three
# and eight units of k (fewer steps per item than the records are requested ahead, and more), items of 32 pairs and fewer between
# longer ones
@pytest.mark.parametrize("E,hidden,inter", [(30, 256, 2048), (30, 2048, 256), (36, 512, 1536), (60, 768, 1024), (64, 256, 2048),
                                            (120, 2048, 256)])
def test_many_items_per_workgroup(qa, E, hidden, inter):
    import torch
    from izwi_amd import capi
    rng = np.random.default_rng(4800 + hidden)

    def stack(n, k):
        blocks = rng.integers(0, 256, size=(E * n * k // 256, 144), dtype=np.uint8)
        blocks[:, :4] = (1e-3 * rng.uniform(0.5, 2.0, size=(blocks.shape[0], 2))).astype(np.float16).view(np.uint8)
        return qa.QTensor.from_blocks(qa.GgmlDType.Q4K, blocks.reshape(-1), (E, n, k))

    experts = qa.MoeExperts(stack(inter, hidden), stack(inter, hidden), stack(hidden, inter))
    counts = rng.integers(300, 900, size=E)
    counts[:4] = [0, 1, 640, 609]
    t = int(counts.sum())
    ids = torch.from_numpy(rng.permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(t, 1)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(4801)
    x = torch.randn(t, hidden, device="cuda", generator=gen)
    wts = torch.rand(t, 1, device="cuda", generator=gen)
    perm, offsets = qa.moe_sort(ids, E)
    got = [experts.forward(x, ids, wts, perm, offsets) for _ in range(3)]
    try:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(1))
        tiles = experts.forward(x, ids, wts, perm, offsets)
    finally:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(-1))
    for g in got:
        assert torch.equal(g.view(torch.int32), tiles.view(torch.int32))


@pytest.mark.parametrize("t", [129, 144, 500, 2100])  # 129: just over eight pairs per expert; 144 * 8 pairs: the one-workgroup sort; beyond 2048 pairs two launches
def test_layer_equals_the_tile_kernels(qa, oracle, t):
    import torch
    from izwi_amd import capi
    E, hidden, inter = 128, 512, 256
    _, experts = _stacks(qa, oracle, E, hidden, inter, 4300)
    x = torch.from_numpy(oracle.randn(4400 + t, (t, hidden))).cuda()
    logits = torch.from_numpy(oracle.randn(4401 + t, (t, E))).cuda()
    got = [experts.layer(logits, x, 8, return_routing=True) for _ in range(2)]
    try:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(1))
        tiles = experts.layer(logits, x, 8, return_routing=True)
    finally:
        capi.check(capi.lib().izwi_qmm_set_moe_expert_form(-1))
    for g in got:
        for a, b in zip(g, tiles):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("pairs,experts", [
    (2048, 128), (2049, 128), (2049, 511), (4097, 1), (5000, 512),  # around one workgroup's sort
    (2688, 513), (2689, 513), (2049, 589), (16384, 513),  # more experts than the wide sort counts: as many pairs as one workgroup's LDS holds, more
    (64, 1023), (16385, 128),
    (17 * 1024, 1), (40001, 3), (20000, 511), (20000, 512),
    (20000, 513),   # more experts than a workgroup of the wide sort counts
    (512 * 1024, 128), (512 * 1024 + 1, 128),  # the most workgroups, and one pair beyond them
])
def test_sort_of_many_pairs(qa, pairs, experts):
    import torch
    rng = np.random.default_rng(pairs + experts)
    ids = rng.integers(0, experts, size=pairs).astype(np.int32)
    ids[rng.integers(0, pairs, size=9)] = [-1, experts, 1 << 30, -(1 << 31), -7, experts + 1, -1, experts, 99999]
    for _ in range(2):  # the scratch memory of the call before is not clean
        perm, offsets = qa.moe_sort(torch.from_numpy(ids.reshape(-1, 1)).cuda(), experts)
    valid = np.flatnonzero((ids >= 0) & (ids < experts))
    want = valid[np.argsort(ids[valid], kind="stable")]
    assert np.array_equal(perm.cpu().numpy()[:len(want)], want)
    assert np.array_equal(offsets.cpu().numpy(), np.concatenate([[0], np.cumsum(np.bincount(ids[valid], minlength=experts))]))


@pytest.mark.parametrize("t", [1, 16, 24, 56, 144])
def test_routing_goes_to_the_callers_buffers(qa, oracle, t):
    """ids and weights from buffers of the caller: plain ones (written by the routing kernel), one inside the
    logits and the same one for both (copied afterwards, the weights last)."""
    import torch
    from izwi_amd import capi
    E, hidden, inter = 128, 256, 256
    _, experts = _stacks(qa, oracle, E, hidden, inter, 4500)
    x = torch.from_numpy(oracle.randn(4600 + t, (t, hidden))).cuda()
    logits = torch.from_numpy(oracle.randn(4601 + t, (t, E))).cuda()
    want, want_ids, want_w = experts.layer(logits, x, 8, return_routing=True)

    def call(lg, ids, w):
        out = torch.empty_like(x)
        capi.check(capi.lib().izwi_moe_layer_f32(experts.gate._h, experts.up._h, experts.down._h, lg.data_ptr(),
                                                 x.data_ptr(), t, 8, out.data_ptr(), ids.data_ptr(), w.data_ptr(), capi.DEVICE,
                                                 torch.cuda.current_stream().cuda_stream))
        return out

    ids, w = torch.empty_like(want_ids), torch.empty_like(want_w)
    cases = [(logits, ids, w)]
    if t > 8:  # (up to 8 tokens the one-launch kernels write both buffers themselves)
        both = torch.empty_like(want_ids)
        inside = logits.clone()
        cases += [(logits, both, both.view(torch.float32)), (inside, inside.view(torch.int32).view(-1)[:t * 8], w)]
    for i, (lg, a, b) in enumerate(cases):
        out = call(lg, a, b)
        assert torch.equal(out, want)
        if i != 1:
            assert torch.equal(a.view(-1), want_ids.view(-1))
        assert torch.equal(b.view(-1), want_w.view(-1))
