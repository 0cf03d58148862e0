"""One Qwen3 decoder layer at one token, composed from the library's calls (izwi_amd/qwen3_layer.py),
against the same composition of the CPU oracle's functions (pytest -m gpu)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

Q4_K = 12


@pytest.fixture(scope="module")
def qa():
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible: the HIP path cannot run (there is no fallback)")
    import izwi_amd
    izwi_amd.lib()
    torch.cuda.set_device(0)
    return izwi_amd


def silu(v):
    return v / (1.0 + np.exp(-v))


@pytest.mark.parametrize("fuse_prep,fuse_norm,fuse_step", [(True, True, True), (False, False, False), (True, False, False),
                                                           (True, True, False)])
@pytest.mark.parametrize("hidden,heads,kv_heads,d,inter,steps", [(1024, 8, 2, 128, 3072, 5), (512, 8, 8, 64, 1024, 3)])
def test_decode_layer_matches_the_oracle_composition(qa, oracle, hidden, heads, kv_heads, d, inter, steps, fuse_prep, fuse_norm,
                                                     fuse_step):
    from izwi_amd.qwen3_layer import Qwen3DecodeLayer
    shapes = {"q": (heads * d, hidden), "k": (kv_heads * d, hidden), "v": (kv_heads * d, hidden),
              "o": (hidden, heads * d), "gate": (inter, hidden), "up": (inter, hidden), "down": (hidden, inter)}
    blocks = {n: oracle.quantize(Q4_K, oracle.randn(10 + i, s, std=0.03)) for i, (n, s) in enumerate(shapes.items())}
    mm = {n: qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType.Q4K, blocks[n], shapes[n])) for n in shapes}
    w_in = oracle.randn(30, (hidden,), mean=1.0, std=0.1)
    w_post = oracle.randn(31, (hidden,), mean=1.0, std=0.1)
    qk_w = oracle.randn(32, (2 * d,), mean=1.0, std=0.1)
    dev = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    layer = Qwen3DecodeLayer(dev(w_in), dev(w_post), mm["q"], mm["k"], mm["v"], dev(qk_w), mm["o"], mm["gate"],
                             mm["up"], mm["down"], heads, kv_heads, d, 1e-6, fuse_prep=fuse_prep, fuse_norm=fuse_norm,
                             fuse_step=fuse_step)
    cap = 16
    kc_d, vc_d = torch.zeros(1, kv_heads, cap, d, device="cuda"), torch.zeros(1, kv_heads, cap, d, device="cuda")
    kc, vc = np.zeros((1, kv_heads, cap, d), np.float32), np.zeros((1, kv_heads, cap, d), np.float32)
    qm = lambda n, x: oracle.qmatmul(Q4_K, x, blocks[n], shapes[n][0])  # noqa: E731
    for pos in range(steps):
        x = oracle.randn(100 + pos, (1, hidden))
        ang = (pos * (10000.0 ** (-np.arange(d // 2) / (d // 2)))).astype(np.float32)
        cos_sin = np.concatenate([np.cos(ang), np.sin(ang)]).astype(np.float32).reshape(1, d)
        got = layer.forward(dev(x), dev(cos_sin), kc_d, vc_d, pos).cpu().numpy()
        # the same steps with the oracle's functions
        normed = oracle.rms_norm(x, w_in, 1e-6)
        q, k, v = qm("q", normed), qm("k", normed), qm("v", normed)
        q4, k4 = oracle.qk_rms_norm(q.reshape(1, 1, heads, d), k.reshape(1, 1, kv_heads, d), qk_w, 1e-6)
        q4, k4 = oracle.rope_pair_bshd(q4, k4, cos_sin)
        kc[0, :, pos], vc[0, :, pos] = k4.reshape(kv_heads, d), v.reshape(kv_heads, d)
        attn = oracle.decode_gqa_attention(q4.reshape(1, heads, 1, d), kc, vc, pos + 1, d ** -0.5)
        x1 = x + qm("o", attn.reshape(1, heads * d))
        normed = oracle.rms_norm(x1, w_post, 1e-6)
        hid = (silu(qm("gate", normed)) * qm("up", normed)).astype(np.float32)
        want = x1 + qm("down", hid)
        assert np.abs(got - want).max() <= 2e-3 * np.abs(want).max(), pos
        assert np.abs(kc_d.cpu().numpy() - kc).max() <= 1e-4 * np.abs(kc).max()


@pytest.mark.parametrize("hidden,heads,kv_heads,d,inter", [(1024, 8, 2, 128, 3072), (512, 8, 8, 64, 1024), (768, 6, 2, 64, 1280)])
@pytest.mark.parametrize("types", [(12, 12), (8, 8), (12, 14)])  # of all projections, of v and down
def test_one_call_layer_equals_its_calls(qa, oracle, hidden, heads, kv_heads, d, inter, types):
    """The layer as one library call gives the bits of the calls it stands for, output and caches."""
    from izwi_amd.decode_ops import decode_attention_step
    from izwi_amd.qmatmul import forward_group
    from izwi_amd.qwen3_layer import Qwen3DecodeLayer
    shapes = {"q": (heads * d, hidden), "k": (kv_heads * d, hidden), "v": (kv_heads * d, hidden),
              "o": (hidden, heads * d), "gate": (inter, hidden), "up": (inter, hidden), "down": (hidden, inter)}
    if any(k % 256 for _, k in shapes.values()) and types[0] != 8:
        pytest.skip("k is no whole number of blocks")
    rng = np.random.default_rng(3)
    mm = {}
    for i, (n, s) in enumerate(shapes.items()):
        t = types[1] if n in ("v", "down") else types[0]
        if t == 14:  # Q6_K block bytes: any quants and scales, a small block scale
            b = rng.integers(0, 256, (s[0] * s[1] // 256, 210), dtype=np.uint8)
            b[:, 208:] = np.array([1e-4], np.float16).view(np.uint8)
        else:
            b = oracle.quantize(t, oracle.randn(50 + i, s, std=0.03))
        mm[n] = qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType(t), b.reshape(-1), s))
    dev = lambda seed, shape, **kw: torch.from_numpy(oracle.randn(seed, shape, **kw)).cuda()  # noqa: E731
    w_in, w_post, qk_w = dev(60, (hidden,), mean=1.0, std=0.1), dev(61, (hidden,), mean=1.0, std=0.1), dev(62, (2 * d,), mean=1.0, std=0.1)
    layer = Qwen3DecodeLayer(w_in, w_post, mm["q"], mm["k"], mm["v"], qk_w, mm["o"], mm["gate"], mm["up"], mm["down"], heads,
                             kv_heads, d, 1e-6)
    cap = 40
    caches = [dev(63 + i, (1, kv_heads, cap, d)) for i in range(2)]
    ref = [c.clone() for c in caches]
    for pos in (0, 17, cap - 1):
        x, cos_sin = dev(70 + pos, (1, hidden)), dev(71 + pos, (1, d))
        assert layer._forward_one_call(x, cos_sin, caches[0].transpose(1, 2), caches[1].transpose(1, 2), pos) is None
        got = layer.forward(x, cos_sin, caches[0], caches[1], pos)
        q, k, v = forward_group(layer.qkv, x, norm_weight=w_in, eps=1e-6)
        attn = decode_attention_step(q, k, v, qk_w, cos_sin, ref[0], ref[1], pos, 1e-6, d ** -0.5)
        mid = mm["o"].forward_fused(attn.view(1, heads * d), residual=x)
        want = mm["down"].forward_fused(layer.gate_up.forward_silu_mul(mid, norm_weight=w_post, eps=1e-6), residual=mid)
        assert torch.equal(got, want) and torch.equal(caches[0], ref[0]) and torch.equal(caches[1], ref[1])
    with pytest.raises(qa.QmmError):
        layer.forward(x, cos_sin, caches[0], caches[1], cap)


def test_one_call_layer_refuses_before_it_launches(qa, oracle):
    """Gate and up of two block types, heads that do not divide and a position outside the caches: refused with the caches and
    the workspace as they were; the layer raises."""
    from izwi_amd import capi
    from izwi_amd.qwen3_layer import Qwen3DecodeLayer
    hidden, heads, kv_heads, d, inter, cap = 512, 4, 2, 64, 512, 8
    shapes = {"q": (heads * d, hidden), "k": (kv_heads * d, hidden), "v": (kv_heads * d, hidden), "o": (hidden, heads * d),
              "gate": (inter, hidden), "up": (inter, hidden), "up8": (inter, hidden), "down": (hidden, inter)}
    mm = {}
    for i, (n, s) in enumerate(shapes.items()):
        t = 8 if n == "up8" else 12
        mm[n] = qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType(t), oracle.quantize(t, oracle.randn(80 + i, s, std=0.03)).reshape(-1), s))
    dev = lambda seed, shape: torch.from_numpy(oracle.randn(seed, shape)).cuda()  # noqa: E731
    x, w_in, w_post, qk_w, cos_sin = dev(90, (1, hidden)), dev(91, (hidden,)), dev(92, (hidden,)), dev(93, (2 * d,)), dev(94, (1, d))
    caches = [dev(95 + i, (1, kv_heads, cap, d)) for i in range(2)]
    workspace, y = torch.full((4096,), 7.0, device="cuda"), torch.full((1, hidden), 7.0, device="cuda")

    def call(up, kv, pos):
        h = [mm[n].qtensor._h for n in ("q", "k", "v", "o", "gate", up, "down")]
        return capi.lib().izwi_qmm_decode_layer_f32(
            *h, *(t.data_ptr() for t in (x, w_in, w_post, qk_w, cos_sin)), heads, kv, d, 1e-6, caches[0].data_ptr(), caches[1].data_ptr(),
            cap, pos, workspace.data_ptr(), 4 * workspace.numel(), y.data_ptr(), torch.cuda.current_stream().cuda_stream)

    before = [c.clone() for c in caches]
    for args in (("up8", kv_heads, 0), ("up", kv_heads, cap), ("up", kv_heads, -1), ("up", 3, 0)):
        assert call(*args) == capi.ERR_INVALID, args
        torch.cuda.synchronize()
        assert bool((workspace == 7.0).all()) and bool((y == 7.0).all()) and all(torch.equal(a, b) for a, b in zip(caches, before)), args
    assert call("up", kv_heads, 0) == 0
    layer = Qwen3DecodeLayer(w_in, w_post, mm["q"], mm["k"], mm["v"], qk_w, mm["o"], mm["gate"], mm["up8"], mm["down"], heads, kv_heads, d)
    with pytest.raises(qa.QmmError):
        layer.forward(x, cos_sin, caches[0], caches[1], 0)
