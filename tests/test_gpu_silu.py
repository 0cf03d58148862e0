"""silu(gate) * up over the whole range of f32 arguments; the kernels share one definition, which is to be no further off than
v / (1 + expf(-v)) in f32."""
import numpy as np
import pytest

from oracle import oracle

pytestmark = pytest.mark.gpu


def silu_f32(v):
    """The same f32 steps with a correctly rounded exponential."""
    with np.errstate(over="ignore", invalid="ignore"):
        e = np.exp(-v.astype(np.float64)).astype(np.float32)
        return (v / (np.float32(1.0) + e)).astype(np.float32)


def records_of(gate, up):
    """silu(gate[i]) * up[i], each the constant of a unit of 256 values of its own row: a Q8_K unit of one value v has
    d = 1 / (-128 / v), both divisions correctly rounded, so v comes back as -128 d to two roundings."""
    import torch
    import izwi_amd as qa
    g, u = (torch.from_numpy(np.repeat(a.reshape(-1, 1), 256, axis=1).astype(np.float32)).cuda() for a in (gate, up))
    data = qa.ActivationRecords.from_silu_mul(qa.GgmlDType.Q4K, g, u).data.cpu().numpy().view(np.uint8)
    tiles = -(-len(gate) // 16)
    side = data[:tiles * 4416].reshape(tiles, 4416)[:, 4096:4160].copy().view(np.float32).reshape(-1)[:len(gate)]
    return -128.0 * side.astype(np.float64)


def test_ordinary_arguments():
    """A grid over [-110, 110] with the neighbourhoods of the magnitudes at which an exponential changes its form."""
    at = [np.linspace(-110, 110, 4001)]
    at += [np.linspace(c - 1e-3, c + 1e-3, 65) for s in (1, -1) for c in (s * 17.0, s * 64.0, s * 87.0, s * 88.7, s * 88.72284, s * 104.0)]
    gate = np.concatenate(at).astype(np.float32)
    want = silu_f32(gate)
    up = np.where(np.abs(want) < 1e-20, np.float32(2.0 ** 100), np.float32(1.0)).astype(np.float32)
    got = records_of(gate, up)
    want = want.astype(np.float64) * up
    # expf one ulp (2^-23), the sum, the division and the two of the record half an ulp each: 2^-23 + 4 * 2^-24
    near = np.abs(got - want) <= 3.0 * 2.0 ** -23 * np.abs(want)
    # where e^-v overflows the result is 0; a last bit of expf decides on which side the largest finite value lies
    edge = np.abs(gate + 88.72284) < 1e-4
    assert np.all(near | edge), gate[~(near | edge)][:10]


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_small_arguments_lose_no_bits(sign):
    """Down to the smallest subnormal silu(v) is v / 2 rounded once: 1 + e^-v is 2 there."""
    rng = np.random.default_rng(1)
    bits = np.concatenate([rng.integers(1 << e, 2 << e, size=40) for e in range(0, 23)] +
                          [rng.integers((e + 1) << 23, (e + 2) << 23, size=40) for e in range(0, 8)] + [[1, 2, 3, 5, 7, (1 << 23) - 1]])
    gate = (np.float32(sign) * bits.astype(np.uint32).view(np.float32)).astype(np.float32)
    half = (gate * np.float32(0.5)).astype(np.float32)
    up = np.full_like(gate, np.float32(2.0 ** 126))
    got, want = records_of(gate, up), half.astype(np.float64) * 2.0 ** 126
    assert np.all(np.abs(got - want) <= 2.0 ** -23 * np.abs(want)), gate[np.abs(got - want) > 2.0 ** -23 * np.abs(want)][:10]


@pytest.mark.parametrize("m", [1, 3, 20])
def test_infinities_nan_and_large_sums(m):
    """gate sums of +-inf, NaN, the largest magnitudes and +-0 through the projections' own epilogues."""
    import torch
    import izwi_amd as qa
    n, k = 64, 256
    rng = np.random.default_rng(2)
    scales = np.array([np.inf, -np.inf, np.nan, 65504.0, -65504.0, 0.0, 1.0, -1.0] * 8, np.float16)

    def matrix(d):
        blocks = np.zeros((n, 144), np.uint8)
        blocks[:, 0:2] = d.astype(np.float16).reshape(n, 1).view(np.uint8)
        blocks[:, 4:12] = 1  # scales of sub-blocks 0 .. 3 one; mins zero
        blocks[:, 8:12] = 0
        blocks[:, 16:144] = 0x11
        return qa.QMatMul.from_qtensor(qa.QTensor.from_blocks(qa.GgmlDType.Q4K, blocks.reshape(-1), (n, k)))

    gate, up = matrix(scales), matrix(np.full(n, 0.5))
    x = torch.from_numpy((rng.uniform(0.5, 1.0, size=(m, k)) * np.array([1.0, 1e30, 1e-30])[np.arange(m) % 3].reshape(m, 1)).astype(np.float32)).cuda()
    g, u = gate.forward(x).cpu().numpy(), up.forward(x).cpu().numpy()
    got = qa.Qwen3GateUpProjection.new_separate(gate, up).forward_silu_mul(x).cpu().numpy()
    with np.errstate(over="ignore", invalid="ignore"):
        want = (silu_f32(g) * u).astype(np.float32)
    assert np.isinf(want).any() and np.isnan(want).any() and (want == 0).any()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    finite = np.isfinite(want)
    assert np.array_equal(got[~finite & ~np.isnan(want)], want[~finite & ~np.isnan(want)])
    tiny = 2.0 ** -149  # below the normal range one spacing a step
    assert np.all(np.abs(got[finite].astype(np.float64) - want[finite]) <= 4.0 * 2.0 ** -23 * np.abs(want[finite]) + 2 * tiny)
