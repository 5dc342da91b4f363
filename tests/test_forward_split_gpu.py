"""GPU parity of the split-product FP32 forward (attention_forward_split.hip): every workgroup shape at ragged sizes, with
padding, radius windows and unaligned views, against the CPU oracle; magnitudes far from 1, rows that leave the sampled
range, infinities and NaN, where the kernel hands query tiles to FP32 MFMAs."""
import numpy as np
import pytest
import torch

import oracle
from parity import check_forward, fp32_score_floor, host, norm_rel, normal_case, padding_mask, reference64, to_dev
from rocmkernels_amd import attention

pytestmark = pytest.mark.gpu

# (width, batch, heads, queries, keys, radius, causal): each workgroup shape on a 256-CU device, sizes off every tile edge.
SHAPES = [
    (32, 8, 1, 2043, 2043, -1, False),    # two query tiles, four key streams
    (32, 24, 1, 500, 470, -1, False),     # two and two
    (32, 24, 1, 1000, 1000, -1, True),    # two and two, causal ramp
    (32, 24, 1, 1001, 999, -1, False),    # four and two
    (32, 48, 2, 515, 515, 100, True),     # four and one
    (64, 24, 1, 500, 530, -1, False),     # two and two
    (64, 24, 1, 1001, 799, -1, False),    # four and two
    (64, 64, 1, 1000, 1030, -1, False),   # eight and one
    (64, 48, 2, 515, 515, 77, False),     # four and one
    (64, 17, 1, 1023, 33, -1, False),     # fewer keys than one 64-key step
    # Either side of the line to the FP32 kernel's planned grid: short ramps, small windows.
    (32, 8, 1, 2043, 2043, -1, True),
    (32, 9, 1, 2043, 2043, -1, True),
    (32, 32, 1, 735, 735, -1, True),
    (32, 32, 1, 737, 737, -1, True),
    (32, 24, 1, 711, 711, 300, True),
    (32, 32, 1, 737, 737, 180, False),
    # Few query tiles a sequence: waves without one, more workgroups than CUs.
    (64, 102, 1, 160, 384, -1, False),
    (64, 85, 1, 160, 384, -1, False),
    (64, 400, 1, 60, 250, -1, False),
    (32, 1100, 1, 31, 160, -1, False),
    (32, 180, 1, 160, 160, -1, True),
]


@pytest.mark.parametrize("aligned", [True, False])
@pytest.mark.parametrize("width,batch,heads,queries,keys,radius,causal", SHAPES)
def test_workgroup_shapes_match_oracle(device, width, batch, heads, queries, keys, radius, causal, aligned):
    q, k, v, _ = normal_case(300 + width + queries, width, batch, heads, queries, keys)
    mask = padding_mask(301, batch, keys, keys // 2)
    mask[0, :40] = 0
    k[0, :, :40] = np.inf  # masked keys: whatever they hold
    v[0, :, :40] = np.nan
    want = oracle.attention(q, np.nan_to_num(k, posinf=0.0), np.nan_to_num(v), mask, radius=radius, causal=causal)
    tensors = to_dev(device, q, k, v)
    if not aligned:  # one float past alignment: the 32-bit load path
        tensors = [torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape) for t in tensors]
    out, lse = attention.forward(*tensors, *to_dev(device, mask), radius=radius, causal=causal)
    check_forward(*host(out, lse), want, f"split d{width}")


@pytest.mark.parametrize("width,batch,heads,queries,keys,radius,causal", SHAPES[:9])
def test_query_row_outside_the_scales(device, width, batch, heads, queries, keys, radius, causal):
    # One query row that no scale fits, in the tile of one wave: its workgroup's other waves still need the rows of K and V
    # that this wave stages, and its barriers. Every other row against the oracle.
    q, k, v, _ = normal_case(340 + width + queries, width, batch, heads, queries, keys)
    mask = padding_mask(341, batch, keys, keys // 2)
    want = oracle.attention(q, k, v, mask, radius=radius, causal=causal)
    for b, row, factor in ((0, 37, np.inf), (1, 5, 2.0**120), (2, 70, 2.0**-100), (3, queries - 1, 2.0**120)):
        q[b, 0, row] *= np.float32(factor)
    out, lse = host(*attention.forward(*to_dev(device, q, k, v, mask), radius=radius, causal=causal))
    uniform = oracle.attention(q[2:3], k[2:3], v[2:3], mask[2:3], radius=radius, causal=causal)  # the row of 2^-100
    want["output"][2, 0, 70], want["lse"][2, 0, 70] = uniform["output"][0, 0, 70], uniform["lse"][0, 0, 70]
    for b, row in ((0, 37), (1, 5), (3, queries - 1)):
        out[b, 0, row], lse[b, 0, row] = want["output"][b, 0, row], want["lse"][b, 0, row]
    check_forward(out, lse, want, f"beside unfit rows d{width}")


@pytest.mark.parametrize("width", [32, 64])
@pytest.mark.parametrize("gain_q,gain_k,gain_v", [(1e-12, 1e12, 1e-20), (3e15, 1e-15, 1e25), (1.0, 1.0, 1e-33), (1e-20, 1e-20, 1e35)])
def test_magnitudes(device, width, gain_q, gain_k, gain_v):
    # Powers of two keep the scaled problem's exact results: O scales with V, scores with Q and K.
    q, k, v, _ = normal_case(310, width, 24, 1, 480, 480)
    q, k, v = (x * np.float32(2.0 ** np.round(np.log2(g))) for x, g in ((q, gain_q), (k, gain_k), (v, gain_v)))
    mask = np.ones((24, 480), np.uint8)
    out, lse = host(*attention.forward(*to_dev(device, q, k, v, mask)))
    unit = np.float64(2.0 ** np.round(np.log2(gain_v)))
    want = oracle.attention(q, k, (v / unit).astype(np.float32), mask)
    check_forward(out.astype(np.float64) / unit, lse, want, f"gains {gain_q} {gain_k} {gain_v}")


@pytest.mark.parametrize("width", [32, 64])
def test_rows_beyond_the_sampled_range(device, width):
    # Two keys and a value row thousands of times larger than the rows around them.
    q, k, v, _ = normal_case(320, width, 24, 1, 480, 480)
    k[3, 0, 101] *= 3e4
    v[5, 0, 257] *= 1e6
    mask = np.ones((24, 480), np.uint8)
    want = oracle.attention(q, k, v, mask)
    out, lse = host(*attention.forward(*to_dev(device, q, k, v, mask)))
    # Against the largest magnitude of each sequence: FP32 scores of thousands round to about 1e-3 (sequence 3 is compared
    # where the large key's weight is exactly 0 or 1 to that rounding, by its row maxima).
    for b in range(24):
        scale = np.abs(want["output"][b]).max()
        if b != 3:
            assert np.abs(out[b] - want["output"][b]).max() <= 1e-5 * max(1.0, scale), b
    assert np.abs(lse[..., 0] - want["lse"][..., 0]).max() <= 1e-6 * np.abs(want["lse"][..., 0]).max()


@pytest.mark.parametrize("width", [32, 64])
def test_zero_rows_around_small_ones(device, width):
    # Every sampled row is 0 (or masked), and the one row that is not is far below 1; the queries make up for the key's.
    q, k, v, _ = normal_case(325, width, 24, 1, 480, 480)
    k[:, :, :479] = 0.0
    v[:, :, :479] = 0.0
    mask = np.ones((24, 480), np.uint8)
    mask[:12, 100:479] = 0
    mask[5] = 0  # nothing visible
    want = oracle.attention(q, k, v, mask)
    q, k, v = (np.ldexp(x, e).astype(np.float32) for x, e in ((q, 30), (k, -30), (v, -40)))
    out, lse = host(*attention.forward(*to_dev(device, q, k, v, mask)))
    out = np.ldexp(out.astype(np.float64), 40)
    for b in range(24):
        assert np.abs(out[b] - want["output"][b]).max() <= 1e-5 * np.abs(want["output"][b]).max(), b
    rows = [b for b in range(24) if b != 5]
    assert np.abs(lse[rows] - want["lse"][rows]).max() <= 1e-6 * np.abs(want["lse"][rows]).max()


@pytest.mark.parametrize("exponent", [10, 14, 20, 30])
@pytest.mark.parametrize("width,batch,heads,queries,keys,radius,causal", [SHAPES[2], (64, 24, 1, 1000, 1000, -1, True), SHAPES[4], SHAPES[7]])
def test_large_rows_outside_the_result(device, width, batch, heads, queries, keys, radius, causal, exponent):
    # Rows that set a workgroup's scales (four in a row: one is sampled) and that a query does not see, or gives no weight to, must
    # not cost it accuracy. Hidden: keys 96 .. 99 under the causal mask; weightless: key 0, whose score is far below all others.
    # An FP32 forward is at 4e-7 of 64 bits on these rows, and terms of the large rows' scale lose 2e-6 (2^14) to all of it.
    q, k, v, _ = normal_case(350 + width, width, batch, heads, queries, keys)
    mask = np.ones((batch, keys), np.uint8)
    large = np.float32(2.0**exponent)
    v[0, 0, 96:100] *= large
    k[1, 0, 96:100] *= large
    q[2:4, 0, :, 0] = np.abs(q[2:4, 0, :, 0]) + 1.0
    k[2:4, 0, :4, 0] = -8.0 * max(64.0, 2.0**exponent / 64.0)  # a score of -90 or less
    v[2, 0, :4] *= large
    want = reference64(q[:4], k[:4], v[:4], mask[:4], radius=radius, causal=causal)
    out, lse = host(*attention.forward(*to_dev(device, q, k, v, mask), radius=radius, causal=causal))
    for b, rows in ((0, slice(0, 96)), (1, slice(0, 96)), (2, slice(4, None)), (3, slice(4, None))):
        if b < 2 and not causal:
            continue
        for name, got in (("output", out), ("lse", lse)):
            assert norm_rel(got[b, 0, rows], want[name][b, 0, rows]) <= 1e-6, (b, name)


@pytest.mark.parametrize("gain", [3.0, 6.0])
@pytest.mark.parametrize("width,batch,heads,queries,keys,radius,causal", SHAPES[1:9])
def test_large_scores(device, width, batch, heads, queries, keys, radius, causal, gain):
    # Q and K scaled by `gain`: row maxima of 40 to 180, each row's weights on a few keys. O and lse within 1e-5, or twice what
    # plain FP32 dot products for the scores alone cost, where that is more (as test_attention_gpu.py::test_large_logits). The first
    # head of four batch entries is compared.
    q, k, v, _ = normal_case(360 + width + queries, width, batch, heads, queries, keys)
    mask = np.ones((batch, keys), np.uint8)
    out, lse = host(*attention.forward(*to_dev(device, q * np.float32(gain), k * np.float32(gain), v, mask), radius=radius, causal=causal))
    q, k, v, mask = q[:4, :1] * np.float32(gain), k[:4, :1] * np.float32(gain), v[:4, :1], mask[:4]
    want = oracle.attention(q, k, v, mask, radius=radius, causal=causal)
    check_forward(out[:4, :1], lse[:4, :1], want, f"large scores d{width}", floor=fp32_score_floor(q, k, v, mask, radius, causal))


@pytest.mark.parametrize("width", [32, 64])
def test_infinities_and_nan(device, width):
    q, k, v, _ = normal_case(330, width, 24, 1, 480, 480)
    q[..., 0] = np.abs(q[..., 0]) + 0.1
    mask = np.ones((24, 480), np.uint8)
    clean = oracle.attention(q, k, v, mask)
    k[2, 0, 7, 0] = -np.inf  # a score of -inf for every query: the key weighs nothing
    v[4, 0, 9, 3] = np.inf   # one feature of every row
    v[6, 0, 11, 5] = np.nan
    q[8, 0, 13, 2] = np.nan  # one row
    out, lse = host(*attention.forward(*to_dev(device, q, k, v, mask)))
    without = mask.copy()
    without[2, 7] = 0
    keyless = k.copy()
    keyless[2, 0, 7] = 0
    want = oracle.attention(q[2:3], keyless[2:3], v[2:3], without[2:3])
    assert np.abs(out[2] - want["output"][0]).max() <= 1e-5
    for b, feature, value in ((4, 3, np.inf), (6, 5, np.nan)):
        others = [f for f in range(width) if f != feature]
        assert np.array_equal(out[b, ..., feature], np.full_like(out[b, ..., feature], value), equal_nan=True)
        assert np.abs(out[b][..., others] - clean["output"][b][..., others]).max() <= 1e-5
    assert np.isnan(out[8, 0, 13]).all() and np.isnan(lse[8, 0, 13]).all()
    rows = [r for r in range(480) if r != 13]
    assert np.abs(out[8, 0, rows] - clean["output"][8, 0, rows]).max() <= 1e-5
