"""Fused attention parity on the GPU vs torch softmax(q k^T * scale) v (CPU fp32, or float64 for config 4)."""
import pytest
import torch

from musc_hip import _attention_hip, synthetic

pytestmark = pytest.mark.gpu


def reference(q, k, v, scale):
    q, k, v = (x.detach().cpu().float() for x in (q, k, v))
    return torch.softmax((q * scale) @ k.transpose(1, 2), -1) @ v


@pytest.mark.parametrize('bh,t', [(4, 1), (3, 33), (2, 77), (8, 1370)])
def test_fp32(device, bh, t):
    g = torch.Generator().manual_seed(bh * 10000 + t)
    q, k, v = (torch.randn((bh, t, 64), generator=g) * 0.64 for _ in range(3))
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu()
    ref = reference(q, k, v, 0.125)
    torch.testing.assert_close(out, ref, rtol=1e-4, atol=2e-5)


def test_fp16_storage(device):
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn((8, 1370, 64), generator=g).half() for _ in range(3))
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu()
    assert out.dtype == torch.float16
    ref = reference(q, k, v, 0.125)
    torch.testing.assert_close(out.float(), ref, rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize('bh,t', [(4, 1), (3, 31), (3, 33), (2, 64), (2, 65), (2, 77), (2, 97), (2, 129), (2, 161)])
def test_fp16_ragged(device, bh, t):
    # every tail of the fp16 kernel's three-stage key pipeline (1 to 6 key blocks, ragged
    # last block) against the CPU fp32 reference of the same fp16 inputs
    g = torch.Generator().manual_seed(bh * 10000 + t + 7)
    q, k, v = (torch.randn((bh, t, 64), generator=g).half() * 0.64 for _ in range(3))
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu()
    torch.testing.assert_close(out.float(), reference(q, k, v, 0.125), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('t,slope', [(700, 0.1), (1370, 0.05), (300, 0.6)])
def test_growing_logits(device, dtype, t, slope):
    # logits rising along the keys: the running maximum is raised every few blocks, so
    # the accumulator rescaling (and, in the fp16 kernel, the rescaling of probabilities
    # whose P V product is still pending) runs many times per query
    g = torch.Generator().manual_seed(t)
    q = torch.zeros((2, t, 64))
    k = torch.randn((2, t, 64), generator=g) * 0.1
    q[:, :, 0] = 1.0
    k[:, :, 0] += slope * torch.arange(t).float()
    v = torch.randn((2, t, 64), generator=g)
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 1.0).cpu().float()
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    torch.testing.assert_close(out, reference(q, k, v, 1.0), rtol=tol, atol=tol)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_huge_logits(device, dtype):
    # logits near 2400 (about 3460 in log2 units): past the range in which the fp16 kernel
    # keeps its running maximum an integer and folds it into the logits MFMA, so it issues
    # the logits unshifted and re-bases every block
    g = torch.Generator().manual_seed(17)
    t = 160
    q = torch.zeros((2, t, 64))
    q[:, :, 0] = 60.0
    k = torch.randn((2, t, 64), generator=g) * 0.1
    k[:, :, 0] += 40.0 + 0.05 * torch.randn((2, t), generator=g)
    v = torch.randn((2, t, 64), generator=g)
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 1.0).cpu().double()
    q64, k64, v64 = (x.double() for x in (q, k, v))
    ref = torch.softmax(q64 @ k64.transpose(1, 2), -1) @ v64
    tol = 1e-4 if dtype == torch.float32 else 1e-2
    assert torch.isfinite(out).all()
    torch.testing.assert_close(out, ref, rtol=tol, atol=tol)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_sharp_logits_select_one_row_dtypes(device, dtype):
    t = 100
    q = torch.zeros((1, t, 64))
    k = torch.zeros((1, t, 64))
    q[0, :, 0] = 50.0
    k[0, 37, 0] = 1.0
    v = torch.randn((1, t, 64))
    out = _attention_hip.attention(q.to(dtype).to(device), k.to(dtype).to(device), v.to(dtype).to(device), 1.0)
    expect = v[0, 37].to(dtype).float().expand(t, 64)
    torch.testing.assert_close(out.cpu().float()[0], expect, rtol=0, atol=1e-5 if dtype == torch.float32 else 1e-3)


def test_sharp_logits_select_one_row(device):
    t = 100
    q = torch.zeros((1, t, 64))
    k = torch.zeros((1, t, 64))
    q[0, :, 0] = 50.0
    k[0, 37, 0] = 1.0
    v = torch.randn((1, t, 64))
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 1.0).cpu()
    torch.testing.assert_close(out[0], v[0, 37].expand(t, 64), rtol=0, atol=1e-5)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_config4_all_blocks(device, dtype):
    # Config 4: B=4, T=1370, 16 heads of 64; q, k, v = N(0,1) tokens @ N(0, 0.02^2) weights,
    # every one of the 24 blocks against softmax(q k^T / 8) v in float64 (on the GPU, from
    # the same stored inputs).
    tol = 2e-5 if dtype == torch.float32 else 2e-4
    for blk, (q, k, v) in enumerate(synthetic.attention_blocks(24, device=device)):
        q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
        out = _attention_hip.attention(q, k, v, 0.125)
        q64, k64, v64 = q.double(), k.double(), v.double()
        ref = torch.softmax(torch.bmm(q64 * 0.125, k64.transpose(1, 2).contiguous()), -1)
        ref = torch.bmm(ref, v64)
        err = (out.double() - ref).abs().max().item()
        print(f'block {blk}: max |err| {err:.3e}', flush=True)
        assert err <= tol + tol * ref.abs().max().item(), (blk, err)


def _f64(q, k, v, scale):
    q, k, v = (x.detach().cpu().double() for x in (q, k, v))
    return torch.softmax(torch.bmm(q * scale, k.transpose(1, 2).contiguous()), -1) @ v


@pytest.mark.parametrize('t', [1, 31, 32, 33, 64, 65, 96, 129, 383, 384, 385, 417])
def test_fp32_split_edges(device, t):
    # key blocks, groups of blocks and 384-query tiles at their edges.  A logit is off by at most a
    # few 2^-22 |q||k| scale (about 5e-6 here at |q| |k| = 26 and scale 1/8), and the output by that
    # times the spread of v; fp32 sums of 417 terms add less
    g = torch.Generator().manual_seed(t)
    q, k, v = (torch.randn((3, t, 64), generator=g) * 0.64 for _ in range(3))
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu().double()
    torch.testing.assert_close(out, _f64(q, k, v, 0.125), rtol=0, atol=1e-5)


@pytest.mark.parametrize('change', ['v_rows', 'k_rows', 'tiny_v', 'huge_k', 'first_block_zero', 'q_rows', 'none'])
@pytest.mark.parametrize('scale', [0.125, -0.125, 0.0])
def test_fp32_inputs_outside_the_split_range(device, change, scale):
    # rows far larger or smaller than the head's first block, which the fp16 split does not hold to
    # 22 bits: those tiles are computed in fp32, so the result stays an fp32 result everywhere
    g = torch.Generator().manual_seed(len(change))
    q, k, v = (torch.randn((2, 200, 64), generator=g) for _ in range(3))
    if change == 'v_rows':
        v[0, 100:] *= 1e6
        v[1, 40] *= 1e-7
    elif change == 'k_rows':
        k[0, 70] *= 1e-6
        k[1, 150:160] *= 30.0
    elif change == 'tiny_v':
        v *= 1e-30
    elif change == 'huge_k':
        k, q = k * 1e25, q * 1e-25
    elif change == 'first_block_zero':
        k[:, :32] = 0
        v[:, :32] = 0
        k[1, 32:] *= 1e-4
        v[1, 32:] *= 1e-4
    elif change == 'q_rows':
        q[:, ::7] *= 1e-12
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), scale).cpu().double()
    ref = _f64(q, k, v, scale)
    # relative to the largest value each output is a mean of: logits within 2^-20 of |q||k| scale
    span = (q.double().norm(dim=-1).max() * k.double().norm(dim=-1).max()).item() * abs(scale)
    tol = (2.0 ** -20 * max(span, 1.0)) * v.abs().amax((1, 2), keepdim=True).double()
    assert torch.all((out - ref).abs() <= tol), ((out - ref).abs() / tol).max()


@pytest.mark.parametrize('where', ['q', 'k', 'v'])
@pytest.mark.parametrize('value', [float('nan'), float('inf'), -float('inf')])
def test_fp32_non_finite_entries(device, where, value):
    # a non-finite entry of one head: that head as fp32 arithmetic gives it (NaN and infinities where
    # torch's fp32 softmax has them), the other head untouched
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn((2, 77, 64), generator=g) for _ in range(3))
    {'q': q, 'k': k, 'v': v}[where][1, 50, 3] = value
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu()
    ref = reference(q, k, v, 0.125)
    torch.testing.assert_close(out[0], ref[0], rtol=1e-4, atol=2e-5)
    if where != 'k':      # a +-inf key gives some queries a -inf logit, whose NaN the two maxima treat alike
        torch.testing.assert_close(out[1], ref[1], rtol=1e-4, atol=2e-5, equal_nan=True)
    else:
        sure = ~torch.isfinite(ref[1])
        assert not torch.isfinite(out[1][sure]).any()
        torch.testing.assert_close(out[1][~sure], ref[1][~sure], rtol=1e-4, atol=2e-5)


@pytest.mark.parametrize('a', [1e2, 1e3, 1e4, 3e4, 1e5, 1e6])
def test_fp32_large_logits(device, a):
    # logits of 1e4 to 1e12.  An fp32 logit is off by at most 2 x 64 x 2^-24 |q||k| scale; where the
    # two largest are further apart than that (and than 20 for exp(-20)) the output is the value row
    # of the largest, elsewhere it lies within the values' range
    g = torch.Generator().manual_seed(11)
    q, k = (torch.randn((2, 256, 64), generator=g) * a for _ in range(2))
    v = torch.randn((2, 256, 64), generator=g)
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu().double()
    assert torch.isfinite(out).all()
    logits = torch.bmm(q.double() * 0.125, k.double().transpose(1, 2).contiguous())
    top = logits.topk(2, dim=-1)
    bound = 2.0 ** -17 * q.double().norm(dim=-1) * k.double().norm(dim=-1).max() * 0.125
    sure = top.values[..., 0] - top.values[..., 1] > 2 * bound + 20
    assert sure.float().mean() > (0.9 if a >= 1e3 else 0.5)
    ref = torch.stack([v[b].double()[top.indices[b, :, 0]] for b in range(2)])
    torch.testing.assert_close(out[sure], ref[sure], rtol=0, atol=1e-5)
    assert (out <= v.double().amax(1, keepdim=True) + 1e-5).all()
    assert (out >= v.double().amin(1, keepdim=True) - 1e-5).all()


@pytest.mark.parametrize('factors', [((5, 1e-5), (20, 1e-6), (40, 1e-11)), ((41, 1e-20), (63, 1e4), (17, 1e12))])
def test_fp32_channels_of_very_different_size_in_v(device, factors):
    # an output column is a mean of its own V column, so its error is that column's: logits within
    # 2^-20 of |q||k| scale (below 8 here), products within 2^-22 of the column's largest entry
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn((3, 300, 64), generator=g) for _ in range(3))
    for c, f in factors:
        v[:, :, c] *= f
    v[1] *= 1e-20
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.0625).cpu().double()
    err = (out - _f64(q, k, v, 0.0625)).abs().amax(1)
    assert (err <= 2.0 ** -17 * v.double().abs().amax(1)).all(), (err / v.double().abs().amax(1)).max()


@pytest.mark.parametrize('fold', [1e6, 1e-6, 1e9])
def test_fp32_channels_of_very_different_size_in_q_and_k(device, fold):
    # channels large in q and as much smaller in k: each logit is still a sum of ordinary products,
    # off by a few 2^-22 of the sum of |q_c k_c| scale (about 5, 2^-22 per split entry and fp32 sum),
    # and an output by that times the spread of v (2-norm: the standard deviation)
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn((3, 300, 64), generator=g) for _ in range(3))
    for c in (7, 8, 33):
        q[:, :, c] *= fold
        k[:, :, c] /= fold
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu().double()
    ref = _f64(q, k, v, 0.125)
    products = torch.bmm(q.double().abs(), k.double().abs().transpose(1, 2).contiguous()).mean() * 0.125
    assert (out - ref).norm() / ref.norm() <= 2.0 ** -21 * products.item(), (out - ref).norm() / ref.norm()


@pytest.mark.parametrize('size', [1e-33, 1e-35, 1e-37, 3e-39])
def test_fp32_smallest_values(device, size):
    # V down to denormal numbers: relative to the largest entry as any other V, but for the last
    # place of a denormal result (2^-149) and of denormal entries
    g = torch.Generator().manual_seed(6)
    q, k, v = (torch.randn((2, 150, 64), generator=g) for _ in range(3))
    v *= size
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu().double()
    err = (out - _f64(q, k, v, 0.125)).abs().max().item()
    assert err <= 2.0 ** -18 * v.abs().max().item() + 2.0 ** -148


@pytest.mark.parametrize('q_size,k_size', [(1e-25, 1e25), (1e-36, 1e36), (1e25, 1e-25), (1e36, 1e-36), (1e-36, 1e-2)])
def test_fp32_sizes_of_q_and_k_that_cancel(device, q_size, k_size):
    g = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn((2, 150, 64), generator=g) for _ in range(3))
    q, k = q * q_size, k * k_size
    k[:, :, 9] *= 1e-3
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu().double()
    torch.testing.assert_close(out, _f64(q, k, v, 0.125), rtol=0, atol=2.0 ** -18 * v.abs().max().item())


@pytest.mark.parametrize('where', ['k', 'v', 'logit'])
@pytest.mark.parametrize('at', [0, 31, 32, 63, 64, 95, 96, 128, 300, 383, 384, 415, 416])
def test_fp32_tiles_left_at_any_key_block(device, where, at):
    # one key that the split does not hold (or whose logits it does not), in the first blocks, at
    # the edges of the pairs of blocks between barriers and in the last, ragged block
    g = torch.Generator().manual_seed(at)
    q, k, v = (torch.randn((2, 417, 64), generator=g) for _ in range(3))
    if where == 'v':
        v[1, at] *= 1e6
    elif where == 'k':
        k[1, at] *= 1e-6
    else:
        k[1, at] *= 40.0
        q[1, ::50] *= 1e5
    out = _attention_hip.attention(q.to(device), k.to(device), v.to(device), 0.125).cpu().double()
    ref = _f64(q, k, v, 0.125)
    if where == 'logit':     # those queries select one key; their logits' gap may be within fp32's error
        assert torch.isfinite(out).all()
        q, out, ref = (torch.cat([x[:, i::50] for i in range(1, 50)], 1) for x in (q, out, ref))
    span = (q.double().norm(dim=-1).max() * k.double().norm(dim=-1).max()).item() * 0.125
    assert ((out - ref).abs() <= 2.0 ** -20 * span * v.double().abs().amax((1, 2), keepdim=True)).all()
