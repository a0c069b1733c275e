"""RsCIN on the GPU vs the oracle restatement of models/modules/_RsCIN.py."""
import numpy as np
import pytest
import torch

from oracle import rscin as orc
from musc_hip._RsCIN_hip import RsCIN

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,d,ks', [(83, 768, [1, 2, 3]), (160, 768, [1, 8, 9]), (7, 16, [2])])
def test_matches_oracle(device, n, d, ks):
    rng = np.random.default_rng(n)
    cls = rng.standard_normal((n, d)).astype(np.float32)
    cls /= np.linalg.norm(cls, axis=1, keepdims=True)
    raw = rng.random(n) * 2.0 + 0.5
    got = RsCIN(raw, list(cls), ks)
    assert isinstance(got, np.ndarray) and got.dtype == np.float32
    np.testing.assert_allclose(got, orc.rscin(raw, list(cls), ks), rtol=0, atol=2e-6)
    # tensors in -> tensor out on the device
    t = RsCIN(torch.from_numpy(raw).to(device), torch.from_numpy(cls).to(device), ks)
    assert t.is_cuda
    np.testing.assert_allclose(t.cpu().numpy(), got, rtol=0, atol=0)


def test_passthrough(device):
    raw = np.arange(5.0)
    assert RsCIN(raw, None, [1]) is raw
    assert RsCIN(raw, [np.ones(4, np.float32)] * 5, [0, 1]) is raw


@pytest.mark.parametrize('n,d', [(1, 4), (2, 3), (63, 772), (64, 769), (65, 768), (128, 1024), (129, 5), (512, 8),
                                 (513, 12), (1025, 7)])
@pytest.mark.parametrize('offset', [0, 1])
def test_row_widths_and_pool_sizes(device, n, d, offset):
    # widths with and without 16-byte rows (offset 1: an unaligned view of aligned rows) and pools
    # at the sizes where the lanes per ranked entry change, against the float64 definition.  The
    # kernel rounds the normalised scores (<= 1) and the result to fp32: 2 x 2^-25 in all, the
    # weights being positive (a shared mean keeps every similarity positive)
    rng = np.random.default_rng(n * 100 + d)
    cls = (rng.standard_normal((n, d)) * 0.3 + 1.0).astype(np.float32)
    cls /= np.linalg.norm(cls, axis=1, keepdims=True)
    raw = rng.random(n) + np.arange(n) * 1e-3
    flat = torch.zeros(n * d + offset, device=device)
    flat[offset:] = torch.from_numpy(cls).reshape(-1).to(device)
    ks = [k for k in (1, 3, 16) if k <= n]
    if n == 1:
        raw = np.array([0.5])
    got = RsCIN(torch.from_numpy(raw).to(device), flat[offset:].view(n, d), ks).cpu().numpy()
    if n == 1:                       # one score: 0 / 0 in the min-max normalisation
        assert np.isnan(got).all()
        return
    np.testing.assert_allclose(got, orc.rscin_bruteforce_f64(raw, cls, ks), rtol=0, atol=1.2e-7)


@pytest.mark.parametrize('n', [3, 16, 17, 64, 129, 512, 513, 700, 1024, 1030, 2100])
def test_equal_similarities_rank_by_index(device, n):
    # few distinct class tokens, so that whole groups of similarities are equal and every cut of
    # k_list falls inside one: the entries with the lower indices are kept.  4-bit channels: the
    # sums are exact in any order
    rng = np.random.default_rng(n)
    distinct = rng.integers(1, 5, (5, 8)).astype(np.float32)
    cls = distinct[rng.integers(0, 5, n)]
    raw = rng.permutation(n) / n + 0.25
    ks = sorted({1, min(2, n), min(16, n), max(1, n // 7), n // 2 + 1, n})
    got = RsCIN(torch.from_numpy(raw).to(device), torch.from_numpy(cls).to(device), ks).cpu().numpy()
    w = cls.astype(np.float64) @ cls.astype(np.float64).T
    s01 = ((raw - raw.min()) / (raw.max() - raw.min())).astype(np.float32).astype(np.float64)
    order = np.argsort(-w, axis=1, kind='stable')
    ref = np.zeros(n)
    for k in ks:
        top = order[:, :k]
        v = np.take_along_axis(w, top, 1)
        ref += (v * s01[top]).sum(1) / v.sum(1)
    np.testing.assert_allclose(got, ref / len(ks), rtol=0, atol=1.2e-7)
