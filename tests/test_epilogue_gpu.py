"""Epilogue parity on the GPU (float64; the reference computes it in float64 too)."""
import numpy as np
import pytest
import torch

from oracle import epilogue as oe
from musc_hip import _epilogue_hip

pytestmark = pytest.mark.gpu


def test_golden_bilinear(golden, device):
    g = golden('bilinear_small.npz')
    scores = torch.from_numpy(g['grid'].reshape(1, 1, 1, 25)).to(device)
    for size, key in ((13, 'up13'), (37, 'up37')):
        maps, img = _epilogue_hip.maps_and_scores(scores, size)
        np.testing.assert_allclose(maps[0, 0].cpu().numpy(), g[key], rtol=0, atol=1e-13)
        assert img[0].item() == pytest.approx(g[key].max(), abs=1e-13)


def test_full_size_vs_oracle(device):
    rng = np.random.default_rng(0)
    raw = rng.random((3, 4, 5, 1369))
    maps, img = _epilogue_hip.maps_and_scores(torch.from_numpy(raw).to(device), 518)
    ref_maps, ref_img = oe.maps_and_scores([[torch.from_numpy(raw[r, l]) for l in range(4)] for r in range(3)], 518)
    assert maps.shape == (5, 1, 518, 518)
    np.testing.assert_allclose(maps.cpu().numpy(), ref_maps.numpy(), rtol=0, atol=1e-12)
    np.testing.assert_allclose(img.cpu().numpy(), ref_img.numpy(), rtol=0, atol=1e-12)
    _, img_only = _epilogue_hip.maps_and_scores(torch.from_numpy(raw).to(device), 518, want_maps=False)
    assert torch.equal(img_only.cpu(), img.cpu())


@pytest.mark.parametrize('p,size', [(1, 7), (4, 1), (784, 518), (9, 2), (1369, 37)])
def test_degenerate_and_other_sizes(device, p, size):
    # one-patch grids (every pixel = the score), a 1x1 output (torch's align_corners maps it to
    # grid[0, 0]), the super_fast 28x28 grid, identity size: against the float64 brute force
    rng = np.random.default_rng(p * 10 + size)
    raw = rng.random((2, 3, 4, p))
    maps, img = _epilogue_hip.maps_and_scores(torch.from_numpy(raw).to(device), size)
    ref_maps, ref_img = oe.maps_and_scores([[torch.from_numpy(raw[r, l]) for l in range(3)] for r in range(2)], size)
    np.testing.assert_allclose(maps.cpu().numpy(), ref_maps.numpy(), rtol=0, atol=1e-12)
    np.testing.assert_allclose(img.cpu().numpy(), ref_img.numpy(), rtol=0, atol=1e-12)
    side = int(round(p ** 0.5))
    mean = raw.mean(axis=(0, 1)).reshape(4, side, side)
    brute = np.stack([oe.bilinear_align_corners_f64(m, size) for m in mean])
    np.testing.assert_allclose(maps[:, 0].cpu().numpy(), brute, rtol=0, atol=1e-12)


@pytest.mark.parametrize('n,side,size', [(2, 37, 518), (35, 37, 518), (62, 37, 518), (40, 28, 517), (1, 5, 1030),
                                         (33, 128, 1025), (3, 100, 33), (70, 2, 500), (64, 1, 512)])
def test_band_heights_and_wide_rows(device, n, side, size):
    # 8-, 16- and 32-row bands, rows wider than a workgroup, bands cut by the last row, downsampling
    rng = np.random.default_rng(n * 1000 + size)
    raw = rng.random((1, 2, n, side * side))
    maps, img = _epilogue_hip.maps_and_scores(torch.from_numpy(raw).to(device), size)
    ref_maps, ref_img = oe.maps_and_scores([[torch.from_numpy(raw[0, l]) for l in range(2)]], size)
    np.testing.assert_allclose(maps.cpu().numpy(), ref_maps.numpy(), rtol=0, atol=1e-12)
    np.testing.assert_allclose(img.cpu().numpy(), ref_img.numpy(), rtol=0, atol=1e-12)


@pytest.mark.parametrize('n', [1, 8, 83])
@pytest.mark.parametrize('side,size', [(3, 1), (4, 2), (5, 7), (12, 31), (12, 32), (6, 33), (14, 63), (14, 64), (9, 65),
                                       (20, 100), (37, 127), (16, 128), (16, 129), (100, 33), (128, 9)])
def test_narrow_maps(device, n, side, size):
    # rows of up to 32, 64 and 128 columns, whose bands are shared by groups of threads
    rng = np.random.default_rng(n * 1000 + size)
    raw = rng.random((2, 1, n, side * side))
    maps, img = _epilogue_hip.maps_and_scores(torch.from_numpy(raw).to(device), size)
    ref_maps, ref_img = oe.maps_and_scores([[torch.from_numpy(raw[r, 0])] for r in range(2)], size)
    np.testing.assert_allclose(maps.cpu().numpy(), ref_maps.numpy(), rtol=0, atol=1e-12)
    np.testing.assert_allclose(img.cpu().numpy(), ref_img.numpy(), rtol=0, atol=1e-12)
