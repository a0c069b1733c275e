"""MSM on pools of more tiles than one grid dimension launches (2^32 threads, 16.7 million
workgroups): the tiles go on in the grid's third dimension.  Sampled rows against float64."""
import pytest
import torch

from musc_hip import _MSM_hip

pytestmark = pytest.mark.gpu
ATOL = 2e-5


def _row_score(z, row, a, b):
    n, p, c = z.shape
    q = z.reshape(-1, c)[row].double()
    best = torch.cat([((part.double() - q) ** 2).sum(-1).amin(1) for part in z.split(512)])
    best = torch.cat([best[:row // p], best[row // p + 1:]]).sqrt()
    return best.sort().values[a:b].mean().item()


# 64-tiles (17.2 million), 128-tiles (17.0 million), the split engine's 256-tiles (16.9 million)
@pytest.mark.parametrize('engine,n,p,c', [('fp32', 3000, 125, 128), ('fp32', 4096, 182, 32), ('split16', 4096, 363, 32)])
def test_more_tiles_than_one_grid_dimension(device, engine, n, p, c):
    g = torch.Generator(device=device).manual_seed(n + p)
    z = torch.randn((n, p, c), generator=g, device=device)
    z /= z.norm(dim=-1, keepdim=True)
    got = _MSM_hip.MSM(z, engine=engine).reshape(-1)
    a, b = _MSM_hip.rank_window(n)
    rows = [0, 1, p - 1, p, 63, 64, 128, n * p // 3, n * p // 2, n * p // 2 + 64, n * p - 129, n * p - 65, n * p - p,
            n * p - 1] + torch.randint(0, n * p, (12,), generator=torch.Generator().manual_seed(p)).tolist()
    ref = torch.tensor([_row_score(z, r, a, b) for r in rows], dtype=torch.float64)
    err = (got[torch.tensor(rows, device=device)].cpu() - ref).abs().max().item()
    print(f'{engine} N={n} P={p} C={c}: {err:.3e}', flush=True)
    assert err <= ATOL
    assert torch.isfinite(got).all()
