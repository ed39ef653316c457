"""The cell sort at the edges of its rules, dense addressing against occupied-cell
addressing (another sorting method), every output bit-identical: 255 to 257
and 511 buckets of 2^11 cells, the first grids with 256 buckets of 2^12 to 2^14,
1281 buckets (the first with two partition levels), and particle counts around
whole tiles of 2048, 4096 and 7168."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L
from test_gpu_cell_sort import linked

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,n", [
    ((64, 120, 68), 2047), ((64, 64, 128), 2048), ((257, 64, 32), 4097), ((73, 448, 32), 100000),
    ((128, 128, 64), 6144), ((128, 128, 128), 1024 * 2048), ((256, 128, 128), 1024 * 2049),
    ((244, 448, 192), 5_700_000), ((100, 100, 100), 1024 * 7168), ((100, 100, 100), 1024 * 7168 - 1)])
def test_edges(ctx, grid, n):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    hi = [float(c - 1) for c in grid]
    ext = torch.tensor(hi, device="cuda")
    rec = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    # every cell within reach: the faces, the last cells and clumps among them
    rec[:, 2:5] = torch.minimum(torch.rand((n, 3), generator=g, device="cuda") * ext, ext)
    rec[: n // 4, 2:5] = torch.minimum(rec[: n // 4, 2:5] * 0.05 + ext * 0.95, ext)
    rec[:, 5:8] = torch.randn((n, 3), generator=g, device="cuda")
    rec = rec[torch.randperm(n, generator=g, device="cuda")].contiguous()
    dom = L.domain([0] * 3, hi, [0] * 3, hi, [1.0] * 3, 0.2, 2)
    a = linked(ctx, rec, n, dom, 0)
    b = linked(ctx, rec, n, dom, L.OPT_SPARSE)
    assert a[4].sparse == 0 and b[4].sparse == 1
    assert a[4].ncells == int(np.prod(grid))
    assert a[3] == b[3]
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)
