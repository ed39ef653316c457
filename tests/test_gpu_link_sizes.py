"""The link kernels' ways by the number of cells and particles of a call: the
parts a small dense cell is split into and the workgroup size for the larger
ones.  Bar: bit-identical labels, ring and halos against a call that links the
same particles another way."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu


def cells_of(torch, per, grid, seed):
    """Unit cells of grid^3, `per` particles in each (one of `per` at random),
    gathered near a random point of the cell; 32-byte records and the domain."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n3 = grid ** 3
    num = torch.tensor(per, device="cuda")[torch.randint(0, len(per), (n3,), generator=g, device="cuda")]
    cell = torch.repeat_interleave(torch.arange(n3, device="cuda"), num)
    low = torch.stack([cell % grid, cell // grid % grid, cell // grid ** 2], 1).float()
    cen = torch.rand((n3, 3), generator=g, device="cuda")[cell]
    x = cen + 0.2 * torch.randn((len(cell), 3), generator=g, device="cuda")
    rec = torch.zeros((len(cell), 8), dtype=torch.float32, device="cuda")
    rec[:, 2:5] = low + x.clamp(0.001, 0.999)
    rec[:, 5:8] = torch.randn((len(cell), 3), generator=g, device="cuda")
    rec = rec[torch.randperm(len(cell), generator=g, device="cuda")].contiguous()
    dom = L.domain([0] * 3, [grid] * 3, [0] * 3, [grid] * 3, [1.0] * 3, 0.16, 10)
    return rec, dom


def linked(ctx, torch, rec, dom, T=0, copies=1):
    n = len(rec)
    recs = rec.repeat(copies, 1).contiguous()
    vols = []
    for k in range(copies):
        v = L.Volume()
        v.offset, v.n, v.domain = k * n, n, dom
        vols.append(v)
    N = n * copies
    nxt = torch.zeros(N, dtype=torch.int32, device="cuda")
    lab = torch.zeros(N, dtype=torch.int32, device="cuda")
    hal = torch.zeros((N // 10 + 1, 8), dtype=torch.float64, device="cuda")
    off = np.zeros(copies + 1, np.uint64)
    st = L.Stats()
    rc, nh = ctx.link_ex(L.particles(recs, N), vols, L.opts(0, 0.0, T), nxt, lab, None, hal, None,
                         N // 10 + 1, off, st)
    L.check(rc)
    return nxt.view(copies, n), lab.view(copies, n), hal.view(torch.int32)[:nh], off, st


@pytest.mark.parametrize("grid,lo,hi", [(8, 1, 512), (9, 513, 16384), (27, 16385, 49152),
                                        (38, 49153, 60000)])
def test_small_cell_parts(ctx, grid, lo, hi):
    # as dense cells (split over waves by their number) and, with the
    # threshold above every cell, particle by particle
    import torch

    rec, dom = cells_of(torch, [24, 30, 64, 65, 95, 96, 130, 159, 160, 200, 255] if grid < 30 else [24, 40, 97], grid, grid)
    print("grid", grid, "n", len(rec), flush=True)
    a = linked(ctx, torch, rec, dom, T=24)
    b = linked(ctx, torch, rec, dom, T=512)
    assert lo <= a[4].ndense <= hi and b[4].ndense == 0
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)


@pytest.mark.parametrize("copies", [4, 32])
def test_dense_cell_workgroups(ctx, copies):
    # one volume below 2^20 particles, and copies of it in one call of more
    # than 2^20 and 2^23: 1024, 512 and 256 threads a cell
    import torch

    rec, dom = cells_of(torch, [3, 10, 257, 400, 900, 2500], 8, 5)
    rec = rec[:300000]
    print("n", len(rec), "copies", copies, flush=True)
    assert len(rec) * copies > (1 << 20 if copies == 4 else 1 << 23)
    a = linked(ctx, torch, rec, dom)
    b = linked(ctx, torch, rec, dom, copies=copies)
    assert a[4].pair_tests_kernel[1] > 0
    nh = int(a[3][1])
    for k in range(copies):
        assert torch.equal(a[0][0], b[0][k]) and torch.equal(a[1][0], b[1][k])
        assert torch.equal(a[2], b[2][int(b[3][k]):int(b[3][k + 1])])
    assert len(b[2]) == nh * copies
