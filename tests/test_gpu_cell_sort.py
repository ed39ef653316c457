"""The cell sort's ways over grid and particle counts: dense addressing (fine
buckets of 2^11 to 2^14 cells, one or two partition levels, tiles of 1024
particles upwards) against occupied-cell addressing, which sorts by another
method.  Bar: every output bit-identical."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu


def linked(ctx, P, n, dom, flags):
    import torch

    v = L.Volume()
    v.offset, v.n, v.domain = 0, n, dom
    nxt = torch.zeros(n, dtype=torch.int32, device="cuda")
    lab = torch.zeros(n, dtype=torch.int32, device="cuda")
    hal = torch.zeros((n // 2 + 1, 8), dtype=torch.float64, device="cuda")
    st = L.Stats()
    rc, nh = ctx.link_ex(L.particles(P, n), [v], L.opts(flags), nxt, lab, None, hal, None,
                         n // 2 + 1, None, st)
    L.check(rc)
    return nxt, lab, hal.view(torch.int32), nh, st


# cells per axis (lcell = 1): one bucket; 255, 256 and 257 buckets of 2^11;
# 512 and 513 of 2^14; 1280 (one level) and 1284 (two levels)
@pytest.mark.parametrize("grid,n", [
    ((2, 2, 2), 1), ((16, 16, 8), 1023), ((16, 16, 8), 1025), ((64, 64, 127), 200001),
    ((64, 64, 128), 2049), ((65, 64, 128), 70000), ((256, 256, 128), 1500000),
    ((256, 256, 64), 1048577), ((256, 256, 129), 1500001), ((256, 256, 320), 5700000), ((256, 256, 321), 5800001)])
def test_dense_sort_matches_occupied_cells(ctx, grid, n):
    import torch

    print("grid", grid, "n", n, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    ext = torch.tensor([float(c - 1) for c in grid], device="cuda")
    rec = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    pos = torch.rand((n, 3), generator=g, device="cuda") * ext
    # a third of them gathered near a few points, some on the upper faces
    k = n // 3
    cen = torch.rand((17, 3), generator=g, device="cuda") * ext
    who = torch.randint(0, 17, (k,), generator=g, device="cuda")
    pos[:k] = cen[who] + torch.randn((k, 3), generator=g, device="cuda")
    pos[: k // 50] = ext
    rec[:, 2:5] = torch.minimum(pos.clamp_min(0.0), ext)
    rec[:, 5:8] = torch.randn((n, 3), generator=g, device="cuda")
    rec = rec[torch.randperm(n, generator=g, device="cuda")].contiguous()
    hi = [float(c - 1) for c in grid]
    dom = L.domain([0] * 3, hi, [0] * 3, hi, [1.0] * 3, 0.2, 2)
    a = linked(ctx, rec, n, dom, 0)
    b = linked(ctx, rec, n, dom, L.OPT_SPARSE)
    assert a[4].sparse == 0 and b[4].sparse == 1
    assert a[4].ncells == int(np.prod(grid))
    assert a[3] == b[3]
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)


@pytest.mark.parametrize("full,thin", [(1, 1), (1, 40), (1, 400), (3, 2000), (130, 131)])
def test_occupied_rows_of_uneven_density(ctx, full, thin):
    # rows of 4000 cells holding a particle in every `full`-th or `thin`-th
    # cell, alternating: a wave's stretch of one row meets fewer or many times
    # more occupied cells in the next, against the oracle
    from test_gpu_parity import check_against_oracle

    rng = np.random.default_rng(full * 7 + thin)
    nx, parts = 4000, []
    for z in range(3):
        for y in range(7):
            x = np.arange(0, nx, full if (y + z) % 2 else thin)
            parts.append(np.stack([x, np.full(len(x), y), np.full(len(x), z)], 1) + rng.random((len(x), 3)))
    blob = np.array([1999.5, 3.5, 1.5]) + rng.normal(0, 0.3, (600, 3))  # a dense cell among them
    pos = np.concatenate(parts + [blob.clip([1998, 2, 0.01], [2002, 5, 2.99])])
    P = np.zeros(len(pos), L.PART_DTYPE)
    P["Pos"] = pos[rng.permutation(len(pos))].astype(np.float32).clip([0, 0, 0], [3999.9, 6.999, 2.999])
    P["ID"] = np.arange(len(pos))
    dom = L.domain([0] * 3, [nx, 7, 3], [0] * 3, [nx, 7, 3], [1] * 3, 0.8, 2)
    check_against_oracle(ctx, P, dom, flags=L.OPT_SPARSE)


# two levels: buckets of 2^12 cells, tiles of one and of several sub-tiles
# (7168 particles, 1024 tiles) with a remainder
@pytest.mark.parametrize("grid,n", [((300, 301, 280), 7340031), ((256, 256, 449), 14680065)])
def test_two_level_sort_matches_occupied_cells(ctx, grid, n):
    test_dense_sort_matches_occupied_cells(ctx, grid, n)


# labels and ring through the partition by index or straight, where the members
# end just before, at and after a tile of 1024 and an eighth of the list
@pytest.mark.parametrize("n", [1, 2, 255, 1023, 1024, 1025, 8191, 8192, 8193, 65537, 300007])
def test_partitioned_writes_match_direct_ones(ctx, n):
    import torch

    print("n", n, flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    side = max(4.0, (n / 6.0) ** (1.0 / 3.0))  # most particles have a neighbour within l
    rec = torch.zeros((n, 8), dtype=torch.float32, device="cuda")
    rec[:, 2:5] = torch.rand((n, 3), generator=g, device="cuda") * side
    dom = L.domain([0] * 3, [side] * 3, [0] * 3, [side] * 3, [1.0] * 3, 0.4, 2)
    a = linked(ctx, rec, n, dom, L.OPT_WRITE_DIRECT)
    b = linked(ctx, rec, n, dom, L.OPT_WRITE_PAIRS)
    assert a[3] == b[3]
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)
