"""Group and member lists beyond one block's run of bitmap words, one scan's
tiles and one sort's LDS, against their closed form."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu


# up to 2^25 particles a block of the group list takes one run of words, beyond
# two and more; above 2048 * 4096 * 4096 / 256 the index partition's scan has
# a launch of its own for the tiles' sums
@pytest.mark.parametrize("half,flags", [
    (17_000_003, 0), (17_000_003, L.OPT_WRITE_PAIRS), (2 ** 24, 0), (68_000_003, 0)])
def test_pairs_far_apart_in_the_list(half, flags):
    # sites of a unit lattice; particle half + i lies beside particle i, or
    # (every third) half a cell away
    import torch

    dev, n, side = "cuda", 2 * half, int(np.ceil(half ** (1 / 3)))
    i = torch.arange(half, device=dev)
    alone = i % 3 == 0
    rec = torch.zeros((n, 8), dtype=torch.float32, device=dev)
    for h, off in ((slice(0, half), None), (slice(half, n), torch.where(alone, 0.5, 0.0625))):
        rec[h, 2] = (i % side).float() + 0.25 + (0 if off is None else off)
        rec[h, 3] = (i // side % side).float() + 0.25
        rec[h, 4] = (i // side ** 2).float() + 0.25
        rec[h, 5] = (i % 1000).float() + (0.0 if off is None else 0.5)
    dom = L.domain([0] * 3, [side] * 3, [0] * 3, [side] * 3, [1] * 3, 0.2, 2)
    vol = L.Volume()
    vol.offset, vol.n, vol.domain = 0, n, dom
    nxt = torch.empty(n, dtype=torch.int32, device=dev)
    lab = torch.empty(n, dtype=torch.int32, device=dev)
    pairs = i[~alone]
    halos = torch.zeros((len(pairs), 8), dtype=torch.float64, device=dev)
    ctx, off = L.Context(0), np.zeros(2, np.uint64)
    torch.cuda.synchronize()
    rc = ctx.link_batch(L.particles(rec, n), [vol], L.opts(L.OPT_OUT_DEVICE | flags), nxt, lab, halos, len(pairs), off)
    L.check(rc)
    assert off.tolist() == [0, len(pairs)]
    assert torch.equal(lab[:half], i.int())
    assert torch.equal(lab[half:], torch.where(alone, i + half, i).int())
    assert torch.equal(nxt[:half], torch.where(alone, i + 1, i + half + 1).int())
    assert torch.equal(nxt[half:], torch.where(alone, i + half + 1, i + 1).int())
    head = halos[:, 0].contiguous().view(torch.int32).view(-1, 2)
    assert torch.equal(head[:, 0], pairs.int()) and bool((head[:, 1] == 2).all())
    sums = rec[pairs, 2:8].double() + rec[half + pairs, 2:8].double()
    assert torch.equal(halos[:, 2:8], sums)
    ctx.close()


@pytest.mark.parametrize("sizes", [
    (16384, 16385), (32768, 32769), (65536, 65537, 40000), (131072, 131073, 5000, 3)])
def test_large_groups(ctx, sizes):
    # members of a group at one place, in random input order: above 16384 the
    # sort's passes go through scratch, two of them or three (by the bits of an
    # index), so that a group ends in either buffer
    rng = np.random.default_rng(sum(sizes))
    who = np.repeat(np.arange(len(sizes)), sizes)
    at = np.stack([2.5 * np.arange(len(sizes)) + 0.3] + 2 * [np.full(len(sizes), 1.7)], 1)
    who = who[rng.permutation(len(who))]
    n, box = len(who), 2.5 * len(sizes) + 1
    P = np.zeros(n, L.PART_DTYPE)
    P["Pos"] = at[who]
    P["Vel"] = rng.normal(0, 100, (n, 3))
    dom = L.domain([0] * 3, [box] * 3, [0] * 3, [box] * 3, [1] * 3, 0.2, 2)
    nxt, lab, halos = np.empty(n, np.uint32), np.empty(n, np.uint32), np.empty(n, L.HALO_DTYPE)
    rc, nh = ctx.link(L.particles(P), dom, L.opts(), nxt, lab, halos, n)
    L.check(rc, "fof_link_gpu")
    members = sorted((np.flatnonzero(who == g) for g in range(len(sizes))), key=lambda m: m[0])
    assert nh == len(sizes)
    for h, m in zip(halos, members):
        assert h["head"] == m[0] and h["n"] == len(m)
        assert (lab[m] == m[0]).all() and np.array_equal(nxt[m], np.roll(m, -1) + 1)
        assert np.array_equal(h["sum_vel"], np.cumsum(P["Vel"][m].astype(np.float64), 0)[-1])
