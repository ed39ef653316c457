"""Pairs of sub-cells with many particles each, linked through few of their
particle pairs or through none: particle pairs below and above the number
from which a whole wave takes them (65536), and beyond 2^32.  Labels, ring and
halos against their closed form."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu


def piles(many, near):
    """x of two piles in sub-cells of [2, 3) (cells of side 1, 9 sub-cells an axis,
    l = 0.2): many + 1 particles in [2, 2.11), all but `near` of them 0.245 from
    the `many` of the second, in [2.22, 2.33); and each particle's pile."""
    x = np.concatenate([np.full(near, 2.106), np.full(many + 1 - near, 2.005), np.full(many, 2.25)])
    return x, np.repeat([0, 1], [many + 1, many])


def check(ctx, pos, who, box):
    """who: the group of each particle."""
    n = len(pos)
    order = np.random.default_rng(n).permutation(n)
    who = who[order]
    P = np.zeros(n, L.PART_DTYPE)
    P["Pos"] = pos[order]
    P["Vel"] = np.random.default_rng(1).normal(0, 100, (n, 3))
    dom = L.domain([0] * 3, box, [0] * 3, box, [1] * 3, 0.2, 2)
    nxt, lab, halos, st = np.empty(n, np.uint32), np.empty(n, np.uint32), np.empty(n, L.HALO_DTYPE), L.Stats()
    rc, nh = ctx.link(L.particles(P), dom, L.opts(), nxt, lab, halos, n, st)
    L.check(rc, "fof_link_gpu")
    at = np.argsort(who, kind="stable")
    members = np.split(at, np.flatnonzero(np.diff(who[at])) + 1)
    members.sort(key=lambda m: m[0])
    assert st.ngroups == nh == len(members)
    for h, m in zip(halos, members):
        assert (lab[m] == m[0]).all() and np.array_equal(nxt[m], np.roll(m, -1) + 1)
        assert h["head"] == m[0] and h["n"] == len(m)
        for f, s in (("Pos", "sum_pos"), ("Vel", "sum_vel")):
            assert np.array_equal(h[s], np.cumsum(P[f][m].astype(np.float64), 0)[-1])
    return st


@pytest.mark.parametrize("many,near", [
    (255, 0), (255, 1), (256, 0), (256, 1), (1000, 1), (65536, 0), (65536, 1), (65536, 256)])
def test_two_piles(ctx, many, near):
    x, pile = piles(many, near)
    pos = np.stack([x, np.full(len(x), 2.05), np.full(len(x), 2.05)], 1)
    st = check(ctx, pos, pile * (near == 0), [5] * 3)
    assert st.ndense == 1


def test_more_pairs_than_are_listed(ctx):
    # 400 cells three apart, every other one's piles linked through one particle
    k = np.arange(400)
    off = 3.0 * np.stack([k % 8, k // 8 % 8, k // 64], 1)
    pos, who = [], []
    for c in k:
        x, pile = piles(300, c % 2)
        pos.append(np.stack([x, np.full(len(x), 2.05), np.full(len(x), 2.05)], 1) + off[c])
        who.append(2 * c + pile * (c % 2 == 0))
    st = check(ctx, np.concatenate(pos), np.concatenate(who), [26.0] * 3)
    assert st.ndense == 400
