"""Two sub-cells whose particle pairs number more than 2^32, linked through few
of them only: one group.  Labels, ring and halo against their closed form (all
particles one group, heads and sums in index order)."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("many,near", [(65536, 256), (1000, 1)])
def test_runs_linked_by_a_few_pairs(ctx, many, near):
    # cells of side 1, 9 sub-cells an axis: the first run in x in [2, 2.11), all
    # but `near` of its particles 0.245 from the second run (l = 0.2), whose
    # particles lie in [2.22, 2.33); (many + 1) * many pairs
    x = np.concatenate([np.full(near, 2.106), np.full(many + 1 - near, 2.005), np.full(many, 2.25)])
    n = len(x)
    order = np.random.default_rng(many).permutation(n)
    P = np.zeros(n, L.PART_DTYPE)
    P["Pos"] = 2.05
    P["Pos"][:, 0] = x[order]
    P["Vel"] = np.random.default_rng(1).normal(0, 100, (n, 3))
    dom = L.domain([0] * 3, [5] * 3, [0] * 3, [5] * 3, [1] * 3, 0.2, 2)
    nxt, lab, halos, st = np.empty(n, np.uint32), np.empty(n, np.uint32), np.empty(n, L.HALO_DTYPE), L.Stats()
    rc, nh = ctx.link(L.particles(P), dom, L.opts(), nxt, lab, halos, n, st)
    L.check(rc, "fof_link_gpu")
    assert st.ndense == 1 and st.ngroups == 1 and nh == 1
    assert (lab == 0).all()
    assert np.array_equal(nxt, np.r_[2:n + 1, 1])
    assert halos["n"][0] == n and halos["head"][0] == 0
    assert np.array_equal(halos["sum_pos"][0], np.cumsum(P["Pos"].astype(np.float64), 0)[-1])
    assert np.array_equal(halos["sum_vel"][0], np.cumsum(P["Vel"].astype(np.float64), 0)[-1])
