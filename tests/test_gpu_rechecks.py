"""The FP64 re-decisions a call reports: of the tests it counts, however the
link kernels share a cell out."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu

TIE = np.array([15, 20, 0]) / 128  # as long as the linking length
LINK = 25 / 128


def cells(k, here, there):
    """k cells of a grid, three apart: `here` particles at one place and `there`
    at one place exactly a linking length away."""
    side = int(np.ceil(k ** (1 / 3)))
    q = np.arange(k)
    at = 3.0 * np.stack([q % side, q // side % side, q // side ** 2], 1) + 0.25
    pos = np.concatenate([np.repeat(at, here, 0), np.repeat(at + TIE, there, 0)])
    P = np.zeros(len(pos), L.PART_DTYPE)
    P["Pos"] = pos[np.random.default_rng(k).permutation(len(pos))]
    box = 3.0 * side
    return P, L.domain([0] * 3, [box] * 3, [0] * 3, [box] * 3, [1] * 3, LINK, 2)


def stats(ctx, P, dom, T):
    n = len(P)
    st = L.Stats()
    rc, _ = ctx.link(L.particles(P), dom, L.opts(0, 0.0, T), np.empty(n, np.uint32), np.empty(n, np.uint32),
                     np.empty(n, L.HALO_DTYPE), n, st)
    L.check(rc, "fof_link_gpu")
    return st


@pytest.mark.parametrize("here,there,T", [(1, 1, 2), (60, 60, 24), (100, 100, 24)])
@pytest.mark.parametrize("k", [600, 17000])
def test_small_cells_in_parts(ctx, here, there, T, k):
    # one cell is linked by eight waves, of 600 the largest by four, of 17000 by two
    if k * (here + there) > 1_000_000:
        k = 1_000_000 // (here + there)
    one, many = (stats(ctx, *cells(c, here, there), T) for c in (1, k))
    assert one.ndense == 1 and many.ndense == k and many.ngroups == k
    assert one.rechecks >= here * there
    assert many.pair_tests == k * one.pair_tests
    assert many.rechecks == k * one.rechecks


def test_short_run_against_a_long_one(ctx):
    # the first pair of the two runs links; the tile past the short run's end is no test
    P, dom = cells(1, 1, 300)
    st = stats(ctx, P, dom, 0)
    assert st.ndense == 1 and st.ngroups == 1
    assert st.pair_tests == 1 and st.rechecks == 1
