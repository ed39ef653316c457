"""Dense cells of 256 particles or more with chosen numbers of occupied
sub-cells and neighbour items, against the oracle: few runs (every pair
tested) and many (the window bitmap), runs from one particle to hundreds,
neighbour items below, at and above a chunk.  Bar: bit-exact labels, ring and
halo table (test_gpu_parity.check_against_oracle)."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu


def block(occupied, per_run, around, l, seed):
    """A 5^3 grid of unit cells: the central cell holds `per_run` particles in
    each of `occupied` sub-cells, its 26 neighbours `around` particles each
    spread over the cell, the outer cells a few."""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(np.sqrt(3.0) / (l * (1 - 1e-6))))
    bins = rng.permutation(m ** 3)[:occupied]
    sub = np.stack([bins % m, bins // m % m, bins // m ** 2], 1)
    n = np.broadcast_to(per_run, occupied) if np.isscalar(per_run) else rng.choice(per_run, occupied)
    who = np.repeat(np.arange(occupied), n)
    parts = [2 + (sub[who] + 0.05 + 0.9 * rng.random((len(who), 3))) / m]
    for z in range(5):
        for y in range(5):
            for x in range(5):
                if (x, y, z) == (2, 2, 2):
                    continue
                near = max(abs(x - 2), abs(y - 2), abs(z - 2)) == 1
                k = around if near else 3
                parts.append(np.array([x, y, z]) + rng.random((k, 3)))
    pos = np.concatenate(parts)
    P = np.zeros(len(pos), L.PART_DTYPE)
    P["Pos"] = pos[rng.permutation(len(pos))].clip(0, 4.999).astype(np.float32)
    P["Vel"] = rng.normal(0, 100, (len(pos), 3)).astype(np.float32)
    P["ID"] = np.arange(len(pos))
    return P, L.domain([0] * 3, [5] * 3, [0] * 3, [5] * 3, [1] * 3, l, 2)


@pytest.mark.parametrize("l", [0.2, 0.34, 0.15])
@pytest.mark.parametrize("occupied,per_run", [
    (1, 300), (2, 200), (23, 12), (24, 11), (25, 11), (63, 5), (64, 4), (65, (1, 2, 4, 5, 40)),
    (129, (1, 3, 4, 5, 9)), (216, (2, 4, 300))])
@pytest.mark.parametrize("around", [0, 17, 18, 60])
def test_dense_cell(ctx, occupied, per_run, around, l):
    if l == 0.34 and occupied > 125:
        occupied = 200
    P, dom = block(occupied, per_run, around, l, seed=occupied * 100 + around)
    check_against_oracle(ctx, P, dom)


def test_dense_cells_full_neighbourhood(ctx):
    # every cell dense: the neighbours' runs fill several chunks
    rng = np.random.default_rng(3)
    n = 125 * 700
    P = np.zeros(n, L.PART_DTYPE)
    P["Pos"] = (5 * rng.random((n, 3))).clip(0, 4.999).astype(np.float32)
    dom = L.domain([0] * 3, [5] * 3, [0] * 3, [5] * 3, [1] * 3, 0.15, 2)
    lab, st = check_against_oracle(ctx, P, dom)
    assert st.ndense >= 100
