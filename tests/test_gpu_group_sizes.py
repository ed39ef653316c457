"""Groups of chosen sizes against the oracle: the sizes where the halo sums'
blocks (64 members, 256 ahead) and the member sorts' ways of sorting change.

Bar: test_gpu_outputs.check_volume (bit-exact labels, ring, canonical labels,
halo table and raw second moments; centred moments within 1e-12 of their
scale)."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L
from test_gpu_outputs import check_volume, link_ex

pytestmark = pytest.mark.gpu

BLOCKS = [1, 2, 3, 4, 5, 7, 8, 9, 63, 64, 65, 127, 128, 129, 255, 256, 257, 319, 320, 321, 511, 512,
          513, 575, 577, 769]
SORTS = [1, 2, 4, 5, 64, 65, 512, 513, 1023, 1024, 1025, 2047, 2049, 3071, 4095, 4096, 4097]
LARGE = [3, 1024, 1025, 5000, 8191, 8192, 8193, 16383, 16384, 16385, 20001]


def clusters(sizes, seed, l=0.2):
    """Compact clusters of the given sizes (every pair linked) on a lattice
    of spacing 2, members shuffled over the input order."""
    rng = np.random.default_rng(seed)
    k = int(np.ceil(len(sizes) ** (1 / 3)))
    cen = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[: len(sizes)]
    cen = 2.0 * cen[rng.permutation(len(sizes))] + 1.0
    pos = np.repeat(cen, sizes, 0) + rng.uniform(-0.05, 0.05, (sum(sizes), 3))
    n = len(pos)
    P = np.zeros(n, L.PART_DTYPE)
    P["Pos"] = pos[rng.permutation(n)].astype(np.float32)
    P["Vel"] = rng.normal(0, 300, (n, 3)).astype(np.float32)
    P["ID"] = rng.permutation(n) + 7
    box = [2.0 * k + 1.0] * 3
    dom = L.domain([0] * 3, box, [0] * 3, box, [0.9] * 3, l, 1)
    v = L.Volume()
    v.offset, v.n, v.domain = 0, n, dom
    return P, v


@pytest.mark.parametrize("moments", [False, True])
@pytest.mark.parametrize("nphalomin", [1.0, 5.0])
@pytest.mark.parametrize("sizes", [BLOCKS, SORTS, LARGE], ids=["blocks", "sorts", "large"])
def test_group_sizes(ctx, sizes, nphalomin, moments):
    print("sizes", sizes, nphalomin, moments, flush=True)
    P, v = clusters(sizes, seed=len(sizes))
    v.domain.nphalomin = nphalomin
    rc, nh, nxt, lab, mid, halos, mom, hoff, st = link_ex(ctx, P, [v], moments=moments)
    L.check(rc)
    check_volume(P, v, lab, nxt, mid, halos[:nh], mom[:nh] if moments else None)
    assert nh == sum(s >= nphalomin for s in sizes)
