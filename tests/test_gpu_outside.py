"""Device-resident particles outside their volume: FOF_E_DOMAIN, whatever cells
they would fall into, and a context that links right afterwards."""
import time

import numpy as np
import pytest

from cm_halofinder_amd import _lib as L
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

BOX, CELL, LINK = 12.0, 1.0, 0.2


def particles(seed, n=6000, corner=400):
    """Uniform, with a first cell dense enough for sub-cells."""
    rng = np.random.default_rng(seed)
    P = np.zeros(n + corner, L.PART_DTYPE)
    pos = np.concatenate([rng.random((n, 3)) * BOX, rng.random((corner, 3)) * CELL])
    P["Pos"] = pos[rng.permutation(len(pos))].clip(0, 11.999)
    P["Vel"] = rng.normal(0, 100, P["Vel"].shape)
    return P


def domain(variable, nphalomin=2):
    vl = L.VarLinkTable([0] * 3, 3 * BOX ** 2, np.linspace(0.15, 0.25, 64) ** 2) if variable else None
    return L.domain([0] * 3, [BOX] * 3, [0] * 3, [BOX] * 3, [CELL] * 3, LINK, nphalomin, varlink=vl)


def outside(P, how, rng):
    P = P.copy()
    if how == "all":  # the wrong domain: everything beyond it, on every side
        P["Pos"] += rng.choice([-40, 40], (len(P), 3))
    else:
        k = rng.choice(len(P), 1 if how == "one" else 700, replace=False)
        bad = rng.choice([-3.0, 5.0, 11.5, 12.5, 1e6, np.nan, np.inf, -np.inf], (len(k), 3))
        bad[np.arange(len(k)), rng.integers(0, 3, len(k))] = rng.choice([-3.0, 12.5, 1e6, np.nan, np.inf], len(k))
        P["Pos"][k] = bad
    return P


def call(ctx, P, vols, flags=0, bufs=None):
    import torch

    n = len(P)
    if bufs is None:
        bufs = [torch.zeros(n * 32, dtype=torch.uint8, device="cuda"),
                *(torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2)),
                torch.zeros(n * 64, dtype=torch.uint8, device="cuda")]
    bufs[0].copy_(torch.from_numpy(P.view(np.uint8)))
    off = np.zeros(len(vols) + 1, np.uint64)
    rc = ctx.link_batch(L.particles(bufs[0], n), vols, L.opts(L.OPT_OUT_DEVICE | flags), bufs[1], bufs[2], bufs[3],
                        n, off)
    return rc, bufs


def volumes(n, dom):
    vols = [L.Volume(), L.Volume()]  # the second one small and empty of dense cells
    for v, (a, b) in zip(vols, ((0, n - 500), (n - 500, n))):
        v.offset, v.n, v.domain = a, b - a, dom
    return vols


@pytest.mark.parametrize("variable", [False, True])
@pytest.mark.parametrize("flags", [0, L.OPT_SPARSE])
@pytest.mark.parametrize("how", ["one", "many", "all"])
def test_outside_is_refused(ctx, how, flags, variable):
    rng = np.random.default_rng(len(how) + flags + variable)
    for k, nph in enumerate((2, 1)):
        P, dom = particles(k), domain(variable, nph)
        vols = volumes(len(P), dom)
        fresh = L.Context(0)
        rc, want = call(fresh, P, vols, flags)
        L.check(rc)
        fresh.close()
        rc, bufs = call(ctx, outside(P, how, rng), vols, flags)
        assert rc == L.E_DOMAIN
        rc, bufs = call(ctx, P, vols, flags, bufs)
        L.check(rc)
        for a, b in zip(want[1:3], bufs[1:3]):
            assert np.array_equal(a.cpu().numpy(), b.cpu().numpy())
        if not variable:
            check_against_oracle(ctx, P, dom, flags=flags)


def test_graph_replays_after_a_refused_call():
    ctx, rng = L.Context(0), np.random.default_rng(5)
    P, dom = particles(9), domain(False)
    vols = volumes(len(P), dom)
    rc, bufs = call(ctx, outside(P, "many", rng), vols, L.OPT_GRAPH)  # captured
    assert rc == L.E_DOMAIN
    rc, _ = call(ctx, P, vols, L.OPT_GRAPH, bufs)
    L.check(rc)
    lab = bufs[2].cpu().numpy()
    rc, _ = call(ctx, outside(P, "one", rng), vols, L.OPT_GRAPH, bufs)
    assert rc == L.E_DOMAIN
    rc, _ = call(ctx, P, vols, 0, bufs)
    L.check(rc)
    assert np.array_equal(lab, bufs[2].cpu().numpy())
    ctx.close()


def test_one_outside_of_many_is_quick(ctx):
    # its cell by coordinates lies at the far end of the particles sorted in
    # between: no thread walks those
    rng = np.random.default_rng(1)
    n = 4_000_000
    P = np.zeros(n, L.PART_DTYPE)
    P["Pos"] = (rng.random((n, 3), np.float32) * 158).clip(0, 157.999)
    dom = L.domain([0] * 3, [158] * 3, [0] * 3, [158] * 3, [1] * 3, 0.2, 20)
    vol = L.Volume()
    vol.offset, vol.n, vol.domain = 0, n, dom
    rc, bufs = call(ctx, P, [vol])
    L.check(rc)
    P["Pos"][12345] = 1e9
    t = time.perf_counter()
    rc, _ = call(ctx, P, [vol], 0, bufs)
    assert rc == L.E_DOMAIN and time.perf_counter() - t < 1.0
