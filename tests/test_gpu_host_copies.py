"""Host particles and outputs, whose copies go through page-locked pieces from
8 MiB on.  Bar: every output equal, byte for byte, to the call on device memory,
and a particle outside its domain found wherever in the records it stands."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L

pytestmark = pytest.mark.gpu

MIB8 = 8 << 20


def records(n, stride, seed):
    """n records of stride bytes, in pairs a tenth of a linking length apart."""
    g = np.random.default_rng(seed)
    half = g.random(((n + 1) // 2, 3), np.float32) * np.float32(14.0) + np.float32(1.0)
    pos = np.concatenate([half, half + np.float32(0.02)])[:n]
    rec = np.zeros((n, stride), np.uint8)
    rec[:, 0:8] = g.permutation(n).astype(np.uint64)[:, None].view(np.uint8)
    rec[:, 8:20] = np.ascontiguousarray(pos).view(np.uint8)
    rec[:, 20:32] = g.standard_normal((n, 3), np.float32).view(np.uint8)
    return rec


def volumes(sizes):
    dom = L.domain([0] * 3, [16] * 3, [0] * 3, [16] * 3, [0.25] * 3, 0.05, 2)
    vols, at = [], 0
    for m in sizes:
        v = L.Volume()
        v.offset, v.n, v.domain = at, m, dom
        vols.append(v)
        at += m
    return vols


@pytest.mark.parametrize("sizes,stride", [
    ([MIB8 // 32 - 1], 32),             # the last that is copied at once
    ([MIB8 // 32], 32),                 # the first in pieces
    ([MIB8 // 44 + 1], 44),             # pieces that whole records do not fill
    ([2 * MIB8 // 32 + 1, 0, 5], 32),   # a last piece of a few records, several volumes
    ([(1 << 21) + 3], 32),              # outputs in pieces too, buffers used again
    ([1 << 21, (1 << 21) + 77], 32),
])
def test_host_copies(ctx, sizes, stride):
    import torch

    n = sum(sizes)
    print("n", n, "stride", stride, flush=True)
    rec, vols = records(n, stride, n), volumes(sizes)
    cap = n // 2 + 1

    def outputs(make):
        return [make(n * 4), make(n * 4), make(n * 8), make(cap * 64), make(cap * 192)]

    host = outputs(lambda b: np.zeros(b, np.uint8))
    off = np.zeros(len(vols) + 1, np.uint64)
    rc, nh = ctx.link_ex(L.particles(rec.reshape(-1), n, stride), vols, L.opts(), *host, cap, off)
    L.check(rc)
    dev = outputs(lambda b: torch.zeros(b, dtype=torch.uint8, device="cuda"))
    drec = torch.from_numpy(rec.reshape(-1)).cuda()
    doff = np.zeros(len(vols) + 1, np.uint64)
    rc, dnh = ctx.link_ex(L.particles(drec, n, stride), vols, L.opts(), *dev, cap, doff)
    L.check(rc)
    torch.cuda.synchronize()
    assert nh == dnh and nh > 0 and np.array_equal(off, doff)
    for h, d, b in zip(host, dev, (n * 4, n * 4, n * 8, nh * 64, nh * 192)):
        assert np.array_equal(h[:b], d[:b].cpu().numpy())

    for at in {0, n // 2, n - 1}:
        bad = rec.copy()
        bad[at, 8:12] = np.frombuffer(np.float32(np.nan).tobytes(), np.uint8)
        rc, nh = ctx.link_ex(L.particles(bad.reshape(-1), n, stride), vols, L.opts(), *host, cap, off)
        assert rc == L.E_DOMAIN and nh == 0
