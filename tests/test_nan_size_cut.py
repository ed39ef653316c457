"""A size cut that is not a number: no group is below it (src_v2/FOF.c:202), so
every particle may be a halo and the workspace has room for that."""
import numpy as np
import pytest

from cm_halofinder_amd import _lib as L


def volumes(n, cuts):
    vols = []
    for k, c in enumerate(cuts):
        v = L.Volume()
        v.offset, v.n = k * n, n
        v.domain = L.domain([0] * 3, [8] * 3, [0] * 3, [8] * 3, [1] * 3, 0.3, c)
        vols.append(v)
    return vols


@pytest.mark.parametrize("cuts", [[np.nan], [20, np.nan], [np.nan, 20]])
def test_workspace_holds_every_group(cuts):
    n = 3000
    parts = L.particles(np.zeros(len(cuts) * n, L.PART_DTYPE))
    keep_all = [0 if np.isnan(c) else c for c in cuts]
    assert L.plan(parts, volumes(n, cuts)).workspace_bytes == L.plan(parts, volumes(n, keep_all)).workspace_bytes


@pytest.mark.gpu
def test_every_group_is_a_halo(ctx):
    from test_gpu_parity import check_against_oracle

    rng = np.random.default_rng(2)
    P = np.zeros(3000, L.PART_DTYPE)
    P["Pos"] = (8 * rng.random((3000, 3))).clip(0, 7.999)
    P["Vel"] = rng.normal(0, 100, P["Vel"].shape)
    lab, st = check_against_oracle(ctx, P, volumes(3000, [np.nan])[0].domain)
    assert st.nhalos == st.ngroups > 1000
