"""Tile lists by direct placement against the oracle and the sorting modes, bit
for bit (whole numbers: no tolerance): pair counts around a wave, a group of the
pairs kernel and a window, grids around a 32 x 32 patch, several cameras whose
rows share a patch, boxes over the whole grid, all pairs in one tile, equal
depths, culled pairs; and the forms that stay with the sort (a negative depth, a
grid past the packed fields)."""
import numpy as np
import pytest
import torch

from gsplat.cuda import _wrapper as W
from oracle import ubs_oracle as O

pytestmark = pytest.mark.gpu


def _inputs(C, N, tw, th, ts, kind, seed):
    g = np.random.Generator(np.random.PCG64(seed))
    m2 = g.uniform((-ts, -ts), ((tw + 1) * ts, (th + 1) * ts), (C, N, 2))
    radii = g.integers(-1, 3 * ts, (C, N))
    if kind == "one_tile":
        m2[:] = (tw // 2 + 0.5) * ts, (th // 2 + 0.5) * ts
        radii[:] = ts // 4
    elif kind == "whole_grid":
        radii[:, ::3] = 2 * ts * max(tw, th)
    depths = g.uniform(1.0, 9.0, (C, N))
    if kind == "ties":
        depths = np.round(depths)
    return m2.astype(np.float32), radii.astype(np.int32), depths.astype(np.float32)


def _run(mode, m2, radii, depths, ts, tw, th):
    before = W.isect_sort_mode()
    W.set_isect_sort_mode(mode)
    try:
        tpg, ids, flat, offs = W.isect_tiles_offsets(*(torch.tensor(a, device="cuda") for a in (m2, radii, depths)),
                                                     ts, tw, th)
    finally:
        W.set_isect_sort_mode(before)
    return [None if t is None else t.cpu().numpy() for t in (tpg, ids, flat, offs)]


@pytest.mark.parametrize("C,N,tw,th,ts,kind", [
    (1, 1, 1, 1, 16, "random"), (1, 63, 5, 3, 16, "random"), (1, 65, 32, 32, 8, "ties"), (1, 1023, 33, 31, 16, "random"),
    (1, 1025, 31, 33, 16, "whole_grid"), (1, 2049, 20, 20, 16, "one_tile"), (1, 5000, 65, 40, 16, "ties"),
    (3, 1500, 40, 21, 16, "random"), (2, 700, 120, 68, 16, "whole_grid"), (5, 90, 3, 13, 32, "ties"),
    (1, 150000, 16, 16, 16, "random"), (1, 70000, 12, 9, 16, "one_tile")])
def test_placement_matches_the_oracle(device, C, N, tw, th, ts, kind):
    m2, radii, depths = _inputs(C, N, tw, th, ts, kind, 7 * N + tw)
    assert W.lib().ubs_isect_bins_workspace_bytes(C, N, tw, th) > 0
    want_tpg, want_ids, want_flat = O.isect_tiles(m2, radii, depths, ts, tw, th)
    tpg, ids, flat, offs = _run("depth_first", m2, radii, depths, ts, tw, th)
    assert np.array_equal(tpg.ravel(), np.asarray(want_tpg).ravel())
    assert np.array_equal(ids, want_ids) and np.array_equal(flat, want_flat)
    assert np.array_equal(offs, O.isect_offset_encode(want_ids, C, tw, th))


@pytest.mark.parametrize("case", ["negative_depth", "wide_grid", "all_culled"])
def test_forms_beside_the_placement(device, case):
    C, N, tw, th, ts = 2, 900, 30, 20, 16
    if case == "wide_grid":
        tw, th = 70000, 1
        assert W.lib().ubs_isect_bins_workspace_bytes(C, N, tw, th) == 0
    m2, radii, depths = _inputs(C, N, tw, th, ts, "random", 3)
    if case == "negative_depth":
        depths[0, ::5] *= -1
    if case == "all_culled":
        radii[:] = 0
    got, want = (_run(mode, m2, radii, depths, ts, tw, th) for mode in ("depth_first", "onesweep"))
    for a, b in zip(got[:3], want[:3]):
        assert np.array_equal(a, b)
    if case == "all_culled":
        assert got[1].size == 0 and (got[3] is None or not got[3].any())
