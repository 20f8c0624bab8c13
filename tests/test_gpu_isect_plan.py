"""Tile lists by direct placement at the sizes where its plan changes, bit for bit
against the sort of all id bits (whole numbers: no tolerance): more blocks of pairs
than the cutting workgroup has threads, more tasks than the counting and placing
grids, all pairs in one patch (fuller tasks), more than 12.8k blocks, exactly 512
patches, and a patch more (which stays with the sort)."""
import pytest
import torch

from gsplat.cuda import _wrapper as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,N,tw,th,radius,placed", [
    (2, 600_000, 120, 68, 20, True),      # 1172 blocks
    (3, 1_000_000, 120, 68, 12, True),    # about 6000 tasks
    (1, 1_200_000, 32, 16, 6, True),      # one patch: tasks of 2300 pairs
    (1, 457_729, 30, 12, 40, True),       # 448 blocks of which the last holds one pair: the first with 1024 tasks
    (1, 457_728, 33, 12, 10, True),       # 447 blocks
    (5, 2_700_000, 60, 34, 5, True),      # 13184 blocks
    (1, 300_000, 512, 512, 40, True),     # 512 patches
    (8, 30_000, 64, 512, 30, True),       # 512 patches in rows of cameras
    (1, 40_000, 1, 1, 6, True), (1, 40_000, 5, 6, 20, True), (1, 40_000, 8, 4, 20, True),  # 1, 30 and 32 tiles
    (4, 500_000, 120, 68, 6, True),       # 68 patches: planned after the count is known
    (8, 300_000, 120, 68, 2, True),       # 136 patches, few entries
    (1, 50_000, 512, 513, 40, False),     # 528 patches
    (1, 50_000, 513, 512, 40, False)])    # 544
def test_plan_matches_the_sort(device, C, N, tw, th, radius, placed):
    assert (W.lib().ubs_isect_bins_workspace_bytes(C, N, tw, th) > 0) == placed
    ts = 16
    g = torch.Generator(device=device).manual_seed(N + tw)
    m2 = torch.rand((C, N, 2), device=device, generator=g) * torch.tensor([tw * ts, th * ts], device=device)
    radii = torch.randint(-1, radius, (C, N), device=device, generator=g, dtype=torch.int32)
    depths = torch.rand((C, N), device=device, generator=g) * 4.0 + 2.0
    depths = torch.where(radii % 3 == 0, (depths * 64).round() / 64, depths)  # a third of them tied
    out = []
    before = W.isect_sort_mode()
    try:
        for mode in ("depth_first", "onesweep"):
            W.set_isect_sort_mode(mode)
            tpg, ids, flat, offs = W.isect_tiles_offsets(m2, radii, depths, ts, tw, th)
            if offs is None:
                offs = W.isect_offset_encode(ids, C, tw, th)
            out.append((tpg, ids, flat, offs))
    finally:
        W.set_isect_sort_mode(before)
    if placed:  # also where the sort is taken for its speed
        st = W.isect_begin(m2, radii, depths, ts, tw, th)
        if st.bins is None:
            W._plan_bins(st)
        out.append(W.isect_finish(st, *W.isect_read_info([st])[0]))
        assert out[-1][3] is not None
    assert out[0][1].numel() > N // 8
    for got in out[1:]:
        for a, b in zip(out[0], got):
            assert torch.equal(a, b)


def test_a_state_can_be_finished_twice(device):
    g = torch.Generator(device=device).manual_seed(5)
    m2 = torch.rand((2, 5000, 2), device=device, generator=g) * 300.0
    radii = torch.randint(0, 30, (2, 5000), device=device, generator=g, dtype=torch.int32)
    depths = torch.rand((2, 5000), device=device, generator=g) + 1.0
    st = W.isect_begin(m2, radii, depths, 16, 20, 20)
    info = W.isect_read_info([st])[0]
    first, second = W.isect_finish(st, *info), W.isect_finish(st, *info)
    for a, b in zip(first[:3], second[:3]):
        assert torch.equal(a, b)
