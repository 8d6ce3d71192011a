"""Host side of the depth selector in culbm_amd.calibrate (no GPU)."""
from __future__ import annotations

import math

from culbm_amd.calibrate import SELECT_CELLS, depth_candidates


def test_depth_candidates_cover_the_launch_sizes_within_the_domain():
    for dom in ((288, 272, 280), (128, 128, 128), (512, 512, 512), (64, 64, 8), (1000, 1000, 3)):
        nx, ny, nz = dom
        c = depth_candidates(dom)
        assert c[0] == 0 and c == sorted(set(c))                # the automatic choice, then ascending
        assert all(2 <= d <= nz for d in c[1:]) or nz < 2
        for cells in SELECT_CELLS:                              # every target size is represented
            d = max(2, min(nz, math.ceil(cells / (nx * ny))))
            assert d in c


def test_depth_candidates_at_the_optimised_workload():
    # 288x272 planes of 78,336 cells: 1.4M cells is 18 planes, 2.6M is 34
    c = depth_candidates((288, 272, 280))
    assert 18 in c and 34 in c and 16 in c


def test_select_rejects_an_empty_candidate_list():
    import pytest

    from culbm_amd.calibrate import select

    with pytest.raises(ValueError):
        select((16, 16, 16), depths=())
    with pytest.raises(ValueError):
        select((16, 16, 16), inner_loops=())


def test_selector_does_not_report_a_depth_that_did_not_run():
    """Pull left to the library takes pairs at this size: no wavefront depth is
    reported for it, and a context's info names the depth that an explicit setting
    would take, not the two-step kernel's."""
    import fakehip

    fakehip.run("""
    from culbm_amd.calibrate import select
    dim = (112, 104, 96)
    rows = select(dim, stream_policy=0, depths=(0, 24), steps=4, develop=2)["candidates"]
    assert [(r["requested_depth"], r["wave_depth"], r["pairs"]) for r in rows] == [(0, 0, True), (24, 24, False)], rows
    rows = select(dim, stream_policy=1, depths=(0, 24), steps=4, develop=2)["candidates"]
    assert [(r["wave_depth"], r["pairs"]) for r in rows] == [(96, False), (24, False)], rows
    for op in (1, 3):
        lat = Lattice(LatticeConfig(domain=dim, opt_policy=op))
        assert lat.info()["launches_per_pass"] == 3
        auto = lat.info()["wave_depth"]
        lat.close()
        lat = Lattice(LatticeConfig(domain=dim, opt_policy=op, wave_depth=auto))
        assert lat.info()["wave_depth"] == auto == 60
        lat.close()
    """)
