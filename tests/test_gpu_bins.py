"""Binning at the edges of its blocks: primitive counts around one group (64) and
one block of eight (512), framebuffers around 64 tile columns and at the widest,
and rows of one tile.  A bit missing or out of order shows in the framebuffer;
whole numbers, exact."""
import pytest

import harness
import rdp_streams as rs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,prims", [(8, 8, 63), (504, 16, 64), (505, 9, 65), (512, 24, 511), (513, 17, 512),
                                                (520, 8, 513), (1016, 40, 577), (1023, 7, 130)])
def test_bins_match_oracle(width, height, prims):
    s = rs.config0_stream(seed=width * 1000 + prims, num_triangles=prims, width=width, height=height)
    print(f"[case] {prims} triangles on {width}x{height}", flush=True)
    total, lines = harness.compare(harness.run_gpu(s), harness.run_oracle(s))
    assert total == 0, lines
