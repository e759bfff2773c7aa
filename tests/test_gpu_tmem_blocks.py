"""TMEM snapshots where the gather's blocks of uploads start and end: passes of
1 to a few hundred uploads, each sampled by the primitive after it, so a wrong
snapshot shows in the framebuffer.  Whole numbers: exact."""
import numpy as np
import pytest

import harness
import rdp_streams as rs

pytestmark = pytest.mark.gpu

BLOCK = 8


@pytest.mark.parametrize("uploads", [1, BLOCK - 1, BLOCK, BLOCK + 1, 2 * BLOCK + 1, 8 * BLOCK, 301])
def test_every_snapshot_matches_oracle(uploads):
    s = rs.config1_stream(frames=1, tris_per_frame=2 * uploads, width=96, height=72, tris_per_texture=2)
    print(f"[case] {uploads} tile uploads", flush=True)
    total, lines = harness.compare(harness.run_gpu(s), harness.run_oracle(s))
    assert total == 0, lines


@pytest.mark.parametrize("prims", [10, 64, 200])
def test_mip_and_tlut_uploads_match_oracle(prims):
    """Five uploads per texture that each write part of TMEM: blocks begin inside
    a texture, and most halfwords keep values carried from earlier blocks."""
    rng_tile = np.random.default_rng(prims)
    s = rs.config2_stream(frames=2, prims_per_frame=prims, width=int(rng_tile.integers(64, 200)), height=75,
                          num_textures=5)
    print(f"[case] {prims} two-cycle primitives", flush=True)
    total, lines = harness.compare(harness.run_gpu(s), harness.run_oracle(s))
    assert total == 0, lines
