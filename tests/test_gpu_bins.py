"""Binning at the edges of its blocks: primitive counts around one group (64) and
one block of eight (512), framebuffers around 64 tile columns and at the widest,
and rows of one tile.  A bit missing or out of order shows in the framebuffer;
whole numbers, exact."""
import numpy as np
import pytest

import harness
import rdp_streams as rs

pytestmark = pytest.mark.gpu


SIZES = [(8, 8, 63), (504, 16, 64), (505, 9, 65), (512, 24, 511), (513, 17, 512), (520, 8, 513), (1016, 40, 577),
         (1023, 7, 130)]


@pytest.mark.parametrize("width,height,prims", SIZES)
def test_bins_match_oracle(width, height, prims):
    s = rs.config0_stream(seed=width * 1000 + prims, num_triangles=prims, width=width, height=height)
    print(f"[case] {prims} triangles on {width}x{height}", flush=True)
    total, lines = harness.compare(harness.run_gpu(s), harness.run_oracle(s))
    assert total == 0, lines


def test_bins_of_a_wide_batch_match_oracle():
    """24 processors and more in a round: setup, spans and bins in blocks of one
    wave, beside the raster."""
    import rdp_mi
    streams = [rs.config0_stream(seed=width * 1000 + prims + 1 + 7 * k, num_triangles=prims, width=width, height=height)
               for k, (width, height, prims) in enumerate(2 * SIZES + [(64, 64, 1), (320, 240, 4160)] + 6 * [(40, 40, 70)])]
    print(f"[case] {len(streams)} processors in one batch", flush=True)
    procs = [rdp_mi.CommandProcessor(rs.RDRAM_SIZE) for _ in streams]
    for p, s in zip(procs, streams):
        p.hold_submissions()
        p.write_rdram(np.zeros(rs.RDRAM_SIZE // 4, np.uint32))
        p.write_hidden_rdram(np.full(rs.RDRAM_SIZE // 2, s.hidden_init, np.uint8))
        p.enqueue_commands(s.all_words())
    rdp_mi.batch_flush(procs)
    for p in procs:
        p.idle()
    outs = [(p.read_rdram(), p.read_hidden_rdram(), p.read_tmem()) for p in procs]
    for p in procs:
        p.close()
    for s, out in zip(streams, outs):
        total, lines = harness.compare(out, harness.run_oracle(s))
        assert total == 0, (s.name, lines)
