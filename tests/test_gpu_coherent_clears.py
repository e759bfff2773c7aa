"""Host-coherent RDRAM where a submission's own clears decide which pages are
copied in: full-width, partial, scissored, interlaced and odd clear rectangles
over random memory the caller rewrites between frames, drawn over with depth
and blending.  Every byte of RDRAM and hidden RDRAM must be the oracle's."""
import numpy as np
import pytest

import harness
import rdp_streams as rs

pytestmark = pytest.mark.gpu

W, H = 100, 70
# Clear rectangle (x0, y0, x1, y1 in quarter pixels) and scissor (xlo, ylo, xhi, yhi, field, odd).
FULL = (0, 0, (W - 1) << 2, (H - 1) << 2)
OPEN = (0, 0, W << 2, H << 2, False, False)
CASES = {
    "full": (FULL, OPEN),
    "fraction": ((3, 2, (W - 1) * 4 + 3, (H - 1) * 4 - 1), OPEN),
    "one_column_short": ((0, 0, (W - 2) << 2, (H - 1) << 2), OPEN),
    "from_second_column": ((4, 0, (W - 1) << 2, (H - 1) << 2), OPEN),
    "middle_rows": ((0, 21, (W - 1) << 2, 161), OPEN),
    "scissored_rows": (FULL, (0, 35, W << 2, 190, False, False)),
    "scissored_columns": (FULL, (8, 0, (W << 2) - 12, H << 2, False, False)),
    "interlaced": (FULL, (0, 0, W << 2, H << 2, True, True)),
}


def frame(rng, rect, scissor, size, depth_rect):
    cl = rs.CommandList()
    cl.set_other_modes(rs.OtherModes(cycle_type=3))
    cl.set_scissor(*scissor[:4], field=scissor[4], keep_odd=scissor[5])
    cl.set_color_image(rs.DEPTH_ADDR, W, rs.SIZ_16)
    cl.set_fill_color(0xFFFCFFFC)
    if depth_rect:
        cl.fill_rectangle(*rect)
    cl.sync_pipe()
    cl.set_color_image(rs.COLOR_ADDR, W, size)
    cl.set_mask_image(rs.DEPTH_ADDR)
    cl.set_fill_color(int(rng.integers(0, 1 << 32, dtype=np.int64)))
    cl.fill_rectangle(*rect)
    cl.sync_pipe()
    cl.set_scissor(0, 0, W << 2, H << 2)
    cl.set_other_modes(rs.OtherModes(cycle_type=0, depth_test=True, depth_write=True, force_blend=True,
                                     blend=((0, 0, 1, 0), (0, 0, 1, 0))))
    cl.set_combine(*rs.SHADE_COMBINE)
    n = 24
    xy = np.stack([rng.integers(0, W * 4, size=(n, 3)), rng.integers(0, H * 4, size=(n, 3))], axis=-1)
    cl.extend_array(rs.triangle_commands(xy, rgba=rng.integers(0, 256, size=(n, 3, 4)).astype(np.float64),
                                         z=rng.integers(0, 0x40000, size=(n, 3)).astype(np.float64)))
    cl.sync_full()
    return cl.words()


@pytest.mark.parametrize("size", [rs.SIZ_16, rs.SIZ_32])
@pytest.mark.parametrize("case", CASES)
def test_clears_over_caller_memory(oracle_mod, case, size):
    import rdp_mi
    rng = np.random.default_rng(len(case) * 7 + size)
    rect, scissor = CASES[case]
    host = rng.integers(0, 1 << 32, size=rs.RDRAM_SIZE // 4, dtype=np.uint64).astype(np.uint32)
    o = oracle_mod.Oracle(rs.RDRAM_SIZE)
    o.rdram[:] = host
    p = rdp_mi.CommandProcessor(rs.RDRAM_SIZE, host_rdram=host)
    hidden = rng.integers(0, 4, size=rs.RDRAM_SIZE // 2).astype(np.uint8)
    p.write_hidden_rdram(hidden)
    o.hidden[:] = hidden
    for k in range(3):
        print(f"[case] clear {case} size {size} frame {k}", flush=True)
        words = frame(rng, rect, scissor, size, depth_rect=k != 1)
        p.enqueue_commands(words)
        o.process(words)
        p.idle()
        o.flush()
        total, lines = harness.compare((host, p.read_hidden_rdram(), p.read_tmem()), (o.rdram.copy(), o.hidden.copy(), o.tmem.copy()))
        assert total == 0, lines
        # The caller rewrites both images and what surrounds them.
        for base in (rs.COLOR_ADDR, rs.DEPTH_ADDR):
            span = slice(base // 4 - 64, base // 4 + W * H + 64)
            new = rng.integers(0, 1 << 32, size=span.stop - span.start, dtype=np.uint64).astype(np.uint32)
            host[span] = new
            o.rdram[span] = new
    p.close()
    o.close()
