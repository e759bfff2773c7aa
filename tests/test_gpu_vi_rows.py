"""The one-kernel scanout where a wave's row of filter texels is largest, smallest
or ragged: every horizontal step at its limits (one texel for 64 pixels, four per
pixel), vertical steps with and without a fraction (one or two rows per line),
crops that leave a partial last wave, the fetch bug's rows, and the same image
through a waiting and an asynchronous scanout.  Whole numbers: exact."""
import numpy as np
import pytest

import rdp_streams as rs
import test_gpu_vi as gv
import vi_cases

pytestmark = pytest.mark.gpu

STEPS = [(1, 1024), (512, 1023), (1023, 1025), (1024, 2048), (1025, 2049), (4095, 4095), (2048, 1), (640, 1000)]


@pytest.mark.parametrize("xs,ys", STEPS)
@pytest.mark.parametrize("fmt", [2, 3])
def test_rows_match_oracle(oracle_mod, xs, ys, fmt):
    import rdp_mi
    rng = np.random.default_rng(xs * 4096 + ys)
    rdram, hidden, _ = vi_cases.random_case(xs + fmt, frames=1)
    p = rdp_mi.CommandProcessor(rs.RDRAM_SIZE)
    p.write_rdram(rdram)
    p.write_hidden_rdram(hidden)
    o = oracle_mod.Oracle(rs.RDRAM_SIZE)
    o.rdram[:] = rdram
    o.hidden[:] = hidden
    buf = rdp_mi.ScanoutBuffer()
    for k in range(4):
        control = fmt | ((1 << 16) | (1 << 4) if k & 1 else 0) | (1 << 6 if k == 3 else 0) | ((k % 3) << 8)
        regs = {rs.VI_CONTROL: control, rs.VI_ORIGIN: 0x100000 + 4 * k, rs.VI_WIDTH: 61 + 193 * k, rs.VI_V_SYNC: 525,
                rs.VI_V_START: vi_cases.start_reg(34 + 2 * k, 34 + 478), rs.VI_H_START: vi_cases.start_reg(108 - k, 108 + 641),
                rs.VI_X_SCALE: vi_cases.scale_reg(xs, int(rng.integers(0, 4096)) if k else 0),
                rs.VI_Y_SCALE: vi_cases.scale_reg(ys, int(rng.integers(0, 4096)) if k else 0), rs.VI_V_CURRENT_LINE: k & 1}
        opts = dict(upscale_deinterlacing=0 if k == 3 else 1, blend_previous_frame=k & 1)
        if k == 2:
            opts.update(crop_enable=1, crop_left=1, crop_right=64, crop_top=3, crop_bottom=2)
        print(f"[case] step {xs} {ys} format {fmt} frame {k}", flush=True)
        vi_cases.apply_frame(p, regs, None)
        vi_cases.apply_frame(o, regs, None)
        if k == 1:
            p.scanout_async(buf, gv.gpu_opts(opts))
            got = buf.wait()
        else:
            got = p.scanout_sync(gv.gpu_opts(opts))
        exp = o.scanout(gv.oracle_opts(opts))
        assert got.shape == exp.shape and np.array_equal(got, exp)
    buf.close()
    o.close()
    p.close()
