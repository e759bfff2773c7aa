"""Small rounds that share their setup, TMEM and bin launches (groups of rounds),
where a group or a submission begins and ends: many passes in one flush, passes
whose TMEM comes from an earlier pass of the group, uploads that read what an
earlier pass of the group renders, passes whose scratch fills a group, and the
same with upscaling and super-sampled readback.  Whole numbers: exact."""
import numpy as np
import pytest

import harness
import rdp_streams as rs
import test_gpu_rounds as tr

pytestmark = pytest.mark.gpu


def check(streams, batched, flags=0):
    """The streams' frames held and handed over at once, by the plain path or one
    batched flush."""
    import rdp_mi
    procs = [rdp_mi.CommandProcessor(rs.RDRAM_SIZE, flags=flags) for _ in streams]
    for p, s in zip(procs, streams):
        p.hold_submissions()
        p.write_rdram(s.rdram_init if s.rdram_init is not None else np.zeros(rs.RDRAM_SIZE // 4, np.uint32))
        p.write_hidden_rdram(np.full(rs.RDRAM_SIZE // 2, s.hidden_init, np.uint8))
        p.enqueue_commands(s.all_words())
    if batched:
        rdp_mi.batch_flush(procs)
    for p in procs:
        p.idle()
    for p, s in zip(procs, streams):
        got = (p.read_rdram(), p.read_hidden_rdram(), p.read_tmem())
        total, lines = harness.compare(got, harness.run_oracle(s))
        assert total == 0, f"{s.name}: {lines}"
    for p in procs:
        p.close()


def chained(seed: int, passes: int) -> rs.Stream:
    """Passes that alternate between two images; every third one uploads (half
    of those from the image rendered before), the others draw with the TMEM an
    earlier pass left."""
    frames = []
    for k in range(passes):
        s = tr.texture_stream(seed + k, from_pass_a=k % 6 == 0)
        words = s.frames[0].words
        if k % 3:
            # Without the uploads: drop SetTextureImage (0x3d) and LoadTile (0x34).
            keep = [w for w in np.split(words, np.cumsum([_len(w) for w in _commands(words)])[:-1])
                    if (int(w[0]) >> 24) & 63 not in (0x3D, 0x34)]
            words = np.concatenate(keep)
        frames.append(rs.Frame(words))
    first = tr.texture_stream(seed, True)
    return rs.Stream(name=f"chain{seed}:{passes}", seed=seed, frames=frames, rdram_init=first.rdram_init, hidden_init=3)


def _len(cmd):
    return cmd[1] - cmd[0]


def _commands(words):
    import rdp_mi
    out, i = [], 0
    while i < words.size:
        n = int(rdp_mi.COMMAND_LENGTHS[(int(words[i]) >> 24) & 63])
        out.append((i, i + n))
        i += n
    return out


@pytest.mark.parametrize("passes", [1, 2, 5, 33, 70])
@pytest.mark.parametrize("batched", [False, True])
def test_chained_passes_match_oracle(passes, batched):
    print(f"[case] {passes} chained frames, batched {batched}", flush=True)
    check([chained(900 + passes, passes)] if not batched else [chained(1000 + i, passes) for i in range(3)], batched)


def test_passes_larger_than_a_group_match_oracle():
    """Each pass takes tens of MB of scratch, so groups split between them."""
    frames = [rs.config0_stream(seed=7000 + k, num_triangles=1400, width=320, height=480).frames[0] for k in range(4)]
    print("[case] four passes of 1400 full-screen triangles", flush=True)
    check([rs.Stream(name="large", seed=0, frames=frames)], False)


@pytest.mark.parametrize("ssaa", [False, True])
def test_upscaled_groups_match_oracle(ssaa):
    """Native passes, their upscaled copies and (ssaa) resolves in one group; the
    second frame draws with the first one's TMEM."""
    import rdp_mi
    import test_gpu_upscale as tu
    s = rs.config2_stream(seed=4242, frames=3, prims_per_frame=40, width=256, height=40)
    print(f"[case] upscaled group ssaa {ssaa}", flush=True)
    ref = tu.oracle_state(s, 2, ssaa=False if ssaa else None)
    p = rdp_mi.CommandProcessor(rs.RDRAM_SIZE, flags=rdp_mi.FLAG_UPSCALING[2] |
                                (rdp_mi.FLAG_SUPER_SAMPLED_READ_BACK if ssaa else 0))
    p.hold_submissions()
    p.write_rdram(s.rdram_init)
    p.write_hidden_rdram(np.full(rs.RDRAM_SIZE // 2, s.hidden_init, np.uint8))
    p.enqueue_commands(s.all_words())
    p.idle()
    got = (p.read_rdram(), p.read_hidden_rdram(), p.read_tmem(), p.read_upscaled_rdram(), p.read_upscaled_hidden_rdram())
    p.close()
    for name, a, b in zip(("rdram", "hidden", "tmem", "planes", "hidden planes"), got, ref):
        assert np.array_equal(np.ascontiguousarray(a).view(np.uint8).ravel(), np.ascontiguousarray(b).view(np.uint8).ravel()), name
