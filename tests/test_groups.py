"""Groups of rounds (parallel-rdp_amd/csrc/rdp_groups.hpp) on the CPU: the index of
a pass in its group fits the 15 bits a work item has for it however many rounds
hold an upscaled pass, an upscaled pass's round leaves the scratch of the round
before it alone, rounds of one group never share scratch, and a group has few
enough rounds to compare each with all before it."""
import os
import random
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PASS_BITS, SCRATCH, MOST_ROUNDS = 15, 64 << 20, 64


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("groups") / "probe")
    subprocess.run(["g++", "-std=c++17", "-O2", "-o", out, os.path.join(ROOT, "tests", "groups_probe.cpp")], check=True)
    return out


def walk(probe, rounds, own=False):
    text = "".join(f"{p} {s} {int(u)}\n" for p, s, u in rounds)
    out = subprocess.run([probe, str(int(own))], input=text, capture_output=True, text=True, check=True).stdout
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


def rounds_of(kind):
    rng = random.Random(kind)
    if kind == "upscaled":  # two processors one pass out of phase: every round has an upscaled pass
        return [(7, 4096, True)] * 20000
    if kind == "native":
        return [(rng.randint(1, 7), rng.randint(1, 30 << 20), False) for _ in range(3000)]
    if kind == "large":
        return [(1, 40 << 20, k % 2 == 1) for k in range(200)]
    if kind == "small":
        return [(2, 12288, False)] * 2000
    return [(rng.randint(1, 7), rng.randint(1, 4 << 20), rng.random() < 0.5 and k > 0) for k in range(6000)]


@pytest.mark.parametrize("kind", ["upscaled", "native", "large", "small", "mixed"])
def test_groups(probe, kind):
    rounds = rounds_of(kind)
    out = walk(probe, rounds)
    assert len(out) == len(rounds) and out[0][0] == 1
    end = 0  # of the scratch of the round before
    length = 0  # rounds of the group
    for k, ((passes, scratch, upscaled), (begins, base, total)) in enumerate(zip(rounds, out)):
        assert total <= 1 << PASS_BITS, k
        length = 1 if begins else length + 1
        assert length <= MOST_ROUNDS, k
        if upscaled or not begins:
            assert base == end, k
        else:
            assert base == 0, k
        if not begins and not upscaled:
            assert base + scratch <= SCRATCH, k
        end = base + scratch


def test_rounds_of_their_own(probe):
    rounds = [(30000, 1 << 20, k % 3 == 0) for k in range(50)]
    for k, (begins, base, total) in enumerate(walk(probe, rounds, own=True)):
        assert (begins, base, total) == (1, k << 20, 30000)
