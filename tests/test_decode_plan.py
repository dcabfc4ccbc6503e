"""The decode reader's choice for a batch (slots by one launch, splits by two, or
either by its lengths), on the CPU: the plan itself, printed by
lib/pbe_decode_plan."""
import random
import subprocess

import pytest

import pbe_handoff as P

SLOTS, SPLITS, EITHER = 0, 1, 2
TOOL = P.LIB_PATH.parent / "pbe_decode_plan"


def plan(*cases):
    """(batch, kv_heads, query heads of one, head_dim, fp8, max_blocks, splits, compute units, atomics, address) -> rows."""
    lines = "".join(" ".join(str(int(x)) for x in (c[0], c[1], c[1] * c[2], *c[3:])) + "\n" for c in cases)
    got = subprocess.run([str(TOOL)], input=lines, capture_output=True, text=True, check=True, timeout=60).stdout.split("\n")
    return [dict(zip(("mode", "slots", "hshift", "one_round", "used", "given"), map(int, g.split()))) for g in got[:len(cases)]]


def auto(batch, kv, group, dim, fp8, blocks, cus=256, atomics=1, address=4096):
    """The case with its automatic split count (of 256 compute units)."""
    return (batch, kv, group, dim, fp8, blocks, P.decode_splits(batch, kv, blocks, P.PBE_KV_FP8_E4M3 if fp8 else P.PBE_KV_BF16), cus, atomics, address)


@pytest.mark.parametrize("case,mode", [
    # few sequences: the second launch combines them
    ((1, 2, 7, 64, 0, 315), SPLITS), ((1, 2, 6, 128, 0, 1024), SPLITS), ((2, 2, 6, 128, 1, 315), SPLITS), ((3, 1, 8, 128, 0, 315), SPLITS),
    ((2, 2, 6, 128, 0, 160), SLOTS), ((2, 2, 6, 128, 0, 161), SPLITS), ((3, 2, 6, 128, 0, 315), SLOTS), ((4, 8, 4, 128, 1, 125), SPLITS),
    ((1, 2, 6, 128, 0, 24), SLOTS), ((1, 2, 7, 64, 0, 25), SPLITS),  # at most 24 blocks: one slot, one launch
    # small batches of 64-dim heads
    ((16, 2, 7, 64, 0, 63), SPLITS), ((4, 2, 7, 64, 0, 275), SPLITS), ((4, 2, 7, 64, 0, 276), SLOTS),
    # 64-byte rows that nothing joins
    ((32, 5, 4, 64, 1, 250), SPLITS), ((32, 5, 4, 64, 0, 250), EITHER), ((16, 16, 2, 64, 1, 250), SPLITS), ((32, 4, 4, 64, 1, 250), SLOTS),
    # equal lengths would leave compute units idle: the lengths decide
    ((130, 2, 6, 128, 0, 145), EITHER), ((170, 2, 6, 128, 0, 125), EITHER), ((171, 2, 6, 128, 0, 125), SLOTS), ((128, 2, 6, 128, 0, 125), SLOTS),
    ((87, 2, 6, 128, 0, 125), EITHER), ((66, 2, 6, 128, 0, 125), SLOTS), ((65, 4, 7, 128, 0, 125), EITHER), ((65, 4, 7, 128, 1, 125), EITHER),
    ((96, 4, 7, 128, 1, 125), SLOTS), ((89, 4, 7, 128, 1, 125), EITHER), ((130, 2, 7, 64, 0, 125), EITHER), ((130, 2, 7, 64, 1, 125), SLOTS),
    ((48, 8, 4, 128, 1, 250), EITHER), ((130, 2, 6, 128, 0, 30), SLOTS),  # short ones have nothing to win
    # large and mixed batches: one launch
    ((64, 2, 6, 128, 1, 315), SLOTS), ((64, 2, 6, 128, 0, 440), SLOTS), ((8, 4, 7, 128, 1, 1024), SLOTS), ((256, 2, 6, 128, 0, 440), SLOTS),
])
def test_how_a_batch_is_read(case, mode):
    assert plan(auto(*case))[0]["mode"] == mode


def test_no_atomics_no_tickets():
    """A workspace in host memory: splits, or (a single one) whole sequences."""
    cases = [auto(b, 2, 6, 128, f, n, atomics=0) for b in (1, 64, 130, 300) for f in (0, 1) for n in (10, 315)]
    for c, got in zip(cases, plan(*cases)):
        assert got["mode"] == (SPLITS if c[6] > 1 else SLOTS), c
        assert got["mode"] == SPLITS or got["slots"] == c[0]


@pytest.mark.parametrize("cus", [32, 64, 128, 256, 304])
def test_the_width_follows_the_gpu(cus):
    for fp8 in (0, 1):
        for kv in (1, 2, 4):
            for got in plan((24, kv, 6, 128, fp8, 400, 64, cus, 1, 4096)):
                assert got["one_round"] == max(1, cus // (kv >> got["hshift"]))
                assert got["slots"] <= 2 * max(24, got["one_round"])


def test_the_plan_stays_in_its_workspace():
    """Whatever the shape, split count and address, slots and splits end inside
    the bytes asked for, and there is a slot for every sequence."""
    r = random.Random(5)
    cases = []
    for _ in range(4000):
        batch = int(2 ** r.uniform(0, 13))
        cases.append((batch, r.choice([1, 2, 3, 4, 5, 6, 8, 16, 32]), r.randint(1, 8), r.choice([64, 128]), r.randint(0, 1), int(2 ** r.uniform(0, 13)),
                      r.choice([1, 2, 3, 7, 16, 64, 1024]), r.choice([32, 256]), r.randint(0, 1), 4096 + 4 * r.randint(0, 8)))
    for c, got in zip(cases, plan(*cases)):
        assert got["used"] <= got["given"], (c, got)
        assert got["slots"] >= c[0] and got["hshift"] in (0, 1) and (not got["hshift"] or c[1] % 2 == 0), (c, got)
        assert got["mode"] == SLOTS or c[6] > 1, (c, got)
        if got["mode"] == EITHER:
            assert c[0] * c[1] * c[2] <= 3072 and got["slots"] >= c[0], (c, got)
        if got["mode"] == SPLITS and c[8]:  # its launches have fewer than 2^32 threads
            assert c[0] * c[1] * c[6] * 64 < 1 << 32 and c[0] * c[1] * c[2] * 256 < 1 << 32, (c, got)
