"""Sums over lanes that are halved among them (``codegen/channelwise.py``): the emitted steps, run lane by lane on the host, leave
every sum complete in the one lane that ``emit_slot_of_lane`` names for it."""

import re

import numpy as np
import pytest

from cuequivariance_amd.codegen.channelwise import emit_lane_sums, emit_slot_of_lane

LANE = np.arange(64)


def _partner(v, bit):
    """cw_common.h: lane_partner inside a row of 16 lanes (8: rotation by 8, 4: mirror of 8 lanes, 2 and 1: quad permutations)."""
    return v[LANE ^ (7 if bit == 4 else bit)]


def _fold(bit, a, b=None):
    b = a if b is None else b
    is_set = (LANE & bit) != 0
    if bit >= 16:  # the swap: the set lanes of a change places with the clear lanes of b
        a, b = np.where(is_set, b[LANE ^ bit], a), np.where(is_set, b, a[LANE ^ bit])
        return np.where(is_set, b + a, a + b)
    return np.where(is_set, b, a) + _partner(np.where(is_set, a, b), bit)


@pytest.mark.parametrize("lanes", [64, 32, 16])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 9, 16])
def test_sums_end_in_the_lanes_that_store_them(n, lanes):
    rng = np.random.default_rng(n)
    values = {f"v{i}": rng.integers(0, 1000, 64).astype(np.int64) for i in range(n)}
    lines = []
    name = emit_lane_sums(lines.append, "", "float", list(values), lanes, "r")
    env = dict(values)
    for line in lines:
        target, bit, args = re.fullmatch(r"const float (\w+) = lane_fold<(\d+)>\((.*)\);", line).groups()
        env[target] = _fold(int(bit), *[env[a.strip()] for a in args.split(",") if a.strip() != "lane"])
    lines = []
    emit_slot_of_lane(lines.append, "", "slot", n, lanes)
    text = " ".join(lines)
    slots = []
    for lane in LANE:
        scope = {"lane": int(lane), "slot": 0}
        scope["mine"] = eval(re.search(r"bool mine = (.*?);", text).group(1), {}, scope)
        for bit, before in re.findall(r"slot = 2 \* slot \+ \(\(lane & (\d+)\) \? 1 : 0\); mine = mine && slot < (\d+);", text):
            scope["slot"] = 2 * scope["slot"] + (1 if lane & int(bit) else 0)
            scope["mine"] = scope["mine"] and scope["slot"] < int(before)
        slots.append(scope["slot"] if scope["mine"] else -1)
    for group in range(64 // lanes):
        own = slice(group * lanes, (group + 1) * lanes)
        assert sorted(s for s in slots[own] if s >= 0) == list(range(n))
        for lane in range(64)[own]:
            if slots[lane] >= 0:
                assert env[name][lane] == values[f"v{slots[lane]}"][own].sum()
