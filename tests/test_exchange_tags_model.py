"""What earlier launches may have left in the slots of a GroupNorm unit, on the CPU model of the exchange between its slices
(test_exchange_protocol_model.py; csrc/groupnorm.hip: gn_exchange_enter).

Launches that follow one another leave words of their own tags, in any mix of splits.  Launches that overlapped on one scratch,
which the header forbids, leave words of any of their tags in any slot, a mean beside an M2 of another one: never above the
number of launches so far, which the unit's count stands for once they are over.  The next launch in order must take
none of these words, whatever its split, and its slices must agree.
"""
import random

import pytest

from test_exchange_protocol_model import MAX_SPLIT, Launch, Unit


def left_by_overlapping_launches(rng, launches):
    unit = Unit()
    unit.count = launches * MAX_SPLIT
    for slots in (unit.slot_mean, unit.slot_m2):
        for l in range(MAX_SPLIT):
            tag = rng.choice([launches, launches, launches - 1, rng.randrange(launches + 1)])
            slots[l] = (tag, "left behind")
    return unit


@pytest.mark.parametrize("split", [2, 4, 64])
@pytest.mark.parametrize("seed", range(20))
def test_launches_in_order_are_right_whatever_the_slots_hold(seed, split):
    rng = random.Random(seed)
    unit = left_by_overlapping_launches(rng, rng.choice([1, 2, 7, 1000]))
    before = unit.count
    for launch in range(1, 5):
        spin_limit = rng.choice([1, 2, 50, 10 ** 9])
        starve = rng.randrange(split) if rng.random() < 0.5 and spin_limit < 10 ** 9 else None
        Launch(unit, rng.choice([split, split, 2, 8]), launch, rng, spin_limit).run(starve)  # asserts that no stale word is accepted
        assert unit.count == before + launch * MAX_SPLIT


def test_patient_slices_never_give_up():
    rng = random.Random(11)
    unit = left_by_overlapping_launches(rng, 5)
    for launch, split in enumerate([8, 2, 64, 4, 4, 2, 16, 8], 1):
        Launch(unit, split, launch, rng, 10 ** 9).run()
    assert unit.fallbacks == 0
