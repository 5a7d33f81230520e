"""The tags of the exchange between the slices of a GroupNorm unit (csrc/groupnorm.hip: gn_exchange), on the CPU model
of test_exchange_protocol_model.py, whose other steps (publishing, polling, giving up, storing) are the kernels' own.

A slice's tag is one more than that of its own first word, read at kernel start; there is no launch count and no
counter of finished slices.  When a slice has its statistics it puts the tag also into the first words l of the slots
that no slice of the launch uses, l % split == slice: between launches all slots of a unit carry one tag, so a launch
with any other split finds its slices agreed.  The stores are relaxed: they become visible in any order, and all of
them before the next launch on the stream starts.
"""
import random

import pytest

from test_exchange_protocol_model import MAX_SPLIT, Launch, Unit


class TaggedLaunch(Launch):
    def slice_program(self, s):
        u = self.unit
        u.epoch = u.slot_mean[s][0]  # the step that the model calls reading the epoch
        program = super().slice_program(s)
        ops = 0
        for _ in program:
            if ops == 0:
                tag = u.slot_mean[s][0] + 1
            u.done = 0  # no counter: never split - 1, so the model's last step is not taken
            yield
            ops += 1
        for l in range(s + self.split, MAX_SPLIT, self.split):
            self.store(s, "mean", l, (tag, 0.0))
            yield


@pytest.mark.parametrize("seed", range(40))
def test_slots_carry_one_tag_between_launches(seed):
    rng = random.Random(seed)
    unit = Unit()
    for launch in range(1, 13):
        split = rng.choice([2, 2, 4, 4, 8, 16, 64])
        spin_limit = rng.choice([1, 1, 2, 5, 50, 10 ** 9])
        starve = rng.randrange(split) if rng.random() < 0.5 and spin_limit < 10 ** 9 else None
        TaggedLaunch(unit, split, launch, rng, spin_limit).run(starve)  # asserts that no stale word is accepted
        assert [tag for tag, _ in unit.slot_mean] == [launch] * MAX_SPLIT


def test_patient_slices_never_give_up():
    rng = random.Random(11)
    unit = Unit()
    for launch, split in enumerate([8, 2, 64, 4, 4, 2, 16, 8], 1):
        TaggedLaunch(unit, split, launch, rng, 10 ** 9).run()
    assert unit.fallbacks == 0
