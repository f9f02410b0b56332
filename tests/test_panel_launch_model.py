"""Panels whose workgroups wait for each other, launched from several contexts at
once: a model of how workgroups find room on the card.

A launch's workgroups become resident one by one, in launch order, while the card has
room; a panel of more than one workgroup holds its room until all of its groups are
resident.  Cooperative launches go through one queue, one after another; regular ones
of different streams are placed side by side."""
import random
import re
from pathlib import Path

ROOM = 512  # resident workgroups of the column-exchange kernel


def _drains(launches, rng):
    """launches: (groups, cooperative) of different streams, in any interleaving."""
    coop = [g for g, c in launches if c]
    live = [[g, 0] for g, c in launches if not c]
    current = None
    while live or coop or current:
        if current is None and coop:
            current = [coop.pop(0), 0]
            live.append(current)
        # launches whose groups are all resident finish and give their room back
        done = [x for x in live if x[1] == x[0]]
        if done:
            x = rng.choice(done)
            live.remove(x)
            if x is current:
                current = None
            continue
        if sum(x[1] for x in live) >= ROOM:
            return False  # every resident group waits for one that has no room
        rng.choices(live, [x[0] - x[1] for x in live])[0][1] += 1
    return True


def test_waiting_launches_beside_cooperative_ones_can_stall():
    rng = random.Random(0)
    assert not all(_drains([(512, True), (32, False)], rng) for _ in range(500))


def test_cooperative_panels_and_single_workgroups_drain_in_any_order():
    rng = random.Random(1)
    for _ in range(2000):
        launches = [(rng.choice([1, 2, 32, 480, 512]), None) for _ in range(rng.randint(1, 6))]
        assert _drains([(g, g > 1) for g, _ in launches], rng), launches


def test_only_single_workgroup_panels_are_launched_regularly():
    src = (Path(__file__).resolve().parent.parent / "evd4sc2025_amd" / "csrc" / "panel_qr.hip").read_text()
    guards = re.findall(r"if \(([^\n]*)\)\n\s*EVD_HIP\(ctx, hipLaunchKernel\(\(const void \*\)panel_qr_kernel", src)
    assert guards == ["G == 1"]
    assert "panel_qr_kernel<<<" not in src
