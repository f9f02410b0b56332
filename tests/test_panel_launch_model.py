"""Panels whose workgroups wait for each other, launched from several contexts at
once: a model of how workgroups find room on the card.

A launch's workgroups become resident one by one while the card has room; a panel
of more than one workgroup holds its room until all of its groups are resident.
Cooperative launches go through one queue, one after another; regular ones of different
streams are placed side by side.  The groups of a gated launch wait for a bounded
time; then one closes the gate and works alone, and the others leave, those that
find room later too."""
import random
import re
from pathlib import Path

ROOM = 512  # resident workgroups of the column-exchange kernel


class _Launch:
    def __init__(self, groups, kind):
        self.groups, self.kind = groups, kind
        self.started = self.resident = 0
        self.closed = False

    def finished(self):
        return self.started == self.groups and (self.closed or self.resident == self.groups)


def _drains(launches, rng, worked=None):
    """launches: (groups, kind) of different streams with kind "cooperative", "regular"
    (waiting, without a gate) or "gated", in any interleaving of arrivals and time-outs."""
    coop = [_Launch(g, k) for g, k in launches if k == "cooperative"]
    live = [_Launch(g, k) for g, k in launches if k != "cooperative"]
    current = None
    while live or coop:
        if current is None and coop:
            current = coop.pop(0)
            live.append(current)
        done = [x for x in live if x.finished()]
        if done:
            x = rng.choice(done)
            if worked is not None:
                worked.append("alone" if x.closed else "together")
            live.remove(x)
            if x is current:
                current = None
            continue
        room = ROOM - sum(x.resident for x in live)
        arrive = [x for x in live if x.started < x.groups and (x.closed or room > 0)]
        expire = [x for x in live if x.kind == "gated" and not x.closed and 0 < x.resident < x.groups]
        if not arrive and not expire:
            return False  # every resident group waits for one that has no room
        if arrive and (not expire or rng.random() < 0.98):
            x = rng.choices(arrive, [y.groups - y.started for y in arrive])[0]
            x.started += 1
            x.resident += not x.closed  # behind a closed gate it leaves at once
        else:
            x = rng.choice(expire)
            x.closed, x.resident = True, 1
    return True


def test_waiting_launches_beside_cooperative_ones_can_stall():
    rng = random.Random(0)
    assert not all(_drains([(512, "cooperative"), (32, "regular")], rng) for _ in range(500))


def test_gated_and_cooperative_panels_drain_in_any_order():
    rng = random.Random(1)
    worked = []
    for _ in range(1500):
        launches = [(rng.choice([1, 2, 32, 480, 512]), rng.choice(["gated", "gated", "cooperative"]))
                    for _ in range(rng.randint(1, 6))]
        n = len(worked)
        assert _drains(launches, rng, worked), launches
        assert len(worked) - n == len(launches)  # every panel is factored, and once
    assert "alone" in worked and "together" in worked


def test_waiting_panels_are_launched_cooperatively_or_gated():
    src = (Path(__file__).resolve().parent.parent / "evd4sc2025_amd" / "csrc" / "panel_qr.hip").read_text()
    guards = re.findall(r"if \(([^\n]*)\)\n\s*EVD_HIP\(ctx, hipLaunchKernel\(\(const void \*\)panel_qr_kernel", src)
    assert guards == ["G == 1 || gate"]
    assert "panel_qr_kernel<<<" not in src
