"""CPU model of the bulge chase's message protocol (chase.hip, chase_kernel):
sweeps run concurrently and hand each other the window of every step through
slots that are doubled by the sweep's parity and hold EMPTY until a message
element arrives.  Stores complete late and in random order, and each wave sees
its own rows of a window by itself; the only ordering the model grants is the
kernel's: a wave that has its part of a window has completed its stores of the
steps before, and in a sweep's last step it completes its empties before it
sends.  Every interleaving must give the oracle's sequential result, no element
may land in a slot that is not empty or be left behind in one that is loaded
again, and without the start word, or either ordering of empties, the model
must fail.  With units, the messages inside a run of sweeps go through the box
of the run's XCD, those between runs through the common one.  A second model
hands out the sweeps (next_sweep)."""
import random

import numpy as np
import pytest

from oracle import evd_oracle as O

EMPTY = object()


def _refl(x):
    nrm = np.sqrt(x @ x)
    if nrm > 0:
        u = x / nrm
        u[0] += 1.0 if x[0] >= 0 else -1.0
        u /= np.sqrt(abs(u[0]))
        return u, (-nrm if x[0] >= 0 else nrm)
    return np.zeros_like(x), x[0]


class Stale(Exception):
    pass


def _lens(n, b, p):
    ln = min(b, n - p)
    return ln, max(0, min(b, n - p - ln))


def _window(n, b, p):
    """The elements of a step's window that are loaded: ('S' | 'N', i, k)."""
    ln, ln2 = _lens(n, b, p)
    w = [("S", i, k) for i in range(ln) for k in range(ln)]
    w += [("N", i, k) for i in range(ln2) for k in range(ln) if not (i == b - 1 and k < b - 1)]
    return w


def chase(Bd, b, seed, start_word=True, ordered=True, last_wait=True, window=7, unit=None, members=1, waves=2):
    n = Bd.shape[0]
    rng = random.Random(seed)
    nsw = n - 2
    mem = {}  # (box and parity, slot | 'X', element) -> value; absent = EMPTY

    def half(s):
        """Where sweep s sends: its parity, in the common box or that of its unit's XCD."""
        return s % 2 if not unit or (s + 1) % unit == 0 else (s // unit % members, s % 2)

    for j in range(-(-n // b)):
        p = 1 + j * b
        if p < n:
            ln, _ = _lens(n, b, p)
            for what, i, k in _window(n, b, p):
                r, c = (p + max(i, k), p + min(i, k)) if what == "S" else (p + ln + i, p + k)
                mem[1, j, what, i, k] = Bd[r, c]
    for i in range(min(b, n - 1)):
        mem[1, "X", i] = Bd[1 + i, 0]
    D, E, U = np.zeros(n), np.zeros(n - 1), np.zeros((n + b, n))
    D[0] = Bd[0, 0]
    started = set()

    def flush(x, wave=None, upto=None, kinds=("empty", "send")):
        """Complete stores of sweep x: those of a wave up to step `upto`, or a random one."""
        q = x["stores"]
        if wave is None:
            pick = [rng.randrange(len(q))] if q else []
        else:
            pick = [i for i, e in enumerate(q) if e[1] <= upto and e[4] == wave and e[0] in kinds]
        for i in reversed(pick):
            kind, _, key, v, _ = q.pop(i)
            if kind == "empty":
                mem.pop(key, None)
            else:
                if key in mem:
                    raise Stale(f"{key} written twice")
                mem[key] = v

    def program(s):
        """The sweep as a generator: yields None to be rescheduled."""
        x = st[s]
        rd, wr = half(s - 1), half(s)
        p = s + 1
        ln, ln2 = _lens(n, b, p)
        wv = lambda row: row * waves // b  # the wave of a row
        store = lambda kind, j, row, key, v=None: x["stores"].append((kind, j, key, v, wv(row)))
        while start_word and s > 0 and s - 1 not in started:
            yield
        keys = [(rd, "X", i) for i in range(ln)]
        got = {}
        while len(got) < len(keys):
            for k in keys:
                if k not in got and k in mem:
                    got[k] = mem[k]
            yield
        for k in keys:
            store("empty", -1, 0, k)
        u, beta = _refl(np.array([got[k] for k in keys]))
        U[p:p + ln, s] = u
        E[s] = beta
        j, B1 = 0, None
        while True:
            send = lambda row, key, v: store("send", j, row, key, v)
            if j > 0:  # before the window, and before the empties are known to be complete
                B1 = B1 - np.outer(u, u @ B1)
                for k in range(1, b):
                    send(k, (wr, j - 1, "S", b - 1, k - 1), B1[0, k])
                    send(k, (wr, j - 1, "S", k - 1, b - 1), B1[0, k])
                    for i in range(1, ln):
                        send(k, (wr, j - 1, "N", i - 1, k - 1), B1[i, k])
            keys = [(rd, j, *e) for e in _window(n, b, p)]
            got, seen = {}, set()
            while len(seen) < waves:  # elements are seen one by one, in any order
                for k in keys:
                    if k not in got and k in mem and rng.random() < 0.7:
                        got[k] = mem[k]
                for w in set(range(waves)) - seen:
                    if all(k in got for k in keys if wv(k[3]) == w):
                        seen.add(w)
                        if ordered:  # loads of this window were issued after the last step's stores
                            flush(x, w, j - 1)
                yield
            S = np.array([[got[rd, j, "S", i, k] for k in range(ln)] for i in range(ln)])
            N = np.array([[got.get((rd, j, "N", i, k), 0.0) for k in range(ln)] for i in range(ln2)]).reshape(ln2, ln)
            for k in keys:
                store("empty", j, k[3], k)
            yield
            if ln2 == 0 and last_wait:
                for w in range(waves):
                    flush(x, w, j, ("empty",))
            y = S @ u
            w = y - 0.5 * (u @ y) * u
            S = S - np.outer(u, w) - np.outer(w, u)
            N = N - np.outer(N @ u, u)
            if j == 0:
                started.add(s)
                D[s + 1] = S[0, 0]
                for i in range(1, ln):
                    send(i, (wr, "X", i - 1), S[i, 0])
                if s == nsw - 1:
                    E[n - 2], D[n - 1] = S[1, 0], S[1, 1]
            else:
                send(0, (wr, j - 1, "S", b - 1, b - 1), S[0, 0])
                for i in range(1, ln):
                    send(i, (wr, j - 1, "N", i - 1, b - 1), S[i, 0])
            for i in range(1, ln):
                for k in range(1, ln):
                    send(i, (wr, j, "S", i - 1, k - 1), S[i, k])
            if ln2 == 0:
                break
            un, betan = _refl(N[:, 0].copy()) if ln2 > 1 else (np.zeros(1), N[0, 0])
            send(0, (wr, "X", b - 1) if j == 0 else (wr, j - 1, "N", b - 1, b - 1), betan)
            yield
            p += ln
            U[p:p + ln2, s] = un
            u, B1 = un, N
            ln, ln2 = _lens(n, b, p)
            j += 1
        while x["stores"]:
            yield

    st, ticket, idle = {}, 0, 0
    while ticket < nsw or st:
        cand = list(st)
        if ticket < nsw and len(st) < window:
            cand.append(-1)
        s = rng.choice(cand)
        if s == -1:
            st[ticket] = {"stores": []}
            st[ticket]["run"] = program(ticket)
            ticket += 1
            continue
        if rng.random() < 0.5:
            flush(st[s])
        else:
            try:
                next(st[s]["run"])
            except StopIteration:
                del st[s]
        idle += 1
        if idle > 2_000_000:
            raise Stale("no progress")
    left = [k for k in mem if k[0] == half(nsw - 2)]  # what sweep nsw - 2 sent: all of it was loaded
    if left:
        raise Stale(f"{len(left)} elements left behind")
    return D, E, U


def _band(n, b):
    A = O.gen_symmetric(n, 3, 0).astype(np.float64)
    return np.tril(np.triu(A, -b), b)


@pytest.mark.parametrize("n,b", [(3, 4), (4, 3), (9, 4), (22, 4), (23, 4), (24, 4), (25, 4), (26, 5), (17, 2), (19, 7)])
def test_messages_match_sequential_chase(n, b):
    B = _band(n, b)
    ref = O.sb2st(B, b)
    for seed in range(40 if n < 23 else 12):
        res = chase(B, b, seed)
        assert max(np.abs(a - r).max() for a, r in zip(res, ref)) < 1e-11


@pytest.mark.parametrize("unit,members", [(2, 1), (2, 3), (3, 2), (5, 2), (100, 1)])
@pytest.mark.parametrize("n,b", [(9, 4), (24, 4), (26, 5), (17, 2)])
def test_messages_through_unit_boxes(n, b, unit, members):
    B = _band(n, b)
    ref = O.sb2st(B, b)
    for seed in range(8):
        res = chase(B, b, 70 * unit + 10 * members + seed, unit=unit, members=members)
        assert max(np.abs(a - r).max() for a, r in zip(res, ref)) < 1e-11


@pytest.mark.parametrize("unsafe,n,b,seeds", [({"start_word": False}, 25, 4, 30), ({"ordered": False, "waves": 1}, 17, 2, 200),
                                              ({"last_wait": False}, 9, 4, 300)])
def test_model_catches_unsafe_protocols(unsafe, n, b, seeds):
    B = _band(n, b)
    ref = O.sb2st(B, b)
    bad = 0
    for seed in range(seeds):
        try:
            res = chase(B, b, seed, **unsafe)
            bad += max(np.abs(a - r).max() for a, r in zip(res, ref)) > 1e-6
        except Stale:
            bad += 1
    assert bad


def hand_out(nsweeps, count, length, members, groups, seed):
    """next_sweep for groups[x] workgroups on XCD x, every atomic access an
    interleaving point, on a chain in which a sweep ends only after its
    predecessor.  Returns {(problem, sweep): XCD}."""
    rng = random.Random(seed)
    total = -(-nsweeps // length) * count
    DONE = 0x7FFFFFFF
    word = {"unit": 0, "members": 0}
    state = {x: (0, 0, 0) for x in range(len(groups))}  # member, unit + 1, handed out
    owner, ended = {}, set()

    def take(x):
        while True:
            m, unit, idx = state[x]
            state[x] = (m, unit, idx + 1)
            yield
            if unit == DONE:
                return None
            if unit and idx < length:
                s = (unit - 1) // count * length + idx
                if s < nsweeps:
                    return (unit - 1) % count, s
                continue
            if idx == (length if unit else 0):
                if not unit:
                    m, word["members"] = word["members"], word["members"] + 1
                    yield
                u = None
                if m < members:
                    t, word["unit"] = word["unit"], word["unit"] + 1
                    yield
                    u = t if t < total else None
                state[x] = (m, DONE, 1) if u is None else (m, u + 1, 1)
                yield
                return None if u is None else (u % count, u // count * length)
            while state[x][1] == unit:
                yield

    def workgroup(x):
        while True:
            job = yield from take(x)
            if job is None:
                return
            assert job not in owner
            owner[job] = x
            q, s = job
            while s > 0 and (q, s - 1) not in ended:
                yield
            ended.add(job)

    live = [workgroup(x) for x in range(len(groups)) for _ in range(groups[x])]
    for _ in range(2_000_000):
        if not live:
            return owner
        g = rng.choice(live)
        try:
            next(g)
        except StopIteration:
            live.remove(g)
    raise Stale("no progress")


@pytest.mark.parametrize("nsweeps,count,length,members,groups", [
    (1, 1, 2, 1, [1, 1]), (9, 1, 9, 1, [2, 3, 1]), (23, 1, 4, 3, [2, 1, 4, 1]), (10, 5, 3, 2, [3, 3, 3]),
    (7, 3, 1, 1, [4]), (12, 2, 5, 2, [1, 0, 0]), (2, 6, 2, 8, [1] * 8)])
def test_hand_out_reaches_every_sweep(nsweeps, count, length, members, groups):
    for seed in range(5):
        owner = hand_out(nsweeps, count, length, members, groups, seed)
        assert set(owner) == {(q, s) for q in range(count) for s in range(nsweeps)}
        assert len(set(owner.values())) <= members
        for (q, s), x in owner.items():  # a unit stays on one XCD
            assert s % length == 0 or owner[q, s - 1] == x
