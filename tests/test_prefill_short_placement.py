"""Host-side model of the short prefill's task lists under any placement of its workgroups (CPU).

The single-launch prefill (up to 256 tokens) runs as tasks that 256 workgroups take from lists.
A workgroup holds its CU until its list is done, so launches that overlap on one device may each
hold CUs that the other waits for. This model restates the lists, the flags a task waits for and
the relays, places the workgroups of two launches on 8 XCDs of 32 CUs in any proportion (a
workgroup that ends makes room for a waiting one) and runs them until both launches are done
or nobody can go on:

* with a list per XCD from the start, two launches that hold an XCD each stop for good;
* with the kernel's rule (a list per XCD once two workgroups are on every XCD, otherwise a
  single list) both always finish.
"""

import random

import pytest

NXCD, CUS, NW, GROUPS = 8, 32, 8, 4
TASKS = {"qkv": 4, "att": 2, "o": 2, "gu": 6, "down": 4}  # an XCD's tasks of a step (and row block)
RELAYED = ("att", "o", "gu", "down")
BEFORE = {"o": "att", "gu": "o", "down": "gu"}  # the step whose tasks, on every XCD, a step waits for


class Launch:
    def __init__(self, nb, layers, rule):
        self.nb, self.layers, self.rule = nb, layers, rule
        self.mode = "xcd" if rule == "xcd lists" else None
        self.roles, self.tickets, self.any_ticket = [0] * NXCD, [0] * NXCD, 0
        self.flags = {}   # (xcd, step, row block, task) -> layers done
        self.words = {}   # relays: (step, wave, xcd) and (own, step, wave, xcd) -> layers done
        self.pending = [CUS] * NXCD  # workgroups not yet placed

    def done(self):
        return all(self.flags.get((g, "down", rb, j), 0) == self.layers
                   for g in range(NXCD) for rb in range(self.nb) for j in range(TASKS["down"]))

    def tasks(self, nq):
        """An XCD's list of one layer: (step, task, first row block)."""
        nat = [(s, i) for s in TASKS for i in range(TASKS[s] * (self.nb if s == "att" else nq))]
        return [(s, i % TASKS[s], i // TASKS[s]) for s, i in nat]

    def step_done(self, g, step, rb, want):
        """What a task on XCD g looks at for a step of all XCDs and row block rb."""
        if self.mode == "any":
            return all(self.flags.get((x, step, rb, j), 0) >= want for x in range(NXCD) for j in range(TASKS[step]))
        G = -(-self.nb // NW)
        return self.words.get(("own", step, rb // G, g), 0) >= want

    def relay(self, g):
        G = -(-self.nb // NW)
        waves = [self.relay_wave(g, wv, list(range(wv * G, min(self.nb, wv * G + G)))) for wv in range(NW)]
        while waves:
            waves = [w for w in waves if next(w, None) is not None]
            yield True

    def relay_wave(self, g, wv, blocks):
        for layer in range(1, self.layers + 1 if blocks else 1):
            for step in RELAYED:
                while not all(self.flags.get((g, step, rb, j), 0) >= layer for rb in blocks for j in range(TASKS[step])):
                    yield True
                self.words[(step, wv, g)] = layer
                while not all(self.words.get((step, wv, x), 0) >= layer for x in range(NXCD)):
                    yield True
                self.words[("own", step, wv, g)] = layer

    def worker(self, g, mode):
        nq = self.nb if mode == "any" else min(self.nb, GROUPS)
        per_layer = self.tasks(nq)
        while True:
            if mode == "any":
                t, self.any_ticket = self.any_ticket, self.any_ticket + 1
                g, t = t % NXCD, t // NXCD
            else:
                t, self.tickets[g] = self.tickets[g], self.tickets[g] + 1
            if t >= len(per_layer) * self.layers:
                return
            layer, (step, j, rb0) = 1 + t // len(per_layer), per_layer[t % len(per_layer)]
            for rb in [rb0] if mode == "any" or step == "att" else range(rb0, self.nb, nq):
                while True:
                    if self.mode not in (None, mode):
                        return  # (the launch runs from the other kind of list; nothing published yet)
                    if self.mode is None:
                        ok = False
                    elif step == "att":
                        ok = all(self.flags.get((g, "qkv", r, q), 0) >= layer
                                 for r in range(rb + 1) for q in (2, 3)) and self.flags.get((g, "qkv", rb, j), 0) >= layer
                    elif step == "qkv":
                        ok = layer == 1 or self.step_done(g, "down", rb, layer - 1)
                    else:
                        ok = self.step_done(g, BEFORE[step], rb, layer)
                    if ok:
                        break
                    yield True
                assert self.flags.get((g, step, rb, j), 0) == layer - 1
                self.flags[(g, step, rb, j)] = layer

    def workgroup(self, g):
        first = self.roles[g] == 0
        self.roles[g] += 1
        if not first:
            yield from self.worker(g, "xcd")
        while self.mode is None:
            if all(r >= 2 for r in self.roles):
                self.mode = "xcd"
            else:
                yield True
        if self.mode == "any":
            yield from self.worker(0, "any")
        elif first:
            yield from self.relay(g)


def run(placement, nb, layers, rule):
    """placement[x]: how many of XCD x's 32 CUs launch 0 gets at first, launch 1 the others.
    True if both launches finish."""
    ls = [Launch(nb, layers, rule) for _ in range(2)]
    resident = []

    def place(which, x):
        ls[which].pending[x] -= 1
        resident.append((which, x, ls[which].workgroup(x)))

    for x in range(NXCD):
        for _ in range(placement[x]):
            place(0, x)
        for _ in range(CUS - placement[x]):
            place(1, x)

    def state():
        return [(dict(l.flags), dict(l.words), l.mode, list(l.tickets), l.any_ticket) for l in ls], len(resident)

    while resident:
        before = state()
        for wg in list(resident):
            if next(wg[2], None) is None:
                resident.remove(wg)
                for which in range(2):
                    if ls[which].pending[wg[1]]:
                        place(which, wg[1])
                        break
        if state() == before:
            waiting = [l for l in ls if l.mode is None]
            if not waiting:
                return False  # nobody can go on
            waiting[0].mode = "any"  # its wait for workgroups on every XCD has run out
    return all(l.done() for l in ls)


SPLITS = {"an XCD each": [32, 0, 16, 16, 16, 16, 16, 16], "one workgroup each": [31, 1, 16, 16, 16, 16, 16, 16],
          "halves of the device": [32] * 4 + [0] * 4, "all but one": [32] * 7 + [31], "even": [16] * 8,
          "one after another": [32] * 8}


@pytest.mark.parametrize("nb", [1, 2, 9])
@pytest.mark.parametrize("split", sorted(SPLITS))
def test_overlapping_launches_finish(split, nb):
    assert run(SPLITS[split], nb, 2, "kernel")


def test_overlapping_launches_finish_however_they_are_placed():
    rng = random.Random(1)
    for _ in range(6):
        assert run([rng.choice([0, 1, 2, 16, 30, 31, 32]) for _ in range(NXCD)], rng.randint(1, 5), 1, "kernel")


@pytest.mark.parametrize("split,finish", [("an XCD each", False), ("one workgroup each", False), ("even", True),
                                          ("one after another", True)])
def test_lists_per_xcd_alone_would_not_do(split, finish):
    """The model sees what the rule is for: without it, launches that hold an XCD each never end."""
    assert run(SPLITS[split], 1, 2, "xcd lists") == finish
