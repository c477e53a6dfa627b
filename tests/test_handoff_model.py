"""CPU model of LDS hand-offs under random interleavings: the parts that every
kernel's model shares, and the small-batch egress kernel.

Each wave of a fused workgroup is modelled as a generator that yields after
every shared-memory step and spins (yields 'blocked') at every bounded wait
of the kernel.  A scheduler runs the generators in a random order; a run in
which every live wave stays blocked is a deadlock.  The models also check that
the MAC / verify wave reads every payload row in order with the right
contents.  Sizes are read from the kernel sources, so the models follow the
constants the kernels are built with.

The row pipelines' models (tasks of four rows by sixteen pages) are in
test_handoff_tasks.py, with the tests of the bounded waits.
"""
import random
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "vlx-tee_amd" / "csrc"


def _const(fname, name):
    m = re.search(rf"constexpr int {name} = (\d+);", (CSRC / fname).read_text())
    assert m, (fname, name)
    return int(m.group(1))


# code rows per unit of each section kind (code_rows_per_unit, ztcp_layout.h):
# the reference's int8 / int4 / raw, and the extension kinds e4m3 (16-element
# groups), int4 per 32 and int8 asymmetric per 64 (16 groups per unit, so 16
# code rows and one parameter row).  Every kind but raw has one parameter row
# per unit.
NBLK = {"i8": 8, "i4": 4, "raw": 16, "e4": 8, "i4g32": 8, "a8": 16}
CONFIGS = {  # sections (kind, units) of the layouts the kernels meet
    "k8v4": [("i8", 16), ("i8", 16), ("i4", 32)],
    "int4": [("i8", 16), ("i4", 16), ("i4", 32)],
    "fp8only": [("i8", 32), ("i8", 32)],
    "mla": [("i8", 8), ("i4", 64)],
    "raw_rope": [("raw", 4), ("i4", 8), ("i4", 16)],
    "tiny": [("i8", 1), ("i4", 1)],
    "one_unit_sections": [("i8", 1), ("i8", 3), ("i4", 2)],
    # extension kinds (egress kind families 1 / 2, ingress family 1), the
    # 16-token x 8-head x 128 pages and 64-token MLA pages of the workloads
    "k8v4asym_e4rope": [("e4", 16), ("a8", 8), ("i4g32", 16)],
    "e4m3": [("e4", 32), ("e4", 32)],
    "mla_int4g32_e4rope": [("e4", 8), ("i4g32", 32)],
    "asym8_small": [("a8", 1), ("a8", 3), ("i4g32", 2)],
    "mixed_raw_ext": [("raw", 2), ("a8", 2), ("e4", 3)],
}


def payload_rows(secs, padding=0):
    """Payload rows in order: ('code', section, unit, j) / ('scale', g) /
    ('pad', i); code rows also get their code index."""
    rows, g = [], 0
    for si, (kind, nu) in enumerate(secs):
        for u in range(nu):
            for j in range(NBLK[kind]):
                rows.append(("code", si, u, j))
        if kind != "raw":
            rows += [("scale", g + u) for u in range(nu)]
            g += nu
    rows += [("pad", i) for i in range(padding)]
    return rows


class Sched:
    def __init__(self, seed):
        self.rng = random.Random(seed)

    def run(self, actors, max_steps=5_000_000):
        live = list(range(len(actors)))
        blocked = 0
        for _ in range(max_steps):
            if not live:
                return True
            i = self.rng.choice(live)
            try:
                s = next(actors[i])
            except StopIteration:
                live.remove(i)
                blocked = 0
                continue
            if s == "blocked":
                blocked += 1
                # with bounded waits every wait ends by itself
                if BOUND is None and blocked > 50 * len(live) + 1000:
                    return False
            else:
                blocked = 0
        raise RuntimeError("step limit")


class Bounded:
    """The kernels' bounded waits (wait_ge, vlx-tee_amd/csrc/ztcp_rows.h): a
    wait gives up after `limit` polls, records the expiry in the workgroup's
    LDS word and returns; with `short_circuit` (the kernels' rule) a wait that
    finds the word set returns at its next poll.  After an expiry rows are
    handed over out of turn, so the model's content checks no longer apply
    (the kernel fails such a workgroup closed)."""

    def __init__(self, limit, short_circuit=True):
        self.limit, self.short_circuit = limit, short_circuit
        self.expired = False
        self.expiries = 0   # waits that ran out their own bound
        self.polls = 0      # polls of all waits together

    def wait(self, cond):
        spins = 0
        while not cond():
            if self.short_circuit and self.expired:
                return
            if spins >= self.limit:
                self.expired = True
                self.expiries += 1
                return
            spins += 1
            self.polls += 1
            yield "blocked"


BOUND = None  # a Bounded while a test runs the model with bounded waits


def wait(cond):
    if BOUND is not None:
        yield from BOUND.wait(cond)
        return
    while not cond():
        yield "blocked"


def check(cond, *msg):
    """The model's content checks; void once a bounded wait has expired."""
    if BOUND is not None and BOUND.expired:
        return
    assert cond, msg


MAC_GROUP_OFF = False  # planted mistake: the MAC wave tests only the first row of each group


def mac_groups(prow, ring, ring_flag, st, KRING):
    """The MAC / verify wave (mac_rows, vlx-tee_amd/csrc/ztcp_rows.h): rows
    in groups of kMacGroup.  One test of the group's flags: a group whose rows
    are all in the ring is read at once and `used` is published once for it;
    otherwise the group is taken a row at a time, each row once its flag is
    set, and `used` is published after each.  The last total % kMacGroup
    rows are always taken a row at a time."""
    G = _const("ztcp_rows.h", "kMacGroup")
    assert KRING % G == 0, "ring lengths are multiples of the MAC group"
    for g0 in range(0, len(prow), G):
        rows = range(g0, min(g0 + G, len(prow)))
        tested = rows[:1] if MAC_GROUP_OFF else rows
        if len(rows) == G and all(ring_flag[m % KRING] >= m + 1 for m in tested):
            for m in rows:
                check(ring[m % KRING] == prow[m], (m, ring[m % KRING], prow[m]))
                yield "ok"
            st["used"] = rows[-1] + 1
            yield "ok"
            continue
        for m in rows:
            yield from wait(lambda: ring_flag[m % KRING] >= m + 1)
            check(ring[m % KRING] == prow[m], (m, ring[m % KRING], prow[m]))
            yield "ok"
            st["used"] = m + 1
            yield "ok"


# ---------------------------------------------------------------------------
# The small-batch egress kernel (egress_small_kernel): three producer waves
# make task t = 192 k + 64 w + lane of pass k (code row t // ppw of page
# t % ppw) and publish pass counts; after every wave's last pass they make
# the scale rows and count themselves done.  The MAC wave reads payload rows
# in order, a code row once every wave has published the pass that holds its
# last page's task (need = (c ppw + ppw - 1) // 192 + 1 passes; rows below
# need * 192 // ppw are then complete), a scale row once all three waves are
# done.  The model runs the waves lane by lane in random order and checks
# that every row the MAC wave reads has been written for every page.
# ---------------------------------------------------------------------------
PASS_OFF_BY_ONE = False  # planted mistake: the MAC wave waits for one pass fewer than it needs


def small_egress_model(secs, ppw, seed):
    waves = _const("ztcp_egress.hip", "kSmallWaves") - 1
    tasks_per_pass = 64 * waves
    rows = payload_rows(secs)
    code_rows = [r for r in rows if r[0] == "code"]
    ncode, nq = len(code_rows), sum(1 for r in rows if r[0] == "scale")
    ntask = ncode * ppw
    npass = -(-ntask // tasks_per_pass)
    written = set()     # (page, payload row) written to the LDS copy
    passes = [0] * waves
    done = [0]

    def producer(w):
        for k in range(npass):
            lanes = list(range(64))
            random.Random(seed * 31 + w * 7 + k).shuffle(lanes)
            for lane in lanes:
                t = k * tasks_per_pass + w * 64 + lane
                if t < ntask:
                    c, i = divmod(t, ppw)
                    written.add((i, rows.index(code_rows[c])))
                    yield "step"
            passes[w] = k + 1
            yield "step"
        yield from wait(lambda: min(passes) >= npass)
        for t in range(w * 64, nq * ppw, tasks_per_pass):
            for lane_t in range(t, min(t + 64, nq * ppw)):
                g, i = divmod(lane_t, ppw)
                written.add((i, rows.index(("scale", g))))
                yield "step"
        done[0] += 1

    def mac():
        ready, scales, c = 0, False, 0
        for r, row in enumerate(rows):
            if row[0] == "code":
                if c >= ready:
                    need = (c * ppw + ppw - 1) // tasks_per_pass + 1 - (1 if PASS_OFF_BY_ONE else 0)
                    yield from wait(lambda: min(passes) >= need)
                    ready = min(ncode, need * tasks_per_pass // ppw)
                c += 1
            elif not scales:
                yield from wait(lambda: done[0] >= waves)
                scales = True
            for i in range(ppw):
                check((i, r) in written, "row read before it was written", r, i, row)
            yield "step"

    assert Sched(seed).run([mac()] + [producer(w) for w in range(waves)])


@pytest.mark.parametrize("cfg", ["k8v4", "int4", "raw_rope", "tiny", "one_unit_sections"])
@pytest.mark.parametrize("ppw", [1, 2, 3, 4])
def test_small_egress_passes(cfg, ppw):
    for seed in range(3):
        small_egress_model(CONFIGS[cfg], ppw, seed)


def test_small_egress_model_catches_a_missing_pass():
    global PASS_OFF_BY_ONE
    PASS_OFF_BY_ONE = True
    try:
        with pytest.raises(AssertionError, match="before it was written"):
            for seed in range(20):
                small_egress_model(CONFIGS["k8v4"], 3, seed)
    finally:
        PASS_OFF_BY_ONE = False
