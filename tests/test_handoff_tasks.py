"""The row pipelines' hand-offs with tasks of four rows and groups of 16 pages.

A CPU model of egress_fused_kernel and ingress_fused_kernel (workgroups of one
to four page groups): producers / decoders take tasks in order, one ahead; the
ring, its flags, the staging slots, their counts and flags are per page group;
the storer passes four rows at a time and stores a scale group behind the code
rows, encrypting it for some page groups of a full workgroup; the feeder puts
the scale rows; the MAC wave takes rows that every page group has filled.
Random interleavings must neither deadlock nor read a slot that holds another
row.  Sizes come from the kernel sources; planted mistakes show that the model
sees the faults it is for.
"""
import re

import pytest

import test_handoff_model as M
from test_handoff_model import CONFIGS, CSRC, NBLK, Bounded, Sched, _const, check, mac_groups, payload_rows, wait

ROWS = 4
STORER_SKIPS_ITS_SHARE = False  # planted mistake: the storer stores a scale group without encrypting its share
STORE_WHOLE_SECTION = False   # planted mistake: the storer stores scale groups only at a section's end
FREE_ON_FIRST_TASK = False    # planted mistake: a unit's staging slot is freed by its first task
ONE_GROUP_FLAG = False        # planted mistake: the MAC wave looks at page group 0's flags only
IGNORE_STORER = False         # planted mistake: a ring slot is reused once the MAC wave alone has passed it
LAZY_PUBLISH = False          # planted mistake: the storer publishes stored scale rows only when it is done
WHOLE_GROUPS_ONLY = False     # planted mistake: a section's last scale group is stored only if it is whole


class AllGroups:
    """Row slots of every page group, as the MAC wave sees them."""

    def __init__(self, per_group, value):
        self.g, self.value = per_group, value

    def __getitem__(self, slot):
        vals = [x[slot] for x in (self.g[:1] if ONE_GROUP_FLAG and self.value == "flag" else self.g)]
        return min(vals) if self.value == "flag" else (vals[0] if all(v == vals[0] for v in vals) else tuple(vals))


class Ring:
    def __init__(self, n_groups, length):
        self.n = length
        self.data = [[None] * length for _ in range(n_groups)]
        self.flag = [[0] * length for _ in range(n_groups)]

    def put(self, g, m, row):
        s = m % self.n
        check(self.flag[g][s] <= max(0, m - self.n + 1), "ring slot overwritten before use", m)
        self.data[g][s] = row

    def mac(self, prow, st):
        yield from mac_groups(prow, AllGroups(self.data, "data"), AllGroups(self.flag, "flag"), st, self.n)


def code_items(secs, prow):
    """Code items (four rows of a unit) in payload order: section, unit, first row in unit, payload row, g."""
    first = {}
    for m, r in enumerate(prow):
        if r[0] == "code" and r[3] % ROWS == 0:
            first[r[1:]] = m
    out, q = [], 0
    for si, (kind, nu) in enumerate(secs):
        for u in range(nu):
            for j in range(0, NBLK[kind], ROWS):
                out.append(dict(si=si, u=u, j=j, m=first[(si, u, j)], kind=kind, g=q + u, nu=nu))
        if kind != "raw":
            q += nu
    return out


def producer_scale_groups(ng, nblk):
    """The kernel's rule of the same name: page groups whose scale rows the producers encrypt."""
    m = re.search(r"return ng < 4 \? ng : 4 - min\(nblk / (\d+), 4\);", (CSRC / "ztcp_egress.hip").read_text())
    return ng if ng < 4 else 4 - min(nblk // int(m.group(1)), 4)


def egress(secs, n_prod, ng, seed):
    KR, KS, KG = (_const("ztcp_egress.hip", k) for k in ("kRing", "kStage", "kScaleGroup"))
    prow = payload_rows(secs)
    items = code_items(secs, prow)
    tasks = [(it, g) for it in items for g in range(ng)]
    ring, st = Ring(ng, KR), dict(task=0, used=0, stored=0)
    stage = [[None] * KS for _ in range(ng)]            # unit whose scales a slot holds
    count = [[0] * KS for _ in range(ng)]
    enc = [[0] * KS for _ in range(ng)]
    cipher = [set() for _ in range(ng)]                 # units whose staged scales are encrypted
    free = [0] * KS
    scale_stored = set()

    def passed():
        return st["used"] if IGNORE_STORER else min(st["used"], st["stored"])

    def producer():
        t = st["task"]; st["task"] += 1
        yield "ok"
        while t < len(tasks):
            tn = st["task"]; st["task"] += 1
            yield "ok"
            it, g = tasks[t]
            quant = it["kind"] != "raw"
            if quant:
                u = it["g"]
                yield from wait(lambda: free[u % KS] >= u - KS + 1)
                check(stage[g][u % KS] in (None, u) or stage[g][u % KS] <= u - KS, "staging slot in use")
                stage[g][u % KS] = u
                yield "ok"
            m = it["m"]
            yield from wait(lambda: passed() >= m + ROWS - KR)
            for i in range(ROWS):
                ring.put(g, m + i, prow[m + i])
            yield "ok"
            for i in range(ROWS):
                ring.flag[g][(m + i) % KR] = m + i + 1
            yield "ok"
            if quant and g < producer_scale_groups(ng, NBLK[it["kind"]]):
                u0 = it["u"] - it["u"] % KG
                n, g0 = min(KG, it["nu"] - u0), it["g"] - (it["u"] - u0)
                count[g][g0 % KS] += 1
                if count[g][g0 % KS] == n * (NBLK[it["kind"]] // ROWS):
                    count[g][g0 % KS] = 0
                    check(all(stage[g][(g0 + i) % KS] == g0 + i for i in range(n)), "encrypts another unit")
                    cipher[g].update(range(g0, g0 + n))
                    yield "ok"
                    enc[g][g0 % KS] = g0 + 1
                yield "ok"
            t = tn

    def storer():
        made, pub, q = [], 0, 0
        r = 0

        for kind, nu in secs:
            nblk, quant, us = NBLK[kind], kind != "raw", 0
            ngp = producer_scale_groups(ng, nblk)
            eg, cr = ngp, 0
            while True:
                tail = cr >= nu * nblk
                rows = range(r, r + ROWS)
                ready = lambda: all(ring.flag[g][m % KR] >= m + 1 for g in range(ng) for m in rows)  # noqa: E731,B023
                done = cr // nblk
                while quant and us < nu and (tail or done - us >= KG):
                    n, g0 = min(KG, nu - us), q + us
                    if WHOLE_GROUPS_ONLY and n < KG:
                        us = nu
                        break
                    due = tail or (done - us >= 2 * KG and not STORE_WHOLE_SECTION)
                    if eg < ng and not STORER_SKIPS_ITS_SHARE:
                        if not due and ready():
                            break
                        check(all(stage[eg][(g0 + i) % KS] == g0 + i for i in range(n)), "encrypts another unit")
                        cipher[eg].update(range(g0, g0 + n))
                        eg += 1
                        yield "ok"
                        continue
                    if not due:
                        break
                    yield from wait(lambda: all(enc[g][g0 % KS] >= g0 + 1 for g in range(ngp)))  # noqa: B023
                    for g in range(ng):
                        check(all(stage[g][(g0 + i) % KS] == g0 + i for i in range(n)), "stores another unit")
                        check(all(g0 + i in cipher[g] for i in range(n)), "stores scales in the clear")
                    yield "ok"
                    for i in range(n):
                        free[(g0 + i) % KS] = g0 + i + 1
                        made.append(g0 + i)
                    if len(made) - pub >= 2 * KG and not LAZY_PUBLISH:
                        scale_stored.update(made[pub:]); pub = len(made)
                    us, eg = us + KG, ngp
                    yield "ok"
                if tail:
                    break
                if pub < len(made) and not ready() and not LAZY_PUBLISH:
                    scale_stored.update(made[pub:]); pub = len(made)
                    yield "ok"
                yield from wait(ready)
                for m in rows:  # one row after the other
                    check(all(ring.data[g][m % KR] == prow[m] for g in range(ng)), "stores another row", m)
                    yield "ok"
                r += ROWS
                cr += ROWS
                st["stored"] = r
                yield "ok"
            if quant:
                r += nu
                st["stored"] = r
                q += nu
                yield "ok"
        scale_stored.update(made[pub:])
        yield "ok"

    def feeder():
        rows = [(m, x[1]) for m, x in enumerate(prow) if x[0] == "scale"]
        for i, (m, g) in enumerate(rows):
            if i == 0 or rows[i - 1][0] != m - 1:
                yield from wait(lambda: g in scale_stored)
            if i + 1 < len(rows) and rows[i + 1][0] == m + 1:
                gn = rows[i + 1][1]
                yield from wait(lambda: gn in scale_stored)
            yield from wait(lambda: passed() >= m - KR + 1)
            for p in range(ng):
                ring.put(p, m, prow[m])
            yield "ok"
            for p in range(ng):
                ring.flag[p][m % KR] = m + 1
            yield "ok"

    return Sched(seed).run([producer() for _ in range(n_prod)] + [storer(), feeder(), ring.mac(prow, st)])


def section_items(nu, qpu, L):
    """section_item (ztcp_ingress.hip) written out: code items >= 0, ~q for scale group q."""
    nsg, per = (nu + L - 1) // L, L * qpu
    out = [~q for q in range(min(2, nsg))]
    for q in range(nsg):
        code = list(range(q * per, min((q + 1) * per, nu * qpu)))
        if 1 <= q <= nsg - 2:
            code.insert(per // 2, ~(q + 1))
        out += code
    return out


def ingress(secs, n_dec, ng, seed, padding=0):
    KR, KS, L = (_const("ztcp_ingress.hip", k) for k in ("kRing", "kStage", "kLookahead"))
    prow = payload_rows(secs, padding)
    by_key = {(it["si"], it["u"], it["j"]): it for it in code_items(secs, prow)}
    items, q = [], 0
    for si, (kind, nu) in enumerate(secs):
        qpu = NBLK[kind] // ROWS
        for x in (section_items(nu, qpu, L) if kind != "raw" else range(nu * qpu)):
            if x < 0:
                items.append(("scale", q + ~x * L, min(L, nu - ~x * L)))
            else:
                items.append(("code", by_key[(si, x // qpu, (x % qpu) * ROWS)]))
        q += nu if kind != "raw" else 0
    tasks = [(it, g) for it in items for g in range(ng)]
    ring, st = Ring(ng, KR), dict(task=0, used=0)
    stage = [[None] * KS for _ in range(ng)]
    ready = [[0] * KS for _ in range(ng)]
    free = [[0] * KS for _ in range(ng)]
    count = [[0] * KS for _ in range(ng)]

    def decoder():
        t = st["task"]; st["task"] += 1
        yield "ok"
        while t < len(tasks):
            tn = st["task"]; st["task"] += 1
            yield "ok"
            it, g = tasks[t]
            if it[0] == "scale":
                units = range(it[1], it[1] + it[2])
                yield from wait(lambda: all(free[g][u % KS] >= u - KS + 1 for u in units))
                for u in units:
                    check(count[g][u % KS] == 0, "slot still read")
                    stage[g][u % KS] = u
                yield "ok"
                for u in units:
                    ready[g][u % KS] = u + 1
                yield "ok"
            else:
                c = it[1]
                m, u = c["m"], c["g"]
                yield from wait(lambda: st["used"] >= m + ROWS - KR)
                for i in range(ROWS):
                    ring.put(g, m + i, prow[m + i])
                yield "ok"
                for i in range(ROWS):
                    ring.flag[g][(m + i) % KR] = m + i + 1
                yield "ok"
                if c["kind"] != "raw":
                    yield from wait(lambda: ready[g][u % KS] >= u + 1)
                    check(stage[g][u % KS] == u, "scales of another unit", stage[g][u % KS], u)
                    yield "ok"
                    count[g][u % KS] += 1
                    if FREE_ON_FIRST_TASK or count[g][u % KS] == NBLK[c["kind"]] // ROWS:
                        count[g][u % KS] = 0
                        free[g][u % KS] = u + 1
                    yield "ok"
            t = tn

    def feeder():
        for m, x in enumerate(prow):
            if x[0] == "code":
                continue
            yield from wait(lambda: st["used"] >= m - KR + 1)
            for p in range(ng):
                ring.put(p, m, x)
            yield "ok"
            for p in range(ng):
                ring.flag[p][m % KR] = m + 1
            yield "ok"

    return Sched(seed).run([decoder() for _ in range(n_dec)] + [feeder(), ring.mac(prow, st)])


@pytest.mark.parametrize("cfg", sorted(CONFIGS))
@pytest.mark.parametrize("waves,ng", [(1, 1), (11, 1), (3, 2), (8, 3), (11, 4)])
def test_egress_tasks(cfg, waves, ng):
    for seed in range(2):
        assert egress(CONFIGS[cfg], waves, ng, seed), f"deadlock {cfg} waves={waves} groups={ng} seed={seed}"


@pytest.mark.parametrize("cfg", sorted(CONFIGS))
@pytest.mark.parametrize("waves,ng", [(1, 1), (12, 1), (3, 2), (12, 3), (12, 4)])
def test_ingress_tasks(cfg, waves, ng):
    for seed in range(2):
        assert ingress(CONFIGS[cfg], waves, ng, seed), f"deadlock {cfg} waves={waves} groups={ng} seed={seed}"
    assert ingress(CONFIGS[cfg], waves, ng, 7, padding=5)


def test_scale_groups_held_to_the_section_end_deadlock():
    global STORE_WHOLE_SECTION
    STORE_WHOLE_SECTION = True
    try:
        assert not all(egress(CONFIGS["k8v4"], 11, 2, s) for s in range(2))
    finally:
        STORE_WHOLE_SECTION = False


def test_model_catches_a_storer_that_skips_its_share():
    global STORER_SKIPS_ITS_SHARE
    STORER_SKIPS_ITS_SHARE = True
    try:
        with pytest.raises(AssertionError, match="in the clear"):
            egress(CONFIGS["k8v4"], 11, 4, 0)
    finally:
        STORER_SKIPS_ITS_SHARE = False


def test_model_catches_a_slot_freed_by_the_first_task():
    global FREE_ON_FIRST_TASK
    FREE_ON_FIRST_TASK = True
    try:
        with pytest.raises(AssertionError):
            for s in range(5):
                ingress(CONFIGS["k8v4"], 12, 1, s)
    finally:
        FREE_ON_FIRST_TASK = False


def test_model_catches_a_mac_wave_that_reads_one_groups_flags():
    global ONE_GROUP_FLAG
    ONE_GROUP_FLAG = True
    try:
        with pytest.raises(AssertionError):
            for s in range(5):
                egress(CONFIGS["int4"], 11, 4, s)
    finally:
        ONE_GROUP_FLAG = False


@pytest.mark.parametrize("qpu", [1, 2, 4])
def test_section_item_order(qpu):
    """The kernel's index arithmetic (section_item) against the order written out."""
    L = _const("ztcp_ingress.hip", "kLookahead")

    def section_item(i, nsg):
        pre, per = min(2, nsg), L * qpu
        if i < pre:
            return ~i
        i -= pre
        if i < per or nsg <= 2:
            return i
        i -= per
        span = per + 1
        b = i // span
        if b >= nsg - 2:
            return per * (nsg - 1) + i - (nsg - 2) * span
        off = i - b * span
        if off == per // 2:
            return ~(b + 2)
        return per * (b + 1) + off - (off > per // 2)

    for nu in range(1, 70):
        nsg = (nu + L - 1) // L
        assert [section_item(i, nsg) for i in range(nu * qpu + nsg)] == section_items(nu, qpu, L)




def _planted(name, run):
    """run() with the module's planted mistake `name` on."""
    globals()[name] = True
    try:
        return run()
    finally:
        globals()[name] = False


@pytest.mark.parametrize("name,cfgs", [("LAZY_PUBLISH", ["k8v4"]), ("WHOLE_GROUPS_ONLY", ["tiny", "one_unit_sections"])])
@pytest.mark.parametrize("ng", [1, 4])
def test_scale_rows_published_or_stored_too_late_deadlock(name, cfgs, ng):
    """The feeder, through it the MAC wave and through the ring the producers
    wait for scale rows that the storer has not published or never stores."""
    for cfg in cfgs:
        assert not all(_planted(name, lambda: egress(CONFIGS[cfg], 11, ng, s)) for s in range(3)), cfg  # noqa: B023


def test_model_catches_a_slot_reused_before_the_storer_read_it():
    with pytest.raises(AssertionError, match="stores another row|stores another unit"):
        for s in range(20):
            _planted("IGNORE_STORER", lambda: egress(CONFIGS["fp8only"], 11, 1, s))  # noqa: B023


def test_model_catches_a_group_read_on_its_first_flag_only():
    M.MAC_GROUP_OFF = True
    try:
        with pytest.raises(AssertionError):
            for s in range(20):
                egress(CONFIGS["k8v4"], 11, 1, s)
    finally:
        M.MAC_GROUP_OFF = False


def _with_stage(n, run):
    """run() with kStage = n instead of the kernels' (fewer slots than the schedule needs)."""
    global _const
    real = _const
    try:
        _const = lambda f, name: n if name == "kStage" else real(f, name)  # noqa: E731
        return run()
    finally:
        _const = real


@pytest.mark.parametrize("ng", [1, 4])
def test_a_staging_ring_smaller_than_the_schedule_deadlocks(ng):
    """Scale groups of four units cannot be staged in fewer than two groups'
    slots (ingress), nor kept by the storer a group behind (egress)."""
    assert not _with_stage(3, lambda: ingress(CONFIGS["k8v4"], 12, ng, 0))
    assert not _with_stage(4, lambda: egress(CONFIGS["k8v4"], 11, ng, 0))


def _run_bounded(limit, short_circuit, model):
    M.BOUND = Bounded(limit, short_circuit)
    try:
        done = model()
        return done, M.BOUND
    finally:
        M.BOUND = None


@pytest.mark.parametrize("cfg", ["k8v4", "k8v4asym_e4rope"])
@pytest.mark.parametrize("ng", [1, 4])
def test_bounded_waits_never_expire_in_a_healthy_workgroup(cfg, ng):
    for model in (lambda: egress(CONFIGS[cfg], 11, ng, 0), lambda: ingress(CONFIGS[cfg], 12, ng, 0)):
        done, b = _run_bounded(10**6, True, model)
        assert done and not b.expired


@pytest.mark.parametrize("ng", [1, 4])
def test_one_expired_wait_ends_every_later_wait_of_the_workgroup(ng):
    """A planted deadlock (the storer holding back its stored scale rows) with
    the kernels' bounded waits: the first wait to run out its bound marks the
    workgroup, every other wait returns at its next poll, and the workgroup
    finishes after at most one expiry per wave.  Without that rule each later
    wait spins out its own bound again, so the time to failure grows with the
    number of waits left (hundreds of bounds per wave in the kernel)."""
    n_prod, limit = 11, 400
    waves = n_prod + 3  # producers, storer, feeder, MAC wave
    for seed in range(2):
        model = lambda: _planted("LAZY_PUBLISH", lambda: egress(CONFIGS["k8v4"], n_prod, ng, seed))  # noqa: E731,B023
        done, b = _run_bounded(limit, True, model)
        assert done and b.expired
        assert 1 <= b.expiries <= waves
        assert b.polls <= waves * limit
        done, old = _run_bounded(limit, False, model)
        assert done and old.expiries > 2 * waves
        assert old.polls > 2 * waves * limit


def test_one_expired_wait_ends_a_broken_ingress_workgroup():
    for seed in range(2):
        done, b = _run_bounded(400, True, lambda: _with_stage(3, lambda: ingress(CONFIGS["k8v4"], 12, 1, seed)))  # noqa: B023
        assert done and b.expired and 1 <= b.expiries <= 14
