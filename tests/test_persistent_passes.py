"""The persistent kernels run compaction passes until one queues something.  A pass that queues nothing
(its pairs wait for the window to rise, or for held vertices) is followed by the next without a grid
barrier, so the next must not add to counters that a slow workgroup is still to read."""
import os
import random
import re

import pytest

from conftest import PKG_DIR

KERNELS = open(os.path.join(PKG_DIR, "csrc", "np_kernels.hip")).read()


def _pass_loop(kernel):
    """The kernel's loop over passes, without what only pushed frontiers run."""
    body = KERNELS[KERNELS.index("void %s(DevState st, SchedDev sp) {" % kernel):]
    loop = body[body.index("for (;;) {"):]
    return loop[:loop.index("__syncthreads()")].replace("PUSH ? it % 3 : ", "")


def _counters(by, it, p):
    return {"iteration": it, "pass": p}[by] % 3


def _run(by, queued, rng):
    """Three workgroups over passes that queue queued[p] vertices each, in a random order of their steps;
    True if every workgroup read the same totals.  clear, add, barrier, read, and after a pass that
    queued something the expansion's barrier."""
    n, cnt = 3, [0, 0, 0]
    seen = [[] for _ in range(n)]
    arrived = [0] * n

    def workgroup(b):
        it = 0
        for p, q in enumerate(queued):
            first = p == 0 or seen[b][-1] > 0
            if b == 0 and (by == "pass" or first):
                cnt[_counters(by, it, p + 1) if by == "pass" else (it + 2) % 3] = 0
            yield None
            cnt[_counters(by, it, p)] += q
            arrived[b] += 1
            yield arrived[b]
            seen[b].append(cnt[_counters(by, it, p)])
            if seen[b][-1] > 0:
                it += 1
                arrived[b] += 1
                yield arrived[b]

    wgs = {b: workgroup(b) for b in range(n)}
    waits = {b: None for b in wgs}
    while wgs:
        ready = [b for b in wgs if waits[b] is None or min(arrived[x] for x in wgs) >= waits[b]]
        if not ready:
            return False
        b = rng.choice(ready)
        try:
            waits[b] = next(wgs[b])
        except StopIteration:
            arrived[b] = 1 << 30
            del wgs[b]
    return all(s == [n * q for q in queued] for s in seen)


@pytest.mark.parametrize("by, safe", [("pass", True), ("iteration", False)])
def test_model_of_the_counters(by, safe):
    rng = random.Random(7)
    ok = all(_run(by, [1] + [rng.choice([0, 0, 1, 2]) for _ in range(7)], rng) for _ in range(3000))
    assert ok == safe


@pytest.mark.parametrize("kernel", ["k_persistent", "k_pk_persistent"])
def test_kernels_rotate_the_counters_by_pass(kernel):
    loop = _pass_loop(kernel)
    assert not re.search(r"\bit\b", re.sub(r"//.*", "", loop)), loop
    slot = {"k_persistent": ("slot", "next"), "k_pk_persistent": (r"\(pass % 3\)", r"\(\(pass \+ 1\) % 3\)")}[kernel]
    barrier = loop.index("grid_sync")
    for x in slot:
        assert re.search(r"st\.cnt \+ %s \* NCLS" % x, loop[:barrier]), (kernel, x)
    assert loop.index("st_coherent(st.cnt") < loop.index("compaction")
