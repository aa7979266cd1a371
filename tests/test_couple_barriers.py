"""The barriers of the one-launch coupling call (k_couple), as a model of the
counters its workgroups share: the sequence of arrivals and waits is read from
the kernel's source, every interleaving of three workgroups is walked, each
with and without the wait that only workgroups with long entry lists make.  A
wait may end only when every workgroup has arrived where it waits, and no
interleaving may get stuck."""
import itertools
import os
import re

import pytest

from fsilbm3d_amd.build import CSRC

ROUNDS = 3


def _kernel_ops():
    """[("arrive", word) | ("wait", word, count, optional)] of k_couple, its round loop unrolled."""
    src = open(os.path.join(CSRC, "fsil_ibm_kernels.h")).read()
    body = src[src.index("void k_couple(CoupleArgs a)"):]
    body = body[:body.index("\ntimeout:")]
    word = {"arrived": re.search(r"\*const arrived = &ctl\[(\w+)\]", body).group(1)}
    pat = re.compile(r"couple_(barrier|arrive|wait)\((?:&ctl\[(\w+)\]|(\w+))(?:, ([^,]+), &late)?\)")
    once, loop = [], []
    for what, ctl, name, nth in pat.findall(body):
        w = ctl or word[name]
        ops = once
        if nth.endswith("+ r"):
            ops, nth = loop, nth.split()[0]
        if what != "wait":
            ops.append(("arrive", w))
        if what != "arrive":
            ops.append(("wait", w, int(nth), what == "wait"))
    assert len(once) >= 2 and len(loop) == 2
    for r in range(ROUNDS):
        once += [loop[0], ("wait", loop[1][1], loop[1][2] + r, False)]
    return once


def _walk(ops, groups=3):
    """The first fault of any interleaving, or None."""
    words = sorted({o[1] for o in ops})
    arrive_of = {}
    for i, o in enumerate(ops):
        if o[0] == "wait":
            arrive_of[i] = max(k for k in range(i) if ops[k][0] == "arrive" and ops[k][1] == o[1])
    for skips in itertools.product((False, True), repeat=groups):
        start = ((0,) * groups, (0,) * len(words))
        seen, todo = {start}, [start]
        while todo:
            pcs, counts = todo.pop()
            moved = False
            for g, pc in enumerate(pcs):
                if pc == len(ops):
                    continue
                o, new = ops[pc], list(counts)
                if o[0] == "arrive":
                    new[words.index(o[1])] += 1
                elif not (o[3] and skips[g]):
                    if counts[words.index(o[1])] < groups * o[2]:
                        continue
                    if any(p <= arrive_of[pc] for p in pcs):
                        return f"a wait on {o[1]} for {o[2]} ends with workgroups at {pcs}"
                moved = True
                nxt = (pcs[:g] + (pc + 1,) + pcs[g + 1:], tuple(new))
                if nxt not in seen:
                    seen.add(nxt)
                    todo.append(nxt)
            if not moved and any(p < len(ops) for p in pcs):
                return f"stuck at {pcs}"
    return None


def test_every_wait_ends_with_all_workgroups_arrived():
    ops = _kernel_ops()
    assert sum(o[0] == "wait" and o[3] for o in ops) == 1  # the lists' wait
    assert _walk(ops) is None


@pytest.mark.parametrize("word,fault", [("a", "ends"), ("b", None)])
def test_a_shared_count_does_not_bear_a_skipped_wait(word, fault):
    """The model itself: a wait that some skip, on the running count of the others or on its own word."""
    shared = word == "a"
    ops = [("arrive", "a"), ("wait", "a", 1, False), ("arrive", word), ("wait", word, 2 if shared else 1, True),
           ("arrive", "a"), ("wait", "a", 3 if shared else 2, False)]
    found = _walk(ops)
    assert (found is None) if fault is None else (fault in found)
