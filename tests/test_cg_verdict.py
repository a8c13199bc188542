"""The end of a resident CG solve (mfem_amd/csrc/k_cg_resident.hip, "Verdict") as
a state machine: three workgroups, every interleaving, any wait running out at
any poll. On the GPU the interleavings that matter need a stall of the length of
a wait between two polls, so they are enumerated here.

A workgroup publishes its sums of the last iteration or gives up before (a wait
for q); then it polls for all sums. Each transition below is one atomic access of
the kernel with what follows from it."""
import pytest

WGS = 3
RUN, POLL, AGREE, WROTE, LEFT = "run", "poll", "agree", "wrote", "left"


def moves(s, rule):
    """The states that one access of one workgroup leads to. State: a position per
    workgroup, the published sums, the flag, the verdict, workgroup 0's report."""
    pos, sums, flag, verdict, report = s

    def to(i, p, sums=sums, flag=flag, verdict=verdict, report=report):
        return (pos[:i] + (p,) + pos[i + 1:], sums, flag, verdict, report)

    def give_up(i):
        if rule == "alone":  # every workgroup by itself
            return to(i, LEFT, flag=True, report="expired" if i == 0 else report)
        if verdict == "done":  # the compare-exchange lost: keep polling
            return None
        return to(i, LEFT, flag=True, verdict="expired",
                  report="expired" if i == 0 else report)

    for i, p in enumerate(pos):
        if p == RUN:
            yield to(i, POLL, sums=sums | {i})
        if p in (RUN, POLL):  # the wait runs out, or the flag is up
            n = give_up(i)
            if n:
                yield n
        if p == POLL and len(sums) == WGS:  # the sums that stop the solve
            if rule == "alone":
                yield to(i, WROTE, report="done" if i == 0 else report)
            elif i == 0 and verdict != "expired":
                yield to(i, WROTE, verdict="done", report="done")
            elif i == 0:
                yield to(i, LEFT, report="expired")
            else:
                yield to(i, AGREE)
        if p == AGREE and verdict:  # waits for the verdict, then writes x or leaves
            yield to(i, WROTE if verdict == "done" else LEFT)


def ends(rule):
    start = ((RUN,) * WGS, frozenset(), False, None, None)
    seen, todo = {start}, [start]
    while todo:
        s = todo.pop()
        nxt = list(moves(s, rule))
        if not nxt:
            yield s
        for n in nxt:
            if n not in seen:
                seen.add(n)
                todo.append(n)


def whole(s):
    pos, report = s[0], s[4]
    wrote = [p == WROTE for p in pos]
    return all(wrote) if report == "done" else report == "expired" and not any(wrote)


def test_every_solve_ends_with_one_answer():
    finals = list(ends("verdict"))
    assert {s[4] for s in finals} == {"done", "expired"}
    for s in finals:
        assert all(p in (WROTE, LEFT) for p in s[0]), s  # nobody waits for ever
        assert whole(s), s


def test_the_model_sees_a_part_written_solution():
    """Without the verdict workgroup 0 reports success over rows that a workgroup
    left unwritten."""
    assert any(s[4] == "done" and not whole(s) for s in ends("alone"))
