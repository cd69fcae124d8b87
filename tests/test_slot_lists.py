"""The voxel lists of the speculative kernel: no list is written while another wavefront
still reads it, whatever the schedule.

Every schedule of the evaluating wavefronts is walked on the CPU.  What an evaluator
does, in which order, and how many lists there are comes from the kernel's source: after
its evaluation (which writes its list) a wavefront waits for its turn, and from there on
the statements of the turn are its steps.
"""
import re
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "chromo_amd" / "csrc"


def _body(text, start):
    """The braces' text that follows `start`."""
    i = text.index("{", text.index(start))
    depth, j = 0, i
    while True:
        depth += {"{": 1, "}": -1}.get(text[j], 0)
        j += 1
        if depth == 0:
            return text[i:j]


def _reads_list(name):
    """Whether evaluator function `name` reads the list (EvLds::uv)."""
    return "S.uv[" in _body((CSRC / "chromo_eval.hpp").read_text(), f"void {name}(")


def _turn_steps():
    """From the turn on: 'read' (a function that reads the list), 'pass' (the turn)."""
    src = re.sub(r"//[^\n]*", "", (CSRC / "chromo_spec.hpp").read_text())
    text = src[src.index("if (turn && S.kind == SLOT_SMALL && (res.resample"):]
    text = text[text.index("if (turn) {"):text.index("ctl_set(&ctl->idle[wv], 1)")]
    steps = []
    for m in re.finditer(r"(ev_\w+)(?:<\w+>)?\(|ctl_set\(&ctl->(resolved),", text):
        if m.group(2):
            steps.append("pass")
        elif _reads_list(m.group(1)):
            steps.append("read")
    assert steps.count("pass") == 1 and "read" in steps
    return steps


def _lists(ev):
    src = (CSRC / "chromo_spec.hpp").read_text()
    expr = re.search(r"constexpr int LISTS = ([^;]+);", src).group(1)
    return eval(expr, {}, {"EV": ev})


def _overlaps(ev, lists, steps, slots):
    """Whether some schedule writes a list that another wavefront has still to read.

    A wavefront: (slot, place), place -1 before its evaluation, 0 waiting for its turn
    with its list written, 1.. after that many steps of the turn.  While it waits it may
    still look the ev - 1 slots before its own up in their lists."""
    seen, todo = set(), [(0, 0, ((None, 0),) * ev)]
    while todo:
        state = todo.pop()
        if state in seen:
            continue
        seen.add(state)
        nxt, resolved, waves = state
        for w, (slot, place) in enumerate(waves):
            def go(n, r, v):
                todo.append((n, r, waves[:w] + (v,) + waves[w + 1:]))
            if slot is None:
                if nxt < slots:
                    go(nxt + 1, resolved, (nxt, -1))
            elif place == -1:
                for x, (other, at) in enumerate(waves):
                    if x == w or other is None:
                        continue
                    mine = at >= 0 and "read" in steps[at:] and other % lists == slot % lists
                    waits = at <= 0 and any(q >= 0 and q != slot and q % lists == slot % lists
                                            for q in range(other - ev + 1, other))
                    if mine or waits:
                        return True
                go(nxt, resolved, (slot, 0))
            elif place > 0 or resolved == slot:
                r = slot + 1 if steps[place] == "pass" else resolved
                go(nxt, r, (None, 0) if place + 1 == len(steps) else (slot, place + 1))
    return False


@pytest.mark.parametrize("ev", [2, 3])
def test_no_list_is_written_while_it_is_read(ev):
    lists = _lists(ev)
    assert not _overlaps(ev, lists, _turn_steps(), 2 * lists + ev)
    # the walk finds the overlaps it looks for: one list fewer, or a read after the turn
    assert _overlaps(ev, lists - 1, ["read", "pass"], 2 * lists + ev)
    assert _overlaps(ev, lists, ["read", "pass", "read"], 2 * lists + ev)
