"""The FP64 walk's hand-over of a team's next group: the team's first wave writes it to LDS, every wave
reads it, and the team's waits order the two. The order of the write, the waits and the read is taken
from the kernel's source, and every interleaving of a team's waves over some groups is followed: each
wave takes the groups in turn, and no wave waits for ever. (A wave held up between a read and the
wait before it is one of the interleavings; on a GPU it is rare.)"""
import os
import re

import pytest

SOURCE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lageunha_amd", "csrc", "tree.hip")


def kernel_order():
    """'W' write of the next group, 'S' team wait, 'R' read, as they stand at the end of a group."""
    with open(SOURCE) as f:
        text = f.read()
    body = text[text.index("walk_f64_kernel(walk64_args A)"):text.index("unsigned blocks_for")]
    body = re.sub(r"//[^\n]*", "", body)
    order = ""
    for m in re.finditer(r"s_next\[team\]\s*=[^=]|s_next\[team\]|(?<!auto )team_sync\(\)", body):
        order += "S" if m.group().startswith("team_sync") else ("W" if "=" in m.group() else "R")
    return order


def failures(order, waves, groups):
    """Follows all interleavings; returns what goes wrong in some of them ('wrong', 'stuck')."""
    # a wave: its place in the order, the group it is on, the value it has read; wave 0 alone writes
    start = (tuple((0, 0, 0) for _ in range(waves)), 0, (0,) * waves)  # waves, s_next, waits arrived at
    todo, seen, bad = [start], {start}, set()
    while todo:
        state = todo.pop()
        ws, nxt, arrived = state
        moved, done = False, 0
        for w, (at, g, val) in enumerate(ws):
            if g == groups:
                done += 1
                continue
            op = order[at]
            n2, a2, v2 = nxt, arrived, val
            if op == "W" and w == 0:
                n2 = g + 1
            elif op == "R":
                v2 = nxt
            elif op == "S":
                if val >= 0:  # arrive: once, then wait until every wave has arrived as often
                    a2 = arrived[:w] + (arrived[w] + 1,) + arrived[w + 1:]
                    nw = ws[:w] + ((at, g, -1 - val),) + ws[w + 1:]
                    s2 = (nw, nxt, a2)
                    moved = True
                    if s2 not in seen:
                        seen.add(s2)
                        todo.append(s2)
                    continue
                if min(arrived) < arrived[w]:
                    continue  # waits
                v2 = -1 - val
            at2, g2 = at + 1, g
            if at2 == len(order):
                at2, g2 = 0, v2
                if v2 != g + 1:
                    bad.add("wrong")
                    continue
            moved = True
            s2 = (ws[:w] + ((at2, g2, v2),) + ws[w + 1:], n2, a2)
            if s2 not in seen:
                seen.add(s2)
                todo.append(s2)
        if not moved and done < waves:
            bad.add("stuck")
    return bad


def test_the_interleavings_tell_a_sound_order_from_an_unsound_one():
    assert failures("WSSR", 2, 3) and failures("WR", 2, 3) and not failures("WSRS", 2, 3)


@pytest.mark.parametrize("waves", [2, 4])
def test_every_wave_of_a_team_takes_the_same_groups(waves):
    order = kernel_order()
    assert order.count("W") == 1 and order.count("R") == 1 and "S" in order, order
    assert not failures(order, waves, 3), order
