"""A launch of the persistent solve (mke_amd/csrc/persist_run.h) whose
workgroups do not all find a CU, as a model on the CPU: every order of their
steps, with fewer CUs than workgroups and every moment at which one may give
up.  A launch that is going to be repeated must leave what the repeated one
reads as it was, and a column that gives up must not stop another one.

Model: a workgroup stores its slot of exchange 0, waits until the slots of
its column are all there, and so on; the first thing that a repeated launch
would read is written after exchange `quiet` - 1.  While a slot of exchange 0 is
missing a workgroup may give up: it sets the abort flag and leaves its CU to
the next.  A workgroup that waits may see the flag and leave."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HOPS = 3


def outcomes(quiet, columns, cus, shared_flag):
    """(a column was given up, it has written, it has finished) for each
    column, over every reachable end.  columns: workgroups of each."""
    col = [c for c, k in enumerate(columns) for _ in range(k)]
    n = len(col)
    flag = lambda c: 0 if shared_flag else c  # noqa: E731
    # a workgroup: -1 not started, 2 h: before storing slot h, 2 h + 1: waiting
    # for exchange h, "left", "done"; slots stored per workgroup; flags; writes
    start = ((-1,) * n, (0,) * n, (False,) * len(columns), (False,) * n)
    seen, todo, ends = {start}, [start], set()
    while todo:
        at, slots, flags, wrote = todo.pop()
        nexts = []

        def go(i, state, slot=None, raised=None, write=False):
            a, s, f, w = list(at), list(slots), list(flags), list(wrote)
            a[i] = state
            if slot is not None:
                s[i] = slot
            if raised is not None:
                f[raised] = True
            w[i] = w[i] or write
            nexts.append((tuple(a), tuple(s), tuple(f), tuple(w)))

        running = sum(isinstance(a, int) and a >= 0 for a in at)
        for i in range(n):
            a = at[i]
            if a == -1:
                if running < cus and all(b != -1 for b in at[:i]):  # dispatched in order
                    go(i, 0)
            elif a in ("left", "done"):
                continue
            elif a % 2 == 0:
                go(i, a + 1, slot=a // 2 + 1)
            else:
                h, mine = a // 2, [j for j in range(n) if col[j] == col[i]]
                if all(slots[j] > h for j in mine):
                    go(i, "done" if h + 1 == HOPS else a + 1, write=h + 1 >= quiet)
                else:
                    if h == 0:
                        go(i, "left", raised=flag(col[i]))
                    if flags[flag(col[i])]:
                        go(i, "left")
        if not nexts:
            ends.add(tuple((any(at[i] == "left" for i in range(n) if col[i] == c),
                            any(wrote[i] for i in range(n) if col[i] == c),
                            all(at[i] == "done" for i in range(n) if col[i] == c))
                           for c in range(len(columns))))
        for s in nexts:
            if s not in seen:
                seen.add(s)
                todo.append(s)
    return ends


@pytest.mark.parametrize("columns,cus", [((3,), 2), ((3,), 3), ((4,), 3), ((2, 2), 3)])
def test_repeated_launch_finds_its_input(columns, cus):
    ends = outcomes(2, columns, cus, False)
    assert ends and not any(left and wrote for e in ends for left, wrote, _ in e)
    assert all(left or done for e in ends for left, _, done in e)
    # with the first write after exchange 0, which the launches that continue
    # a solve once began with, the model does find the lost input
    assert any(left and wrote for e in outcomes(1, columns, cus, False) for left, wrote, _ in e)


def test_column_goes_on_beside_one_that_gives_up():
    """With a flag per column each column finishes or has written nothing;
    with one flag for both, a column could be stopped after it had written."""
    def stopped(ends):
        return any(left and wrote for e in ends for left, wrote, _ in e)

    assert not stopped(outcomes(2, (2, 3), 4, False))
    assert stopped(outcomes(2, (2, 3), 4, True))


TURNS = r"""
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
#include "persist_turns.h"
using phg::PersistTurns;

// threads that each hold a turn until `together` of them do at once, or 2 s
static bool meet(PersistTurns& t, std::vector<int> workgroups, int together)
{
    std::atomic<int> in{0}, most{0};
    std::vector<std::thread> threads;
    for (int w : workgroups)
        threads.emplace_back([&, w] {
            t.enter(w);
            const int now = ++in;
            for (int m = most; now > m && !most.compare_exchange_weak(m, now);) {}
            for (int k = 0; k < 2000 && most < together; ++k)
                std::this_thread::sleep_for(std::chrono::milliseconds(1));
            --in;
            t.leave(w);
        });
    for (auto& th : threads) th.join();
    return most >= together;
}

int main()
{
    PersistTurns t(256);
    // as many small ones as have a shader engine's CUs to themselves
    if (!meet(t, {22, 22}, 2) || !meet(t, {161, 64}, 2)) return 1;
    if (!meet(t, {1, 9, 32, 7, 11, 22, 3, 5}, 8)) return 2;
    // 33 workgroups put two on an engine: 4 x 2 + 1 are more than its 8 CUs
    for (int w : {33, 33, 64, 50})
        if (!t.try_enter(w)) return 3;
    if (t.try_enter(1)) return 4;
    for (int w : {33, 33, 64, 50}) t.leave(w);
    // a whole device's launch alone, also on a device with fewer CUs
    if (!t.try_enter(256) || t.try_enter(1)) return 5;
    t.leave(256);
    PersistTurns small(32);
    if (!small.try_enter(64) || small.try_enter(1)) return 6;
    small.leave(64);
    // who waits is not passed: a small launch comes after the big one that
    // came before it
    if (!t.try_enter(22)) return 7;
    std::atomic<int> order{0};
    int big = 0;
    std::thread first([&] { t.enter(256); big = ++order; t.leave(256); });
    std::this_thread::sleep_for(std::chrono::milliseconds(100));
    if (t.try_enter(22)) return 8;
    t.leave(22);
    first.join();
    if (big != 1 || !t.try_enter(22)) return 9;
    t.leave(22);
    std::puts("ok");
    return 0;
}
"""


def test_turns_of_a_process(tmp_path):
    """Launches of several threads run at the same time where they are sure to
    be resident together, and only there (csrc/persist_turns.h)."""
    src, exe = tmp_path / "turns.cpp", tmp_path / "turns"
    src.write_text(TURNS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I",
                    os.path.join(ROOT, "mke_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r
