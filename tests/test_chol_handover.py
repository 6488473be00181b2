"""The hand-overs between the workgroups of a region of the Cholesky chain (csrc/chol_region.h): a model of what each wave
stores, counts, waits for and reads, with the kernel's own words and targets (csrc/chol_handover.h, compiled for the host),
in which no wait may end before everything that is read behind it has been stored.

Waits end once a count is large enough, so a state with more progress enables more: if a read can ever be reached without a
certain store, it is reached by running everything else as far as it goes while the store's wave is held in front of it.
One such run per store covers all interleavings."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-compressor_amd", "csrc")
WRAPPER = """
#define __host__
#define __device__
#include "chol_handover.h"
using namespace cholregion;
extern "C" {
int x(int m) { return word_x(m); }
int spine_row(int j) { return word_spine_row(j); }
int row(int b) { return word_row(b); }
int next(int b) { return word_next(b); }
int diag(int b) { return word_diag(b); }
int ticket() { return WORD_TICKET; }
int words() { return SYNC_WORDS / SYNC_LINE; }
unsigned one(unsigned done) { return target_one(done); }
unsigned rows(unsigned done, int b, int blocks) { return target_row(done, b, blocks); }
unsigned hand_over() { return HAND_OVER; }
int max_blocks() { return MAX_BLOCKS; }
}
"""
WAVES = 8


@pytest.fixture(scope="module")
def header(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("handover") / "handover.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", "-x", "c++", "-", "-o", lib],
                   input=WRAPPER.encode(), check=True)
    return ctypes.CDLL(lib)


class Task:
    """The program of every wave of a workgroup: ("store", item), ("count", word, add), ("wait", word, target),
    ("read", item, whose), ("meet",).  An item is stored wave by wave; `whose` are the waves that store it."""

    def __init__(self):
        self.waves = [[] for _ in range(WAVES)]

    def all(self, *op, waves=range(WAVES)):
        for w in waves:
            self.waves[w].append(op)

    def wait_for(self, *awaited):  # the first wave polls between two barriers
        self.all("meet")
        for word, target in awaited:
            self.all("wait", word, target, waves=[0])
        self.all("meet")


STORERS = range(4, WAVES)  # of the spine


def region(h, nb, done):
    """The tasks of one region, one set of rows below it."""
    add = lambda waves: h.hand_over() // len(waves)  # noqa: E731
    spine = Task()
    for m in range(nb):
        more = m + 1 < nb
        if m > 0:
            spine.all("store", ("solved", m, m - 1), waves=STORERS)
        spine.all("meet")
        if m > 0:
            spine.all("count", h.spine_row(m), add(STORERS), waves=STORERS)
        if m > 1 and not more:  # block (1, 0) takes the place of what the row blocks read
            for b in range(2, nb):
                spine.all("read", ("taken", b), range(WAVES), waves=STORERS)
        for _ in range(4):
            spine.all("meet")
        spine.all("store", ("x", m), waves=STORERS)
        if not more:
            spine.all("count", h.x(m), add(STORERS), waves=STORERS)
            break
        if m > 0:
            spine.all("wait", h.next(m + 1), h.one(done), waves=STORERS)
            spine.all("read", ("next", m + 1), range(WAVES), waves=STORERS)
        spine.all("meet")
        spine.all("meet")
        spine.all("count", h.x(m), add(STORERS), waves=STORERS)
        if m > 0:
            spine.all("wait", h.diag(m + 1), h.one(done), waves=STORERS)
            spine.all("read", ("diag", m + 1), range(WAVES), waves=STORERS)
        spine.all("meet")
    tasks = [spine]
    every = range(WAVES)
    for b in range(2, nb):
        t = Task()
        t.all("store", ("taken", b))
        for m in range(b - 1):
            if m > 0:
                t.wait_for((h.next(m + 1), h.one(done)))
                t.all("read", ("next", m + 1), every)
            t.wait_for((h.x(m), h.one(done)))
            t.all("read", ("x", m), STORERS)
            t.all("meet")
            t.all("meet")
            if m + 2 == b:
                t.all("store", ("next", b))
                t.all("count", h.next(b), add(every))
                t.all("store", ("diag", b))
                t.all("count", h.diag(b), add(every))
            t.all("store", ("solved", b, m))
            t.all("count", h.row(b), add(every))
            for c in range(m + 2, b):
                t.wait_for((h.row(c), h.rows(done, c, m + 1)))
                t.all("read", ("solved", c, m), every)
            if m + 2 != b:
                t.all("meet")
        tasks.append(t)
    below = Task()
    for j in range(nb):
        if j > 0:
            below.wait_for((h.spine_row(j), h.one(done)), *([(h.row(j), h.rows(done, j, j - 1))] if j > 1 else []))
            for i in range(j):
                below.all("read", ("solved", j, i), STORERS if i == j - 1 else every)
        below.wait_for((h.x(j), h.one(done)))
        below.all("read", ("x", j), STORERS)
    tasks.append(below)
    return tasks


def run(tasks, counts, held=None):
    """As far as the tasks go with wave `held` = (task, wave, index) kept in front of that operation -> (finished, the
    counts, reads that were reached without a store of theirs)."""
    counts, at = dict(counts), [[0] * WAVES for _ in tasks]
    stored, early = set(), []
    moved = True
    while moved:
        moved = False
        for t, task in enumerate(tasks):
            for w in range(WAVES):
                while at[t][w] < len(task.waves[w]) and (t, w, at[t][w]) != held:
                    op = task.waves[w][at[t][w]]
                    if op[0] == "store":
                        stored.add((op[1], w))
                    elif op[0] == "count":
                        counts[op[1]] = counts.get(op[1], 0) + op[2]
                    elif op[0] == "wait" and counts.get(op[1], 0) < op[2]:
                        break
                    elif op[0] == "read":
                        early += [(op[1], v) for v in op[2] if (op[1], v) not in stored]
                    elif op[0] == "meet":
                        behind = [sum(o[0] == "meet" for o in task.waves[v][:at[t][v]]) for v in range(WAVES)]
                        there = [at[t][v] < len(task.waves[v]) and task.waves[v][at[t][v]][0] == "meet" for v in range(WAVES)]
                        if not all(behind[v] > behind[w] or (behind[v] == behind[w] and there[v]) for v in range(WAVES)):
                            break
                    at[t][w] += 1
                    moved = True
    return all(at[t][w] == len(task.waves[w]) for t, task in enumerate(tasks) for w in range(WAVES)), counts, early


def check(h, nb, regions):
    """Every region finishes, and no store of the last one can be missing from a read -> the reads that can do without."""
    counts = {}
    for done in range(regions - 1):
        finished, counts, early = run(region(h, h.max_blocks(), done), counts)
        assert finished and not early
    tasks = region(h, nb, regions - 1)
    finished, _, early = run(tasks, counts)
    assert finished and not early
    found = set()
    for t, task in enumerate(tasks):
        for w in range(WAVES):
            for i, op in enumerate(task.waves[w]):
                if op[0] == "store":
                    found |= {item for item, _ in run(tasks, counts, (t, w, i))[2]}
    return found


@pytest.mark.parametrize("nb", [1, 2, 3, 4])
@pytest.mark.parametrize("regions", [1, 3])
def test_no_wait_ends_before_what_is_read_behind_it(header, nb, regions):
    assert check(header, nb, regions) == set()


def test_one_producer_to_a_word(header):
    producers = {}
    for t, task in enumerate(region(header, header.max_blocks(), 0)):
        for op in sum(task.waves, []):
            if op[0] == "count":
                assert 0 <= op[1] < header.ticket() < header.words()
                producers.setdefault(op[1], set()).add(t)
    assert len(producers) == 4 + 3 + 2 + 2 + 2 and all(len(p) == 1 for p in producers.values())


def test_a_word_with_two_producers_is_found(header):
    """The spine's block (j, j - 1) counted in the word of row block j: four waves that are ahead stand in for those of the
    other workgroup that are not."""

    class Shared:
        def __getattr__(self, name):
            return getattr(header, name)

        def spine_row(self, j):
            return header.row(j) if j > 1 else header.spine_row(j)

        def one(self, done):
            return header.one(done)

        def rows(self, done, b, blocks):
            return (done * b + blocks) * header.hand_over()

    shared = Shared()
    plain = region(shared, 4, 0)
    for task in plain[-1:]:  # the rows below wait for both producers' counts together
        for ops in task.waves:
            for i, op in enumerate(ops):
                if op[0] == "wait" and op[1] in (header.row(2), header.row(3)):
                    ops[i] = ("wait", op[1], header.hand_over() * (2 if op[1] == header.row(2) else 3))
    finished, _, early = run(plain, {})
    assert finished and not early
    found = set()
    for w in range(WAVES):
        held = plain[1].waves[w].index(("store", ("solved", 2, 0)))
        found |= set(run(plain, {}, (1, w, held))[2])
    assert found == {(("solved", 2, 0), w) for w in range(WAVES)}
