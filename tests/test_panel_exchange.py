"""CPU model of the row exchange that ends a sub-block of the grouped LU panel (pyvl_amd/csrc/lu.hip,
panel_kernel; which rows move through which words: lu_exchange.hpp, compiled here as it stands).
Between two barriers the four waves of a group run in any order, so no wave may overwrite a row that
another one of its group still has to publish, and the result has to be that of the interchanges made
one after the other, whatever the order of the waves and groups."""

import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

HDR = Path(__file__).resolve().parents[1] / "pyvl_amd" / "csrc" / "lu_exchange.hpp"
KB = 8


@pytest.fixture(scope="module")
def row_move(tmp_path_factory):
    d = tmp_path_factory.mktemp("exchange")
    (d / "x.cpp").write_text(f'#include "{HDR}"\n'
                             'extern "C" void row_move(int t, int from, int j0, int kb, int *o)\n'
                             '{ const pvl::RowMove m = pvl::row_move(t, from, j0, kb);\n'
                             '  o[0] = m.up; o[1] = m.down; o[2] = m.buf; o[3] = m.idx; }\n')
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", str(d / "x.cpp"), "-o", str(d / "x.so")], check=True)
    lib = C.CDLL(str(d / "x.so"))

    def call(t, frm, j0, kb):
        o = (C.c_int * 4)()
        lib.row_move(t, frm, j0, kb, o)
        return bool(o[0]), bool(o[1]), (o[2], o[3])

    return call


def _pivots(kind, m, j0, kb, rng):
    if kind == "exchange":  # two rows of the sub-block change places, in waves 0 and 1
        return [j0 + 1] + [j0 + t for t in range(1, kb)]
    if kind == "cycle":  # every row of the sub-block moves on
        return [j0 + kb - 1] * kb
    if kind == "inside":
        return [int(rng.integers(j0 + t, j0 + kb)) for t in range(kb)]
    if kind == "repeat":  # the same position below again and again
        return [int(rng.choice([min(m - 1, j0 + kb + 1), j0 + t])) for t in range(kb)]
    return [int(rng.integers(j0 + t, m)) for t in range(kb)]


def _jobs(row_move, m, G, j0, kb, piv):
    """(group, wave) -> (rows it publishes with their words, words it reads with the rows they replace)."""
    at = list(range(m))  # the row now at each position
    for t, p in enumerate(piv):
        at[j0 + t], at[p] = at[p], at[j0 + t]
    jobs = {(g, w): ([], []) for g in range(G) for w in range(4)}
    pivot_rows = {}  # word of each new pivot row: every group reads it (columns right of the sub-block)
    for t in range(kb):
        frm = at[j0 + t]
        up, down, word = row_move(t, frm, j0, kb)
        if up:
            jobs[frm % G, t % 4][0].append((frm, (0, t)))
        if down:
            jobs[(j0 + t) % G, t % 4][0].append((j0 + t, (1, t)))
        pivot_rows[t] = word
        if frm != j0 + t:
            jobs[(j0 + t) % G, t % 4][1].append((word, j0 + t))
        if frm >= j0 + kb:  # its place is taken by a row of the sub-block
            jobs[frm % G, t % 4][1].append(((1, at[frm] - j0), frm))
    return at, jobs, pivot_rows


CASES = [(kind, G, j0, kb, seed) for kind in ("exchange", "cycle", "inside", "repeat", "any") for G in (2, 3, 5)
         for j0, kb in ((8, 8), (16, 5), (0, 2)) for seed in range(6)]


@pytest.mark.parametrize("kind", ["exchange", "cycle", "inside", "repeat", "any"])
def test_rows_move_as_interchanges_in_every_order(row_move, kind):
    for _, G, j0, kb, seed in (c for c in CASES if c[0] == kind):
        rng = np.random.default_rng(1000 * G + 10 * j0 + seed)
        m = j0 + kb + 4 * G + 3
        piv = _pivots(kind, m, j0, kb, rng)
        at, jobs, pivot_rows = _jobs(row_move, m, G, j0, kb, piv)
        for g in range(G):
            for a in range(4):
                for b in range(4):
                    if a != b:
                        read = {r for r, _ in jobs[g, a][0]}
                        assert not read & {r for _, r in jobs[g, b][1]}, (kind, G, j0, kb, piv, g, a, b)
        # the same as a run: waves in random order, each publishing before it reads and overwrites; a wave
        # whose words are not there yet waits
        for _ in range(4):
            L, words = {r: r for r in range(m)}, {}
            todo = [list(("p", *x) for x in jobs[k][0]) + [("w", jobs[k][1])] for k in jobs]
            while any(todo):
                ready = [q for q in todo if q and (q[0][0] == "p" or all(w in words for w, _ in q[0][1]))]
                assert ready, "a wave waits for a word that nobody publishes"
                q = ready[rng.integers(len(ready))]
                act = q.pop(0)
                if act[0] == "p":
                    words[act[2]] = L[act[1]]
                else:
                    for word, dst in act[1]:
                        L[dst] = words[word]
            assert [L[r] for r in range(m)] == at
            assert all(words[w] == at[j0 + t] for t, w in pivot_rows.items())
