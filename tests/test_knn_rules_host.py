"""Host (g++) test of mhip_knn_rules.hpp: over every course that a row can take
through the search's launches, exactly one launch finishes it, and only that
one appends it to the list of ambiguous rows, which has one place per row."""
import ctypes
import itertools
import os
import subprocess

import pytest

SRC = """
#include "%s"
extern "C" int is_new(int redo, int missed) { return mhip::row_is_new(redo, missed); }
extern "C" int mark() { return mhip::ROW_DEFERRED; }
extern "C" int was_deferred(int st) { return mhip::row_was_deferred(st); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text(SRC % os.path.join(root, "meshoid_amd", "csrc", "mhip_knn_rules.hpp"))
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", d / "r.so", d / "r.cpp"], check=True)
    return ctypes.CDLL(str(d / "r.so"))


MISS, AMBIGUOUS = 128, 1


def test_each_row_is_finished_and_listed_once(rules):
    # a wavefront of three rows; per row: its radius seed is too small, and it
    # is ambiguous; per launch: the wavefront defers
    for miss in itertools.product((False, True), repeat=3):
        for amb in itertools.product((False, True), repeat=3):
            for defer1, defer2 in itertools.product((False, True), repeat=2):
                st = [0, 0, 0]
                finished, listed, on_list = [0] * 3, [0] * 3, 0

                def finish(r, bits):
                    finished[r] += 1
                    listed[r] += amb[r]
                    st[r] = bits | (AMBIGUOUS if amb[r] else 0)

                # first launch
                if defer1:
                    on_list += 1
                    st = [rules.mark() if rules.is_new(0, 0) else s for s in st]
                else:
                    for r in range(3):
                        if miss[r]:
                            st[r] = MISS
                        else:
                            finish(r, 0)
                # redo launch: wavefronts with a row that missed
                missed = [bool(s & MISS) for s in st]
                if any(missed):
                    if defer2:
                        on_list += 1
                        st = [rules.mark() if rules.is_new(1, m) else s for m, s in zip(missed, st)]
                    else:
                        for r in range(3):
                            if rules.is_new(1, missed[r]):
                                finish(r, MISS)
                # the deferred wavefronts
                assert on_list <= 1
                if on_list:
                    for r in range(3):
                        if rules.was_deferred(st[r]):
                            finish(r, MISS if miss[r] else 0)
                assert finished == [1, 1, 1]
                assert listed == [int(a) for a in amb] and sum(listed) <= 3
                assert [bool(s & MISS) for s in st] == [bool(m) for m in miss]
                assert all(s < rules.mark() for s in st)
