"""Status codes of in-memory Faith PD for trees and tables that do not fit together:
the same for tables that its filter leaves whole and for those it changes.  All are
returned before any device work."""
import ctypes as C

import numpy as np
import pytest


def table_of(ssu, tree, kind):
    """Three rows over three samples; filtered: the last sample has no counts and the last row no entry."""
    st, le, nm = tree
    if kind == "whole":
        return ssu.Inputs(st, le, nm, ["a", "b", "c"], ["x", "y", "z"], np.array([0, 1, 2, 3], np.uint32),
                          np.array([0, 1, 2], np.uint32), np.array([4.0, 5.0, 6.0]))
    return ssu.Inputs(st, le, nm, ["a", "b", "c"], ["x", "y", "z"], np.array([0, 1, 2, 2], np.uint32),
                      np.array([0, 1], np.uint32), np.array([4.0, 5.0]))


def status(ssu, inp):
    res = C.POINTER(ssu.RVec)()
    return ssu.lib().ssu_faith_pd_inmem(C.byref(inp.table), C.byref(inp.tree), C.byref(res))


@pytest.mark.parametrize("kind", ["whole", "filtered"])
def test_faith_status(ssu, kind):
    inp = table_of(ssu, ssu.newick_to_bp("((a:1,b:1):1,d:1);"), kind)
    assert status(ssu, inp) == ssu.TABLE_AND_TREE_DO_NOT_OVERLAP   # no tip c (dropped rows count too)
    st, le, nm = ssu.newick_to_bp("((a:1,b:1):1,c:1);")
    inp = table_of(ssu, (st, le, nm), kind)
    inp.tree.n_parens = 0
    assert status(ssu, inp) == ssu.TABLE_AND_TREE_DO_NOT_OVERLAP   # a tree without nodes has no tips
    inp = table_of(ssu, (st, le, nm), kind)
    inp.tree.n_parens = len(st) - 1
    assert status(ssu, inp) == ssu.TREE_MISSING                    # unbalanced
    inp = table_of(ssu, (st, le, nm), kind)
    inp.table.n_samples = 0
    assert status(ssu, inp) == ssu.TABLE_EMPTY
