"""Slots of the block CG that a program replaces in a solver's table: the solver
calls them, and a slot that only passes on to the backend's gives the same solve."""
import ctypes as C

import numpy as np
import pytest

from gcge_hip import Matrix, api, capi
from gcge_hip import problems as P

pytestmark = pytest.mark.gpu

SLOTS = {"MatDotMultiVecInnerProdDiag": capi.F_MatDotMultiVecInnerProdDiag,
         "BlockCGResidualUpdate": capi.F_BlockCGResidualUpdate,
         "BlockPCGResidualUpdate": capi.F_BlockPCGResidualUpdate}


@pytest.mark.parametrize("name,precond", [("MatDotMultiVecInnerProdDiag", 0), ("BlockCGResidualUpdate", 0),
                                          ("MatDotMultiVecInnerProdDiag", 1), ("BlockPCGResidualUpdate", 1)])
def test_replaced_slot_is_called(name, precond):
    A, nev = P.lap2d(20)[0], 4
    X0, calls, results = P.random_x0(A.shape[0], nev, 3), [0], []
    for replace in (False, True):
        S = api.Solver(Matrix(A), None, nev, precision="fp64", ev_tol=1e-9, conv_type="NS", ev_max_it=200,
                       bcg_precond=precond)
        ops = S.solver.contents.ops.contents
        own = C.cast(getattr(ops, name), SLOTS[name])

        def forward(*args):
            calls[0] += 1
            own(*args)

        slot = SLOTS[name](forward)
        if replace:
            setattr(ops, name, C.cast(slot, C.c_void_p))
        results.append(S.solve(X0))
    assert calls[0] > 20
    assert results[0]["num_iter"] == results[1]["num_iter"]
    assert np.array_equal(results[0]["eval"], results[1]["eval"])
    assert np.array_equal(results[0]["evec"], results[1]["evec"])
