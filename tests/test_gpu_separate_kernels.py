"""The solver's operator forms on the separate SpMV and vector kernels: the tests of test_gpu_lattice.py
and test_gpu_elemop.py, whose systems are small enough to be solved in one launch, once more in
contexts with an explicit launch shape of the vector step (8 elements a pass, its default), which
selects the separate kernels."""
import pytest

import ferrite_amd as fa
from test_gpu_elemop import *  # noqa: F401,F403
from test_gpu_lattice import *  # noqa: F401,F403

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def separate_kernels(monkeypatch):
    allocate, solve = fa.allocate_matrix, fa.solve

    def allocate_separate(*args, **kw):
        K = allocate(*args, **kw)
        fa.set_tuning(K, cg_elems=8)
        return K

    def solve_separate(*args, **kw):
        res = solve(*args, **kw)
        assert res.kernels in ("separate", None)
        return res

    monkeypatch.setattr(fa, "allocate_matrix", allocate_separate)
    monkeypatch.setattr(fa, "solve", solve_separate)
