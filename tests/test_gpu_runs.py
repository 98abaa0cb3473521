"""GPU test of the flux kernels' runs per cube, which follow the number of
resident cubes: one inner iteration on both sides of every line of that rule
against the oracle (state arrays bitwise, norms at 1e-12 of their magnitude:
the summation order differs)."""
import numpy as np
import pytest

from test_gpu_parity import STATE, compare, er_close

pytestmark = pytest.mark.gpu

# 1, 7, 100 | 101, 700 | 701, 1,100 | 1,101 cubes (whole and ragged groups of 8)
LATTICES = [(1, 1, 1), (7, 1, 1), (5, 5, 4), (101, 1, 1), (10, 10, 7), (701, 1, 1), (11, 10, 10),
            (367, 3, 1)]


@pytest.mark.parametrize("dims", LATTICES, ids=lambda d: str(int(np.prod(d))))
def test_runs_per_cube_bitwise(B, O, dims):
    size = 1.0 / max(dims)
    case = B.Case(B.case_params("tiny", lattice=dims, cube_size=size, ico_level=3,
                                sphere_center=tuple(0.5 * d * size for d in dims),
                                sphere_diameter=0.3 * min(dims) * size))
    e = B.Engine(0)
    try:
        e.load_case(case)
        h = e.run(1, 1)
        orc = O.OracleRun(case, nthreads=16)
        ho = orc.run(1, 1)
        compare(e, orc, STATE)
        assert er_close(h, ho)
    finally:
        e.close()
