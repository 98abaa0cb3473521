"""GPU test of the IB fill on both sides of its LDS capacity of 3072 value slots:
spheres that fill one cube and need 3069 (in LDS) and 3074 (on memory).  FP64
bitwise the oracle; mixed bitwise the fill on memory."""
import numpy as np
import pytest

from test_gpu_parity import STATE, compare, er_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("diameter,centre,in_lds", [(1.072, (0.52, 0.47, 0.5), True),
                                                    (1.084, (0.5, 0.5, 0.45), False)],
                         ids=["3069", "3074"])
def test_fill_at_the_lds_capacity(B, O, diameter, centre, in_lds):
    case = B.Case(B.case_params("cfg2", lattice=(1, 1, 1), cube_size=1.0, sphere_center=centre,
                                sphere_diameter=diameter, ico_level=4))
    e = B.Engine(0)
    try:
        e.load_case(case)
        levels = e.ghost_stats()["levels"]
        h = e.run(1, 2)
        orc = O.OracleRun(case, nthreads=8)
        ho = orc.run(1, 2)
        compare(e, orc, STATE)
        assert er_close(h, ho)
        out = []
        for limit in (None, 0):
            if limit is not None:
                e.set_ghost_lds_limit(limit)
            e.alloc_pool(case.ncube - 1, 1, "mixed")
            s = e.add_case(case)
            er = e.run(1, 2)
            out.append((e.case_state(s, "U1_"), er))
        assert (levels < e.ghost_stats()["levels"]) == in_lds
        for a, b in zip(*out):
            assert np.array_equal(a.view(np.int64), b.view(np.int64))
    finally:
        e.close()
