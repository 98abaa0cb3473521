"""GPU test of the flux kernels' runs per cube, which follow the number of
resident cubes: one inner iteration on both sides of every line of that rule
against the oracle (state arrays bitwise, norms at 1e-12 of their magnitude:
the summation order differs)."""
import numpy as np
import pytest

from test_gpu_parity import STATE, compare, er_close

pytestmark = pytest.mark.gpu

# 1, 7, 48 | 49, 64 | 65, 90 | 91, 128 | 129, 240 | 241, 370 | 371, 560 | 561, 800
# cubes (whole and ragged groups of 8; from 561 on the last 192 cubes in four runs)
LATTICES = [(1, 1, 1), (7, 1, 1), (4, 4, 3), (7, 7, 1), (4, 4, 4), (13, 5, 1), (6, 5, 3), (13, 7, 1),
            (8, 4, 4), (43, 3, 1), (8, 6, 5), (241, 1, 1), (37, 5, 2), (53, 7, 1), (8, 10, 7),
            (187, 3, 1), (10, 10, 8)]


@pytest.mark.parametrize("dims", LATTICES, ids=lambda d: str(int(np.prod(d))))
def test_runs_per_cube_bitwise(B, O, dims):
    case = lattice_case(B, dims)
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


def lattice_case(B, dims):
    size = 1.0 / max(dims)
    return B.Case(B.case_params("tiny", lattice=dims, cube_size=size, ico_level=3,
                                sphere_center=tuple(0.5 * d * size for d in dims),
                                sphere_diameter=0.3 * min(dims) * size))


# In place: 1, 100 | 101, 320 | 321 cubes (flux and update as two kernels | one).
@pytest.mark.parametrize("dims", [(1, 1, 1), (5, 5, 4), (101, 1, 1), (8, 8, 5), (107, 3, 1)],
                         ids=lambda d: str(int(np.prod(d))))
def test_in_place_stages_bitwise(B, O, dims):
    case = lattice_case(B, dims)
    out = []
    for fuse in (1, 2):
        e = B.Engine(0)
        try:
            e.load_case(case)
            e.set_flux(1, 1, fuse)
            h = e.run(1, 2)
            if fuse == 1:
                orc = O.OracleRun(case, nthreads=16)
                ho = orc.run(1, 2)
                compare(e, orc, STATE)
                assert er_close(h, ho)
            out.append(h)
        finally:
            e.close()
    # the norms do not depend on the kernel that formed them
    assert np.array_equal(out[0].view(np.int64), out[1].view(np.int64))


# 1, 32 | 33, 64 | 65, 128 | 129, 200 | 201, 370 | 371, 560 | 561, 1,003 cubes
@pytest.mark.parametrize("dims", [(1, 1, 1), (8, 4, 1), (11, 3, 1), (4, 4, 4), (13, 5, 1),
                                  (8, 4, 4), (43, 3, 1), (8, 5, 5), (67, 3, 1), (37, 5, 2),
                                  (53, 7, 1), (8, 10, 7), (187, 3, 1), (59, 17, 1)],
                         ids=lambda d: str(int(np.prod(d))))
def test_mixed_runs_by_rule_are_bitwise(B, dims):
    # The runs the rule picks against a pinned count, on one case.
    case = lattice_case(B, dims)
    out = []
    for pinned in (None, 1, 4):
        e = B.Engine(0)
        try:
            e.alloc_pool(case.ncube - 1, 1, "mixed")
            s = e.add_case(case)
            if pinned:
                e.set_flux(2, pinned, 0)
            er = e.run(1, 1)[:, s, :]
            out.append((e.case_state(s, "U1_"), er))
        finally:
            e.close()
    for st, er in out[1:]:
        assert np.array_equal(st.view(np.int64), out[0][0].view(np.int64))
        assert np.array_equal(er.view(np.int64), out[0][1].view(np.int64))


# Stage opening: IB cubes with BCs on three faces and entries at their edge
# cells; levels of more entries than one pass takes, in more than 1536 slots.
@pytest.mark.parametrize("dims", [(2, 2, 1), (2, 2, 2), (5, 5, 5)],
                         ids=lambda d: str(int(np.prod(d))))
def test_stage_opening_bitwise(B, O, dims):
    size = 1.0 / max(dims)
    case = B.Case(B.case_params("cfg2", lattice=dims, cube_size=size,
                                sphere_center=tuple(0.5 * d * size for d in dims),
                                sphere_diameter=0.25 * min(dims) * size))
    e = B.Engine(0)
    try:
        e.load_case(case)
        h = e.run(1, 2)
        orc = O.OracleRun(case, nthreads=16)
        ho = orc.run(1, 2)
        compare(e, orc, STATE)
        assert er_close(h, ho)
        # mixed: the fill in LDS against the fill on memory
        out = []
        for limit in (None, 0):
            if limit is not None:
                e.set_ghost_lds_limit(limit)
            e.alloc_pool(case.ncube - 1, 1, "mixed")
            s = e.add_case(case)
            er = e.run(1, 2)
            out.append((e.case_state(s, "U1_"), er))
        for a, b in zip(*out):
            assert np.array_equal(a.view(np.int64), b.view(np.int64))
    finally:
        e.close()


# Single stages that write the other copy of the iterate: each leaves the ghost
# regions of the domain BCs where the next one and a reader find them.
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 2, 2), (3, 1, 2)],
                         ids=lambda d: "x".join(map(str, d)))
def test_single_pushing_stages_bitwise(B, O, dims):
    case = lattice_case(B, dims)
    e = B.Engine(0)
    try:
        e.load_case(case)
        e.set_flux(1, 1, 2)
        orc = O.OracleRun(case, nthreads=16)
        for RK in (1, 2, 3, 1):
            e.part("stage", RK)
            e.part("interface")
            orc.stage(RK)
            compare(e, orc, ("U1_",))
    finally:
        e.close()
