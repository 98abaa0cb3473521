"""GPU tests of engine parts next to runs and repeated: a part that writes the
other copy of the iterate leaves the state where the captured step, the next
stage and a reader find it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATE = {"fp64": ("U1_", "U1", "U1q", "U1p1", "U1p2", "Rku1", "Residual1"),
         "mixed": ("U1_", "U1", "U1q")}


def pool(B, case, precision):
    e = B.Engine(0)
    e.alloc_pool(case.ncube - 1, 1, precision)
    e.add_case(case)
    return e


def same(a, b, names):
    for n in names:
        x, y = a.case_state(0, n), b.case_state(0, n)
        assert np.array_equal(x.view(np.int64), y.view(np.int64)), n


PARTS = {
    "stage": lambda e: e.part("stage", 1),
    "flux_push": lambda e: e.part("flux_push", 2),
    "flux_update": lambda e: e.part("flux_update", 1),
    "timed_stage": lambda e: e.time_part("stage", RK=1, reps=3),
    "timed_stage_twice": lambda e: e.time_part("stage", RK=1, reps=2),
    "timed_flux": lambda e: e.time_part("flux_push", RK=1, reps=1),
}


@pytest.mark.parametrize("n_inner", [1, 2])
@pytest.mark.parametrize("part", sorted(PARTS))
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_captured_steps_continue_from_a_part(B, precision, part, n_inner):
    # Steps, parts that swap the copies of the iterate, and steps again: the
    # replays continue from the copy the part wrote, as eager steps do.
    case = B.Case(B.case_params("tiny"))
    graph, eager = pool(B, case, precision), pool(B, case, precision)
    try:
        for rep in range(3):
            h = graph.run(2, n_inner, use_graph=True)
            ho = eager.run(2, n_inner, use_graph=False)
            assert np.array_equal(h.view(np.int64), ho.view(np.int64)), rep
            same(graph, eager, STATE[precision])
            for e in (graph, eager):
                PARTS[part](e)
            same(graph, eager, STATE[precision])
    finally:
        graph.close()
        eager.close()


@pytest.mark.parametrize("reps", [1, 2, 3, 4])
@pytest.mark.parametrize("precision,part", [("fp64", "flux_push"), ("mixed", "flux_push"),
                                            ("mixed", "flux_update")])
def test_repeated_pushing_kernel_carries_the_bc_regions(B, precision, part, reps):
    # The kernel several times with no stage opening in between: each reads the
    # ghost regions of the domain BCs, and the last leaves them in the iterate.
    case = B.Case(B.case_params("tiny"))
    timed, single = pool(B, case, precision), pool(B, case, precision)
    try:
        for e in (timed, single):
            e.run(1, 2)   # (an even number of kernels: the copies differ)
        timed.time_part(part, RK=2, reps=reps)
        for _ in range(reps):
            single.part(part, 2)
        same(timed, single, ("U1_",))
        for e in (timed, single):
            e.run(1, 1)
        same(timed, single, STATE[precision])
    finally:
        timed.close()
        single.close()
