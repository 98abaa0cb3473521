"""GPU test of the IB fill's slot limit: its largest setting stands for the
kernel's capacity, so it takes back a lowered limit."""
import pytest

pytestmark = pytest.mark.gpu


def test_largest_limit_is_the_default(B):
    # A body inside few cubes of 5x5x5: one needs more slots than the largest
    # setting's number, and fits the kernel's capacity.
    case = B.Case(B.case_params("cfg2", lattice=(5, 5, 5), cube_size=0.2,
                                sphere_center=(0.5, 0.5, 0.5), sphere_diameter=0.25))
    e = B.Engine(0)
    try:
        stats = []
        for limit in (None, 0, 1536):
            if limit is not None:
                e.set_ghost_lds_limit(limit)
            e.load_case(case)
            stats.append(e.ghost_stats())
        shipped, memory, restored = stats
        assert memory["levels"] > shipped["levels"]
        assert restored == shipped
        for bad in (-1, 1537):
            with pytest.raises(B.BCMError, match="slot limit"):
                e.set_ghost_lds_limit(bad)
    finally:
        e.close()
