"""GPU test of state downloads around the size where they go through pinned
chunks on several host threads (16 MB: 52 | 53 cubes of 320 kB; whole and
partial last chunks): what was uploaded comes back bitwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncubes", [1, 52, 53, 64, 131])
def test_download_returns_the_upload(B, ncubes):
    case = B.Case(B.case_params("tiny", lattice=(ncubes, 1, 1), cube_size=1.0 / ncubes,
                                sphere_diameter=0.0))
    rng = np.random.default_rng(ncubes)
    a = rng.uniform(-1.0, 1.0, size=(case.ncube, 20, 20, 20, 5))
    a[0] = 0.0
    e = B.Engine(0)
    try:
        e.load_case(case)
        for rep in range(2):
            for name in ("U1_", "U1q"):
                e.set_state(name, a)
                assert np.array_equal(e.get_state(name), a), (name, rep)
                assert np.array_equal(e.case_state(0, name), a), (name, rep)
            a[1:] = -a[1:][::-1]
    finally:
        e.close()
