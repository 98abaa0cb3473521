"""GPU test that a HIP error left by an earlier call is reported, whatever
state download (direct or through pinned chunks) comes before the next call
that looks for one."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncubes", [1, 53])
def test_downloads_do_not_clear_a_pending_error(B, ncubes):
    case = B.Case(B.case_params("tiny", lattice=(ncubes, 1, 1), cube_size=1.0 / ncubes,
                                sphere_diameter=0.0))
    hip = ctypes.CDLL(B.LIB_PATH)   # (the runtime the library is linked with)
    e = B.Engine(0)
    try:
        e.load_case(case)
        e.sync()
        assert hip.hipSetDevice(1 << 20) != 0   # no such device: an error stays pending
        with pytest.raises(B.BCMError):
            e.get_state("U1")
            e.sync()
        e.sync()   # reported once
        assert np.array_equal(e.get_state("U1")[1:], case.array("U1")[1:])
    finally:
        e.close()
