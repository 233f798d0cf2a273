"""The single-reduction coarse iteration on the assembled operator at the row counts where its
block size changes (256 threads to 8192 rows, 512 to 16,384, 1024 above: 23^3 = 12,167 rows and
20^3, 21^3, 25^3, 26^3 around the two lines), against its element form, as in
test_coarse_assembled_matches_element_form: with a fixed count of coarse iterations the p-MG
solves agree to rounding, and repeated solves are bit-identical."""
import numpy as np
import pytest

import libparanumal_amd as lp
from tests.test_gpu_parity import mg_settings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [21, 22, 24, 26, 27])
def test_coarse_block_sizes(n):
    base = mg_settings("FP32", **{"LINEAR SOLVER STOPPING CRITERION": "RELATIVE", "MULTIGRID COARSE TOLERANCE": 0.0,
                                  "MULTIGRID COARSE MAXIT": 40, "BOX NX": n, "BOX NY": n, "BOX NZ": n,
                                  "POLYNOMIAL DEGREE": 2, "MULTIGRID DEGREES": "2,1"})
    elem = lp.Elliptic(dict(base, **{"MULTIGRID COARSE ASSEMBLED": "FALSE"}))
    asm = lp.Elliptic(dict(base, **{"MULTIGRID COARSE ASSEMBLED": "TRUE"}))
    a = elem.run()
    runs = [asm.run() for _ in range(3)]
    b = runs[0]
    assert all(r["norm"] == b["norm"] and r["iterations"] == b["iterations"] for r in runs)
    assert a["iterations"] == b["iterations"]
    assert asm.geti("coarseIterations") == elem.geti("coarseIterations") == 40
    x1, x3 = asm.solution(), elem.solution()
    assert np.max(np.abs(x1 - x3)) <= 1e-9 * np.max(np.abs(x3))
    elem.close()
    asm.close()
