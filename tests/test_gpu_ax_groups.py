"""The partial Ax over element counts around its group sizes.

A workgroup of the Ax kernel takes a group of elements (up to 64 at N = 1) and a
group past the end repeats its last element: counts of 1, one less and one more
than a group, with and without an element list, must give each listed element's
oracle value, leave every other element untouched, and count each element once in
p.Ap. FP64 rounds about 6 (N+1) products per node of size up to max|A_L q|:
6 * 16 * 2^-53 = 1.1e-14, far inside 1e-12; in FP32 the same count of 2^-24 gives
6e-6, the bound 2e-5 with the FP32 copies of the factors.
"""
import numpy as np
import pytest
import torch

import libparanumal_amd as lp
from tests.oracle_lib import OracleElliptic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 13, 14, 15])
def test_ax_counts_and_lists(N):
    shape = (5, 4, 4) if N <= 4 else (3, 2, 1)
    o = OracleElliptic({"MESH FILE": "BOX", "MESH DIMENSION": 3, "ELEMENT TYPE": 12, "BOX NX": shape[0],
                        "BOX NY": shape[1], "BOX NZ": shape[2], "BOX DIMX": 2, "BOX DIMY": 2, "BOX DIMZ": 2,
                        "BOX BOUNDARY FLAG": 1, "POLYNOMIAL DEGREE": N, "BOX CURVED MAP AMPLITUDE": 0.05,
                        "LAMBDA": 0.7, "DATA FILE": "data/ellipticSine3D.h", "PRECONDITIONER": "JACOBI"})
    L = lp.lib()
    E, Np = o.geti("Nelements"), (N + 1) ** 3
    q = np.random.default_rng(N).uniform(-1, 1, o.geti("Ngather"))
    ref = o.partial_ax(q).reshape(E, Np)
    g2lh = o.array("GlobalToLocal")
    qL = np.where(g2lh >= 0, q[np.maximum(g2lh, 0)], 0.0).reshape(E, Np)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    g2l, qd = dev(g2lh), dev(q)
    geo = [dev(o.array(k)) for k in ("wJ", "ggeo", "D")]
    geo32, q32 = [a.float() for a in geo], qd.float()
    st = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(50 + N)
    for n in sorted({1, 2, 3, E - 1, E} | ({7, 8, 9, 31, 33, 63, 64, 65} if E > 65 else {4, 5})):
        for elements in (None, rng.permutation(E)[:n].astype(np.int32)):
            mine = np.arange(n) if elements is None else elements
            other = np.setdiff1d(np.arange(E), mine)
            lst = None if elements is None else dev(elements)
            ptr = None if lst is None else lst.data_ptr()
            for geom, vec, fn, tol in ((geo, qd, L.libp_ax_hex_partial_f64, 1e-12),
                                       (geo32, q32, L.libp_ax_hex_partial_f32, 2e-5)):
                out = torch.full((E * Np,), 3.0, dtype=vec.dtype, device="cuda")
                lp.check(fn(N, n, ptr, g2l.data_ptr(), *[a.data_ptr() for a in geom], 0.7, vec.data_ptr(),
                            out.data_ptr(), st))
                torch.cuda.synchronize()
                got = out.double().cpu().numpy().reshape(E, Np)
                assert np.max(np.abs(got[mine] - ref[mine])) <= tol * np.max(np.abs(ref)), (n, elements is None)
                assert np.all(got[other] == 3.0)
            out = torch.full((E * Np,), 3.0, dtype=torch.float64, device="cuda")
            part = torch.full((L.libp_ax_hex_split_blocks(N, n),), float("nan"), dtype=torch.float64, device="cuda")
            s = torch.zeros(16, dtype=torch.float64, device="cuda")
            s[0] = 1.0
            lp.check(L.libp_pcg_ax_hex_pap_f64(N, n, ptr, g2l.data_ptr(), *[a.data_ptr() for a in geo], 0.7,
                                               qd.data_ptr(), out.data_ptr(), part.data_ptr(), s.data_ptr(), st))
            torch.cuda.synchronize()
            pap = float(np.sum(qL[mine] * ref[mine]))
            assert abs(float(s[4]) - pap) <= 1e-12 * np.sum(np.abs(qL[mine] * ref[mine])), (n, elements is None)
