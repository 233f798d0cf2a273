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


def element_ax(qL, wJ, ggeo, D, lam):
    """A_L q of element-local values [E][k][j][i], from the definition in FP64."""
    E, Nq = qL.shape[0], qL.shape[1]
    G = ggeo.reshape(E, 6, Nq, Nq, Nq)
    qr = np.einsum("im,ekjm->ekji", D, qL, optimize=True)
    qs = np.einsum("jm,ekmi->ekji", D, qL, optimize=True)
    qt = np.einsum("km,emji->ekji", D, qL, optimize=True)
    fr = G[:, 0] * qr + G[:, 1] * qs + G[:, 2] * qt
    fs = G[:, 1] * qr + G[:, 3] * qs + G[:, 4] * qt
    ft = G[:, 2] * qr + G[:, 4] * qs + G[:, 5] * qt
    return (np.einsum("mi,ekjm->ekji", D, fr, optimize=True) + np.einsum("mj,ekmi->ekji", D, fs, optimize=True) +
            np.einsum("mk,emji->ekji", D, ft, optimize=True) + lam * wJ.reshape(qL.shape) * qL)


@pytest.mark.parametrize("N", range(1, 16))
def test_ax_local_values_and_lambda_zero_forms(N):
    """The element-local form (a random E-vector, so copies of a node differ) for lambda 0 and
    not, with part of a group; and every form at lambda = 0 with a wJ full of NaN, which no
    form may read: the E-vector and p.Ap (N = 15: on the matrix cores), with and without a
    list, the split, and the matrix-core entry itself. The definition above is checked against
    the oracle first. Tolerances as above (1e-12 of the largest value)."""
    shape = (5, 3, 3) if N <= 4 else (3, 2, 1)
    o = OracleElliptic({"MESH FILE": "BOX", "MESH DIMENSION": 3, "ELEMENT TYPE": 12, "BOX NX": shape[0],
                        "BOX NY": shape[1], "BOX NZ": shape[2], "BOX DIMX": 2, "BOX DIMY": 2, "BOX DIMZ": 2,
                        "BOX BOUNDARY FLAG": 1, "POLYNOMIAL DEGREE": N, "BOX CURVED MAP AMPLITUDE": 0.05,
                        "LAMBDA": 0.7, "DATA FILE": "data/ellipticSine3D.h", "PRECONDITIONER": "JACOBI"})
    L = lp.lib()
    E, Np, Nq = o.geti("Nelements"), (N + 1) ** 3, N + 1
    rng = np.random.default_rng(200 + N)
    wJ, ggeo, D, g2l = (o.array(k) for k in ("wJ", "ggeo", "D", "GlobalToLocal"))
    D = D.reshape(Nq, Nq)
    q = rng.uniform(-1, 1, o.geti("Ngather"))
    full = np.where(g2l >= 0, q[np.maximum(g2l, 0)], 0.0).reshape(E, Nq, Nq, Nq)
    want = element_ax(full, wJ, ggeo, D, 0.7)
    assert np.max(np.abs(want.ravel() - o.partial_ax(q))) <= 1e-13 * np.max(np.abs(want))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    gd, wd, Dd, g2ld, qd = dev(ggeo), dev(wJ), dev(D), dev(g2l), dev(q)
    wnan = torch.full_like(wd, float("nan"))
    st = torch.cuda.current_stream().cuda_stream
    fresh = lambda n: torch.full((n,), 3.0, dtype=torch.float64, device="cuda")  # noqa: E731

    def check(out, ref, mine, what):
        torch.cuda.synchronize()
        got = out.cpu().numpy()[:E * Np].reshape(E, Nq, Nq, Nq)
        assert np.max(np.abs(got[mine] - ref[mine])) <= 1e-12 * np.max(np.abs(ref)), what
        assert np.all(got[np.setdiff1d(np.arange(E), mine)] == 3.0), what

    qL = rng.uniform(-1, 1, (E, Nq, Nq, Nq))
    qLd = dev(qL)
    for lam, w in ((0.7, wd), (0.0, wnan)):
        ref = element_ax(qL, wJ, ggeo, D, lam)
        for n in {1, E - 1, E}:
            out = fresh(E * Np)
            lp.check(L.libp_ax_hex_local_f64(N, n, w.data_ptr(), gd.data_ptr(), Dd.data_ptr(), lam, qLd.data_ptr(),
                                             out.data_ptr(), st))
            check(out, ref, np.arange(n), ("local", lam, n))

    ref = element_ax(full, wJ, ggeo, D, 0.0)
    geo = (g2ld.data_ptr(), wnan.data_ptr(), gd.data_ptr(), Dd.data_ptr())
    for elements in (None, rng.permutation(E)[:E - 1].astype(np.int32)):
        mine = np.arange(E) if elements is None else elements
        lst = None if elements is None else dev(elements)
        ptr, n = (None if lst is None else lst.data_ptr()), len(mine)
        out = fresh(E * Np)
        lp.check(L.libp_ax_hex_partial_f64(N, n, ptr, *geo, 0.0, qd.data_ptr(), out.data_ptr(), st))
        check(out, ref, mine, "E-vector")
        out, s = fresh(E * Np), torch.zeros(16, dtype=torch.float64, device="cuda")
        s[0] = 1.0
        part = torch.full((L.libp_ax_hex_split_blocks(N, n),), float("nan"), dtype=torch.float64, device="cuda")
        lp.check(L.libp_pcg_ax_hex_pap_f64(N, n, ptr, *geo, 0.0, qd.data_ptr(), out.data_ptr(), part.data_ptr(),
                                           s.data_ptr(), st))
        check(out, ref, mine, "p.Ap")
        products = full[mine] * ref[mine]
        assert abs(float(s[4]) - products.sum()) <= 1e-12 * np.abs(products).sum()
        if N == 15:
            out = fresh(E * Np)
            lp.check(L.libp_ax_hex_partial_mfma_n15(n, ptr, *geo, 0.0, qd.data_ptr(), out.data_ptr(), st))
            check(out, ref, mine, "matrix cores")
    if N <= 14:
        Nface = L.libp_ax_hex_face_nodes(N)
        y, face = fresh(q.size), fresh(E * Nface)
        lp.check(L.libp_ax_hex_split_f64(N, E, None, *geo, 0.0, qd.data_ptr(), y.data_ptr(), face.data_ptr(), None,
                                         None, st))
        torch.cuda.synchronize()
        ix = np.arange(Nq)
        inner = np.zeros((Nq, Nq, Nq), bool)
        inner[np.ix_(ix[1:-1], ix[1:-1], ix[1:-1])] = True
        got = face.cpu().numpy().reshape(E, Nface)
        tol = 1e-12 * np.max(np.abs(ref))
        assert np.max(np.abs(got - ref[:, ~inner])) <= tol
        if inner.any():
            rows = g2l.reshape(E, Nq, Nq, Nq)[:, inner]
            assert np.max(np.abs(y.cpu().numpy()[rows] - ref[:, inner])) <= tol
