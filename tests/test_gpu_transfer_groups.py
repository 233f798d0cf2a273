"""The p-MG transfers over element counts around their group sizes (up to 32 elements per
workgroup; a group past the end repeats its last element), with and without an element
list and weights, for fine and coarse degrees across the range, against the tensor product
in FP64. Three contractions of at most 16 terms round 3 * 16 products: 48 * 2^-53 of the
sum of magnitudes in FP64, 48 * 2^-24 in FP32 (with P and the inputs rounded to FP32
first), plus one rounding for the weight."""
import numpy as np
import pytest
import torch

import libparanumal_amd as lp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nf,Nc", [(2, 1), (3, 1), (3, 2), (4, 2), (5, 4), (6, 4), (7, 3), (7, 5), (8, 1), (9, 6),
                                   (11, 10), (12, 9), (13, 7), (15, 11), (15, 14),
                                   # the 8 x 8 tile, and coarse lines of 5, 6, 7, 9, 12 and 13 in sixes
                                   (7, 1), (7, 2), (7, 4), (6, 5), (10, 6), (9, 8), (12, 11), (14, 12)])
def test_transfers_counts_and_lists(Nf, Nc):
    L = lp.lib()
    F, C = Nf + 1, Nc + 1
    rng = np.random.default_rng(100 * Nf + Nc)
    E = 67 if Nf <= 4 else 11
    nf, nc = E * F**3 // 2, E * C**3 // 2
    g2lf = rng.integers(-1, nf, E * F**3).astype(np.int32)
    g2lc = rng.integers(-1, nc, E * C**3).astype(np.int32)
    g2lf[:3] = -1
    P = rng.uniform(-1, 1, (F, C))
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    gf, gc = dev(g2lf), dev(g2lc)
    st = torch.cuda.current_stream().cuda_stream
    for dt, eps, s in ((np.float64, 2.0**-53, "f64"), (np.float32, 2.0**-24, "f32")):
        Pt, qf, qc, w = (a.astype(dt) for a in (P, rng.uniform(-1, 1, nf), rng.uniform(-1, 1, nc), rng.uniform(0.1, 1, nf)))
        Pd, qfd, qcd, wd = dev(Pt), dev(qf), dev(qc), dev(w)
        P64 = Pt.astype(np.float64)
        local = lambda q, g, n: np.where(g >= 0, q[np.maximum(g, 0)].astype(np.float64), 0.0).reshape(E, n, n, n)  # noqa: E731
        down = lambda q, A: np.einsum("ka,jb,ic,ekji->eabc", A, A, A, q, optimize=True)  # noqa: E731
        up = lambda q, A: np.einsum("ka,jb,ic,eabc->ekji", A, A, A, q, optimize=True)  # noqa: E731
        for n in sorted({1, 2, 3, 4, 5, 8, 9, E - 1, E} | ({31, 32, 33, 64, 65} if E > 65 else set())):
            for elements in (None, rng.permutation(E)[:n].astype(np.int32)):
                mine = np.arange(n) if elements is None else elements
                other = np.setdiff1d(np.arange(E), mine)
                lst = None if elements is None else dev(elements)
                ptr = None if lst is None else lst.data_ptr()
                for weighted in (False, True):
                    vals = qf.astype(np.float64) * w.astype(np.float64) if weighted else qf.astype(np.float64)
                    qL = local(vals, g2lf, F)
                    out = torch.full((E * C**3,), 5.0, dtype=Pd.dtype, device="cuda")
                    if weighted:
                        lp.check(getattr(L, "libp_mg_coarsen_weighted_hex_" + s)(
                            Nf, Nc, n, ptr, gf.data_ptr(), Pd.data_ptr(), wd.data_ptr(), qfd.data_ptr(), out.data_ptr(), st))
                    else:
                        lp.check(getattr(L, "libp_mg_coarsen_hex_" + s)(
                            Nf, Nc, n, ptr, gf.data_ptr(), Pd.data_ptr(), qfd.data_ptr(), out.data_ptr(), st))
                    torch.cuda.synchronize()
                    got = out.double().cpu().numpy().reshape(E, C, C, C)
                    err = np.abs(got - down(qL, P64))[mine]
                    assert np.all(err <= 50 * eps * down(np.abs(qL), np.abs(P64))[mine] + 1e-300), (s, n, weighted)
                    assert np.all(got[other] == 5.0)
                out = torch.full((E * F**3,), 5.0, dtype=Pd.dtype, device="cuda")
                lp.check(getattr(L, "libp_mg_prolong_hex_" + s)(Nf, Nc, n, ptr, gc.data_ptr(), Pd.data_ptr(),
                                                                qcd.data_ptr(), out.data_ptr(), st))
                torch.cuda.synchronize()
                got = out.double().cpu().numpy().reshape(E, F, F, F)
                qL = local(qc, g2lc, C)
                err = np.abs(got - up(qL, P64))[mine]
                assert np.all(err <= 50 * eps * up(np.abs(qL), np.abs(P64))[mine] + 1e-300), (s, n)
                assert np.all(got[other] == 5.0)
