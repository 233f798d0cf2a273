"""The three-launch Jacobi-PCG iteration (libp_pcg_jacobi_iteration_f64) against the
separate calls, bit for bit: p, x, r, z and the scalars after every iteration, over element
counts that give one, a few and many partial sums, up to the iteration that meets the
tolerance and past it (nothing may change after STOP)."""
import ctypes

import numpy as np
import pytest
import torch

import libparanumal_amd as lp
from tests.oracle_lib import OracleElliptic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,shape", [(1, (9, 8, 10)), (2, (2, 2, 2)), (4, (3, 4, 5)), (4, (16, 16, 16)), (7, (5, 3, 2)),
                                     (9, (3, 2, 2)), (15, (2, 1, 1))])
def test_folded_iteration_matches_separate_calls(N, shape):
    L = lp.lib()
    s = {"MESH FILE": "BOX", "MESH DIMENSION": 3, "ELEMENT TYPE": 12, "BOX NX": shape[0], "BOX NY": shape[1],
         "BOX NZ": shape[2], "BOX DIMX": 2, "BOX DIMY": 2, "BOX DIMZ": 2, "BOX BOUNDARY FLAG": 1,
         "POLYNOMIAL DEGREE": N, "LAMBDA": 1, "BOX CURVED MAP AMPLITUDE": 0.05, "DATA FILE": "data/ellipticSine3D.h",
         "PRECONDITIONER": "JACOBI"}
    el = lp.Elliptic(s)
    E, Ng, NL = el.geti("Nelements"), el.geti("Ngather"), el.geti("Nelements") * el.geti("Np")
    assert L.libp_pcg_jacobi_iteration_folds(N, E, Ng) == 1
    P = {k: el.array_info(k)[0] for k in ("GlobalToLocal", "wJ", "ggeo", "D", "rowStartsT", "colIdsT", "invDiag")}
    st = torch.cuda.current_stream().cuda_stream
    new = lambda n: torch.zeros(n, dtype=torch.float64, device="cuda")  # noqa: E731
    r0 = torch.from_numpy(np.random.default_rng(N).uniform(-1, 1, Ng)).cuda()
    ws = torch.zeros(L.libp_reduce_ws_bytes(), dtype=torch.uint8, device="cuda")
    tol = 0.05 * float(r0 @ r0)  # met within a few iterations
    sets = []
    for _ in range(2):
        sets.append(dict(p=new(Ng), x=new(Ng), r=r0.clone(), z=new(Ng), AqL=new(NL),
                         pap=new(L.libp_ax_hex_split_blocks(N, E)), part=new(L.libp_pcg_gather_jacobi_partials(Ng))))
    a, b = sets
    sa, sb = new(16), new(32)
    sa[7] = tol
    sb[16 + 7] = tol
    for t, sc in ((a, sa.data_ptr()), (b, sb.data_ptr() + 16 * 8)):
        lp.check(L.libp_pcg_jacobi_rdotz_f64(Ng, P["invDiag"], t["r"].data_ptr(), t["z"].data_ptr(), t["p"].data_ptr(), 0,
                                             sc, ws.data_ptr(), st))
    host = torch.zeros(16, dtype=torch.float64).pin_memory()
    dptr = ctypes.c_void_p()
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipHostGetDevicePointer(ctypes.byref(dptr), ctypes.c_void_p(host.data_ptr()), 0) == 0
    stopped = 0
    for it in range(60):
        lp.check(L.libp_pcg_update_p_f64(Ng, int(it == 0), a["z"].data_ptr(), a["p"].data_ptr(), sa.data_ptr(), st))
        lp.check(L.libp_pcg_ax_hex_pap_f64(N, E, None, P["GlobalToLocal"], P["wJ"], P["ggeo"], P["D"], 1.0,
                                           a["p"].data_ptr(), a["AqL"].data_ptr(), a["pap"].data_ptr(), sa.data_ptr(),
                                           st))
        lp.check(L.libp_pcg_gather_jacobi_update_f64(Ng, P["rowStartsT"], P["colIdsT"], a["AqL"].data_ptr(),
                                                     P["invDiag"], a["p"].data_ptr(), a["x"].data_ptr(),
                                                     a["r"].data_ptr(), a["z"].data_ptr(), sa.data_ptr(),
                                                     a["part"].data_ptr(), st))
        lp.check(L.libp_pcg_jacobi_iteration_f64(N, E, None, P["GlobalToLocal"], P["wJ"], P["ggeo"], P["D"], 1.0, Ng,
                                                 P["rowStartsT"], P["colIdsT"], P["invDiag"], it, b["p"].data_ptr(),
                                                 b["AqL"].data_ptr(), b["x"].data_ptr(), b["r"].data_ptr(),
                                                 b["z"].data_ptr(), b["pap"].data_ptr(), b["part"].data_ptr(),
                                                 sb.data_ptr(), st))
        lp.check(L.libp_pcg_jacobi_iteration_check_f64(Ng, it, sb.data_ptr(), b["part"].data_ptr(), dptr, st))
        torch.cuda.synchronize()
        for k in ("p", "x", "r", "z"):
            assert torch.equal(a[k], b[k]), (it, k)
        h, ref = host.numpy(), sa.cpu().numpy()
        assert [h[i] for i in (0, 5, 7, 8, 9)] == [ref[i] for i in (0, 5, 7, 8, 9)], it
        stopped += int(ref[8] != 0)
        if stopped == 3:
            break
    assert stopped == 3, "the tolerance was not met"
    el.close()


def test_folded_iteration_refuses_large_problems():
    L = lp.lib()
    assert L.libp_pcg_jacobi_iteration_folds(7, 48**3, 37595375) == 0
    assert L.libp_pcg_jacobi_iteration_folds(4, 512, 1024 * 512) == 1
    assert L.libp_pcg_jacobi_iteration_folds(4, 512, 1024 * 512 + 1) == 0
    ptr = ctypes.c_void_p(256)
    assert L.libp_pcg_jacobi_iteration_f64(7, 48**3, None, *[ptr] * 4, 0.0, 37595375, *[ptr] * 3, 0, *[ptr] * 8, None) == 1


@pytest.mark.parametrize("maxit", [1, 3, 4, 5, 9, 400])
def test_folded_solve_iterations(maxit):
    """Whole solves, stopped by the tolerance or by the iteration limit anywhere in a chunk."""
    s = {"MESH FILE": "BOX", "MESH DIMENSION": 3, "ELEMENT TYPE": 12, "BOX NX": 4, "BOX NY": 5, "BOX NZ": 3,
         "BOX DIMX": 2, "BOX DIMY": 2, "BOX DIMZ": 2, "BOX BOUNDARY FLAG": 1, "POLYNOMIAL DEGREE": 4, "LAMBDA": 0,
         "DATA FILE": "data/ellipticSine3D.h", "LINEAR SOLVER": "PCG", "PRECONDITIONER": "JACOBI",
         "MAXIMUM ITERATIONS": maxit, "LINEAR SOLVER STOPPING CRITERION": "RELATIVE"}
    out = []
    for fused in ("TRUE", "FALSE"):
        el = lp.Elliptic(dict(s, **{"PCG FUSED OPERATOR": fused}))
        for _ in range(2):  # the second solve reuses the handle's buffers
            r = el.run()
        out.append((r["iterations"], el.solution(), r["r_final"]))
        el.close()
    assert out[0][0] == out[1][0] and (maxit > 100) == (out[0][0] < maxit)
    assert np.max(np.abs(out[0][1] - out[1][1])) <= 1e-10 * np.max(np.abs(out[1][1]))
    assert abs(out[0][2] - out[1][2]) <= 1e-6 * out[1][2]
