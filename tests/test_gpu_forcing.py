"""The Fourier forcing against extended precision: nodes at integers and half integers (the
ends of the sine's reduction), far from zero, and one to several workgroups. A mode's
argument in half turns is three products, three sums and the phase over pi: five roundings
of at most |t|, pi |t| 5 * 2^-53 in the sine; the series and the products add 8 * 2^-53;
summing 64 modes rounds each partial sum once."""
import numpy as np
import pytest
import torch

import libparanumal_amd as lp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,Np,scale", [(1, 8, 1.0), (3, 125, 1.0), (70, 512, 1.0), (5, 64, 1e4)])
def test_fourier_forcing(E, Np, scale):
    rng = np.random.default_rng(E + Np)
    NL = E * Np
    x, y, z = (rng.uniform(-1, 1, NL) * scale for _ in range(3))
    x[: NL // 2], y[: NL // 2], z[: NL // 2] = (np.round(2 * a[: NL // 2]) / 2 for a in (x, y, z))
    w = rng.uniform(0.1, 1, NL)
    c = np.concatenate([rng.integers(1, 9, (64, 3)), rng.uniform(-1, 1, (64, 1)), rng.uniform(0, 2 * np.pi, (64, 1))], 1)
    c[::2, 4] = 0.0
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    X, Y, Z, W, Cd = (dev(a) for a in (x, y, z, w, c))
    mapB = torch.zeros(NL, dtype=torch.int32, device="cuda")
    out = torch.full((NL + 1,), 5.0, dtype=torch.float64, device="cuda")
    lp.check(lp.lib().libp_rhs_hex_f64(E, Np, 1, Cd.data_ptr(), X.data_ptr(), Y.data_ptr(), Z.data_ptr(), W.data_ptr(),
                                       1.0, mapB.data_ptr(), out.data_ptr(), None,
                                       torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    ld = np.longdouble
    pi = ld("3.14159265358979323846264338327950288")
    ref, bound, eps = np.zeros(NL, ld), np.zeros(NL), 2.0**-53
    for kx, ky, kz, amp, phase in c:
        t = ld(kx) * x.astype(ld) + ld(ky) * y.astype(ld) + ld(kz) * z.astype(ld)
        t -= 2 * np.round(t / 2)  # whole turns, exact
        ref += ld(amp) * np.sin(pi * t + ld(phase))
        size = kx * np.abs(x) + ky * np.abs(y) + kz * np.abs(z) + phase / np.pi
        bound += np.abs(amp) * (np.pi * 5 * size + 8 + 64) * eps
    got = out.cpu().numpy()
    assert np.all(np.abs(got[:NL].astype(ld) - ref * w.astype(ld)) <= bound * w)
    assert got[NL] == 5.0
