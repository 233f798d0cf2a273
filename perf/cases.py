"""The work that users of this framework have it do, as measurable cases.

A case is a dict of plain values; `kind` names the entry point it takes:

- operator:  Elliptic.operator, the C0 operator A q on a hex box. It is what a
             caller with a solver of its own calls, and the inside of every solve.
- smooth:    one Chebyshev-Jacobi smoothing (degree 2, x not zero) of the finest
             p-multigrid level, Elliptic.mg_level_op(0, MG_SMOOTH).
- transfer:  the restriction and the prolongation between the two finest
             p-multigrid levels (MG_COARSEN, then x += P e by MG_PROLONGATE).
- vcycle:    Elliptic.precon, a whole p-multigrid V-cycle with the AMG base level
             (a fixed linear map; the Jacobi-PCG base level runs in `solve`).
- solve:     Elliptic.run and Elliptic.solution, a whole solve to 1e-8: PCG with
             Jacobi, or flexible PCG with p-multigrid.
- learned:   Elliptic.learned_correction, the linear learned smoother at N=7.
- mlp:       the forward and backward layers of the smoother's 896-256-256-512
             network (libp_mlp_linear_*), the products of one training step.

The sizes are the framework's own workloads (8^3 at N=4, 48^3 and 32^3 at N=7,
16^3 at N=15) and generic ragged ones. Vectors are uniform in [-1, 1], as in
power iterations and tests; the solves take the 64-mode smooth random forcing.

`exact` rebuilds the mesh, the operator and the smoothers in torch FP64 from
their definitions, without the library.
"""
import ctypes
import math
import os

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LINEAR_WEIGHTS = os.path.join(ROOT, "libparanumal_amd", "weights", "learned_hex_n7_linear.bin")
MLP_WIDTHS = (896, 256, 256, 512)  # 512 element values + 6 x 64 neighbour values, hidden, hidden, 512


def listed():
    return [
        # the smallest operator: 29,791 dofs, where launches and latency count
        box("op_n4_8", "operator", 4, 8, 8, 8, lam=0.0),
        # a low degree on a ragged screened box, the coarse meshes of many users
        box("op_n2_ragged", "operator", 2, 61, 47, 53, lam=1.0, curve=0.05, bc=2),
        # a degree whose element is no multiple of a wavefront, ragged box
        box("op_n10_ragged", "operator", 10, 19, 23, 17, lam=1.0, curve=0.05),
        # the largest: the framework's headline mesh, Poisson
        box("op_n7_48", "operator", 7, 48, 48, 48, lam=0.0),
        # the highest degree, curved and screened
        box("op_n15_16", "operator", 15, 16, 16, 16, lam=1.0, curve=0.05),
        # the fine smoother of the FP32 p-multigrid solves
        box("smooth_n7_32_f32", "smooth", 7, 32, 32, 32, lam=1.0, curve=0.05, bits=32),
        # a level pair of the default (halved dofs) schedule: 6 -> 4
        box("transfer_n6_f32", "transfer", 6, 29, 31, 27, lam=1.0, bits=32),
        # a whole preconditioner application as an outside Krylov method calls it
        box("vcycle_n7_32_f32", "vcycle", 7, 32, 32, 32, lam=1.0, curve=0.05, bits=32, degrees="7,3,1"),
        # the smallest whole call: the Jacobi-PCG solve of the 8^3 box
        box("solve_pcg_n4_8", "solve", 4, 8, 8, 8, lam=0.0, precon="JACOBI"),
        # a whole p-multigrid solve of ordinary size
        box("solve_pmg_n7", "solve", 7, 18, 20, 16, lam=1.0, curve=0.05, precon="MULTIGRID", bits=32, degrees="7,3,1"),
        # one application of the linear learned smoother on the mesh it was fitted on
        box("learned_n7_32", "learned", 7, 32, 32, 32, lam=0.0, curve=0.05, bits=32, degrees="7,3,1"),
        # the network's training products over the elements of the 32^3 box
        {"name": "mlp_32768", "kind": "mlp", "M": 32768},
    ]


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["operator"] * 5 + ["smooth", "transfer", "vcycle", "solve", "solve", "learned", "mlp"])
    if kind == "mlp":
        return {"kind": "mlp", "M": round(math.exp(rng.uniform(math.log(500), math.log(32768))))}
    lam = rng.choice([0.0, 1.0])
    bc = 1 if lam == 0.0 else rng.choice([1, 2])
    curve = rng.choice([0.0, 0.05])
    small, large = 2e4, {"operator": 16e6, "solve": 1.2e6}.get(kind, 8e6)  # local nodes
    N = {"operator": rng.randint(1, 15), "learned": 7, "solve": rng.randint(2, 8)}.get(kind, rng.randint(3, 9))
    nodes = math.exp(rng.uniform(math.log(small), math.log(large)))
    side = (nodes / (N + 1) ** 3) ** (1 / 3)
    nx, ny, nz = (max(4 if curve else 2, round(side * rng.uniform(0.8, 1.25))) for _ in range(3))
    bits = 32 if kind in ("vcycle", "solve", "learned") else rng.choice([32, 64])
    precon = rng.choice(["JACOBI", "MULTIGRID"]) if kind == "solve" else ""
    return box(None, kind, N, nx, ny, nz, lam, curve, bc, bits=64 if kind == "operator" else bits, precon=precon)


def box(name, kind, N, nx, ny, nz, lam, curve=0.0, bc=1, bits=64, precon="", degrees=""):
    """bc: 1 Dirichlet, 2 Neumann; degrees "" is the default schedule (halved dofs)."""
    c = {"kind": kind, "N": N, "nx": nx, "ny": ny, "nz": nz, "lam": lam, "curve": curve, "bc": bc, "bits": bits,
         "precon": precon, "degrees": degrees}
    return dict(c, name=name) if name else c


# ------------------------------ the framework's side ------------------------------

def settings(case, seed):
    kind = case["kind"]
    s = {"MESH FILE": "BOX", "MESH DIMENSION": 3, "ELEMENT TYPE": 12, "BOX NX": case["nx"], "BOX NY": case["ny"],
         "BOX NZ": case["nz"], "BOX DIMX": 2, "BOX DIMY": 2, "BOX DIMZ": 2, "BOX BOUNDARY FLAG": case["bc"],
         "POLYNOMIAL DEGREE": case["N"], "LAMBDA": case["lam"], "DISCRETIZATION": "CONTINUOUS",
         "DATA FILE": "ellipticFourier3D", "DATA SEED": 1 + seed % 1000003, "LINEAR SOLVER": "PCG",
         "LINEAR SOLVER STOPPING CRITERION": "RELATIVE", "LINEAR SOLVER TOLERANCE": 1e-8, "PRECONDITIONER": "JACOBI"}
    if case["curve"]:
        s["BOX CURVED MAP AMPLITUDE"] = case["curve"]
    if kind in ("smooth", "transfer", "vcycle", "learned") or case["precon"] == "MULTIGRID":
        s.update({"PRECONDITIONER": "MULTIGRID", "LINEAR SOLVER": "FPCG", "MULTIGRID PRECISION": f"FP{case['bits']}"})
        if case["degrees"]:
            s.update({"MULTIGRID COARSENING": "CUSTOM", "MULTIGRID DEGREES": case["degrees"]})
        if kind == "vcycle":
            s["MULTIGRID COARSE SOLVER"] = "AMG"
        if kind == "learned":
            s.update({"MULTIGRID SMOOTHER": "LEARNED", "MULTIGRID LEARNED ARCH": "LINEAR",
                      "MULTIGRID LEARNED WEIGHTS": LINEAR_WEIGHTS})
    return s


def vector(n, seed, dtype=torch.float64):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.rand(n, dtype=torch.float64, device="cuda", generator=g).mul_(2).sub_(1).to(dtype)


def mlp_inputs(case, seed):
    """Weights, biases, unit-variance inputs and an output gradient of a converged net's size, in BF16."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    normal = lambda *shape: torch.randn(*shape, device="cuda", generator=g)  # noqa: E731
    W = [(normal(o, i) * math.sqrt(2.0 / i)).bfloat16() for i, o in zip(MLP_WIDTHS, MLP_WIDTHS[1:])]
    b = [normal(o) * 0.1 for o in MLP_WIDTHS[1:]]
    return W, b, normal(case["M"], MLP_WIDTHS[0]).bfloat16(), (normal(case["M"], MLP_WIDTHS[-1]) * 1e-3).bfloat16()


def prepare(case, seed):
    import libparanumal_amd as lp
    kind = case["kind"]
    if kind == "mlp":
        W, b, X, dY = mlp_inputs(case, seed)
        M, (_, H, _, O) = case["M"], MLP_WIDTHS
        new = lambda *shape, t=torch.bfloat16: torch.empty(*shape, dtype=t, device="cuda")  # noqa: E731
        ws = max(lp.lib().libp_mlp_ws_bytes(M, i, o) for i, o in zip(MLP_WIDTHS, MLP_WIDTHS[1:]))
        return {"case": case, "lp": lp, "W": W, "b": b, "X": X, "dY": dY, "H": [new(M, H), new(M, H)],
                "Y": new(M, O, t=torch.float32), "dH": [new(M, H), new(M, H)],
                "dW": [torch.empty_like(w, dtype=torch.float32) for w in W], "db": [torch.empty_like(v) for v in b],
                "ws": new(ws, t=torch.uint8)}
    el = lp.Elliptic(settings(case, seed))
    st = {"case": case, "el": el}
    n = el.geti("Ngather")
    if kind in ("operator", "vcycle"):
        st.update(q=vector(n, seed), y=torch.zeros(n, dtype=torch.float64, device="cuda"))
    elif kind == "smooth":
        dt = torch.float32 if case["bits"] == 32 else torch.float64
        st.update(r=vector(n, seed, dt), x0=vector(n, seed + 1, dt))
        st.update(x=st["x0"].clone())
    elif kind == "transfer":
        dt = torch.float32 if case["bits"] == 32 else torch.float64
        nc, _ = el.mg_level_ndofs(1)
        st.update(r=vector(n, seed, dt), e=vector(nc, seed + 1, dt), x0=vector(n, seed + 2, dt))
        st.update(x=st["x0"].clone(), rc=torch.zeros(nc, dtype=dt, device="cuda"))
    elif kind == "learned":
        st.update(q=vector(n, seed, torch.float32), y=torch.zeros(n, dtype=torch.float32, device="cuda"))
    if kind in ("smooth", "transfer"):
        st["stream"] = torch.cuda.ExternalStream(el.stream)
    torch.cuda.synchronize()
    return st


def run(st):
    kind = st["case"]["kind"]
    if kind == "mlp":
        return run_mlp(st)
    el = st["el"]
    if kind == "operator":
        el.operator(st["q"], st["y"])
        return st["y"]
    if kind == "vcycle":
        el.precon(st["q"], st["y"])
        return st["y"]
    if kind == "learned":
        el.learned_correction(st["q"], st["y"])
        return st["y"]
    if kind == "solve":
        el.run()
        return el.solution()
    # smooth and transfer update x in place: each pass starts from the same x0
    with torch.cuda.stream(st["stream"]):
        st["x"].copy_(st["x0"])
    if kind == "smooth":
        el.mg_level_op(0, el.MG_SMOOTH, st["r"], st["x"], 0)
        return st["x"]
    el.mg_level_op(0, el.MG_COARSEN, st["r"], st["rc"])
    el.mg_level_op(0, el.MG_PROLONGATE, st["e"], st["x"])
    return st["rc"], st["x"]


def run_mlp(st):
    L, check, M = st["lp"].lib(), st["lp"].check, st["case"]["M"]
    W, b, H, dH, dW, db = st["W"], st["b"], st["H"], st["dH"], st["dW"], st["db"]
    X, Y, dY, ws = st["X"], st["Y"], st["dY"], st["ws"].data_ptr()
    stream = torch.cuda.current_stream().cuda_stream
    for x, w, v, y, relu in ((X, W[0], b[0], H[0], 1), (H[0], W[1], b[1], H[1], 1), (H[1], W[2], b[2], Y, 0)):
        o, i = w.shape
        check(L.libp_mlp_linear_fwd(M, i, o, x.data_ptr(), i, w.data_ptr(), i, v.data_ptr(), relu, y.data_ptr(), o,
                                    stream), "fwd")
    for k, x, d in ((2, H[1], dY), (1, H[0], dH[1]), (0, X, dH[0])):
        o, i = W[k].shape
        check(L.libp_mlp_linear_bwd_weight(M, i, o, d.data_ptr(), o, x.data_ptr(), i, dW[k].data_ptr(),
                                           db[k].data_ptr(), ws, stream), "bwd_weight")
        if k:
            check(L.libp_mlp_linear_bwd_data(M, i, o, d.data_ptr(), o, W[k].data_ptr(), i, x.data_ptr(), i,
                                             dH[k - 1].data_ptr(), i, stream), "bwd_data")
    return [Y] + dW + db


# ---------------------------------- what it takes ----------------------------------

def degrees(case):
    """The p-multigrid degrees: the given ones, or from N the largest degree with at most half the nodes, and so on."""
    if case["degrees"]:
        return [int(d) for d in case["degrees"].split(",")]
    out = [case["N"]]
    while out[-1] > 1:
        n = out[-1]
        m = n - 1
        while m > 1 and (m + 1) ** 3 > (n + 1) ** 3 // 2:
            m -= 1
        out.append(m)
    return out


def counts(case, N=None):
    """(elements, local nodes, gathered dofs)"""
    N = N or case["N"]
    E = case["nx"] * case["ny"] * case["nz"]
    off = -1 if case["bc"] == 1 else 1
    return E, E * (N + 1) ** 3, math.prod(N * case[d] + off for d in ("nx", "ny", "nz"))


def operator_work(case, width, N=None):
    N = N or case["N"]
    _, NL, n = counts(case, N)
    return ((6 + (case["lam"] != 0)) * width + 4) * NL + 2 * width * n, NL * (12 * (N + 1) + 18)


def smoothing_work(case, width, N, applications):
    """A Chebyshev smoothing: its operator applications, then invDiag, r, x in and x out once."""
    by, fl = operator_work(case, width, N)
    n = counts(case, N)[2]
    return applications * by + 4 * width * n, applications * (fl + 6 * n)


def transfer_work(case, width, Nf, Nc):
    """Restriction (r, multiplicities in, coarse r out) and prolongation (e in, x in and out), with their maps."""
    _, Lf, nf = counts(case, Nf)
    _, Lc, nc = counts(case, Nc)
    F, C = Nf + 1, Nc + 1
    sweeps = 2 * (F * F * F * C + F * F * C * C + F * C * C * C) * (Lf // F ** 3)
    return width * (4 * nf + 2 * nc) + 8 * (Lf + Lc), 2 * sweeps


def cycle_work(case, width):
    deg, by, fl = degrees(case), 0, 0
    for Nf, Nc in zip(deg, deg[1:]):
        # two applications before, the residual, three after
        for b, f in (smoothing_work(case, width, Nf, 6), transfer_work(case, width, Nf, Nc)):
            by, fl = by + b, fl + f
    return by, fl


def work(case):
    kind, width = case["kind"], case.get("bits", 64) // 8
    if kind == "mlp":
        M, pairs = case["M"], list(zip(MLP_WIDTHS, MLP_WIDTHS[1:]))
        fl = 2 * M * (2 * sum(i * o for i, o in pairs) + sum(i * o for i, o in pairs[1:]))
        i, h, _, o = MLP_WIDTHS
        return {"bytes": M * (2 * i + 4 * o + 2 * o) + sum(8 * a * c for a, c in pairs), "flops": fl}
    _, NL, n = counts(case)
    if kind == "operator":
        by, fl = operator_work(case, 8)
    elif kind == "smooth":
        by, fl = smoothing_work(case, width, case["N"], 3)
    elif kind == "transfer":
        by, fl = transfer_work(case, width, *degrees(case)[:2])
    elif kind == "vcycle":
        by, fl = cycle_work(case, width)
    elif kind == "learned":
        # the residual, invDiag, correction, both maps and the weights; 896 x 512 products per element
        E = counts(case)[0]
        by, fl = 12 * n + 4 * (512 + 384) * E + 2 * 896 * 512, 2 * 896 * 512 * E
    else:
        # the iterations of the solve: about 9 with p-multigrid, and with Jacobi what the condition number of
        # degree N on elements of width h asks for; each an operator and the four vectors p, x, r, z
        b, f = operator_work(case, 8)
        if case["precon"] == "MULTIGRID":
            vb, vf = cycle_work(case, width)
            by, fl = 9 * (b + vb + 64 * n), 9 * (f + vf + 12 * n)
        else:
            its = 3 * case["N"] ** 1.5 * max(case["nx"], case["ny"], case["nz"]) ** 0.5
            by, fl = its * (b + 64 * n), its * (f + 12 * n)
        by += 8 * NL
    return {"bytes": int(by), "flops": int(fl)}


def tolerance(case):
    """What another order of sums at the same precision shows, about four times over."""
    kind = case["kind"]
    if kind == "mlp":  # 1.4e-3 in the hidden layers' gradients, from BF16 roundings that fall the other way
        return {"rel": 6e-3}
    if kind == "learned":  # 1.3e-3 from the BF16 inputs, some of which another RMS rounds the other way
        return {"rel": 2e-3}
    if kind == "solve":  # 6e-9 where the stopping rule, 1e-8 of the first residual, ends; an iteration more or less
        return {"rel": 1e-7}
    if kind == "operator" or case["bits"] == 64:  # 3.8e-13 at N=15
        return {"rel": 2e-12}
    return {"rel": 1e-6}  # FP32: 0.5e-7 to 2e-7


# ------------------------- the same in torch FP64, from the definitions -------------------------

def gll(N):
    """Gauss-Lobatto-Legendre nodes, weights and the derivative matrix D[i, m] = l'_m(r_i)."""
    from numpy.polynomial import legendre as leg
    PN = [0.0] * N + [1.0]
    r = np.concatenate([[-1.0], np.sort(np.real(leg.legroots(leg.legder(PN)))) if N > 1 else [], [1.0]])
    for _ in range(3):  # Newton on P'_N at the inner nodes
        r[1:-1] -= leg.legval(r[1:-1], leg.legder(PN)) / leg.legval(r[1:-1], leg.legder(PN, 2)) if N > 1 else 0.0
    p = leg.legval(r, PN)
    w = 2.0 / (N * (N + 1) * p * p)
    d = r[:, None] - r[None, :]
    np.fill_diagonal(d, 1.0)
    D = p[:, None] / p[None, :] / d
    np.fill_diagonal(D, 0.0)
    D[0, 0], D[N, N] = -N * (N + 1) / 4.0, N * (N + 1) / 4.0
    return r, w, D


def interpolation(rc, rf):
    """P[f, c] = l_c(rf): degree raising between two GLL node sets."""
    P = np.ones((len(rf), len(rc)))
    for c in range(len(rc)):
        for m in range(len(rc)):
            if m != c:
                P[:, c] *= (rf - rc[m]) / (rc[c] - rc[m])
    return P


def along(A, v, axis):
    """Contract A[out, in] with axis 1, 2 or 3 (t, s, r) of v[element, t, s, r]."""
    return torch.movedim(torch.movedim(v, axis, -1).contiguous() @ A.T.contiguous(), -1, axis)


class Box:
    """The C0 operator on the hex box [-1, 1]^3, in FP64."""

    def __init__(self, case, N=None):
        self.N = N = N or case["N"]
        self.nx, self.ny, self.nz, self.lam, self.curve = (case[k] for k in ("nx", "ny", "nz", "lam", "curve"))
        self.E, self.Nq = self.nx * self.ny * self.nz, N + 1
        r, w, D = gll(N)
        dev = lambda a: torch.tensor(a, dtype=torch.float64, device="cuda")  # noqa: E731
        self.r_host, self.r, self.w, self.D = r, dev(r), dev(w), dev(D)
        e = torch.arange(self.E, device="cuda")
        self.ex, self.ey, self.ez = e % self.nx, (e // self.nx) % self.ny, e // (self.nx * self.ny)
        line = torch.arange(N + 1, device="cuda")
        axis = lambda c, shape: (N * c[:, None] + line).view(self.E, *shape)  # noqa: E731
        X, Y, Z = axis(self.ex, (1, 1, N + 1)), axis(self.ey, (1, N + 1, 1)), axis(self.ez, (N + 1, 1, 1))
        gx, gy, gz = (N * n + 1 for n in (self.nx, self.ny, self.nz))
        gid = (X + gx * (Y + gy * Z)).reshape(-1)
        # rows in the order in which the elements first meet their nodes; Dirichlet nodes have none (-1)
        first = torch.full((gx * gy * gz,), gid.numel(), device="cuda")
        first.scatter_reduce_(0, gid, torch.arange(gid.numel(), device="cuda"), "amin")
        if case["bc"] == 1:
            inside = lambda n: torch.tensor([0] + [1] * (n - 2) + [0], device="cuda", dtype=torch.bool)  # noqa: E731
            keep = (inside(gz)[:, None, None] & inside(gy)[None, :, None] & inside(gx)[None, None, :]).reshape(-1)
        else:
            keep = torch.ones(gx * gy * gz, dtype=torch.bool, device="cuda")
        ids = torch.nonzero(keep).reshape(-1)
        ids = ids[torch.argsort(first[ids])]
        self.n = ids.numel()
        row = torch.full((gx * gy * gz,), -1, device="cuda")
        row[ids] = torch.arange(self.n, device="cuda")
        self.g2l = row[gid]
        self.local = torch.nonzero(self.g2l >= 0).reshape(-1)  # the local nodes that have a row, and their rows
        self.rows = self.g2l[self.local]
        self.mult = self.gather(torch.ones(self.E * self.Nq ** 3, dtype=torch.float64, device="cuda"))

    def scatter(self, q):
        return torch.where(self.g2l >= 0, q[self.g2l.clamp(min=0)], torch.zeros((), dtype=q.dtype, device="cuda"))

    def gather(self, v):
        return torch.zeros(self.n, dtype=v.dtype, device="cuda").index_add_(0, self.rows, v.reshape(-1)[self.local])

    def nodes(self, a=0, b=None):
        """Physical nodes of elements [a, b), each [element, t, s, r]."""
        b = self.E if b is None else b
        at = lambda c, n, shape: (-1 + 2.0 / n * (c[a:b, None] + 0.5 * (1 + self.r))).view(b - a, *shape)  # noqa: E731
        q = self.Nq
        x, y, z = at(self.ex, self.nx, (1, 1, q)), at(self.ey, self.ny, (1, q, 1)), at(self.ez, self.nz, (q, 1, 1))
        x, y, z = (v.expand(b - a, q, q, q) for v in (x, y, z))
        if self.curve:
            x = x + self.curve * torch.sin(2 * math.pi * y) * torch.sin(2 * math.pi * z)
        return x, y, z

    def factors(self, a, b):
        """J w times grad r_i . grad r_j (six of them), and J w."""
        c = [[along(self.D, v, 3), along(self.D, v, 2), along(self.D, v, 1)] for v in self.nodes(a, b)]
        cross = lambda i, j, k, l: c[i][j] * c[k][l] - c[i][l] * c[k][j]  # noqa: E731
        J = c[0][0] * cross(1, 1, 2, 2) - c[0][1] * cross(1, 0, 2, 2) + c[0][2] * cross(1, 0, 2, 1)
        grad = [[cross(1, 1, 2, 2), -cross(0, 1, 2, 2), cross(0, 1, 1, 2)],
                [-cross(1, 0, 2, 2), cross(0, 0, 2, 2), -cross(0, 0, 1, 2)],
                [cross(1, 0, 2, 1), -cross(0, 0, 2, 1), cross(0, 0, 1, 1)]]
        JW = J * self.w[:, None, None] * self.w[None, :, None] * self.w[None, None, :]
        s = JW / (J * J)
        dot = lambda i, j: s * (grad[i][0] * grad[j][0] + grad[i][1] * grad[j][1] + grad[i][2] * grad[j][2])  # noqa: E731
        return [dot(0, 0), dot(0, 1), dot(0, 2), dot(1, 1), dot(1, 2), dot(2, 2)], JW

    def chunks(self):
        step = max(1, 4_000_000 // self.Nq ** 3)
        return [(a, min(a + step, self.E)) for a in range(0, self.E, step)]

    def keep_factors(self):
        self.kept = {c: self.factors(*c) for c in self.chunks()}

    def operator(self, q):
        qL = self.scatter(q).view(self.E, self.Nq, self.Nq, self.Nq)
        out = torch.empty_like(qL)
        for a, b in self.chunks():
            G, JW = getattr(self, "kept", {}).get((a, b)) or self.factors(a, b)
            v = qL[a:b]
            r, s, t = along(self.D, v, 3), along(self.D, v, 2), along(self.D, v, 1)
            DT = self.D.T.contiguous()
            out[a:b] = (along(DT, G[0] * r + G[1] * s + G[2] * t, 3) + along(DT, G[1] * r + G[3] * s + G[4] * t, 2) +
                        along(DT, G[2] * r + G[4] * s + G[5] * t, 1) + self.lam * JW * v)
        return self.gather(out)

    def diagonal(self):
        out = torch.empty(self.E, self.Nq, self.Nq, self.Nq, dtype=torch.float64, device="cuda")
        D2, d = (self.D * self.D).T.contiguous(), torch.diagonal(self.D)
        dr, ds, dt = d[None, None, :], d[None, :, None], d[:, None, None]
        for a, b in self.chunks():
            G, JW = getattr(self, "kept", {}).get((a, b)) or self.factors(a, b)
            out[a:b] = (along(D2, G[0], 3) + along(D2, G[3], 2) + along(D2, G[5], 1) + self.lam * JW +
                        2 * (G[1] * dr * ds + G[2] * dr * dt + G[4] * ds * dt))
        return self.gather(out)


def drand48(n):
    """The first n values of drand48 after srand48(0)."""
    a, c, mask = 0x5DEECE66D, 0xB, (1 << 48) - 1
    block = 1 << 12
    x, first, A, C = 0x330E, [], 1, 0
    for _ in range(block):
        x = (a * x + c) & mask
        first.append(x)
        A, C = (A * a) & mask, (C * a + c) & mask  # block steps at once: x -> A x + C
    out, cur = [], np.array(first, dtype=np.uint64)
    for _ in range(-(-n // block)):
        out.append(cur)
        cur = (cur * np.uint64(A) + np.uint64(C)) & np.uint64(mask)
    return np.concatenate(out)[:n].astype(np.float64) / float(1 << 48)


def largest_eigenvalue(m, inv):
    """Of D^-1 A, by ten Arnoldi steps from the drand48 start: the smoother's definition of it."""
    v = torch.tensor(drand48(m.n), device="cuda")
    V, H = [v / v.norm()], np.zeros((10, 10))
    for j in range(10):
        w = inv * m.operator(V[j])
        for i in range(j + 1):
            H[i, j] = float(V[i] @ w)
            w = w - H[i, j] * V[i]
        if j < 9:
            H[j + 1, j] = float(w.norm())
            V.append(w / H[j + 1, j])
    return float(np.abs(np.linalg.eigvals(H)).max())


def exact_smooth(case, r, x):
    """x + p(D^-1 A) D^-1 (r - A x), p the Chebyshev polynomial of degree 2 + 1 on [rho/10, rho]."""
    m = Box(case)
    inv = 1.0 / m.diagonal()
    hi = largest_eigenvalue(m, inv)
    theta, delta = 0.55 * hi, 0.45 * hi
    sigma = theta / delta
    rho = 1.0 / sigma
    res = inv * (r - m.operator(x))
    d = res / theta
    x = x + d
    for _ in range(2):
        res = res - inv * m.operator(d)
        new = 1.0 / (2 * sigma - rho)
        d = 2 * new / delta * res + new * rho * d
        rho = new
        x = x + d
    return x


def exact_transfer(case, r, e, x):
    Nf, Nc = degrees(case)[:2]
    f, c = Box(case, Nf), Box(case, Nc)
    P = torch.tensor(interpolation(c.r_host, f.r_host), device="cuda")
    PT = P.T.contiguous()
    up = lambda A, v: along(A, along(A, along(A, v, 3), 2), 1)  # noqa: E731
    rc = c.gather(up(PT, f.scatter(r / f.mult).view(f.E, f.Nq, f.Nq, f.Nq)))
    # a fine node takes the mean over its elements of what each interpolates there (they agree but for rounding)
    fine = f.gather(up(P, c.scatter(e).view(c.E, c.Nq, c.Nq, c.Nq))) / f.mult
    return rc, x + fine


def forcing(m, seed):
    """sum a_k sin(pi k.x + phi_k), 64 modes drawn with erand48 from the seed."""
    libc = ctypes.CDLL(None)
    libc.erand48.restype = ctypes.c_double
    xs = (ctypes.c_ushort * 3)(0x330E, seed & 0xffff, (seed >> 16) & 0xffff)
    x, y, z = m.nodes()
    f = torch.zeros_like(x)
    for _ in range(64):
        k = [1 + int(4 * libc.erand48(xs)) for _ in range(3)]
        sign = -1.0 if libc.erand48(xs) < 0.5 else 1.0
        phase = 2 * math.pi * libc.erand48(xs)
        f += sign / sum(i * i for i in k) * torch.sin(math.pi * (k[0] * x + k[1] * y + k[2] * z) + phase)
    return f


def exact_solve(case, seed):
    """The discrete solution by Jacobi-PCG to 1e-13, at every local node (0 at Dirichlet nodes)."""
    m = Box(case)
    m.keep_factors()
    JW = torch.cat([m.kept[c][1] for c in m.chunks()])
    r = m.gather(JW * forcing(m, 1 + seed % 1000003))
    inv = 1.0 / m.diagonal()
    x = torch.zeros_like(r)
    z = inv * r
    p, rz, stop = z, r @ z, 1e-13 * float(r.norm())
    for it in range(4000):
        Ap = m.operator(p)
        alpha = rz / (p @ Ap)
        x += alpha * p
        r -= alpha * Ap
        if it % 20 == 19 and float(r.norm()) < stop:
            break
        z = inv * r
        old, rz = rz, r @ z
        p = z + rz / old * p
    return m.scatter(x).cpu().numpy()


def exact_learned(case, r):
    """Mean over a node's elements of s W (z / s), z = D^-1 r on the element and on the six neighbours' node
    layers next to the shared faces (0 outside the box and at Dirichlet nodes): the input scale s cancels."""
    m = Box(case)
    z = m.scatter(r / m.diagonal()).view(m.E, 8, 8, 8)
    grid = z.view(m.nz, m.ny, m.nx, 8, 8, 8)
    layers = []
    for f in range(6):  # faces t-, s-, r+, s+, r-, t+
        axis, step = [(0, -1), (1, -1), (2, 1), (1, 1), (2, -1), (0, 1)][f]
        layer = grid.select(3 + axis, 6 if step < 0 else 1)
        n = grid.shape[axis]
        moved = torch.zeros_like(layer)
        if n > 1:
            moved.narrow(axis, 0 if step > 0 else 1, n - 1).copy_(layer.narrow(axis, 1 if step > 0 else 0, n - 1))
        layers.append(moved.reshape(m.E, 64))
    X = torch.cat([z.reshape(m.E, 512)] + layers, dim=1)
    theta = torch.tensor(np.fromfile(LINEAR_WEIGHTS, dtype=np.float32, offset=44), device="cuda")
    W = theta[:512 * 896].view(512, 896).bfloat16().double()
    omega = theta[-1].double()
    return m.gather(X @ W.T) / m.mult + omega * r / m.diagonal()


def exact_mlp(case, seed):
    W, b, X, dY = mlp_inputs(case, seed)
    W, b, X, dY = [w.double() for w in W], [v.double() for v in b], X.double(), dY.double()
    H1 = torch.relu(X @ W[0].T + b[0])
    H2 = torch.relu(H1 @ W[1].T + b[1])
    d2 = (dY @ W[2]) * (H2 > 0)
    d1 = (d2 @ W[1]) * (H1 > 0)
    return ([H2 @ W[2].T + b[2], d1.T @ X, d2.T @ H1, dY.T @ H2] + [d1.sum(0), d2.sum(0), dY.sum(0)])


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return exact_mlp(case, seed)
    if kind == "vcycle":  # the aggregates of its base level are the library's own
        return None
    if kind == "solve":
        return exact_solve(case, seed)
    n = counts(case)[2]
    if kind == "operator":
        return Box(case).operator(vector(n, seed))
    dt = torch.float32 if case["bits"] == 32 else torch.float64
    r = vector(n, seed, dt).double()
    if kind == "learned":
        return exact_learned(case, r)
    if kind == "smooth":
        return exact_smooth(case, r, vector(n, seed + 1, dt).double())
    nc = counts(case, degrees(case)[1])[2]
    return exact_transfer(case, r, vector(nc, seed + 1, dt).double(), vector(n, seed + 2, dt).double())
