"""The calls a program makes of this library, as cases to time.

A program holds one context per lattice, gauge fields, operators, solvers and
spinors on the device and calls `multiply`, `multiply_add`, `solve`,
`solve_batch`, `two_flavor_force` and the request server.  Every pass here is
one such call (one burst of requests for the server).  Results stay in the
spinors a program reads on from; `run` returns tensors over those spinors'
device memory, or the host arrays a call fills.

Lattices, representations, kappa, c_sw and tolerances are those of the
benchmark and the tests: SU(3) at kappa 0.12-0.134, SU(2) adjoint at 0.17,
c_sw = 1, links exp(i eps H) at eps = 0.5, antiperiodic in time.

`exact` restates each result in plain torch in complex128.
"""
import ctypes
import math

import numpy as np
import torch

import leonardym_amd as lym

EPS, CSW = 0.5, 1.0
REPS = {"su3": lym.REP_SU3_FUND, "adj": lym.REP_SU2_ADJ}
OPS = {"wilson": lym.OP_WILSON, "clover": lym.OP_CLOVER, "eo": lym.OP_EO_CLOVER}
STORAGE = {"full": lym.LINKS_FULL, "rows": lym.LINKS_RECONSTRUCT}
SOLVERS = {"cg": lym.SOLVER_CG, "bicgstab": lym.SOLVER_BICGSTAB, "eo_bicgstab": lym.SOLVER_PRECOND_BICGSTAB,
           "eo_cg": lym.SOLVER_PRECOND_CG, "eo_mixed": lym.SOLVER_PRECOND_MIXED_CG}
SLOPPY = {"double": None, "single": lym.PREC_SINGLE, "half": lym.PREC_HALF}
KAPPA = {"su3": 0.13, "adj": 0.17}

# most sites of a drawn case, and the sites of the largest listed one, per kind of call
MOST = {"apply": 32 ** 3 * 64, "solve": 24 ** 3 * 48, "batch": 24 ** 3 * 48, "force": 12 ** 3 * 24}


def _case(name, path, dims, **kw):
    c = {"path": path, "lx": dims[0], "ly": dims[1], "lz": dims[2], "lt": dims[3]}
    if name:
        c["name"] = name
    c.update(kw)
    return c


def listed():
    return [
        # the smallest apply of the workloads (8^4 Wilson, as inside its CG): latency and launch bound
        _case("wilson_8", "apply", (8, 8, 8, 8), op="wilson", rep="su3", links="full", power=1, gamma5=True),
        # the benchmark's apply: the full-lattice clover Q of the 16^3x32 workload
        _case("clover_16x32", "apply", (16, 16, 16, 32), op="clover", rep="su3", links="full", power=1, gamma5=True),
        # the same on the largest lattice of the workloads
        _case("clover_32x64", "apply", (32, 32, 32, 64), op="clover", rep="su3", links="full", power=1, gamma5=True),
        # the even-odd Schur complement squared with real adjoint links: what an FP64 CG on the
        # 24^3x48 adjoint lattice applies in every iteration
        _case("eo_square_adj_24x48", "apply", (24, 24, 24, 48), op="eo", rep="adj", links="full", power=2,
              gamma5=True),
        # D v1 + alpha v2 (a shifted operator) on extents that are odd and no multiple of a tile, 12-real links
        _case("shifted_odd", "apply_add", (15, 9, 11, 13), op="clover", rep="su3", links="rows", power=1,
              gamma5=False),
        # ConjugateGradient on the squared Wilson operator, 8^4: the reference's own CPU-size solve
        _case("cg_wilson_8", "solve", (8, 8, 8, 8), op="wilson", rep="su3", links="full", power=2, method="cg",
              sloppy="double"),
        # PreconditionedBiCGStab, the reference's production inverter, on the 16^3x32 clover lattice
        _case("eo_bicgstab_16x32", "solve", (16, 16, 16, 32), op="clover", rep="su3", links="full", power=1,
              method="eo_bicgstab", sloppy="double"),
        # mixed-precision even-odd CG with FP16 storage on the 24^3x48 adjoint lattice
        _case("mixed_half_adj_24x48", "solve", (24, 24, 24, 48), op="clover", rep="adj", links="full", power=1,
              method="eo_mixed", sloppy="half"),
        # the same with FP32 storage on a lattice between the workloads' sizes
        _case("mixed_single_12x24", "solve", (12, 12, 12, 24), op="clover", rep="su3", links="rows", power=1,
              method="eo_mixed", sloppy="single"),
        # a propagator: the 12 point sources of one site on 32^3x64, one batched call
        _case("propagator_32x64", "batch", (32, 32, 32, 64), op="clover", rep="su3", links="full", power=1, nrhs=12,
              sloppy="half"),
        # the solve server taking a burst of requests over three resident lattices, each with its own
        # kappa, tolerance and source
        _case("serve_burst", "serve", (16, 16, 16, 32), requests=18, sloppy="half"),
        # one HMC fermion-force evaluation: two BiCGStab solves and the derivative with respect to every link
        _case("force_8x16", "force", (8, 8, 8, 16), op="wilson", rep="su3", links="full", power=1,
              method="bicgstab", sloppy="double"),
    ]


def _extents(rng, most, even):
    """Four extents, volumes spread over their logarithm from 4^4 to `most` sites."""
    while True:
        v = math.exp(rng.uniform(math.log(256.0), math.log(most)))
        s = (v / 2.0) ** 0.25
        d = [s * rng.uniform(0.7, 1.4) for _ in range(3)] + [2 * s * rng.uniform(0.7, 1.4)]
        d = [max(4, 2 * round(x / 2)) if even else max(4, round(x)) for x in d]
        if not even and all(x % 2 == 0 for x in d):
            d[rng.randrange(4)] += 1
        if d[0] * d[1] * d[2] * d[3] <= most:
            return tuple(d)


def draw(rng):
    path = rng.choice(["apply", "apply", "apply_add", "solve", "solve", "solve", "batch", "serve", "force"])
    rep, links = rng.choice(["su3", "su3", "adj"]), rng.choice(["full", "full", "rows"])
    if path in ("apply", "apply_add"):
        # odd extents: the full-lattice operators only
        even = rng.random() < 0.75
        kinds = ["wilson", "clover", "eo"] if even and path == "apply" else ["wilson", "clover"]
        op, power = rng.choice(kinds), rng.choice([1, 1, 2])
        dims = _extents(rng, MOST["apply"] // power, even)
        return _case(None, path, dims, op=op, rep=rep, links=links, power=power, gamma5=rng.random() < 0.7)
    if path == "solve":
        method = rng.choice(["cg", "eo_bicgstab", "eo_cg", "eo_mixed", "eo_mixed"])
        op = rng.choice(["wilson", "clover"]) if method == "cg" else "clover"
        sloppy = rng.choice(["half", "single"]) if method == "eo_mixed" else "double"
        return _case(None, path, _extents(rng, MOST["solve"], True), op=op, rep=rep, links=links,
                     power=2 if method == "cg" else 1, method=method, sloppy=sloppy)
    if path == "batch":
        return _case(None, path, _extents(rng, MOST["batch"], True), op="clover", rep=rep, links=links, power=1,
                     nrhs=rng.randint(2, 12), sloppy=rng.choice(["half", "half", "single"]))
    if path == "serve":
        return _case(None, path, _extents(rng, 16 ** 3 * 32, True), requests=rng.randint(1, 18),
                     sloppy=rng.choice(["half", "single"]))
    return _case(None, path, _extents(rng, MOST["force"], True), op="wilson", rep="su3", links=links, power=1,
                 method="bicgstab", sloppy="double")


# ---------------------------------------------------------------- inputs
def _dims(case):
    return (case["lx"], case["ly"], case["lz"], case["lt"])


def _rng(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + stream)
    return g


def _su3_links(n, gen):
    """n matrices exp(i EPS H), H = sum_a w_a lambda_a / 2, w ~ N(0, 1)."""
    w = torch.randn(n, 8, dtype=torch.float64, device="cuda", generator=gen) * (0.5 * EPS)
    H = torch.zeros(n, 3, 3, dtype=torch.complex128, device="cuda")
    r3 = 1.0 / math.sqrt(3.0)
    H[:, 0, 0], H[:, 1, 1], H[:, 2, 2] = w[:, 2] + r3 * w[:, 7], -w[:, 2] + r3 * w[:, 7], -2 * r3 * w[:, 7]
    H[:, 0, 1], H[:, 0, 2], H[:, 1, 2] = (torch.complex(w[:, a], -w[:, a + 1]) for a in (0, 3, 5))
    H[:, 1, 0], H[:, 2, 0], H[:, 2, 1] = (torch.complex(w[:, a], w[:, a + 1]) for a in (0, 3, 5))
    H = 1j * H
    U = torch.eye(3, dtype=torch.complex128, device="cuda").expand(n, 3, 3).clone()
    for k in range(14, 0, -1):
        U = (H[:, :, :, None] * U[:, None, :, :]).sum(2) / k
        for i in range(3):
            U[:, i, i] += 1.0
    # unitary to rounding: rows 0 and 1 orthonormal, row 2 their conjugated cross product
    a = U[:, 0] / U[:, 0].abs().square().sum(-1, keepdim=True).sqrt()
    b = U[:, 1] - (a.conj() * U[:, 1]).sum(-1, keepdim=True) * a
    b = b / b.abs().square().sum(-1, keepdim=True).sqrt()
    return torch.stack([a, b, torch.linalg.cross(a, b).conj()], 1)


def _so3_links(n, gen):
    """n rotations: the adjoint form of exp(i EPS sigma.a), a ~ N(0, 1)^3."""
    a = torch.randn(n, 3, dtype=torch.float64, device="cuda", generator=gen) * EPS
    th = a.square().sum(-1).sqrt()
    u = a / th[:, None]
    c, s = torch.cos(2 * th), torch.sin(2 * th)
    R = (1 - c)[:, None, None] * u[:, :, None] * u[:, None, :]
    for i in range(3):
        R[:, i, i] += c
    for i, j, k in ((0, 1, 2), (1, 2, 0), (2, 0, 1)):
        R[:, j, k] += s * u[:, i]
        R[:, k, j] -= s * u[:, i]
    return R


def _links(dims, rep, seed, stream=0):
    """[V, 4, 3, 3] on the GPU, without the boundary sign."""
    n = 4 * math.prod(dims)
    U = _su3_links(n, _rng(seed, stream)) if rep == "su3" else _so3_links(n, _rng(seed, stream))
    return U.reshape(-1, 4, 3, 3)


def _spinor(dims, seed, stream):
    """[V, 4, 3] complex Gaussian on the GPU."""
    z = torch.randn(math.prod(dims), 4, 3, 2, dtype=torch.float64, device="cuda", generator=_rng(seed, stream))
    return torch.view_as_complex(z) * math.sqrt(0.5)


def _host_links(U):
    """Links for Gauge and add_lattice: column-major in memory, as the library stores them."""
    return np.swapaxes(U.transpose(-1, -2).contiguous().cpu().numpy(), -1, -2)


_contexts = {}


def _context(dims, rep):
    """The program's context of a lattice: one per geometry, kept."""
    key = (tuple(dims), rep)
    if key not in _contexts:
        _contexts[key] = lym.Context(dims, REPS[rep], -1)
    return _contexts[key]


def _layout(dims):
    """(stride, even-odd) of a device spinor: double2 [2 parities][12][stride]."""
    even = all(d % 2 == 0 for d in dims)
    vh = math.prod(dims) // (2 if even else 1)
    return (vh + 63) // 64 * 64, even


class _DeviceMemory:
    """A spinor's device memory as an array: the handle is {context, pointer}."""

    def __init__(self, spinor):
        self.spinor = spinor  # lives as long as the tensors over it
        ptr = ctypes.c_void_p.from_address(spinor.h.value + ctypes.sizeof(ctypes.c_void_p)).value
        stride, _ = _layout(spinor.ctx.dims)
        self.__cuda_array_interface__ = {"shape": (2, 12, stride, 2), "typestr": "<f8", "data": (ptr, False),
                                         "version": 2, "strides": None}


def _tensor(spinor):
    return torch.as_tensor(_DeviceMemory(spinor), device="cuda")


def _requests(case, seed):
    """(lattice index, kappa, tolerance, source stream) of a burst, and its lattices."""
    big = _dims(case)
    lattices = [(8, 8, 8, 8), (12, 12, 12, 12), big]
    r = np.random.default_rng(seed)
    return lattices, [(int(q % 3), float(r.uniform(0.120, 0.134)), float(r.choice([1e-10, 1e-12])), 10 + q)
                      for q in range(case["requests"])]


def _point_sites(case, seed):
    return [int(v) for v in np.random.default_rng(seed).integers(0, _dims(case))]


def prepare(case, seed):
    dims, path = _dims(case), case["path"]
    if path == "serve":
        lattices, reqs = _requests(case, seed)
        srv = lym.Server(workers=4, hbm_budget=16 << 30, max_batch=4, sloppy=SLOPPY[case["sloppy"]])
        ids = [srv.add_lattice(d, _host_links(_links(d, "su3", seed, i)), csw=CSW) for i, d in enumerate(lattices)]
        todo = []
        for li, kappa, tol, stream in reqs:
            src, out = (lym.pinned_empty((math.prod(lattices[li]), 4, 3)) for _ in range(2))
            src[...] = _spinor(lattices[li], seed, stream).cpu().numpy()
            todo.append((ids[li], kappa, tol, src, out))
        return {"case": case, "server": srv, "todo": todo}
    ctx = _context(dims, case["rep"])
    gauge = lym.Gauge(ctx, _host_links(_links(dims, case["rep"], seed)), folded=False, storage=STORAGE[case["links"]])
    op = lym.Operator(ctx, OPS[case["op"]], case["power"], KAPPA[case["rep"]], CSW, case.get("gamma5", True),
                      gauge=gauge)
    s = {"case": case, "ctx": ctx, "op": op}
    if path in ("apply", "apply_add"):
        s["in"] = lym.Spinor(ctx, _spinor(dims, seed, 1).cpu().numpy())
        if path == "apply_add":
            s["v2"] = lym.Spinor(ctx, _spinor(dims, seed, 2).cpu().numpy())
        s["out"] = lym.Spinor(ctx)
        s["result"] = _tensor(s["out"])
        op.multiply(s["out"], s["in"])  # builds the operator's clover blocks, once per kappa and gauge field
        return s
    n2 = 1.0
    if path == "batch":
        site = _point_sites(case, seed)
        s["in"] = [lym.Spinor(ctx, lym.point_source(dims, site, q % 4, q // 4)) for q in range(case["nrhs"])]
        s["out"] = [lym.Spinor(ctx) for _ in s["in"]]
        s["result"] = [_tensor(x) for x in s["out"]]
    else:
        s["in"] = lym.Spinor(ctx, _spinor(dims, seed, 1).cpu().numpy())
        s["out"] = lym.Spinor(ctx)
        s["result"] = _tensor(s["out"])
        n2 = s["in"].squared_norm()
    tol = 1e-12 if case["sloppy"] == "double" else 1e-11
    s["solver"] = lym.Solver(ctx, SOLVERS[case.get("method", "eo_mixed")], precision=tol ** 2 * n2, max_steps=20000,
                             sloppy=SLOPPY[case["sloppy"]])
    return s


def run(s):
    path = s["case"]["path"]
    if path == "apply":
        s["op"].multiply(s["out"], s["in"])
    elif path == "apply_add":
        s["op"].multiply_add(s["out"], s["in"], s["v2"], ALPHA)
    elif path == "solve":
        s["solver"].solve(s["op"], s["in"], s["out"])
    elif path == "batch":
        s["solver"].solve_batch(s["op"], s["in"], s["out"])
    elif path == "serve":
        srv = s["server"]
        ids = [srv.submit(*r) for r in s["todo"]]
        return [srv.wait(i)[1] for i in ids]
    else:
        return s["solver"].two_flavor_force(s["op"], s["in"])[0]
    return s["result"]


ALPHA = 0.37 - 0.21j


# ---------------------------------------------------------------- work
# per site: complex multiply-adds are 8 flops; a hop is 2 projected colour vectors times a 3x3 matrix
def _apply_work(case, V, elem, nrhs=1):
    """(bytes, flops) of one apply of the operator (one power) on nrhs vectors."""
    real = case["rep"] == "adj"
    link = (9 if case["links"] == "full" else 6) * (1 if real else 2) * elem
    blocks = 72 * elem if case["op"] != "wilson" else 0
    spinor = 24 * elem
    hop = 8 * (2 * 15 * (2 if real else 4.4) + 12 * 4)
    diag = 2 * 6 * 6 * 8 if case["op"] != "wilson" else 24
    if case["op"] == "eo":  # per odd site: all links, A_oo, R_ee^-1, in and out
        return V / 2 * (8 * link + 2 * blocks + 2 * spinor * nrhs), V / 2 * nrhs * (2 * hop + 2 * diag)
    return V * (4 * link + blocks + 2 * spinor * nrhs), V * nrhs * (hop + diag)


# applies of the squared operator a solve of these lattices takes (iterations, to its tolerance)
ITERATIONS = {"cg": 90, "eo_bicgstab": 62, "eo_cg": 90, "eo_mixed": 85, "bicgstab": 90}


def work(case):
    V = math.prod(_dims(case))
    path = case["path"]
    if path in ("apply", "apply_add"):
        b, f = _apply_work(case, V, 8)
        b, f = case["power"] * b, case["power"] * f
        if case["op"] == "eo":
            b += V / 2 * 2 * 192  # the even half, copied
        if path == "apply_add":
            b, f = b + V * 192, f + V * 96
        return {"bytes": b, "flops": f}
    if path == "serve":
        lattices, reqs = _requests(case, 0)
        c = {"op": "eo", "rep": "su3", "links": "rows"}
        each = [_apply_work(c, math.prod(lattices[li]), 2 if case["sloppy"] == "half" else 4) for li, _, _, _ in reqs]
        return {"bytes": 2 * ITERATIONS["eo_mixed"] * sum(b for b, _ in each),
                "flops": 2 * ITERATIONS["eo_mixed"] * sum(f for _, f in each)}
    elem = {"double": 8, "single": 4, "half": 2}[case["sloppy"]]
    method = case.get("method", "eo_mixed")
    c = dict(case, op="eo" if method.startswith("eo") else case["op"])
    if elem < 8:
        c["links"] = "rows"  # low-precision links hold rows 0 and 1
    b, f = _apply_work(c, V, elem, case.get("nrhs", 1))
    n = ITERATIONS[method] * 2  # two applies an iteration: the squared operator, or BiCGStab's two
    if method == "eo_bicgstab":
        n *= 2  # BiCGStab on the squared Schur complement
    if path == "force":
        n *= 2  # two solves
    return {"bytes": n * b, "flops": n * f}


# ---------------------------------------------------------------- the same results in complex128, plain torch
GAMMA = ((3, 2, 1, 0), (-1j, -1j, 1j, 1j)), ((3, 2, 1, 0), (-1, 1, 1, -1)), ((2, 3, 0, 1), (-1j, 1j, 1j, -1j)), \
    ((2, 3, 0, 1), (1, 1, 1, 1))  # row s of gamma_mu: its column and entry
G5 = (1, 1, -1, -1)


def _spin(v):
    return torch.tensor(v, dtype=torch.complex128, device="cuda")[:, None]


def _mv(M, v):
    """3x3 per site times the colour vectors of every spin."""
    return (M[..., None, :, :] * v[..., :, None, :]).sum(-1)


def _mm(A, B):
    return (A[..., :, :, None] * B[..., None, :, :]).sum(-2)


class _Dirac:
    """D = A - kappa H on [Lx, Ly, Lz, Lt, 4, 3]; A = 1 - kappa c_sw sum_{mu<nu} gamma_mu gamma_nu F_munu."""

    def __init__(self, dims, U, kappa, clover):
        self.dims, self.kappa = dims, kappa
        U = U.to(torch.complex128).reshape(*dims, 4, 3, 3)
        self.U = [U[..., m, :, :].contiguous() for m in range(4)]
        self.W = list(self.U)
        self.W[3] = self.U[3].clone()
        self.W[3][:, :, :, -1] *= -1
        self.Wd = [torch.roll(w, 1, m).conj().transpose(-1, -2).contiguous() for m, w in enumerate(self.W)]
        self.g5 = _spin(G5)
        self.perm = [torch.tensor(p, device="cuda") for p, _ in GAMMA]
        self.ph = [_spin(e) for _, e in GAMMA]
        self.A = self._clover() if clover else None

    def gamma(self, m, v):
        return self.ph[m] * v[..., self.perm[m], :]

    def hop(self, v):
        """-kappa H v"""
        out = torch.zeros_like(v)
        for m in range(4):
            f, b = _mv(self.W[m], torch.roll(v, -1, m)), _mv(self.Wd[m], torch.roll(v, 1, m))
            out += f + b - self.gamma(m, f - b)
        return -self.kappa * out

    def _clover(self):
        """[..., 2 chiralities, 6, 6]"""
        U = self.U
        A = torch.zeros(*self.dims, 2, 2, 3, 2, 3, dtype=torch.complex128, device="cuda")
        gam = []
        for p, e in GAMMA:
            g = torch.zeros(4, 4, dtype=torch.complex128)
            for s in range(4):
                g[s, p[s]] = e[s]
            gam.append(g)
        for m in range(4):
            for n in range(m + 1, 4):
                # the four leaves of the (m, n) plane at every site, from the plaquette and its corners
                um, un = U[m], U[n]
                um_n, un_m = torch.roll(um, -1, n), torch.roll(un, -1, m)
                dag = lambda M: M.conj().transpose(-1, -2)  # noqa: E731
                q = _mm(_mm(um, un_m), dag(_mm(un, um_n)))          # x, m, n, -m, -n
                t = _mm(_mm(un_m, dag(um_n)), _mm(dag(un), um))     # at x + m: n, -m, -n, m
                Q = q + torch.roll(t, 1, m)
                t = _mm(_mm(dag(um_n), dag(un)), _mm(um, un_m))     # at x + m + n: -m, -n, m, n
                Q += torch.roll(t, (1, 1), (m, n))
                t = _mm(_mm(dag(un), um), _mm(un_m, dag(um_n)))     # at x + n: -n, m, n, -m
                Q += torch.roll(t, 1, n)
                F = (Q - dag(Q)) / 8
                gg = (gam[m] @ gam[n]).cuda()
                for h in range(2):
                    s = gg[2 * h:2 * h + 2, 2 * h:2 * h + 2]
                    A[..., h, :, :, :, :] += s[:, None, :, None] * F[..., None, :, None, :]
        A = (-self.kappa * CSW) * A.reshape(*self.dims, 2, 6, 6)
        for k in range(6):
            A[..., k, k] += 1
        return A

    def diag(self, v, M=None):
        M = self.A if M is None else M
        if M is None:
            return v
        return (M * v.reshape(*self.dims, 2, 1, 6)).sum(-1).reshape(v.shape)

    def D(self, v):
        return self.diag(v) + self.hop(v)

    def solve(self, b):
        """D^-1 b by conjugate gradients on D^+ D (D^+ = g5 D g5), restarted on the true residual."""
        x = torch.zeros_like(b)
        n2 = lambda v: torch.view_as_real(v).square().sum().item()  # noqa: E731
        dd = lambda v: self.g5 * self.D(self.g5 * self.D(v))  # noqa: E731
        for _ in range(4):
            r = self.g5 * self.D(self.g5 * (b - self.D(x)))
            p, rr = r.clone(), n2(r)
            if rr < 1e-30 * n2(b):
                break
            stop = max(1e-16 * rr, 1e-31 * n2(b))
            while rr > stop:
                q = dd(p)
                a = rr / torch.linalg.vecdot(p.reshape(-1), q.reshape(-1)).real.item()
                x += a * p
                r -= a * q
                new = n2(r)
                p = r + (new / rr) * p
                rr = new
        return x


def _device_layout(dims, v):
    """[Lx, Ly, Lz, Lt, 4, 3] in the order of a device spinor, as [2, 12, stride, 2] reals."""
    stride, even = _layout(dims)
    out = torch.zeros(2, 12, stride, dtype=torch.complex128, device="cuda")
    v = v.reshape(-1, 12)
    if even:
        odd = _parity(dims).reshape(-1)
        for p in (0, 1):
            out[p, :, :v.shape[0] // 2] = v[odd == p].T
    else:
        out[0, :, :v.shape[0]] = v.T
    return torch.view_as_real(out)


def _parity(dims):
    c = torch.meshgrid(*(torch.arange(d, device="cuda") for d in dims), indexing="ij")
    return (c[0] + c[1] + c[2] + c[3]) % 2


def _exact_apply(case, seed, dims):
    d = _Dirac(dims, _links(dims, case["rep"], seed), KAPPA[case["rep"]], case["op"] != "wilson")
    v = _spinor(dims, seed, 1).reshape(*dims, 4, 3)
    if case["op"] == "eo":
        odd = _parity(dims)[..., None, None].to(torch.complex128)
        Ainv = torch.linalg.inv(d.A)

        def one(w):
            o = odd * w
            e = d.diag((1 - odd) * d.hop(o), Ainv)
            o = odd * (d.diag(o) - d.hop(e))
            return (1 - odd) * w + (d.g5 * o if case["gamma5"] else o)
    else:
        one = lambda w: d.g5 * d.D(w) if case["gamma5"] else d.D(w)  # noqa: E731
    out = one(v)
    if case["power"] == 2:
        out = one(out)
    if case["path"] == "apply_add":
        out = out + ALPHA * _spinor(dims, seed, 2).reshape(*dims, 4, 3)
    return _device_layout(dims, out)


def _exact_force(case, seed, dims):
    d = _Dirac(dims, _links(dims, case["rep"], seed), KAPPA[case["rep"]], False)
    phi = _spinor(dims, seed, 1).reshape(*dims, 4, 3)
    Y = d.solve(d.g5 * phi)
    X = d.solve(d.g5 * Y)
    out = torch.empty(*dims, 4, 3, 3, dtype=torch.complex128, device="cuda")
    outer = lambda a, b: (a[..., :, :, None] * b.conj()[..., :, None, :]).sum(-3)  # noqa: E731
    for m in range(4):
        W, Wd = d.W[m], d.W[m].conj().transpose(-1, -2)
        K = 0
        for A, B in ((X, Y), (Y, X)):
            Bu, Au, b = torch.roll(B, -1, m), torch.roll(A, -1, m), _mv(Wd, B)
            K = K + outer(d.g5 * (Bu - d.gamma(m, Bu)), A) - outer(d.g5 * (b + d.gamma(m, b)), _mv(W, Au))
        K = _mm(d.U[m], -d.kappa * K)
        K = (K - K.conj().transpose(-1, -2)) / 4
        tr = K.diagonal(dim1=-2, dim2=-1).sum(-1) / 3
        for i in range(3):
            K[..., i, i] -= tr
        out[..., m, :, :] = K
    return out.reshape(-1, 4, 3, 3).cpu().numpy()


def exact(case, seed):
    dims, path = _dims(case), case["path"]
    V = math.prod(dims)
    if path in ("apply", "apply_add"):
        return _exact_apply(case, seed, dims)
    if path == "force":
        return _exact_force(case, seed, dims)
    if path == "serve":
        lattices, reqs = _requests(case, seed)
        U = [_links(d, "su3", seed, i) for i, d in enumerate(lattices)]
        out = []
        for li, kappa, _, stream in reqs:
            d = _Dirac(lattices[li], U[li], kappa, True)
            x = d.solve(_spinor(lattices[li], seed, stream).reshape(*lattices[li], 4, 3))
            out.append(x.reshape(-1, 4, 3).cpu().numpy())
        return out
    d = None
    if path == "batch":
        if V * case["nrhs"] > 24 ** 3 * 48:
            return None  # over 20 seconds
        d = _Dirac(dims, _links(dims, case["rep"], seed), KAPPA[case["rep"]], True)
        out = []
        for q in range(case["nrhs"]):
            b = torch.zeros(*dims, 4, 3, dtype=torch.complex128, device="cuda")
            b[(*_point_sites(case, seed), q % 4, q // 4)] = 1
            out.append(_device_layout(dims, d.solve(b)))
        return out
    d = _Dirac(dims, _links(dims, case["rep"], seed), KAPPA[case["rep"]], case["op"] != "wilson")
    b = _spinor(dims, seed, 1).reshape(*dims, 4, 3)
    if case["power"] == 2:  # Q^2 x = b, Q = gamma5 D
        b = d.solve(d.g5 * b)
        return _device_layout(dims, d.solve(d.g5 * b))
    return _device_layout(dims, d.solve(b))
