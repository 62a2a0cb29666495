"""The work that users of invdft_amd have it do, as cases to time.

Kinds of case, each through the entry points of include/idft*.h:

  vmult     one application of the adjoint operator H~ x - eps x to a block of
            device multivectors: what an outer Krylov solver calls once per step
  ends      the two ends of an adjoint block solve, computeRhs and distributeX
            (a caller with its own Krylov solver between them)
  solve     a blocked adjoint solve to its tolerance: right-hand side,
            preconditioned MINRES, the null-space correction
  minres    the same for a fixed number of steps
  force     one getForceVector evaluation of an inversion, warm-started from the
            previous one's orbitals: eigensolve, density, loss, adjoint, force
  forward   the forward half alone (eigensolve, density, loss) of a wide block of
            orbitals
  poisson   the set-up's electrostatic potential of a charge density

A state holds what a user's program holds: the context, device blocks, host
arrays.  Meshes and block widths are those of the package's configurations
(8^3 cells at degree 3 up to 40^3 at degree 4 with 80 columns) and what lies
between; `draw` spreads over the same ranges.
"""
import ctypes as C
import math

import numpy as np
import torch

import invdft_amd
from invdft_amd import abi, synthetic

HALF_WIDTH = 12.0
BOLTZMANN_HA = 3.166811563e-6


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # a small molecule's mesh, a few orbitals: latency and launches
        dict(name="vmult_8c_p3_b5", kind="vmult", n_cells=8, degree=3, ncols=5),
        # a production mesh, the headline block width
        dict(name="vmult_24c_p5_b12", kind="vmult", n_cells=24, degree=5, ncols=12),
        # odd mesh and odd width
        dict(name="vmult_19c_p4_b21", kind="vmult", n_cells=19, degree=4, ncols=21),
        # the largest block the operator takes
        dict(name="vmult_40c_p4_b80", kind="vmult", n_cells=40, degree=4, ncols=80),
        # the ends of an adjoint block solve at the headline mesh, and on a fine
        # mesh with many orbitals
        dict(name="ends_24c_p5_b12", kind="ends", n_cells=24, degree=5, ncols=12),
        dict(name="ends_32c_p5_b32", kind="ends", n_cells=32, degree=5, ncols=32),
        # a whole adjoint solve of a small molecule to its tolerance
        dict(name="solve_16c_p4_b6", kind="solve", n_cells=16, degree=4, ncols=6, n_occ=2),
        # a large adjoint block for a fixed number of steps (such a solve takes
        # thousands: this is its steady state)
        dict(name="minres_40c_p4_b64", kind="minres", n_cells=40, degree=4, ncols=64, steps=48),
        # evaluations of an inversion: small and in FP64, as in an uneven batch
        # of small problems; the production mesh in mixed precision
        dict(name="force_8c_p3", kind="force", n_cells=8, degree=3, n_occ=4, n_eig=8,
             precision="fp64"),
        dict(name="force_24c_p5_mixed", kind="force", n_cells=24, degree=5, n_occ=8, n_eig=12,
             precision="mixed"),
        # many orbitals: the dense block algebra of the eigensolver counts too
        dict(name="forward_20c_p4_n40", kind="forward", n_cells=20, degree=4, n_occ=8, n_eig=40,
             precision="mixed"),
        # once per molecule, before the inversion
        dict(name="poisson_16c_p4", kind="poisson", n_cells=16, degree=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vmult", "vmult", "ends", "solve", "minres", "force", "forward",
                       "poisson"])
    p = rng.randint(2, 5)
    if kind == "vmult":
        b = _log_int(rng, 1, 80)
        n1 = _log_int(rng, 16, min(161, int((161 ** 3 * 80 / b) ** (1 / 3))))
        return dict(kind=kind, n_cells=max(3, n1 // p), degree=p, ncols=b)
    if kind == "ends":
        b = _log_int(rng, 2, 32)
        return dict(kind=kind, n_cells=max(4, _log_int(rng, 24, 150) // p), degree=p, ncols=b)
    if kind == "minres":
        b = _log_int(rng, 2, 40)
        return dict(kind=kind, n_cells=max(6, _log_int(rng, 24, 120) // p), degree=p, ncols=b,
                    steps=rng.randint(16, 64))
    if kind == "poisson":
        return dict(kind=kind, n_cells=max(6, _log_int(rng, 24, 72) // p), degree=p)
    p = rng.randint(3, 5)
    n_occ = rng.randint(1, 8)
    if kind == "solve":
        return dict(kind=kind, n_cells=max(8, rng.randint(24, 72) // p), degree=p, n_occ=n_occ,
                    ncols=n_occ + rng.randint(2, 6))
    if kind == "force":
        return dict(kind=kind, n_cells=max(8, rng.randint(24, 80) // p), degree=p, n_occ=n_occ,
                    n_eig=n_occ + rng.randint(3, 8), precision=rng.choice(["fp64", "mixed"]))
    return dict(kind=kind, n_cells=max(8, rng.randint(24, 80) // p), degree=p, n_occ=n_occ,
                n_eig=n_occ + _log_int(rng, 4, 44), precision=rng.choice(["fp64", "mixed"]))


# ------------------------------------------------- inputs (plain torch and numpy)
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _gll(p):
    """Gauss-Lobatto-Legendre nodes and weights of degree p on [-1, 1]."""
    c = np.zeros(p + 1)
    c[p] = 1.0
    dc = np.polynomial.legendre.legder(c)
    x = np.concatenate([[-1.0], np.sort(np.polynomial.legendre.legroots(dc)), [1.0]])
    for _ in range(3):  # Newton, so that the roots are good to rounding
        f = np.polynomial.legendre.legval(x[1:-1], dc)
        df = np.polynomial.legendre.legval(x[1:-1], np.polynomial.legendre.legder(dc))
        x[1:-1] -= f / df
    w = 2.0 / (p * (p + 1) * np.polynomial.legendre.legval(x, c) ** 2)
    return x, w


def _lagrange(nodes, x):
    """Values [len(x), n] and derivatives of the Lagrange basis on `nodes`."""
    n = len(nodes)
    v, d = np.ones((len(x), n)), np.zeros((len(x), n))
    for a in range(n):
        for m in range(n):
            if m != a:
                v[:, a] *= (x - nodes[m]) / (nodes[a] - nodes[m])
        for k in range(n):
            if k == a:
                continue
            t = np.full(len(x), 1.0 / (nodes[a] - nodes[k]))
            for m in range(n):
                if m not in (a, k):
                    t *= (x - nodes[m]) / (nodes[a] - nodes[m])
            d[:, a] += t
    return v, d


class Mesh:
    """The discretisation of include/idft.h in 64-bit torch: global 1D matrices
    of the uniform tensor-product mesh, applied along each axis in turn."""

    def __init__(self, n_cells, degree, device=None):
        self.nc, self.p, self.n1, self.q = n_cells, degree, degree + 1, degree + 3
        self.N1 = n_cells * degree + 1
        self.N = self.N1 ** 3
        self.nq = n_cells ** 3 * self.q ** 3
        self.h = 2.0 * HALF_WIDTH / n_cells
        self.dev = device or _device()
        gx, gw = _gll(degree)
        qx, qw = np.polynomial.legendre.leggauss(self.q)
        L, dL = _lagrange(gx, qx)
        M = L.T @ (qw[:, None] * L)
        D = dL.T @ (qw[:, None] * dL)
        Mg, Dg = np.zeros((self.N1, self.N1)), np.zeros((self.N1, self.N1))
        Lg = np.zeros((n_cells * self.q, self.N1))
        m = np.zeros(self.N1)
        x1, xq = np.zeros(self.N1), np.zeros(n_cells * self.q)
        for c in range(n_cells):
            s = slice(c * degree, c * degree + self.n1)
            Mg[s, s] += M
            Dg[s, s] += D
            Lg[c * self.q:(c + 1) * self.q, s] = L
            m[s] += gw
            x1[s] = -HALF_WIDTH + c * self.h + 0.5 * self.h * (gx + 1.0)
            xq[c * self.q:(c + 1) * self.q] = -HALF_WIDTH + c * self.h + 0.5 * self.h * (qx + 1.0)
        t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.Mg, self.Dg, self.Lg, self.x1, self.xq = t(Mg), t(Dg), t(Lg), t(x1), t(xq)
        self.J = (0.5 * self.h) ** 3
        m, inside = t(m), torch.ones(self.N1, dtype=torch.float64, device=self.dev)
        inside[0] = inside[-1] = 0.0
        self.inside = inside[:, None, None] * inside[None, :, None] * inside[None, None, :]
        self.mass = self.J * m[:, None, None] * m[None, :, None] * m[None, None, :]
        self.S = self.inside / self.mass.sqrt()
        w1 = t(np.tile(qw, n_cells))
        self.jxw = self.J * w1[:, None, None] * w1[None, :, None] * w1[None, None, :]

    def grid(self, field, x):
        """field(x, y, z) on the tensor grid of x, stored [z][y][x]."""
        return field(x[None, None, :], x[None, :, None], x[:, None, None])

    def to_cells(self, g):
        """[nc Q]^3 grid values as the flat [cell][q] layout."""
        n, q = self.nc, self.q
        return g.reshape(n, q, n, q, n, q).permute(0, 2, 4, 1, 3, 5).reshape(-1)

    def axes(self, Az, Ay, Ax, x):
        """(Az (x) Ay (x) Ax) x for x [z][y][x][col]."""
        nz, ny, nx, b = x.shape
        y = (Az @ x.reshape(nz, -1)).reshape(-1, ny, nx * b)
        y = torch.matmul(Ay, y).reshape(y.shape[0] * Ay.shape[0], nx, b)
        return torch.matmul(Ax, y).reshape(Az.shape[0], Ay.shape[0], Ax.shape[0], b)

    def weighted(self, w, x):
        """N^T diag(w) N x, w on the quadrature grid (JxW included)."""
        y = self.axes(self.Lg, self.Lg, self.Lg, x) * w[..., None]
        t = self.Lg.T.contiguous()
        return self.axes(t, t, t, y)

    def kinetic(self, x):
        """1/2 K x."""
        M, D = self.Mg, self.Dg
        return 0.25 * self.h * (self.axes(D, M, M, x) + self.axes(M, D, M, x)
                                + self.axes(M, M, D, x))

    def hamiltonian(self, v, x):
        """S H S x of the Loewdin Hamiltonian, columns taken a few at a time."""
        x = x.reshape(self.N1, self.N1, self.N1, -1)
        y = torch.empty_like(x)
        S = self.S[..., None]
        for j in range(0, x.shape[-1], 8):
            t = S * x[..., j:j + 8]
            y[..., j:j + 8] = S * (self.kinetic(t) + self.weighted(v * self.jxw, t))
        return y.reshape(self.N, -1)


def _atoms(g, n, spread=2.0):
    pos = (torch.rand(n, 3, generator=g, dtype=torch.float64) * 2 - 1) * spread
    z = torch.randint(2, 9, (n,), generator=g).double()
    return [(float(z[i]), [float(v) for v in pos[i]]) for i in range(n)]


def _wells(atoms):
    def field(x, y, z):
        v = 0.0
        for q, r in atoms:
            v = v - q / torch.sqrt((x - r[0]) ** 2 + (y - r[1]) ** 2 + (z - r[2]) ** 2 + 0.5)
        return v
    return field


def _bumps(g, n=8, amp=0.05):
    a = (torch.rand(n, generator=g, dtype=torch.float64) * 2 - 1) * amp
    s = torch.rand(n, generator=g, dtype=torch.float64) + 1.0
    c = (torch.rand(n, 3, generator=g, dtype=torch.float64) * 2 - 1) * 4.0

    def field(x, y, z):
        v = 0.0
        for k in range(n):
            e = lambda t, m: torch.exp(-(t - float(c[k, m])) ** 2 / (2 * float(s[k]) ** 2))  # noqa: E731
            v = v + float(a[k]) * e(x, 0) * e(y, 1) * e(z, 2)
        return v
    return field


def _potential(mesh, g):
    """Soft-Coulomb wells plus a smooth v_xc, on the quadrature grid."""
    wells, bumps = _wells(_atoms(g, 3)), _bumps(g)
    return mesh.grid(lambda x, y, z: wells(x, y, z) + bumps(x, y, z), mesh.xq)


def _orbitals(mesh, g, b):
    """b smooth orbital-like columns psi [N][b], M-orthonormal, zero on the
    boundary: Gaussians times low-order polynomials about random centres."""
    cols = torch.empty(mesh.N1, mesh.N1, mesh.N1, b, dtype=torch.float64, device=mesh.dev)
    x = mesh.x1
    for j in range(b):
        c = (torch.rand(3, generator=g, dtype=torch.float64) * 2 - 1) * 3.0
        a = 0.15 + 0.5 * float(torch.rand(1, generator=g))
        k = torch.randint(0, 3, (3,), generator=g)
        f = [(x - float(c[m])) ** int(k[m]) * torch.exp(-a * (x - float(c[m])) ** 2)
             for m in range(3)]
        cols[..., j] = f[2][:, None, None] * f[1][None, :, None] * f[0][None, None, :]
    cols *= mesh.inside[..., None]
    y = (mesh.mass.sqrt()[..., None] * cols).reshape(mesh.N, b)
    for _ in range(2):
        R = torch.linalg.cholesky(y.T @ y)
        y = y @ torch.linalg.inv(R).T.contiguous()
    return (y / mesh.mass.sqrt().reshape(-1, 1)).contiguous()


def _adjoint_inputs(case, seed):
    """Orbitals, occupancies, eigenvalues and u of an adjoint block."""
    g = torch.Generator().manual_seed(int(seed))
    mesh = Mesh(case["n_cells"], case["degree"])
    b = case["ncols"]
    v = _potential(mesh, g)
    psi = _orbitals(mesh, g, b)
    eig = np.sort(torch.rand(b, generator=g, dtype=torch.float64).numpy()) * 2.0 - 2.2
    if b >= 2:
        eig[1] = eig[0] + 1e-5  # one degenerate pair
    # the top state partly filled: 500 K smears the Fermi edge over 1.6 mHa
    fermi = eig[-1] + 5e-4
    occ = 1.0 / (1.0 + np.exp((eig - fermi) / (BOLTZMANN_HA * 500.0)))
    pairs = [(i, j) for i in range(b) for j in range(b) if abs(eig[i] - eig[j]) < 0.002]
    bumps = _bumps(g, amp=0.02)
    u = mesh.grid(bumps, mesh.xq)
    x = torch.randn(mesh.N, b, dtype=torch.float64, generator=g.manual_seed(int(seed) + 1)
                    ).to(mesh.dev) if mesh.N * b < 4_000_000 else torch.randn(
        mesh.N, b, dtype=torch.float64, device=mesh.dev,
        generator=torch.Generator(mesh.dev).manual_seed(int(seed) + 1))
    return mesh, dict(v=v, psi=psi, eig=eig, fermi=fermi, occ=occ, pairs=pairs, u=u, x=x)


# ------------------------------------------------------------------- the states
class DeviceBlock(abi.MultiVector):
    """A contract-2 handle over a torch tensor (idft_mv_wrap)."""

    def __init__(self, ctx, tensor):
        wrap = ctx.lib.idft_mv_wrap
        wrap.restype = C.c_int
        wrap.argtypes = [C.c_void_p, C.c_void_p, C.c_int32, C.POINTER(C.c_void_p)]
        self.ctx, self.ncols, self.tensor, self.h = ctx, tensor.shape[1], tensor, None
        h = C.c_void_p()
        ctx._check(wrap(ctx.h, C.c_void_p(tensor.data_ptr()), self.ncols, C.byref(h)))
        self.h = h


class State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def _adjoint_state(case, seed):
    lib = invdft_amd.load()
    mesh, a = _adjoint_inputs(case, seed)
    b = case["ncols"]
    desc = abi.default_desc(lib, n_cells=case["n_cells"], degree=case["degree"],
                            half_width=HALF_WIDTH, n_eig=b, n_electrons=2.0 * b)
    zq = np.zeros(mesh.nq)
    ctx = abi.Context(lib, desc, zq, zq, np.ones(mesh.nq), np.ones(mesh.N))
    ctx.set_veff_quad(mesh.to_cells(a["v"]).cpu().numpy())
    new = lambda: torch.zeros(mesh.N, b, dtype=torch.float64, device=mesh.dev)  # noqa: E731
    s = State(case=case, ctx=ctx, psi=DeviceBlock(ctx, a["psi"]), x=DeviceBlock(ctx, a["x"]))
    if case["kind"] == "vmult":
        s.out = DeviceBlock(ctx, new())
    if case["kind"] == "ends":
        s.out, s.rhs = DeviceBlock(ctx, new()), DeviceBlock(ctx, new())
    torch.cuda.synchronize()
    ctx.adj_update_input_psi(s.psi, a["occ"], mesh.to_cells(a["u"]).cpu().numpy(), a["pairs"],
                             a["fermi"], a["eig"])
    return s


def _well_levels(n_occ, g):
    """Atoms whose n_occ <= 8 lowest levels lie well below the next one: deep
    wells on the corners of a cube, each holding one occupied orbital."""
    atoms = []
    for k in range(n_occ):
        jitter = (torch.rand(3, generator=g, dtype=torch.float64) - 0.5) * 0.4
        corner = [(k >> m & 1) - 0.5 if n_occ > 1 << m else 0.0 for m in range(3)]
        atoms.append((4.0 + 0.06 * k, [3.0 * corner[m] + float(jitter[m]) for m in range(3)]))
    return atoms


def _solve_state(case, seed):
    """A caller of the adjoint problem with the eigenpairs of a potential."""
    lib = invdft_amd.load()
    g = torch.Generator().manual_seed(int(seed))
    mesh = Mesh(case["n_cells"], case["degree"])
    b, n_occ = case["ncols"], case["n_occ"]
    wells, bumps, du = _wells(_well_levels(n_occ, g)), _bumps(g), _bumps(g, amp=0.02)
    desc = abi.default_desc(lib, n_cells=case["n_cells"], degree=case["degree"],
                            half_width=HALF_WIDTH, n_eig=b, n_electrons=2.0 * n_occ)
    zq = np.zeros(mesh.nq)
    ctx = abi.Context(lib, desc, zq, zq, np.ones(mesh.nq), np.ones(mesh.N))
    v = mesh.grid(lambda x, y, z: wells(x, y, z) + bumps(x, y, z), mesh.xq)
    ctx.set_veff_quad(mesh.to_cells(v).cpu().numpy())
    eig, _, _ = ctx.eigensolve(1e-12, 200)
    occ, fermi = ctx.occupancies()
    psi = torch.from_numpy(ctx.eigenvectors()).to(mesh.dev)
    s = State(case=case, ctx=ctx, psi=DeviceBlock(ctx, psi),
              x=DeviceBlock(ctx, torch.zeros_like(psi)))
    pairs = [(i, j) for i in range(b) for j in range(b) if abs(eig[i] - eig[j]) < 0.002]
    torch.cuda.synchronize()
    ctx.adj_update_input_psi(s.psi, occ, mesh.to_cells(mesh.grid(du, mesh.xq)).cpu().numpy(),
                             pairs, fermi, eig)
    return s


def _force_state(case, seed):
    lib = invdft_amd.load()
    g = torch.Generator().manual_seed(int(seed))
    atoms = _well_levels(case["n_occ"], g)
    prob = synthetic.make_problem(
        lib, case["n_cells"], case["degree"], HALF_WIDTH, case["n_eig"], 2.0 * case["n_occ"],
        atoms, seed=int(seed) % 100000, target_tol=1e-8)
    tol = 1e-11
    ctx = prob.context(lib, precision=abi.MIXED if case["precision"] == "mixed" else abi.FP64,
                       cheb_tol=tol, initial_tol_cheb=tol)
    return State(case=case, ctx=ctx, pots=[prob.vxc0, 0.8 * prob.vxc0], turn=0)


def _charge(case, seed):
    """A molecule's electrons (positive) against its smeared nuclei."""
    g = torch.Generator().manual_seed(int(seed))
    mesh = Mesh(case["n_cells"], case["degree"])
    cs = []
    for q, r in _atoms(g, 3):
        for sign, a in ((1.0, 0.5 + 0.5 * float(torch.rand(1, generator=g))), (-0.9, 1.5)):
            cs.append((sign * q * (a / math.pi) ** 1.5, a, r))

    def field(x, y, z):
        v = 0.0
        for c, a, r in cs:
            v = v + c * torch.exp(-a * (x - r[0]) ** 2) * torch.exp(-a * (y - r[1]) ** 2) * \
                torch.exp(-a * (z - r[2]) ** 2)
        return v
    return mesh, mesh.grid(field, mesh.xq)


def _poisson_state(case, seed):
    lib = invdft_amd.load()
    mesh, c = _charge(case, seed)
    desc = abi.default_desc(lib, n_cells=case["n_cells"], degree=case["degree"],
                            half_width=HALF_WIDTH)
    fn = lib.idft_poisson_solve
    dp = C.POINTER(C.c_double)
    fn.restype = C.c_int
    fn.argtypes = [C.POINTER(abi.Desc), dp, dp, C.c_double, C.c_int32, dp, dp, C.c_void_p]
    return State(case=case, fn=fn, desc=desc, charge=mesh.to_cells(c).cpu().numpy(),
                 phi_q=np.zeros(mesh.nq), phi=np.zeros(mesh.N))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("force", "forward"):
        return _force_state(case, seed)
    if kind == "poisson":
        return _poisson_state(case, seed)
    if kind == "solve":
        return _solve_state(case, seed)
    return _adjoint_state(case, seed)


def run(s):
    kind = s.case["kind"]
    if kind == "vmult":
        s.ctx.adj_vmult(s.out, s.x)
        return s.out.tensor
    if kind == "ends":
        # the caller's own solver would leave its solution in s.out
        s.ctx.adj_compute_rhs(None, s.out, s.rhs)
        s.out.tensor.copy_(s.x.tensor)
        torch.cuda.current_stream().synchronize()
        s.ctx.adj_distribute_x()
        return {"rhs": s.rhs.tensor, "x": s.out.tensor}
    if kind in ("solve", "minres"):
        s.ctx.minres_solve(s.x, None, 1e-13, s.case.get("steps", 5000), distribute=True)
        return s.x.tensor
    if kind == "poisson":
        dp = C.POINTER(C.c_double)
        rc = s.fn(C.byref(s.desc), s.charge.ctypes.data_as(dp), None, 1e-12, 5000,
                  s.phi_q.ctypes.data_as(dp), s.phi.ctypes.data_as(dp), None)
        if rc:
            raise abi.IdftError(rc, "poisson")
        return {"phi_q": s.phi_q, "phi": s.phi}
    # an inversion moves the potential between evaluations
    pot = s.pots[s.turn % 2]
    s.turn += 1
    if kind == "force":
        force, loss = s.ctx.get_force(pot)
        return {"force": force, "loss": loss}
    loss = s.ctx.forward(pot)
    return {"loss": loss, "density": s.ctx.density(), "eigenvalues":
            s.ctx.eigenvalues()[:s.case["n_occ"]]}


# ------------------------------------------------------------------- the floor
def work(case):
    """Inputs read once, outputs written once, and the multiply-adds of the 1D
    contractions of the operator (7 kinetic and 6 interpolation products)."""
    nc, p = case["n_cells"], case["degree"]
    N, ncell, n1, q = (nc * p + 1) ** 3, nc ** 3, p + 1, p + 3
    contract = n1 * n1 * n1 * q + n1 * n1 * q * q + n1 * q * q * q
    apply_flops = 2.0 * ncell * (7 * n1 ** 4 + 2 * contract)
    nq = ncell * q ** 3
    kind = case["kind"]
    if kind == "vmult":
        b = case["ncols"]
        return dict(bytes=8.0 * (2 * N * b + nq), flops=apply_flops * b)
    if kind == "ends":
        b = case["ncols"]
        # rhs: psi in, rhs out, u in; distributeX: psi and x in, x out
        return dict(bytes=8.0 * (5 * N * b + nq), flops=4.0 * ncell * contract * b * 3)
    if kind in ("solve", "minres"):
        # a step's operator input and output, the older Lanczos vector, and one
        # pass each for the directions and the solution
        b, steps = case.get("n_occ", case["ncols"]), case.get("steps", 100)
        return dict(bytes=steps * 8.0 * (5 * N * b + nq), flops=steps * apply_flops * b)
    if kind == "poisson":
        steps = 100
        return dict(bytes=steps * 8.0 * 5 * N, flops=steps * 2.0 * ncell * 7 * n1 ** 4)
    # force and forward: a few filter passes of degree 30, then the adjoint steps
    b, s = case["n_eig"], 4 if case["precision"] == "mixed" else 8
    applies, steps = 90, 150 if kind == "force" else 0
    occ = case["n_occ"]
    return dict(bytes=applies * s * (4.0 * N * b + nq) + steps * 8.0 * (5 * N * occ + nq),
                flops=apply_flops * (applies * b + steps * occ))


# -------------------------------------------------------- the values in 64 bits
def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "force", "forward"):
        return None  # a whole eigensolve or adjoint: no quick plain counterpart
    if kind == "poisson":
        return _exact_poisson(case, seed)
    mesh, a = _adjoint_inputs(case, seed)
    if kind == "vmult":
        inside = mesh.inside.reshape(-1, 1)
        eps = torch.as_tensor(a["eig"], dtype=torch.float64, device=mesh.dev)
        return mesh.hamiltonian(a["v"], a["x"]) - eps * inside * a["x"]
    if kind == "ends":
        return _exact_ends(mesh, a)
    return None  # an iteration stopped by its step count


def _exact_ends(mesh, a):
    psi, b = a["psi"], a["psi"].shape[1]
    shape = (mesh.N1, mesh.N1, mesh.N1, b)
    inside = mesh.inside.reshape(-1, 1)
    sq = mesh.mass.sqrt().reshape(-1, 1)
    occ = torch.as_tensor(a["occ"], dtype=torch.float64, device=mesh.dev)

    def columns(w, t):
        y = torch.empty(shape, dtype=torch.float64, device=mesh.dev)
        for j in range(0, b, 8):
            y[..., j:j + 8] = mesh.weighted(w, t.reshape(shape)[..., j:j + 8].contiguous())
        return y.reshape(mesh.N, b)

    R = columns(a["u"] * mesh.jxw, psi)
    keep = torch.zeros(b, b, dtype=torch.float64, device=mesh.dev)
    for i, j in a["pairs"]:
        keep[i, j] = 1.0
    P = (psi.T @ R) * keep
    rhs = inside * (4.0 * occ * R / sq - 2.0 * sq * (psi @ (2.0 * occ[:, None] * P)))
    x = inside * a["x"] / sq
    dot = x.T @ columns(mesh.jxw, psi)
    f = occ
    dF = -f * (1.0 - f) / (BOLTZMANN_HA * 500.0)
    eta_r = -(dF * 2.0 * torch.diagonal(P)).sum()
    eta = 0.0 if abs(float(eta_r)) < 1e-16 else float(eta_r) / float(-dF.sum())
    corr = -dF[:, None] * 2.0 * P
    corr += torch.diag(dF * eta)
    x = x + psi @ ((corr - dot) * keep).T.contiguous()
    return {"rhs": rhs, "x": x}


def _exact_poisson(case, seed):
    """Dirichlet problem by the generalised eigenvectors of the 1D operators."""
    mesh, c = _charge(case, seed)
    w = c * mesh.jxw
    Q = float(w.sum())
    X = mesh.xq
    dip = [float((w * X[None, None, :]).sum()), float((w * X[None, :, None]).sum()),
           float((w * X[:, None, None]).sum())]

    def far(x, y, z):
        r = torch.sqrt(x * x + y * y + z * z).clamp_min(1e-3)
        return Q / r + (dip[0] * x + dip[1] * y + dip[2] * z) / r ** 3

    g = (mesh.grid(far, mesh.x1) * (1.0 - mesh.inside))[..., None]
    t = mesh.Lg.T.contiguous()
    f = 0.5 * mesh.axes(t, t, t, (4.0 * math.pi * w)[..., None]) - mesh.kinetic(g)
    i = slice(1, mesh.N1 - 1)
    M, D = mesh.Mg[i, i], mesh.Dg[i, i]
    R = torch.linalg.cholesky(M)
    Ri = torch.linalg.inv(R)
    lam, U = torch.linalg.eigh(Ri @ D @ Ri.T)
    V = (Ri.T @ U).contiguous()
    Vt = V.T.contiguous()
    y = mesh.axes(Vt, Vt, Vt, f[i, i, i].contiguous())
    y /= 0.25 * mesh.h * (lam[:, None, None] + lam[None, :, None] + lam[None, None, :])[..., None]
    phi = g.clone()
    phi[i, i, i] += mesh.axes(V, V, V, y)
    pq = mesh.axes(mesh.Lg, mesh.Lg, mesh.Lg, phi)[..., 0]
    return {"phi_q": mesh.to_cells(pq), "phi": phi.reshape(-1)}
