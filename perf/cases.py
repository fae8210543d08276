"""The work that programs have this library do, as measurable cases.

A case names a kind of call, an element type and its sizes; ``prepare``
builds the seeded model a Newton driver holds at its second load step (step
1 converged and committed, so every history word is read), ``run`` makes one
pass through the public calls of ``warp3d_amd`` on device buffers, and
``exact`` restates the outputs in plain 64-bit torch.

Kinds
  newton     one Newton iteration: recovery and forces, block tangents,
             sparse assembly (w3d_recover_dev, w3d_tangent,
             w3d_assemble_vss_dev)
  graph      the same iteration as one captured launch (w3d_iteration_dev)
  residual   recovery and forces alone: a line search or a modified-Newton
             residual (w3d_recover_dev)
  stiffness  tangents and assembly alone (w3d_tangent, w3d_assemble_vss_dev)
  asym       the asymmetric assembly's stiffness (w3d_tangent,
             w3d_assemble_csr_dev)
  pcg        the Jacobi-PCG solve of an assembled model (w3d_solve_pcg_dev)
  bicgstab   the nonsymmetric solve of an asymmetric assembly
             (w3d_solve_bicgstab, host vectors as the Fortran driver has)
  serve      a few small crystal-plasticity solves advanced together, from
             the request to the displacements (serve.Problem, serve.Batch)
"""
import math

import numpy as np
import torch

from warp3d_amd import _abi
from warp3d_amd import mesh as M
from warp3d_amd import serve as S
from warp3d_amd.model import BlockModel

# element kinds: (mesh builder, integration order, B-bar, nodes, points)
ELEMS = {
    "hex8": (M.box_hex8, 1, 1, 8, 8),
    "hex20": (M.box_hex20, 1, 0, 20, 27),
    "hex20r": (M.box_hex20, 8, 0, 20, 8),
    "tet10": (M.box_tet10, 4, 0, 10, 4),
}
PREC = {"fp64": _abi.W3D_FP64, "fp32": _abi.W3D_FP32}
SOLVE_RTOL = 1e-8
SERVE_STEPS = 4


def _case(name, kind, elem, nx, ny, nz, prec="fp64", mat="mm01",
          geonl=False):
    return dict(name=name, kind=kind, elem=elem, nx=nx, ny=ny, nz=nz,
                prec=prec, mat=mat, geonl=geonl)


def listed():
    return [
        # the 10^3 verification-size cube of a driver's first runs: launches
        # and host work count, not bandwidth
        _case("newton_hex8_1k", "newton", "hex8", 10, 10, 10),
        # the plain-against-mixed-precision box, 216,000 bricks
        _case("newton_hex8_216k", "newton", "hex8", 60, 60, 60, "fp32"),
        # bricks under finite strains and rotations, odd sizes
        _case("newton_hex8_geonl", "newton", "hex8", 31, 29, 23, "fp32",
              geonl=True),
        # the 27-point quadratic brick in double precision
        _case("newton_hex20_15k", "newton", "hex20", 24, 25, 26, "fp64"),
        # residual evaluations of a line search on the quadratic brick
        _case("residual_hex20_15k", "residual", "hex20", 25, 24, 25),
        # re-forming the stiffness with the reduced rule, FP32 tangent
        _case("stiffness_hex20r_12k", "stiffness", "hex20r", 25, 21, 23,
              "fp32"),
        # quadratic tetrahedra, the usual mesh of a curved part
        _case("newton_tet10_10k", "newton", "tet10", 11, 12, 13, "fp64"),
        # crystal plasticity on a mixed mesh in blocks of uneven spans
        _case("crystal_mixed_17k", "graph", "mixed", 24, 25, 24, "fp32",
              "mm10"),
        # the asymmetric assembly that crystal-plasticity decks switch on
        _case("asym_hex8_crystal", "asym", "hex8", 27, 28, 29, "fp64",
              "mm10"),
        # the equation solve of a Newton iteration
        _case("pcg_hex8_120k_eqs", "pcg", "hex8", 35, 34, 33),
        # the nonsymmetric equation solve
        _case("bicgstab_hex8", "bicgstab", "hex8", 15, 14, 13, "fp64",
              "mm10"),
        # three requests of the RVE server, start to finish of a load step
        _case("serve_rve_3", "serve", "hex8", 8, 9, 10, "fp32", "mm10"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind by its use, sides of the box log-uniform."""
    kind = rng.choice(["newton", "newton", "newton", "residual", "stiffness",
                       "graph", "asym", "pcg", "bicgstab", "serve"])
    mat, prec, geonl = "mm01", rng.choice(["fp64", "fp32"]), False
    if kind in ("newton", "residual", "stiffness"):
        elem = rng.choice(["hex8", "hex20", "hex20r", "tet10"])
        top = {"hex8": 45, "hex20": 22, "hex20r": 22, "tet10": 13}[elem]
        geonl = kind != "stiffness" and rng.random() < 0.2
    elif kind == "graph":
        elem, top, mat = rng.choice([("mixed", 22, "mm10"),
                                     ("hex8", 24, "mm10"),
                                     ("hex8", 40, "mm01"),
                                     ("tet10", 12, "mm10")])
    elif kind == "asym":
        elem, top = rng.choice([("hex8", 26), ("hex20r", 13)])
        prec, mat = "fp64", rng.choice(["mm01", "mm10"])
    elif kind == "pcg":
        elem, top, prec = "hex8", 32, "fp64"
    elif kind == "bicgstab":
        elem, top, prec, mat = "hex8", 15, "fp64", "mm10"
    else:
        elem, top, prec, mat = "hex8", 10, "fp32", "mm10"
    lo = {"mixed": 8, "tet10": 3}.get(elem, 8 if kind == "serve" else 4)
    n = [_logint(rng, lo, top) for _ in range(3)]
    c = _case("", kind, elem, n[0], n[1], n[2], prec, mat, geonl)
    del c["name"]
    return c


# ---------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------
def _material(case):
    if case["mat"] == "mm10":   # copper-like fcc, Voce hardening
        return _abi.mm10_material(tau_y=50.0, tau_v=100.0, theta_0=250.0,
                                  voce_m=1.0, harden_n=20.0, elastic="cubic",
                                  e=66.7e3, nu=0.42, mu=75.0e3)
    if case["elem"] == "hex8":
        return _abi.mm01_material(200e3, 0.3, 350.0, hprime=2000.0)
    return _abi.mm01_material(70e3, 0.33, 300.0, hprime=70e3 / 50)


def _inputs(case, seed):
    """Mesh, model arrays, constraints and the load step's displacement
    increment: an axial stretch that varies across the section, with a
    seeded perturbation of a few per cent of the element strains."""
    rng = np.random.default_rng(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = 1.0 / max(nx, ny, nz)
    size = (nx * h, ny * h, nz * h)
    mat, ang = _material(case), None
    if case["elem"] == "mixed":
        nt = [max(2, v // 4) for v in (nx, ny, nz)]
        nq = [max(2, v // 2) for v in (nx, ny, nz)]
        m = M.MixedMesh([
            (M.box_hex8(nx, ny, nz, size=size, jitter=0.05, seed=seed), 1, 1),
            (M.box_hex20(*nq, size=size, jitter=0.05, seed=seed + 1), 1, 0),
            (M.box_tet10(*nt, size=size, jitter=0.05, seed=seed + 2), 4, 0)])
        ang = M.random_orientations(m.noelem, seed=seed)
        arr = m.model(mat, elblks=m.seeded_blocks(32, 256, seed=seed),
                      angles=ang)
        parts = _parts(case)
    else:
        build, order, bbar, _, _ = ELEMS[case["elem"]]
        m = build(nx, ny, nz, size=size, jitter=0.05, seed=seed)
        if case["mat"] == "mm10":
            ang = M.random_orientations(m.noelem, seed=seed)
        arr = m.model(mat, int_order=order, bbar=bbar, auto_size=128,
                      angles=ang, geonl=case["geonl"])
        parts = [(case["elem"], m.noelem)]
    x = m.coords
    # per load step: past yield at most points by step 2 (for the crystal,
    # short of the increments at which its local solve asks for a cut)
    eps = 6.0e-4 if case["mat"] == "mm10" else 1.5e-3
    if case["geonl"]:
        eps = 2.0e-2
    s = 0.6 + 0.8 * (x[:, 0] - x[:, 0].min()) / np.ptp(x[:, 0])
    du = np.empty_like(x)
    du[:, 2] = eps * x[:, 2] * s
    du[:, 0] = -0.3 * eps * x[:, 2] * (x[:, 0] - x[:, 0].mean())
    du[:, 1] = -0.3 * eps * x[:, 2] * (x[:, 1] - x[:, 1].mean())
    if case["geonl"]:       # a rigid rotation about x grows with the step
        du[:, 1] += -0.05 * x[:, 2]
    du += 0.05 * eps * h * rng.uniform(-1, 1, size=du.shape)
    base = np.abs(x[:, 2]) < 1e-9
    cst = np.zeros(3 * m.nonode, np.int32)
    for k in range(3):
        cst[k::3][base] = 1
    du[base] = 0.0
    return dict(mesh=m, arr=arr, cst=cst, du=du.ravel(), parts=parts, ang=ang)


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def prepare(case, seed):
    """What the program has before the call: the device model at load step
    2, its displacement vectors and the buffers the results go to."""
    if case["kind"] == "serve":
        # the server's 0.2 % a step, to past yield in every grain
        specs = [S.RveSpec(case[k], seed=31 * seed + i,
                           strain=0.002 * SERVE_STEPS, nsteps=SERVE_STEPS)
                 for i, k in enumerate(("nx", "ny", "nz"))]
        return dict(case=case, rves=[S.make_rve(s) for s in specs],
                    opts=S.newton_opts(nsteps=SERVE_STEPS,
                                       precision=PREC[case["prec"]]))
    inp = _inputs(case, seed)
    model = BlockModel(inp["arr"])
    asym = case["kind"] in ("asym", "bicgstab")
    if asym:
        model.set_asymmetric(True)
    neq, nco = model.pattern(inp["cst"])
    nd = inp["du"].size
    st = dict(case=case, model=model, prec=PREC[case["prec"]],
              du=_dev(inp["du"]), u=_dev(np.zeros(nd)), ifv=_dev(np.zeros(nd)))
    torch.cuda.synchronize()
    p = {k: st[k].data_ptr() for k in ("u", "du", "ifv")}
    # load step 1: pseudo-update and one update, committed
    model.recover_dev(1, 0, p["u"], p["du"], p["ifv"])
    model.recover_dev(1, 1, p["u"], p["du"], p["ifv"])
    model.commit_step()
    st["u"].copy_(st["du"])
    torch.cuda.synchronize()
    if case["kind"] in ("stiffness", "asym", "bicgstab"):
        # (pcg: the elastic stiffness of the step's start)
        model.recover_dev(2, 1, p["u"], p["du"], p["ifv"])
    elif case["kind"] == "pcg":
        model.recover_dev(2, 0, p["u"], p["du"], p["ifv"])
    if asym:
        nnz = model.csr_pattern()[1].size
        st["val"] = torch.zeros(max(nnz, 1), dtype=torch.float64,
                                device="cuda")
    else:
        st["diag"] = torch.zeros(neq, dtype=torch.float64, device="cuda")
        st["coef"] = torch.zeros(max(nco, 1), dtype=torch.float64,
                                 device="cuda")
    torch.cuda.synchronize()
    if case["kind"] in ("pcg", "bicgstab"):
        rng = np.random.default_rng(seed + 17)
        rhs = rng.uniform(-1.0, 1.0, neq)
        model.tangent(2, 1, st["prec"])
        if asym:
            model.assemble_csr()
            st["rhs"] = rhs
        else:
            model.assemble_vss_dev(st["diag"].data_ptr(),
                                   st["coef"].data_ptr())
            st["rhs"], st["x"] = _dev(rhs), _dev(np.zeros(neq))
            torch.cuda.synchronize()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "serve":
        batch = S.Batch()
        probs = [S.Problem(r, st["opts"]) for r in st["rves"]]
        try:
            active = list(probs)
            while active:
                status = batch.advance(active)
                active = [p for p, s in zip(active, status)
                          if s in (_abi.W3D_PROBLEM_RUNNING,
                                   _abi.W3D_PROBLEM_STEP_DONE)]
            return [dict(u=p.u(), load=[r["load"] for r in p.records()])
                    for p in probs]
        finally:
            for p in probs:
                p.close()
            batch.close()
    m, prec = st["model"], st["prec"]
    if kind == "pcg":
        st["x"].zero_()
        torch.cuda.current_stream().synchronize()   # the library's own stream
        m.solve_pcg_dev(st["diag"].data_ptr(), st["coef"].data_ptr(),
                        st["rhs"].data_ptr(), st["x"].data_ptr(),
                        rtol=SOLVE_RTOL, maxit=5000)
        return dict(x=st["x"])
    if kind == "bicgstab":
        return dict(x=m.solve_bicgstab(st["rhs"], rtol=SOLVE_RTOL,
                                       maxit=5000)[0])
    out = {}
    p = {k: st[k].data_ptr() for k in ("u", "du", "ifv")}
    if kind == "graph":
        en, pw, _ = m.iteration_dev(2, 1, p["u"], p["du"], p["ifv"], prec,
                                    st["diag"].data_ptr(),
                                    st["coef"].data_ptr())
        return dict(ifv=st["ifv"], energy=en, plastic_work=pw,
                    diag=st["diag"], coef=st["coef"])
    if kind in ("newton", "residual"):
        en, pw, _ = m.recover_dev(2, 1, p["u"], p["du"], p["ifv"])
        out.update(ifv=st["ifv"], energy=en, plastic_work=pw)
    if kind in ("newton", "stiffness"):
        m.tangent(2, 1, prec)
        m.assemble_vss_dev(st["diag"].data_ptr(), st["coef"].data_ptr())
        out.update(diag=st["diag"], coef=st["coef"])
    if kind == "asym":
        m.tangent(2, 1, prec)
        m.assemble_csr_dev(st["val"].data_ptr())
        out.update(val=st["val"])
    return out


# ---------------------------------------------------------------------
# the work a pass cannot do without
# ---------------------------------------------------------------------
def _parts(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["elem"] != "mixed":
        k = 6 if case["elem"] == "tet10" else 1
        return [(case["elem"], k * nx * ny * nz)]
    q = [max(2, v // 2) for v in (nx, ny, nz)]
    t = [max(2, v // 4) for v in (nx, ny, nz)]
    return [("hex8", nx * ny * nz), ("hex20", q[0] * q[1] * q[2]),
            ("tet10", 6 * t[0] * t[1] * t[2])]


# words of the assembled upper triangle per element of a large mesh
UPPER = {"hex8": 123.0, "hex20": 1049.0, "hex20r": 1049.0, "tet10": 190.0}
# FP64 operations of one crystal update at these strains, counted with the
# powers apart: 11 residuals of 820, 8 first Jacobians of 2,900, 3.5 more
# columns of 2,000, 8 small factorisations of 340
MM10_FLOPS = 42.0e3


def work(case):
    b = f = 0.0
    kind = case["kind"]
    if kind == "serve":
        # about 30 Newton iterations over the steps, each an update of every
        # point, a stiffness and a solve of about 90 iterations
        for n in (case["nx"], case["ny"], case["nz"]):
            pts, nnz = 8.0 * n ** 3, 246.0 * n ** 3
            f += 30 * (pts * MM10_FLOPS + 90 * 2 * nnz)
            b += 30 * (pts * (2 * 158 + 45) * 8 + nnz * 8)
        return {"bytes": b, "flops": f}
    for elem, ne in _parts(case):
        _, _, _, nn, g = ELEMS[elem]
        t, pts = 3 * nn, ne * g
        nodes = ne * {"hex8": 1, "tet10": 1.4}.get(elem, 4)
        words = UPPER[elem] * ne
        if kind in ("newton", "graph", "residual"):
            # state words in and out, coordinates, u, du read, forces written
            state = 2 * 158 + 9 + 9 + 6 + 6 + 21 if case["mat"] == "mm10" \
                else 73
            b += pts * state * 8 + nodes * 12 * 8
            f += pts * (MM10_FLOPS if case["mat"] == "mm10" else 400.0)
            f += pts * nn * 60.0
        if kind in ("newton", "graph", "stiffness"):
            if kind == "stiffness":
                b += pts * 21 * 8
            b += words * 8
            f += pts * 2.0 * (36 * t + 6 * (t * (t + 1) // 2))
        if kind == "asym":
            b += pts * (36 if case["mat"] == "mm10" else 21) * 8
            b += 2 * words * 8
            f += pts * 2.0 * (36 * t + 6 * t * t)
        if kind in ("pcg", "bicgstab"):
            # the matrix and vectors once; some 9 iterations per layer of
            # elements, each a product with the matrix
            it = 9.0 * max(case["nx"], case["ny"], case["nz"])
            per = 2 if kind == "bicgstab" else 1
            b += per * words * 8 + 6 * nodes * 8
            f += it * per * 2 * 2 * words
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the difference that displacements perturbed in
    their last bits, the other tangent precision or another stopping
    iteration showed."""
    if case["kind"] == "serve":
        # Newton stops at 1e-4 of the reactions, its solves at 1e-6; one
        # solver iteration more moved the displacements by 1e-10, a Newton
        # iteration more would by 1e-8 and above
        return {"rel": 1e-7, "max": 1e-6}
    if case["kind"] == "pcg":       # stops at a relative residual of 1e-8
        return {"rel": 1e-7, "max": 6e-7}
    if case["kind"] == "bicgstab":  # the same, on a rougher descent
        return {"rel": 2e-6, "max": 6e-6}
    if case["mat"] == "mm10":
        # the local solves stop at a relative residual of 5e-5: forces are
        # within 8e-8 of the root's; the tangent is the last iterate's, so
        # a point that stops one iteration later moves its own entries
        return {"rel": 1e-6, "max": 1e-3}
    if case["prec"] == "fp32" and case["kind"] != "residual":
        return {"rel": 6e-7, "max": 6e-6}
    # points at the yield surface change branch with the last bits
    return {"rel": 4e-10, "max": 2e-7}


# ---------------------------------------------------------------------
# the same outputs in plain 64-bit torch
# ---------------------------------------------------------------------
def _hex_corner():
    return np.array([(-1, -1, 1), (-1, -1, -1), (-1, 1, -1), (-1, 1, 1),
                     (1, -1, 1), (1, -1, -1), (1, 1, -1), (1, 1, 1)], float)


def _rule(elem):
    """Points and weights of the integration rule (any order: the outputs
    are sums over the points)."""
    if elem == "tet10":
        a, b = 0.58541020, 0.13819660   # the tabulated rule, to its digits
        bary = np.full((4, 4), b) + (a - b) * np.eye(4)
        return bary[:, :3], np.full(4, 1.0 / 24.0)
    n = 3 if elem == "hex20" else 2
    p, w = np.polynomial.legendre.leggauss(n)
    i, j, k = [v.ravel() for v in np.meshgrid(range(n), range(n), range(n),
                                              indexing="ij")]
    return np.stack([p[i], p[j], p[k]], 1), w[i] * w[j] * w[k]


def _shape_derivs(elem, pts):
    """(points, 3, nodes) parametric derivatives of the shape functions."""
    if elem == "tet10":
        # barycentric L1..L3 are the coordinates, L4 = 1 - L1 - L2 - L3
        L = np.concatenate([pts, 1 - pts.sum(1, keepdims=True)], 1)
        dL = np.concatenate([np.eye(3), -np.ones((1, 3))])   # (4, 3)
        cols = [(4 * L[:, a, None] - 1) * dL[a] for a in range(4)]
        cols += [4 * (L[:, a, None] * dL[b] + L[:, b, None] * dL[a])
                 for a, b in ((0, 1), (1, 2), (0, 2), (0, 3), (1, 3), (2, 3))]
        return np.stack(cols, 2)
    if elem == "hex8":
        nat = _hex_corner()
        v = 1 + pts[:, None, :] * nat[None]
        d = [nat[:, k] * np.prod(np.delete(v, k, 2), 2) / 8 for k in range(3)]
        return np.stack(d, 1)
    nat = M.HEX20_NAT.astype(float)
    out = np.empty((len(pts), 3, 20))
    for a in range(20):
        c = nat[a]
        v = 1 + pts * c
        zero = np.flatnonzero(c == 0)
        for k in range(3):
            o = [m for m in range(3) if m != k]
            if len(zero) == 0:   # corner: prod(v)/8 (xi.c - 2)
                s = pts @ c - 2
                out[:, k, a] = c[k] * v[:, o[0]] * v[:, o[1]] * \
                    (s + v[:, k]) / 8
            elif k == zero[0]:
                out[:, k, a] = -2 * pts[:, k] * v[:, o[0]] * v[:, o[1]] / 4
            else:
                r = [m for m in o if m != zero[0]][0]
                out[:, k, a] = c[k] * v[:, r] * (1 - pts[:, zero[0]] ** 2) / 4
    return out


def _dvc():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a)).to(_dvc())


class _Kin:
    """Gradients of one element type's shape functions on given coordinates."""

    def __init__(self, elem, x):
        pts, w = _rule(elem)
        dn = _t(_shape_derivs(elem, pts))
        J = torch.einsum("gdj,ejc->egdc", dn, x)
        self.det = torch.linalg.det(J)
        if elem == "tet10" and float(self.det.mean()) < 0:
            self.det = -self.det
        self.grad = torch.einsum("egcd,gdj->egjc", torch.linalg.inv(J), dn)
        self.w = _t(w)
        self.bar = None
        if ELEMS[elem][2]:
            v = (self.grad * self.det[..., None, None]).sum(1)
            self.bar = v / self.det.sum(1)[:, None, None]

    def strain(self, u):
        H = torch.einsum("ejc,egjk->egck", u, self.grad)
        e = torch.stack([H[..., 0, 0], H[..., 1, 1], H[..., 2, 2],
                         H[..., 0, 1] + H[..., 1, 0],
                         H[..., 1, 2] + H[..., 2, 1],
                         H[..., 0, 2] + H[..., 2, 0]], -1)
        if self.bar is not None:
            tr = e[..., 0] + e[..., 1] + e[..., 2]
            trb = (u * self.bar).sum((1, 2))[:, None]
            e[..., :3] += ((trb - tr) / 3)[..., None]
        return e

    def forces(self, sig):
        s = _sym33(sig)
        wd = self.w * self.det
        f = torch.einsum("eg,egck,egjk->ejc", wd, s, self.grad)
        if self.bar is not None:
            p = (sig[..., 0] + sig[..., 1] + sig[..., 2]) / 3 * wd
            f = f + torch.einsum("eg,egjc->ejc", p,
                                 self.bar[:, None] - self.grad)
        return f

    def bmat(self, lo, hi):
        """(elements, points, 6, 3 nodes + component) of elements lo..hi"""
        g = self.grad[lo:hi]
        ne, G, nn, _ = g.shape
        B = torch.zeros(ne, G, 6, nn, 3, dtype=g.dtype, device=g.device)
        for c in range(3):
            B[:, :, c, :, c] = g[..., c]
        for r, a, b in ((3, 0, 1), (4, 1, 2), (5, 0, 2)):
            B[:, :, r, :, a] = g[..., b]
            B[:, :, r, :, b] = g[..., a]
        if self.bar is not None:
            d = (self.bar[lo:hi, None] - g) / 3
            for r in range(3):
                B[:, :, r] += d
        return B.reshape(ne, G, 6, 3 * nn)


def _sym33(v):
    return torch.stack([torch.stack([v[..., 0], v[..., 3], v[..., 5]], -1),
                        torch.stack([v[..., 3], v[..., 1], v[..., 4]], -1),
                        torch.stack([v[..., 5], v[..., 4], v[..., 2]], -1)],
                       -2)


def _vec6(s, shear):
    return torch.stack([s[..., 0, 0], s[..., 1, 1], s[..., 2, 2],
                        shear * s[..., 0, 1], shear * s[..., 1, 2],
                        shear * s[..., 0, 2]], -1)


class _Mises:
    """Isotropic-hardening radial return with its consistent tangent."""

    def __init__(self, mat):
        self.e, self.nu = float(mat.e), float(mat.nu)
        self.y = float(mat.yld_pt)
        f = np.float32   # the property table is single precision
        self.h = float(f(f(mat.e) * f(mat.tan_e) /
                         f(f(mat.e) - f(mat.tan_e))))
        self.g = self.e / 2 / (1 + self.nu)
        self.k = self.e / 3 / (1 - 2 * self.nu)

    def elastic(self, like):
        D = torch.zeros(like.shape[:-1] + (6, 6), dtype=like.dtype,
                        device=like.device)
        D[..., :3, :3] = self.k - 2 * self.g / 3
        for i in range(3):
            D[..., i, i] += 2 * self.g
            D[..., 3 + i, 3 + i] = self.g
        return D

    def update(self, st, de, tangent):
        """st: (stress, plastic strain, energy, plastic work) at n"""
        sig, ep, en, pw = st
        ones = torch.tensor([1., 1, 1, 0, 0, 0], dtype=de.dtype,
                            device=de.device)
        two = torch.tensor([1., 1, 1, 2, 2, 2], dtype=de.dtype,
                           device=de.device)
        half = torch.tensor([1., 1, 1, .5, .5, .5], dtype=de.dtype,
                            device=de.device)
        dv = (de * ones).sum(-1, keepdim=True)
        p = (sig * ones).sum(-1, keepdim=True) / 3 + self.k * dv
        s = sig - (sig * ones).sum(-1, keepdim=True) / 3 * ones + \
            2 * self.g * half * (de - dv / 3 * ones)
        nrm = (s * s * two).sum(-1).sqrt()
        r = math.sqrt(2.0 / 3.0)
        over = nrm - r * (self.y + self.h * ep)
        plastic = over >= 1e-7 * r * (self.y + self.h * ep)
        lam = torch.where(plastic, over / (2 * self.g + 2 * self.h / 3),
                          torch.zeros_like(over))
        scale = 1 - 2 * self.g * lam / nrm.clamp_min(1e-300)
        s1 = s * scale[..., None]
        ep1 = ep + r * lam
        sig1 = s1 + p * ones

        def vm(a):
            d = a - (a * ones).sum(-1, keepdim=True) / 3 * ones
            return (1.5 * (d * d * two).sum(-1)).sqrt()
        en1 = en + 0.5 * (de * (sig1 + sig)).sum(-1)
        pw1 = pw + torch.where(plastic, 0.5 * (vm(sig1) + vm(sig)) *
                               (ep1 - ep), torch.zeros_like(ep))
        D = None
        if tangent:
            D = self.elastic(de)
            bb = r * (self.y + self.h * ep1) / nrm.clamp_min(1e-300)
            gam = 1 / (1 + self.h / (3 * self.g)) - 1 + bb
            n = s / nrm.clamp_min(1e-300)[..., None]
            P = torch.diag(half) - torch.outer(ones, ones) / 3
            Dp = self.k * torch.outer(ones, ones) + \
                2 * self.g * bb[..., None, None] * P - \
                2 * self.g * gam[..., None, None] * n[..., :, None] * \
                n[..., None, :]
            D = torch.where(plastic[..., None, None], Dp, D)
        return (sig1, ep1, en1, pw1), D


def _voigt_rot(R):
    """6x6 rotation of (xx, yy, zz, xy, yz, xz) with tensor shears."""
    pair = ((0, 0), (1, 1), (2, 2), (0, 1), (1, 2), (0, 2))
    rows = []
    for a, b in pair:
        cols = []
        for c, d in pair:
            v = R[..., a, c] * R[..., b, d]
            if c != d:
                v = v + R[..., a, d] * R[..., b, c]
            cols.append(v)
        rows.append(torch.stack(cols, -1))
    return torch.stack(rows, -2)


def _spin_rot(T):
    """Rotation of the skew vectors (yz, xz, xy) under T A T^T."""
    pr = ((1, 2), (0, 2), (0, 1))
    return torch.stack([torch.stack(
        [T[..., a, c] * T[..., b, d] - T[..., a, d] * T[..., b, c]
         for c, d in pr], -1) for a, b in pr], -2)


def _symsw(s, w):
    s0, s1, s2, s3, s4, s5 = s.unbind(-1)
    a, b, c = w.unbind(-1)
    return torch.stack([
        s3 * c - s5 * b, s3 * c - s4 * a, s5 * b + s4 * a,
        0.5 * (c * (s0 - s1) + a * s5 - b * s4),
        0.5 * (a * (s1 - s2) + b * s3 + c * s5),
        0.5 * (b * (s0 - s2) + a * s3 - c * s4)], -1)


class _Crystal:
    """Rate-dependent fcc crystal with Voce hardening: the root of the
    implicit update, one crystal per point."""

    def __init__(self, mat, angles):
        self.m = mat
        psi, th, phi = [_t(np.radians(angles[:, k])) for k in range(3)]
        g = torch.stack([
            -psi.sin() * phi.sin() - psi.cos() * phi.cos() * th.cos(),
            psi.cos() * phi.sin() - psi.sin() * phi.cos() * th.cos(),
            phi.cos() * th.sin(),
            psi.sin() * phi.cos() - psi.cos() * phi.sin() * th.cos(),
            -psi.cos() * phi.cos() - psi.sin() * phi.sin() * th.cos(),
            phi.sin() * th.sin(), psi.cos() * th.sin(),
            psi.sin() * th.sin(), th.cos()], -1).reshape(-1, 3, 3)
        gt = g.transpose(-1, -2)
        n = np.repeat([[1, 1, 1], [-1, -1, 1], [-1, 1, 1], [1, -1, 1]], 3, 0)
        b = np.array([[0, -1, 1], [1, 0, -1], [-1, 1, 0], [0, 1, 1],
                      [1, 0, 1], [1, -1, 0], [0, -1, 1], [-1, 0, -1],
                      [1, 1, 0], [0, 1, 1], [1, 0, -1], [-1, -1, 0]])
        bs = torch.einsum("pij,sj->psi", gt, _t(b / math.sqrt(2.0)))
        ns = torch.einsum("pij,sj->psi", gt, _t(n / math.sqrt(3.0)))
        A = bs[..., :, None] * ns[..., None, :]
        At = A.transpose(-1, -2)
        self.ms0 = _vec6(0.5 * (A + At), 2.0)
        W = 0.5 * (A - At)
        self.q0 = torch.stack([W[..., 1, 2], W[..., 0, 2], W[..., 0, 1]], -1)
        e, v, u = mat.cp_e, mat.cp_nu, mat.cp_mu
        c0 = np.zeros((6, 6))
        c0[:3, :3] = -v / e
        np.fill_diagonal(c0[:3, :3], 1 / e)
        c0[range(3, 6), range(3, 6)] = 2 * (1 + v) / e \
            if mat.elastic_type == 1 else 1 / u
        R = _voigt_rot(gt)
        self.C = R @ _t(np.linalg.inv(c0)) @ R.transpose(-1, -2)

    def update(self, st, D, points, dt=1.0):
        """st: (stress, Rp, tau, energy, plastic work) of points x G"""
        mt = self.m
        sn, Rp, tau_n, en, pw = st
        T = Rp.transpose(-1, -2)
        C, ms0, q0 = self.C[points], self.ms0[points], self.q0[points]
        ms = torch.einsum("pij,psj->psi", _voigt_rot(T), ms0)
        qs = torch.einsum("pij,psj->psi", _spin_rot(T), q0)
        Cm = torch.einsum("pij,psj->psi", C, ms)
        CD = torch.einsum("pij,pj->pi", C, D)
        dg = (2 / 3 * ((D[:, :3] ** 2).sum(-1) +
                       0.5 * (D[:, 3:] ** 2).sum(-1))).sqrt()
        n, th = mt.harden_n, mt.theta_0
        eye = torch.eye(6, dtype=D.dtype, device=D.device)

        def slips(x, tt):
            rs = torch.einsum("psi,pi->ps", ms, x)
            return (dg / tt)[:, None] * (rs / tt[:, None]).abs() ** (n - 1) * \
                rs, rs

        def resid(x, tt):
            gam, _ = slips(x, tt)
            wp = torch.einsum("ps,psk->pk", gam, qs)
            r1 = x - sn - CD + torch.einsum("ps,psi->pi", gam, Cm) + \
                2 * _symsw(x, wp)
            ht = 1 - (tt - mt.tau_y) / mt.tau_v
            f = ht.abs() ** mt.voce_m * torch.sign(ht)
            r2 = tt - tau_n - th * f * gam.abs().sum(-1)
            return torch.cat([r1, r2[:, None]], -1)

        def jac(x, tt):
            gam, rs = slips(x, tt)
            dx = (n * dg / tt)[:, None] * (rs / tt[:, None]).abs() ** (n - 1)
            dgx = dx[..., None] * ms
            cw = Cm + 2 * _symsw(x[:, None].expand(-1, 12, -1), qs)
            wp = torch.einsum("ps,psk->pk", gam, qs)
            lin = torch.stack([_symsw(eye[k].expand(len(x), 6), wp)
                               for k in range(6)], -1)
            J = torch.empty(len(x), 7, 7, dtype=x.dtype, device=x.device)
            J[:, :6, :6] = eye + torch.einsum("psi,psj->pij", cw, dgx) + \
                2 * lin
            J[:, :6, 6] = torch.einsum("ps,psi->pi", -n * gam / tt[:, None],
                                       cw)
            ht = 1 - (tt - mt.tau_y) / mt.tau_v
            f = ht.abs() ** mt.voce_m * torch.sign(ht)
            fp = -mt.voce_m / mt.tau_v * ht.abs() ** (mt.voce_m - 1)
            ga = gam.abs().sum(-1)
            J[:, 6, :6] = -th * f[:, None] * torch.einsum(
                "ps,psi->pi", torch.sign(gam), dgx)
            J[:, 6, 6] = 1 - th * (fp * ga - f * n * ga / tt)
            return J

        x, tt = sn.clone(), tau_n.clone()
        r = resid(x, tt)
        nr = r.norm(dim=-1)
        for _ in range(120):
            if float(nr.max()) < 1e-9:
                break
            d = torch.linalg.solve(jac(x, tt), -r)
            a = torch.ones_like(tt)
            for _ in range(25):
                xn, tn = x + a[:, None] * d[:, :6], tt + a * d[:, 6]
                rn = resid(xn, tn)
                nn = rn.norm(dim=-1)
                bad = ~(nn <= (1 - 1e-4 * a) * nr) & (nr >= 1e-9)
                if not bool(bad.any()):
                    break
                a = torch.where(bad, 0.5 * a, a)
            keep = nr < 1e-9
            x = torch.where(keep[:, None], x, xn)
            tt = torch.where(keep, tt, tn)
            r = torch.where(keep[:, None], r, rn)
            nr = torch.where(keep, nr, nn)
        gam, _ = slips(x, tt)
        wp = torch.einsum("ps,psk->pk", gam, qs)
        W = torch.zeros(len(x), 3, 3, dtype=x.dtype, device=x.device)
        for k, (i, j) in enumerate(((1, 2), (0, 2), (0, 1))):
            W[:, i, j], W[:, j, i] = wp[:, k], -wp[:, k]
        ee = torch.linalg.solve(C, x)
        ep = torch.einsum("ps,psi->pi", gam, ms) + _symsw(ee, wp)
        return (x, torch.linalg.matrix_exp(W) @ Rp, tt,
                en + (x * D).sum(-1), pw + (x * ep).sum(-1))


def _assemble(case, inp, blocks, full):
    """The assembled values of element stiffness blocks: upper triangle
    (diagonal, coefficients) or the full rows, by sorted equation pairs."""
    cst = _t(inp["cst"])
    eq = torch.cumsum((cst == 0).long(), 0) - 1
    eq[cst != 0] = -1
    neq = int((cst == 0).sum())
    keys, vals = [], []
    for conn, Ke in blocks:
        dof = (3 * conn[:, :, None] + torch.arange(3, device=conn.device)) \
            .reshape(len(conn), -1)
        e = eq[dof]
        r, c = e[:, :, None].expand_as(Ke), e[:, None, :].expand_as(Ke)
        ok = (r >= 0) & (c >= 0)
        if not full:
            ok &= c >= r
        keys.append((r * neq + c)[ok])
        vals.append(Ke[ok])
    uniq, inv = torch.unique(torch.cat(keys), return_inverse=True)
    out = torch.zeros(len(uniq), dtype=torch.float64, device=uniq.device)
    out.index_add_(0, inv, torch.cat(vals))
    return neq, uniq // neq, uniq % neq, out


def _cg(neq, row, col, val, b):
    """Jacobi-CG on the upper triangle, to a residual of 1e-14."""
    off = row != col
    r = torch.cat([row, col[off]])
    c = torch.cat([col, row[off]])
    A = torch.sparse_coo_tensor(torch.stack([r, c]),
                                torch.cat([val, val[off]]),
                                (neq, neq)).coalesce().to_sparse_csr()
    d = torch.zeros(neq, dtype=val.dtype, device=val.device)
    d[row[~off]] = val[~off]
    x, res = torch.zeros_like(b), b.clone()
    z = res / d
    p, rz, b0 = z.clone(), res @ z, b.norm()
    for _ in range(4000):
        q = A @ p
        a = rz / (p @ q)
        x += a * p
        res -= a * q
        if float(res.norm()) < 1e-14 * float(b0):
            break
        z = res / d
        rz, old = res @ z, rz
        p = z + rz / old * p
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve" or (kind in ("asym", "bicgstab") and
                           case["mat"] == "mm10"):
        # a path of stopped iterations; the crystal's tangent is its last
        # local iterate's
        return None
    inp = _inputs(case, seed)
    m, arr = inp["mesh"], inp["arr"]
    X, du = _t(m.coords), _t(inp["du"]).reshape(-1, 3)
    incid, incmap = arr.incid - 1, arr.incmap - 1
    ifv = torch.zeros_like(X)
    energy = plastic = 0.0
    blocks, e0 = [], 0
    stiff = kind in ("newton", "stiffness", "asym", "pcg", "graph") and \
        case["mat"] != "mm10" and not case["geonl"]
    for elem, ne in inp["parts"]:
        nn = ELEMS[elem][3]
        conn = _t(incid[incmap[e0]:incmap[e0] + ne * nn].astype(np.int64)
                  .reshape(ne, nn))
        xe, due = X[conn], du[conn]
        G = ELEMS[elem][4]
        z = torch.zeros(ne, G, dtype=torch.float64, device=X.device)
        z6 = torch.zeros(ne, G, 6, dtype=torch.float64, device=X.device)
        k0 = _Kin(elem, xe)
        D, kin, factor = None, k0, k0.det
        if case["mat"] == "mm10":
            cr = _Crystal(arr.materials[0],
                          inp["ang"][e0:e0 + ne].reshape(-1, 3))
            pts = torch.arange(ne, device=X.device).repeat_interleave(G)
            eye = torch.eye(3, dtype=torch.float64, device=X.device)
            st = (z6.reshape(-1, 6), eye.expand(ne * G, 3, 3),
                  z.reshape(-1) + arr.materials[0].tau_y + 1e-5,
                  z.reshape(-1), z.reshape(-1))
            de = k0.strain(due).reshape(-1, 6)
            for _ in range(2):
                st = cr.update(st, de, pts)
            sig, en, pw = (v.reshape(ne, G, *v.shape[1:])
                           for v in (st[0], st[3], st[4]))
        else:
            mm = _Mises(arr.materials[0])
            st = (z6, z, z.clone(), z.clone())
            I = torch.eye(3, dtype=torch.float64, device=X.device)
            for step in range(2):
                de = None
                if case["geonl"]:
                    u0 = due * step

                    def rot(a):
                        F = I + torch.einsum("ejc,egjk->egck", a, k0.grad)
                        U, _, Vh = torch.linalg.svd(F)
                        return U @ Vh, torch.linalg.det(F)
                    mid = _Kin(elem, xe + u0 + 0.5 * due)
                    Rh, _ = rot(u0 + 0.5 * due)
                    R1, dF = rot(u0 + due)
                    d = mid.strain(due)
                    half = torch.tensor([1., 1, 1, .5, .5, .5],
                                        dtype=d.dtype, device=d.device)
                    de = _vec6(Rh.transpose(-1, -2) @ _sym33(d * half) @ Rh,
                               2.0)
                else:
                    de = k0.strain(due)
                elastic = kind == "pcg" and step == 1
                if elastic:
                    D = mm.elastic(de)
                else:
                    st, D = mm.update(st, de, stiff and step == 1)
            sig, _, en, pw = st
            if case["geonl"]:
                kin = _Kin(elem, xe + 2 * due)
                sig = _vec6(R1 @ _sym33(sig) @ R1.transpose(-1, -2), 1.0)
                factor = k0.det * dF
        if kind in ("newton", "graph", "residual"):
            ifv.index_add_(0, conn.reshape(-1),
                           kin.forces(sig).reshape(-1, 3))
            # the reference's energy sums leave out the tetrahedron's 1/6
            wt = kin.w * (6.0 if elem == "tet10" else 1.0)
            energy += float((en * factor * wt).sum())
            plastic += float((pw * factor * wt).sum())
        if stiff:
            step = max(1, 2 ** 27 // (G * 18 * nn * 8))
            for a in range(0, ne, step):
                b = min(ne, a + step)
                B = k0.bmat(a, b)
                wd = (k0.w * k0.det)[a:b]
                DB = torch.einsum("egrs,egst->egrt",
                                  D[a:b] * wd[..., None, None], B)
                g = b - a
                Ke = B.reshape(g, G * 6, -1).transpose(1, 2) @ \
                    DB.reshape(g, G * 6, -1)
                blocks.append((conn[a:b], Ke))
        e0 += ne
    out = {}
    if kind in ("newton", "graph", "residual"):
        out = dict(ifv=ifv.reshape(-1), energy=energy, plastic_work=plastic)
    if kind in ("newton", "graph", "stiffness"):
        out.update(diag=None, coef=None)
    if stiff:
        neq, row, col, val = _assemble(case, inp, blocks, kind == "asym")
        if kind == "asym":
            out["val"] = val
        elif kind == "pcg":
            rng = np.random.default_rng(seed + 17)
            out["x"] = _cg(neq, row, col, val,
                           _t(rng.uniform(-1.0, 1.0, neq)))
        else:
            out["diag"], out["coef"] = val[row == col], val[row != col]
    return out
