"""The work that users of this framework have it do, as cases to measure.

A SIMP program (bin/top3d, top3d_amd.design_loop) spends its time in the MGCG
state solve and, around it, in the sensitivity, the density filter and the
optimality-criteria update.  A program with a driver of its own calls the
same entry points one by one: the operators, smoothers and transfers, the
filter and its transpose, the compliance as a torch.autograd.Function.  The
grids are those of the reference's own command lines (coarse 12x6x6 with 3
levels, coarse 16x8x8 with 4, 5 and 6 levels), of the differentiation check
(64x32x32, 3 levels), and ragged ones whose coarse grids are odd.

A Grid (its levels, element matrices and solver buffers) is what a program
makes once and keeps for the whole optimisation, so the states of one grid
share it.  Densities are fields of an optimisation under way: smooth material
around the volume fraction, drawn towards 0 and 1 as the loop goes on.  The
solves take those of the first design iterations (7 or 8 CG iterations): with
the reference's V-cycle the count of later ones depends on the last bits.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "topopt-in-openmp-gpu_amd"))
import top3d_amd  # noqa: E402

E0, EMIN, NU = 1.0, 1e-6, 0.3
TOL = float(np.float32(1e-5))
VOLFRAC = float(np.float32(0.2))


def listed():
    """Twelve cases, smallest grids first.  `stage`: how far the densities
    are from uniform (0) towards a near 0/1 design (1)."""
    def case(name, kind, nelx, nely, nelz, nl, precision="fp64", bc="reference", stage=0.1,
             rmin=1.5):
        return dict(name=name, kind=kind, nelx=nelx, nely=nely, nelz=nelz, nl=nl,
                    precision=precision, bc=bc, stage=stage, rmin=rmin)

    return [
        # one matvec on the smallest reference grid: a program that applies
        # K to a vector of its own (latency)
        case("operator_48", "operator", 48, 24, 24, 3),
        # a whole design iteration of `top3d -x 12 -y 6 -z 6 -l 3`, FP64
        case("design_fp64_48", "design", 48, 24, 24, 3),
        # the differentiation check: c(x) and dc/dx through the filter for an
        # optimiser of the user's own, symmetric supports, FP64
        case("gradient_fp64_64", "gradient", 64, 32, 32, 3, bc="symmetric"),
        # a ragged grid (odd coarse 15x7x9), mixed form
        case("solve_mixed_120", "solve", 120, 56, 72, 4, "mixed", "symmetric"),
        # `top3d -x 16 -y 8 -z 8 -l 4`: the FP64 state solve
        case("solve_fp64_128", "solve", 128, 64, 64, 4),
        # smoothing and transfers called one by one on that grid: a
        # multigrid cycle that a program writes itself
        case("cycle_128", "cycle", 128, 64, 64, 4),
        # the filter and its transpose at a large radius on a ragged grid
        case("filter_wide_168", "filter", 168, 72, 104, 4, stage=0.6, rmin=3.5),
        # the OC update, change, filter and volume at the benchmark's size
        case("update_256", "update", 256, 128, 128, 5, stage=0.6),
        # the filter and its transpose at the default radius
        case("filter_256", "filter", 256, 128, 128, 5, stage=0.6),
        # the benchmark: a design iteration, mixed; the state solve in FP64
        case("design_mixed_256", "design", 256, 128, 128, 5, "mixed"),
        case("solve_fp64_256", "solve", 256, 128, 128, 5),
        # the largest single-GPU run: autograd compliance and gradient, mixed
        case("gradient_mixed_512", "gradient", 512, 256, 256, 6, "mixed"),
    ]


def draw(rng):
    """A grid of 13 thousand to 33 million elements (spread over the
    logarithm), odd coarse sizes among them, and a kind of call on it."""
    kind = rng.choice(["operator", "design", "gradient", "solve", "solve", "cycle", "filter",
                       "update"])
    while True:
        target = math.exp(rng.uniform(math.log(13e3), math.log(33e6)))
        nl = rng.choice([n for n in (3, 4, 5, 6) if 48 <= target / 8 ** (n - 1) <= 1024] or [3])
        cy, cz = rng.randint(3, 12), rng.randint(3, 12)
        cx = max(3, round(target / 8 ** (nl - 1) / (cy * cz)))
        f = 2 ** (nl - 1)
        if cx <= 24 and (cx + 1) * (cy + 1) * (cz + 1) <= 1377 and cx * cy * cz * f ** 3 < 34e6:
            break
    return dict(kind=kind, nelx=cx * f, nely=cy * f, nelz=cz * f, nl=nl,
                precision=rng.choice(["mixed", "fp64"]) if cx * cy * cz * f ** 3 < 9e6 else "mixed",
                bc=rng.choice(["reference", "symmetric"]), stage=round(rng.uniform(0.0, 0.1), 3),
                rmin=rng.choice([1.5, 1.5, 2.0, 2.5, 3.5]))


# ---- inputs -----------------------------------------------------------------
_kept = {}  # the program's one Grid and what goes with it


def _grid(case):
    key = tuple(case[k] for k in ("nelx", "nely", "nelz", "nl", "precision", "bc"))
    if key not in _kept:
        _kept.clear()
        g = top3d_amd.Grid(*key[:4], precision=case["precision"], bc=case["bc"])
        _kept[key] = (g, g.load())
    return _kept[key]


def _elements(g, a):
    """The real elements of a padded element array, as (x, z, y)."""
    v = a.view(g.nelx + 2, g.nelz + 2, g.nely + 2)
    return v[1:-1, 1:-1, 1:-1]


def _smooth(shape, cells, gen):
    """Smooth random field: normal values `cells` elements apart."""
    size = [max(2, -(-s // cells) + 1) for s in shape]
    f = torch.randn([1, 1] + size, dtype=torch.float64, device="cuda", generator=gen)
    return torch.nn.functional.interpolate(f, size=list(shape), mode="trilinear",
                                           align_corners=True)[0, 0]


def _density(case, g, gen):
    """Design variables of an optimisation under way, in [0.001, 1], mean
    near the volume fraction."""
    shape = (g.nelx, g.nelz, g.nely)
    f = _smooth(shape, 8, gen) + 0.3 * _smooth(shape, 3, gen)
    x = VOLFRAC * (1.0 + 0.15 * f)
    bars = torch.sigmoid(6.0 * (f - 0.8))
    s = case["stage"]
    full = torch.zeros(g.nelem, dtype=torch.float64, device="cuda")
    _elements(g, full).copy_(((1.0 - s) * x + s * bars).clamp(0.001, 1.0))
    return full


def _nodal(g, l, gen):
    """A displacement-like field on the real nodes of level l, zero halo."""
    _, wx, wy, wz, _ = g.padding(l)
    v = torch.zeros(wx, wz, wy, 3, dtype=torch.float64, device="cuda")
    r = torch.randn(wx - 2, wz - 2, wy - 2, 3, dtype=torch.float64, device="cuda", generator=gen)
    v[1:-1, 1:-1, 1:-1] = r
    return v.reshape(-1)


def prepare(case, seed):
    g, F = _grid(case)
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    s = dict(kind=kind, g=g, F=F, rmin=case["rmin"])
    s["x"] = x = _density(case, g, gen)
    if kind == "operator":
        s["v"] = _nodal(g, 0, gen)
    elif kind == "cycle":
        s["u"], s["b"] = _nodal(g, 0, gen), _nodal(g, 0, gen)
        s["invD"] = [g.invdiag(x, l) for l in (0, 1)]
    elif kind == "filter":
        s["up"] = torch.zeros_like(x)
        _elements(g, s["up"]).copy_(-torch.rand(g.nelx, g.nelz, g.nely, dtype=torch.float64,
                                                device="cuda", generator=gen))
    elif kind == "update":
        # sensitivities span orders of magnitude: large along the load path
        e = torch.exp(1.5 * _smooth((g.nelx, g.nelz, g.nely), 8, gen))
        s["dc"] = torch.zeros_like(x)
        _elements(g, s["dc"]).copy_(-e * _elements(g, x) ** 2)
        s["dv"] = _filtered_ones(g, case["rmin"])
    elif kind == "design":
        s["st"] = top3d_amd.DesignState(g, VOLFRAC, case["rmin"])
        s["xp"] = g.filter(s["st"].rmin, x)
    return s


def _filtered_ones(g, rmin):
    return g.filter_grad(rmin, torch.ones(g.nelem, dtype=torch.float64, device="cuda"))


# ---- one pass -----------------------------------------------------------------
def run(s):
    kind, g = s["kind"], s["g"]
    if kind == "operator":
        return {"out": g.apply(s["x"], s["v"])}
    if kind == "solve":
        U = g.zeros(0)
        g.solve(s["x"], s["F"], U, tol=TOL)
        return {"U": U}
    if kind == "gradient":
        xl = s["x"].detach().requires_grad_(True)
        U = g.zeros(0)
        c = top3d_amd.Compliance.apply(top3d_amd.DensityFilter.apply(xl, g, s["rmin"]), g,
                                       s["F"], U, TOL)
        c.backward()
        return {"c": c.detach(), "grad": xl.grad, "U": U}
    if kind == "design":
        st = s["st"]
        # the design the iteration starts from, with a cold state
        st.x.copy_(s["x"])
        st.xPhys = s["xp"]
        st.U.zero_()
        rec = top3d_amd.design_step(st, TOL)
        return {"c": rec["c"], "dc": st.dc, "x": st.x, "xPhys": st.xPhys, "U": st.U}
    if kind == "filter":
        xl = s["x"].detach().requires_grad_(True)
        y = top3d_amd.DensityFilter.apply(xl, g, s["rmin"])
        y.backward(s["up"])
        return {"y": y.detach(), "grad": xl.grad}
    if kind == "update":
        x, xnew = s["x"].clone(), torch.zeros_like(s["x"])
        g.oc(x, xnew, s["dv"], s["dc"], 0.01)
        change = g.change(x, xnew)
        xp = g.filter(s["rmin"], x)
        return {"x": x, "change": change, "xPhys": xp, "volume": g.volume(xp)}
    if kind == "cycle":
        u = g.jacobi(s["x"], 4, s["invD"][0], s["u"].clone(), s["b"], 0)
        r = g.restrict(0, u)
        z = g.jacobi(s["x"], 4, s["invD"][1], g.zeros(1), r, 1)
        return {"u": u, "r": r, "z": z, "p": g.prolong(0, z)}
    raise ValueError(kind)


# ---- what a pass cannot do without --------------------------------------------
def work(case):
    """Bytes and operations of one pass.  A matvec costs 205 operations per
    element in the element's symmetry basis (two 8-point transforms of 3
    components, nine 3x3 blocks, the modulus).  A solve is taken as 8 CG
    iterations, each a V(4,4) cycle (7 sweeps, a sweep from zero, a residual
    and the transfers, on level 0 and an eighth of that on each further one)
    with vectors of the cycle's precision, and the CG's FP64 matvec and
    vector updates."""
    ne = case["nelx"] * case["nely"] * case["nelz"]
    nd = 3 * (case["nelx"] + 1) * (case["nely"] + 1) * (case["nelz"] + 1)
    t = 4 if case["precision"] == "mixed" else 8
    mv = 205 * 2 * ne
    cycle = (7 * (3 * nd + ne) + (2 * nd + ne) + (3 * nd + ne) + 3 * nd) * t * 8 / 7
    solve = {"bytes": 8 * (cycle + (16 * nd + 8 * ne) + (32 + t) * nd + (24 + t) * nd),
             "flops": 8 * (8 * mv * 8 / 7 + mv + 12 * nd)}
    taps = sum(1 for d in _window(case["rmin"]))
    filt = {"bytes": 16 * ne, "flops": 2 * taps * ne}
    sens = {"bytes": 8 * nd + 16 * ne, "flops": 160 * ne}
    parts = {
        "operator": [{"bytes": 16 * nd + 8 * ne, "flops": mv}],
        "solve": [solve],
        "filter": [filt, filt],
        "gradient": [filt, solve, sens, sens, filt],
        "update": [{"bytes": 32 * ne + 16 * ne, "flops": 60 * 8 * ne}, filt, {"bytes": 8 * ne}],
        "cycle": [{"bytes": 1.125 * (24 * nd + 8 * nd + 8 * ne) + 18 * nd, "flops": 4.5 * mv}],
    }
    parts["design"] = [solve, sens, filt] + parts["update"]
    chosen = parts[case["kind"]]
    return {k: float(sum(p.get(k, 0) for p in chosen)) for k in ("bytes", "flops")}


# ---- the same in 64 bits with plain torch ----------------------------------------
#: positions (x, y, z) of an element's nodes
NODES = [(0, 1, 0), (1, 1, 0), (1, 0, 0), (0, 0, 0), (0, 1, 1), (1, 1, 1), (1, 0, 1), (0, 0, 1)]


def _element_matrix():
    """Stiffness of the unit trilinear hexahedron by the 10-point midpoint
    rule per axis, whose moments up to order 2 the two points +-t have;
    u_y points along -y."""
    t = math.sqrt(1 / 3 - 1 / 300)
    C = np.zeros((6, 6))
    C[:3, :3] = NU / ((1 + NU) * (1 - 2 * NU))
    C[range(3), range(3)] = (1 - NU) / ((1 + NU) * (1 - 2 * NU))
    C[range(3, 6), range(3, 6)] = 1 / (2 * (1 + NU))
    K = np.zeros((24, 24))
    for q in range(8):
        p = [0.5 + 0.5 * (t if q >> d & 1 else -t) for d in range(3)]
        B = np.zeros((6, 24))
        for n, pos in enumerate(NODES):
            f = [p[d] if pos[d] else 1 - p[d] for d in range(3)]
            s = [1.0 if pos[d] else -1.0 for d in range(3)]
            dx, dy, dz = s[0] * f[1] * f[2], f[0] * s[1] * f[2], f[0] * f[1] * s[2]
            B[0, 3 * n], B[1, 3 * n + 1], B[2, 3 * n + 2] = dx, dy, dz
            B[3, 3 * n], B[3, 3 * n + 1] = dy, dx
            B[4, 3 * n + 1], B[4, 3 * n + 2] = dz, dy
            B[5, 3 * n], B[5, 3 * n + 2] = dz, dx
        K += B.T @ C @ B / 8
    flip = np.tile([1.0, -1.0, 1.0], 8)
    return K * flip[:, None] * flip[None, :]


def _corner(v, n):
    """Values of node n of every element, from nodal values (x, z, y, ...)."""
    px, py, pz = NODES[n]
    s = v.shape
    return v[px:s[0] - 1 + px, pz:s[1] - 1 + pz, py:s[2] - 1 + py]


class _Plain:
    """The problem on its real nodes (x, z, y, component) and elements."""

    def __init__(self, case):
        self.n = n = (case["nelx"], case["nelz"], case["nely"])
        self.K = torch.from_numpy(_element_matrix()).cuda()
        self.rmin = case["rmin"]
        self.fixed = torch.zeros(n[0] + 1, n[1] + 1, n[2] + 1, 1, dtype=torch.bool, device="cuda")
        lim = n[2] // 4 + 1
        self.fixed[0, :, :lim] = True
        self.fixed[0, :, n[2] + 1 - lim:] = True

    def real(self, v):
        """Real nodes of a halo vector."""
        n = self.n
        return v.view(n[0] + 3, n[1] + 3, n[2] + 3, 3)[1:-1, 1:-1, 1:-1].clone()

    def halo(self, v):
        return torch.nn.functional.pad(v, (0, 0, 1, 1, 1, 1, 1, 1)).reshape(-1)

    def elements(self, x):
        n = self.n
        return x.view(n[0] + 2, n[1] + 2, n[2] + 2)[1:-1, 1:-1, 1:-1].clone()

    def padded(self, x, fill=None):
        if fill is None:
            return torch.nn.functional.pad(x, (1, 1, 1, 1, 1, 1)).reshape(-1)
        out = fill.clone()
        self_view = out.view(self.n[0] + 2, self.n[1] + 2, self.n[2] + 2)
        self_view[1:-1, 1:-1, 1:-1] = x
        return out

    def gather(self, u):
        return torch.cat([_corner(u, n) for n in range(8)], dim=-1)

    def free_apply(self, E, u):
        """K u without supports."""
        f = (self.gather(u) @ self.K.T) * E[..., None]
        out = torch.zeros_like(u)
        for n in range(8):
            _corner(out, n).add_(f[..., 3 * n:3 * n + 3])
        return out

    def apply(self, E, u):
        return torch.where(self.fixed, u, self.free_apply(E, u))

    def invdiag(self, E, KD):
        """Inverse diagonal, KD: the elements' diagonal entries (..., 24)."""
        d = torch.zeros([s + 1 for s in E.shape[:3]] + [3], dtype=torch.float64, device="cuda")
        for n in range(8):
            _corner(d, n).add_(KD[..., 3 * n:3 * n + 3])
        return d

    def solve(self, E, F):
        """K u = F by Jacobi-preconditioned CG on the free nodes."""
        free = ~self.fixed
        KD = E[..., None] * torch.diagonal(self.K)
        inv = free / self.invdiag(E, KD)
        r = F * free
        u = torch.zeros_like(F)
        z = inv * r
        p, rho = z.clone(), (r * z).sum()
        stop = 1e-11 * float(r.norm())
        for it in range(6000):
            q = self.free_apply(E, p) * free
            a = rho / (p * q).sum()
            u += a * p
            r -= a * q
            if it % 50 == 0 and float(r.norm()) < stop:
                return u
            z = inv * r
            new = (r * z).sum()
            p = z + (new / rho) * p
            rho = new
        return None

    def young(self, x):
        return EMIN + x ** 3 * (E0 - EMIN)

    def energy(self, u):
        g = self.gather(u)
        return ((g @ self.K) * g).sum(-1)

    def window(self, v):
        """H v and H 1 over the real elements."""
        n, out, ones = self.n, torch.zeros_like(v), torch.zeros_like(v)
        for (di, dk, dj), w in _window(self.rmin):
            dst, src = [], []
            for d, m in ((di, n[0]), (dk, n[1]), (dj, n[2])):
                dst.append(slice(max(0, -d), min(m, m - d)))
                src.append(slice(max(0, d), min(m, m + d)))
            out[tuple(dst)] += w * v[tuple(src)]
            ones[tuple(dst)] += w
        return out, ones


def _window(rmin):
    cr = math.ceil(rmin)
    for di in range(-(cr - 1), cr + 1):
        for dk in range(-(cr - 1), cr + 1):
            for dj in range(-(cr - 1), cr + 1):
                w = rmin - math.sqrt(di * di + dk * dk + dj * dj)
                if w > 0:
                    yield (di, dk, dj), w


def _oc(x, dv, dc, gval):
    """The bisection on the volume's multiplier, move limit 0.2."""
    l1, l2 = 0.0, 1e9
    while (l2 - l1) / (l1 + l2) > 1e-6:
        lmid = 0.5 * (l2 + l1)
        xnew = torch.sqrt(-dc / (dv * lmid)) * x
        xnew = torch.minimum(xnew, x + 0.2).clamp(max=1.0)
        xnew = torch.maximum(xnew, x - 0.2).clamp(min=0.0)
        if float((dv * (xnew - x)).sum()) + gval > 0:
            l1 = lmid
        else:
            l2 = lmid
    return xnew


def _two_level(P, x, u, b, r_of):
    """Four damped-Jacobi sweeps on each of the levels 0 and 1 with the
    transfers between them."""
    E = P.young(x)
    inv0 = torch.where(P.fixed, 1.0, 1.0 / P.invdiag(E, E[..., None] * torch.diagonal(P.K)))
    for _ in range(4):
        u = u + 0.6 * inv0 * (b - P.apply(E, u))
    r = r_of(u)
    # level 1: K1 = P^T K P on the doubled grid, its diagonal from the
    # sub-cells' projected matrices
    Q = _interpolation()
    n1 = [m // 2 for m in P.n]
    KD = torch.zeros(n1 + [24], dtype=torch.float64, device="cuda")
    for (ox, oy, oz), q in Q.items():
        d = torch.diagonal(q.T @ P.K @ q)
        KD += E[ox::2, oz::2, oy::2][..., None] * d
    fixed1 = torch.zeros(n1[0] + 1, n1[1] + 1, n1[2] + 1, 1, dtype=torch.bool, device="cuda")
    lim = n1[2] // 4 + 1
    fixed1[0, :, :lim] = True
    fixed1[0, :, n1[2] + 1 - lim:] = True
    inv1 = torch.where(fixed1, 1.0, 1.0 / P.invdiag(E[::2, ::2, ::2], KD))
    z = torch.zeros_like(r)
    for _ in range(4):
        kz = torch.where(fixed1, z, r_of(P.free_apply(E, _prolong(z))))
        z = z + 0.6 * inv1 * (r - kz)
    return u, r, z, _prolong(z)


def _interpolation():
    """Per sub-cell (ox, oy, oz) the 24x24 trilinear interpolation from the
    parent's nodes to the sub-cell's."""
    out = {}
    for o in range(8):
        off = (o & 1, o >> 1 & 1, o >> 2)
        q = np.zeros((24, 24))
        for b, pb in enumerate(NODES):
            for a, pa in enumerate(NODES):
                w = 1.0
                for d in range(3):
                    t = 0.5 * (off[d] + pb[d])
                    w *= t if pa[d] else 1 - t
                q[3 * b:3 * b + 3, 3 * a:3 * a + 3] = w * np.eye(3)
        out[off] = torch.from_numpy(q).cuda()
    return out


def _prolong(c):
    for d in range(3):
        n = c.shape[d]
        a, b = c.narrow(d, 0, n - 1), c.narrow(d, 1, n - 1)
        s = list(c.shape)
        s[d] = 2 * n - 1
        f = torch.empty(s, dtype=c.dtype, device=c.device)
        idx = [slice(None)] * c.dim()
        idx[d] = slice(0, None, 2)
        f[tuple(idx)] = c
        idx[d] = slice(1, None, 2)
        f[tuple(idx)] = 0.5 * (a + b)
        c = f
    return c


def _restrict(f):
    for d in range(3):
        n = (f.shape[d] + 1) // 2
        idx = [slice(None)] * f.dim()
        idx[d] = slice(0, None, 2)
        c = f[tuple(idx)].clone()
        idx[d] = slice(1, None, 2)
        odd = 0.5 * f[tuple(idx)]
        c.narrow(d, 0, n - 1).add_(odd)
        c.narrow(d, 1, n - 1).add_(odd)
        f = c
    return f


#: elements up to which the plain CG reaches the solution in a few seconds
PLAIN_SOLVE = 150_000


def exact(case, seed):
    kind = case["kind"]
    ne = case["nelx"] * case["nely"] * case["nelz"]
    if kind in ("solve", "design", "gradient") and ne > PLAIN_SOLVE or ne > 9_000_000:
        return None  # an iterate stopped at 1e-5, and too long a plain solve
    s = prepare(case, seed)
    P = _Plain(case)
    x = P.elements(s["x"])
    if kind == "operator":
        v = P.real(s["v"])
        return {"out": P.halo(P.apply(P.young(x), v))}
    if kind == "cycle":
        u, r, z, p = _two_level(P, x, P.real(s["u"]), P.real(s["b"]), _restrict)
        return {"u": P.halo(u), "r": P.halo(r), "z": P.halo(z), "p": P.halo(p)}
    if kind == "filter":
        h, w = P.window(x)
        t = P.window(P.elements(s["up"]) / w)[0]
        return {"y": P.padded(h / w), "grad": P.padded(t)}
    if kind == "update":
        dv = P.elements(s["dv"])
        new = _oc(x, dv, P.elements(s["dc"]), 0.01)
        h, w = P.window(new)
        return {"x": P.padded(new), "change": float(np.float32(float((new - x).abs().max()))),
                "xPhys": P.padded(h / w), "volume": float((h / w).sum())}
    F = P.real(s["F"])
    if kind == "solve":
        u = P.solve(P.young(x), F)
        return None if u is None else {"U": P.halo(u)}
    h, w = P.window(x)
    xp = h / w
    u = P.solve(P.young(xp), F)
    if u is None:
        return None
    ce = P.energy(u)
    dc = P.window(-3.0 * (E0 - EMIN) * xp ** 2 * ce / w)[0]
    out = {"c": float((P.young(xp) * ce).sum()), "U": P.halo(u)}
    if kind == "gradient":
        return dict(out, grad=P.padded(dc))
    dv = P.window(1.0 / w)[0]
    new = _oc(x, dv, dc, float(xp.sum()) / ne - VOLFRAC)
    h, w = P.window(new)
    return dict(out, dc=P.padded(dc), x=P.padded(new), xPhys=P.padded(h / w))
