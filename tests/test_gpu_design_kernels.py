"""GPU checks of the design-loop kernels at the sizes where they can go
wrong: the OC bisection at its first, second and later passes over the
multipliers and at ragged element counts, the density filter's tiles at the
edges of tiles and at grids narrower than the window."""
import ctypes

import numpy as np
import pytest
import torch

import pyoracle
import top3d_amd

pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def oc_reference(x, dv, dc, gval):
    """The bisection of the optimality-criteria update, one multiplier per
    step, in double precision."""
    l1, l2 = 0.0, 1e9
    xnew = x
    with np.errstate(divide="ignore", invalid="ignore"):
        while (l2 - l1) / (l1 + l2) > 1e-6:
            lmid = 0.5 * (l2 + l1)
            t = x * np.sqrt(-dc / (dv * lmid))
            xnew = np.fmax(0.0, np.fmax(x - 0.2, np.fmin(1.0, np.fmin(x + 0.2, t))))
            if np.sum(dv * (xnew - x)) + gval > 0:
                l1 = lmid
            else:
                l2 = lmid
    return xnew


# scale of the sensitivities: the root lies above 5e8 (no halving), within the
# first 31 halvings of 1e9, within the second and within the third
@pytest.mark.parametrize("scale", [1e9, 1.0, 1e-9, 1e-16])
@pytest.mark.parametrize("n", [1, 1023, 1025, 262145, 524289 + 1024])
def test_oc_update_matches_stepwise_bisection(n, scale):
    print(f"[gpu oc] n {n} scale {scale}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(0.05, 0.95, n)
    dv = rng.uniform(0.5, 1.5, n)
    dc = -scale * rng.uniform(0.5, 1.5, n)
    gval = 0.01 * (1 if n % 2 else -1) * min(1.0, 0.5 * n * 0.05)
    ref = oc_reference(x, dv, dc, gval)
    d = [torch.from_numpy(a).cuda() for a in (x, dv, dc)]
    got = torch.full((n,), -1.0, dtype=torch.float64, device="cuda")
    lib = top3d_amd.library()
    lib.top3d_set_stream(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    lib.update_solution(_p(d[0]), _p(got), _p(d[1]), _p(d[2]), n, gval)
    top3d_amd.check("update_solution")
    # the same multiplier, visited by the same steps: x differs by the
    # rounding of a sqrt(-dc/dv) / sqrt(lmid) (4 roundings of 2^-53)
    assert np.abs(got.cpu().numpy() - ref).max() <= 8 * 2.0 ** -53


@pytest.mark.parametrize("shape", [(8, 4, 4), (36, 12, 20), (16, 32, 8), (12, 36, 44)])
@pytest.mark.parametrize("rmin", [0.7, 1.0, 1.5, 2.0, 2.9, 3.5, 4.5, 6.0, 7.0, 7.5])
def test_filter_tiles(shape, rmin):
    print(f"[gpu filter] {shape} rmin {rmin}", flush=True)
    nelx, nely, nelz = shape
    g, o = top3d_amd.Grid(nelx, nely, nelz, 3), pyoracle.Grid(nelx, nely, nelz, 3)
    rng = np.random.default_rng(3)
    inter = g.interior_elements()
    x = g.density(rng.uniform(0.1, 1.0, inter.size))
    v = g.density(rng.uniform(-1.0, 1.0, inter.size))
    halo = np.ones(g.nelem, bool)
    halo[inter] = False
    v[torch.from_numpy(halo).cuda()] = 7.0  # read by nothing, kept in the result
    r = np.arange(-8, 9)
    d = np.sqrt(r[:, None, None] ** 2 + r[None, :, None] ** 2 + r[None, None, :] ** 2)
    taps = int((d < rmin).sum())
    tol = (2 * taps + 4) * 2.0 ** -53  # each sum in an order of its own, a division
    y = g.filter(rmin, x).cpu().numpy()
    ref = o.filter(rmin, x.cpu().numpy())
    assert np.abs(y[inter] - ref[inter]).max() <= tol * np.abs(ref[inter]).max()
    assert not y[halo].any()
    w = g.filter_grad(rmin, v).cpu().numpy()
    vr = v.cpu().numpy()
    ref = o.filter_grad(rmin, vr.copy())
    size = o.filter_grad(rmin, np.abs(vr))  # the sums' absolute terms
    assert (np.abs(w - ref)[inter] <= tol * size[inter]).all()
    assert (w[halo] == 7.0).all()
    # a NaN reaches the elements within the radius only (the tiles apply no
    # zero weight; beyond radius 7 the loop over the whole window runs)
    c = (nelx // 2 + 1, nelz // 2 + 1, nely // 2 + 1)
    x[(c[0] * (nelz + 2) + c[1]) * (nely + 2) + c[2]] = float("nan")
    i, k, j = np.meshgrid(*(np.arange(1, m + 1) for m in (nelx, nelz, nely)), indexing="ij")
    near = np.sqrt((i - c[0]) ** 2 + (k - c[1]) ** 2 + (j - c[2]) ** 2).ravel() < rmin
    bad = np.isnan(g.filter(rmin, x).cpu().numpy())[inter]
    assert bad[near].all()
    if rmin <= 7.0:
        assert not bad[~near].any()
    g.close()
    o.close()


# Elements at x = 1 that stay there under every multiplier (a solid region with a
# large volume weight) add nothing to the sums: the multiplier is that of the
# others.  Every sum that the bisection
# decides on is far above the rounding of the moving elements' terms (n 2^-53).
@pytest.mark.parametrize("n", [4096, 262145])
def test_oc_update_beside_heavy_elements(n):
    print(f"[gpu oc] heavy elements, n {n}", flush=True)
    rng = np.random.default_rng(n)
    x, dv = rng.uniform(0.05, 0.95, n), rng.uniform(0.5, 1.5, n)
    dc = -rng.uniform(0.5, 1.5, n) * 10.0 ** rng.integers(-2, 3, n)
    heavy = rng.random(n) < 0.25
    x[heavy], dv[heavy], dc[heavy] = 1.0, 1e18, -1e30
    gval = 0.01 * n
    light = ~heavy
    ref = np.ones(n)
    ref[light] = oc_reference(x[light], dv[light], dc[light], gval)
    d = [torch.from_numpy(a).cuda() for a in (x, dv, dc)]
    got = torch.full((n,), -1.0, dtype=torch.float64, device="cuda")
    lib = top3d_amd.library()
    lib.top3d_set_stream(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    lib.update_solution(_p(d[0]), _p(got), _p(d[1]), _p(d[2]), n, gval)
    top3d_amd.check("update_solution")
    assert np.abs(got.cpu().numpy() - ref).max() <= 8 * 2.0 ** -53


def test_oc_update_in_place():
    """xnew may be one of the inputs: the result of the update elsewhere."""
    n = 300_001
    rng = np.random.default_rng(11)
    x, dv, dc = (torch.from_numpy(a).cuda() for a in (
        rng.uniform(0.05, 0.95, n), rng.uniform(0.5, 1.5, n), -rng.uniform(0.5, 1.5, n)))
    lib = top3d_amd.library()
    lib.top3d_set_stream(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    out = torch.empty_like(x)
    torch.cuda.synchronize()
    lib.update_solution(_p(x), _p(out), _p(dv), _p(dc), n, 0.01)
    for k in range(3):
        a = [x.clone(), dv.clone(), dc.clone()]
        torch.cuda.synchronize()
        lib.update_solution(_p(a[0]), _p(a[k]), _p(a[1]), _p(a[2]), n, 0.01)
        top3d_amd.check("update_solution")
        assert torch.equal(a[k], out)
