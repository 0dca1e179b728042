"""GPU parity of the fine operator and its smoother against the CPU oracle at
the sizes where the fine kernel's tiles can go wrong: grids narrower than a
tile, planes of exactly a tile's rows and one more, every shape that the tile
rule chooses from, marches of more planes than one mask of fixed planes holds,
and vectors large enough to be stored past the caches."""
import ctypes

import numpy as np
import pytest
import torch

import pyoracle
import top3d_amd

pytestmark = pytest.mark.gpu

# 24 products of each output's row, the transforms and their sums: 1e-13 in
# double precision, 2e-6 in single, relative to the largest entry; three
# smoother sweeps 1e-12
TOL64, TOL32, TOL_SWEEP = 1e-13, 2e-6, 1e-12


def relerr(got, ref):
    return np.abs(got - ref).max() / np.abs(ref).max()


def check_operator(g, o, seed, sweeps=True):
    assert g.padding(0) == o.padding(0)
    rng = np.random.default_rng(seed)
    x = g.density(rng.uniform(0.1, 1.0, g.nelx * g.nely * g.nelz))
    xo = x.cpu().numpy()
    v = rng.standard_normal(g.ndof(0))
    got = g.apply(x, torch.from_numpy(v).cuda()).cpu().numpy()
    assert relerr(got, o.matvec0(xo, v)) <= TOL64
    v32 = v.astype(np.float32)
    got = g.apply_f32(x, torch.from_numpy(v32).cuda()).cpu().numpy()
    assert relerr(got, o.matvec0(xo, v32.astype(np.float64))) <= TOL32
    if not sweeps:
        return
    inv, b, tmp = o.invdiag(xo, 0), rng.standard_normal(v.size), np.zeros(v.size)
    got = g.jacobi(x, 3, *(torch.from_numpy(a.copy()).cuda() for a in (inv, v, b))).cpu().numpy()
    P = ctypes.c_void_p
    fn = o.lib.or_jacobi0
    fn.argtypes = [P, P, ctypes.c_int, ctypes.c_double, P, P, P, P]
    fn(P(o.h), P(xo.ctypes.data), 3, 0.6, *(P(a.ctypes.data) for a in (inv, v, b, tmp)))
    assert relerr(got, v) <= TOL_SWEEP


@pytest.mark.parametrize("shape", [(4, 4, 4), (8, 16, 12), (12, 20, 44), (16, 24, 8),
                                   (20, 44, 4), (12, 4, 64), (8, 88, 36)])
def test_ragged_tiles(shape):
    print(f"[gpu fine march] {shape}", flush=True)
    g = top3d_amd.Grid(*shape, 3)
    o = pyoracle.Grid(*shape, 3)
    check_operator(g, o, shape[1])
    g.close()
    o.close()


# TY, TZ, NX: the rule's shapes, marches of 65, 66 and 131 planes, one tile row
@pytest.mark.parametrize("tile", ["17,13,0", "18,12,65", "20,11,66", "23,9,131", "2,2,0",
                                  "84,2,1", "2,84,7"])
def test_tile_shapes(tile, monkeypatch):
    print(f"[gpu fine march] tile {tile}", flush=True)
    monkeypatch.setenv("TOP3D_TILE_L0", tile)
    monkeypatch.setenv("TOP3D_TILE_L0_F64", tile)
    g = top3d_amd.Grid(140, 36, 28, 3)
    o = pyoracle.Grid(140, 36, 28, 3)
    check_operator(g, o, 3)
    g.close()
    o.close()


def test_vectors_beyond_the_cache():
    # 2 vectors and the moduli exceed 256 MB in single precision too
    shape = (224, 208, 208, 5)
    print(f"[gpu fine march] {shape}", flush=True)
    g = top3d_amd.Grid(*shape)
    o = pyoracle.Grid(*shape)
    check_operator(g, o, 5, sweeps=False)
    g.close()
    o.close()


# One CG iteration from zero leaves u = alpha z, z the V-cycle of the load:
# checks the V-cycle's own launches, the first two sweeps in one and (mixed)
# the sweep that adds the coarse correction.
def vcycle_of_load(g, seed):
    x = g.density(np.random.default_rng(seed).uniform(0.1, 1.0, g.nelx * g.nely * g.nelz))
    F, U = g.load(), g.zeros(0)
    g.set_max_iter(1)
    g.solve(x, F, U, allow_no_converge=True)
    return x.cpu().numpy(), F.cpu().numpy(), U.cpu().numpy()


# FP64: 1e-10; the FP32 V-cycle: 2^-24 for each of 24 products and 32 sweeps,
# ten times that for what the coarse correction amplifies, 1e-3
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-10), ("mixed", 1e-3)])
@pytest.mark.parametrize("shape", [(16, 24, 8), (12, 20, 44), (8, 88, 36)])
def test_vcycle(shape, precision, tol):
    print(f"[gpu fine march] v-cycle {shape} {precision}", flush=True)
    g = top3d_amd.Grid(*shape, 3, precision=precision)
    o = pyoracle.Grid(*shape, 3)
    x, r, got = vcycle_of_load(g, shape[1])
    assert o.setup(x) == 0
    z = o.vcycle(x, r)
    assert relerr(got, (r @ z) / (z @ o.matvec0(x, z)) * z) <= tol
    g.close()
    o.close()


# Every tile shape forms a node from the same operands in the same order: only
# the order of the sums for alpha changes, 1e-12
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,tile", [((140, 36, 28), "17,12,65"), ((140, 36, 28), "20,11,7"),
                                        ((140, 36, 28), "23,9,131"), ((12, 20, 44), "2,2,3"),
                                        ((16, 24, 8), "5,3,1")])
def test_vcycle_tiles(shape, tile, precision, monkeypatch):
    print(f"[gpu fine march] v-cycle {shape} {tile} {precision}", flush=True)
    g = top3d_amd.Grid(*shape, 3, precision=precision)
    _, _, ref = vcycle_of_load(g, shape[1])
    monkeypatch.setenv("TOP3D_TILE_L0", tile)
    monkeypatch.setenv("TOP3D_TILE_L0_F64", tile)
    _, _, got = vcycle_of_load(g, shape[1])
    assert relerr(got, ref) <= 1e-12
    g.close()


# The level-1 shapes that the rule takes (narrow tiles, 65 x 7 and its clipped
# forms) and a wide tile for all: the same operands in the same order per node,
# so the operator's 1e-13 holds between them with room
@pytest.mark.parametrize("shape,nl", [((168, 72, 104), 4), ((200, 120, 88), 4), ((48, 48, 48), 4),
                                      ((96, 96, 48), 4), ((64, 32, 32), 3), ((512, 16, 24), 3),
                                      ((12, 132, 28), 3)])
def test_level1_shapes(shape, nl, monkeypatch):
    print(f"[gpu fine march] level 1 {shape}", flush=True)
    g = top3d_amd.Grid(*shape, nl, precision="mixed")
    rng = np.random.default_rng(shape[1])
    x = g.density(rng.uniform(0.1, 1.0, g.nelx * g.nely * g.nelz))
    v, b = (torch.from_numpy(rng.standard_normal(g.ndof(1))).cuda() for _ in range(2))
    inv = g.invdiag(x, 1)

    def results():
        return (g.apply_level(1, x, v).cpu().numpy(),
                g.apply_level_f32(1, x, v.float()).cpu().numpy(),
                g.jacobi(x, 2, inv, v.clone(), b, l=1).cpu().numpy())
    got = results()
    monkeypatch.setenv("TOP3D_TILE_L1", "47,9,0")
    for a, r, tol in zip(got, results(), (TOL64, TOL32, TOL_SWEEP)):
        assert relerr(a, r) <= tol
    g.close()
