"""The V-cycle's fused fine launches (the first two sweeps in one, and in the
mixed form the sweep that adds the coarse correction) against the same V-cycle
in launches of its own per sweep and transfer: the node-centric kernel runs it
so, in a child process (the library reads TOP3D_FINE_KERNEL once).  Both
boundary conventions, tiles of the rule and small ones, whose edges meet every
parity of the coarse nodes."""
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.gpu

SHAPES = [(16, 24, 8), (12, 20, 44), (8, 88, 36), (72, 36, 28)]
CASES = [(s, p, bc) for s in SHAPES for p in ("fp64", "mixed") for bc in ("reference", "symmetric")]


def vcycle(shape, precision, bc):
    """alpha z of one CG iteration from zero on a random right-hand side, z its
    V-cycle."""
    import torch

    import top3d_amd
    print(f"[gpu fused sweeps] {shape} {precision} {bc}", flush=True)
    g = top3d_amd.Grid(*shape, 3, precision=precision, bc=bc)
    rng = np.random.default_rng(shape[1])
    x = g.density(rng.uniform(0.1, 1.0, shape[0] * shape[1] * shape[2]))
    _, wx, wy, wz, n = g.padding(0)
    F = np.zeros((wx, wz, wy, 3))
    F[1:-1, 1:-1, 1:-1] = rng.standard_normal((wx - 2, wz - 2, wy - 2, 3))
    F = F.reshape(-1)
    F[g.fixed_dofs(0)] = 0.0
    U = g.zeros(0)
    g.set_max_iter(1)
    g.solve(x, torch.from_numpy(F).cuda(), U, allow_no_converge=True)
    out = U.cpu().numpy()
    g.close()
    return out


@pytest.fixture(scope="module")
def unfused(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("fused") / "unfused.npz")
    run = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), path],
                         env=dict(os.environ, TOP3D_FINE_KERNEL="node"), capture_output=True,
                         text=True, timeout=100)
    assert run.returncode == 0, run.stdout[-2000:] + run.stderr[-2000:]
    return np.load(path)


# 9 applications of the fine operator, each with 24 products and the 8 element
# sums to a row, whose absolute terms are up to 5 times the diagonal's, weighted
# 0.6: 9 x 32 x 3 roundings of 2^-24 or 2^-53 on either side
@pytest.mark.parametrize("tile", ["", "5,3,2", "4,6,9"])
@pytest.mark.parametrize("shape,precision,bc", CASES)
def test_fused_launches(unfused, shape, precision, bc, tile, monkeypatch):
    if tile:
        monkeypatch.setenv("TOP3D_TILE_L0", tile)
        monkeypatch.setenv("TOP3D_TILE_L0_F64", tile)
    ref = unfused[str(CASES.index((shape, precision, bc)))]
    got = vcycle(shape, precision, bc)
    tol = 2 * 9 * 32 * 3 * 2.0 ** (-53 if precision == "fp64" else -24)
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"[gpu fused sweeps] tile {tile} err {err:.1e} of {tol:.1e}", flush=True)
    assert err <= tol


if __name__ == "__main__":
    sys.path.insert(0, os.path.join(os.path.dirname(HERE), "topopt-in-openmp-gpu_amd"))
    np.savez(sys.argv[1], **{str(q): vcycle(*c) for q, c in enumerate(CASES)})
