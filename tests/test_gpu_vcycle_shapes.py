"""The V-cycle's assembly and transfer kernels (k_galerkin_l2_bc,
k_band_assemble, k_restrict_xz_w, k_restrict_once, the prolongation's launch shapes, the
coarsest solve) against the FP64 oracle at the edges of their tiles.

Bars: those of test_gpu_parity, 1e-11 for the V-cycle (two factorisations of
the coarsest matrix with different roundings; everything else agrees to a few
ulps)."""
import numpy as np
import pytest

from oracle import Oracle

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("oracle_lib")]

SHAPES = {
    (4, 4, 4): "padded to 8: one coarsest cell, every level-2 cell void in part",
    (8, 8, 8): "3x3x3 level-2 nodes: less than one block of outputs",
    (28, 24, 8): "level-2 plane of 9x9 nodes: one full block of 64 outputs and a remainder",
    (31, 33, 9): "ragged in every axis",
    (9, 120, 17): "long: 33 level-2 node columns",
    (64, 40, 40): "17 level-2 nodes in y",
    (56, 56, 16): "coarsest plane of 8x8 nodes: one full block of 64 outputs",
    (57, 63, 24): "coarsest plane of 9x9 nodes: a full block and a remainder, padded",
}


def _pair(vox, fix=None, load=None):
    import top3d_xl_amd as t3x
    a = () if fix is None else (fix, load)
    g, o = t3x.Problem(vox, *a), Oracle(vox, *a)
    rng = np.random.default_rng(17)
    E = 1e-6 + rng.random(o.nE) ** 3
    for m in (g, o):
        m.set_modulus(E)
        m.assemble()
    return g, o, rng.standard_normal(3 * o.nN)


def _check(g, o, r):
    z, zo = g.vcycle(r), o.vcycle(r)
    g.close()
    assert np.abs(z - zo).max() < 1e-11 * np.abs(zo).max()


@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_cuboid(shape):
    print(f"\n[gpu-vcycle] {shape}: {SHAPES[shape]}", flush=True)
    _check(*_pair(np.ones(shape, bool)))


def test_supports_on_void_neighbours():
    """Fixed nodes whose level-2 cells hold void children and nodes with fewer
    than 8 solid cells around them, fixed in some components only."""
    print("\n[gpu-vcycle] partly fixed supports next to void", flush=True)
    vox = np.ones((12, 16, 12), bool)
    vox[3:9, 5:11, 2:7] = False
    ny, nx, _ = vox.shape
    nodes = np.array([jy + (ny + 1) * (0 + (nx + 1) * jz) for jz in range(13) for jy in range(0, 13, 2)])
    state = np.zeros((nodes.size, 3), np.uint8)
    state[np.arange(nodes.size), np.arange(nodes.size) % 3] = 1
    state[::4] = 1
    load = np.array([jy + (ny + 1) * (nx + (nx + 1) * 6) for jy in range(13)])
    _check(*_pair(vox, (nodes, state), (load, np.tile([0.0, 0.3, -1.0], (13, 1)))))
