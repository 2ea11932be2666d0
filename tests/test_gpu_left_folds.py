"""Dot products left to the update that needs them (k_pcg_update_late,
k_pcg_pupdate_late) against the FP64 oracle, on both sides of the rule's line:
one partial, a wave's worth, more than a block's threads, more than the
finaliser's 1024 threads, and just past the line.

Bars: those of test_gpu_parity (filter 1e-10 and equal iteration counts; PCG at
its tolerance on moduli in [0.5, 1.5] equal counts and 1e-4)."""
import numpy as np
import pytest

from oracle import Oracle

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("oracle_lib")]

# about 1, 63, 260, 1,030, 1,440 and 1,460 blocks of 256 nodes: the z.r partials of the filter (the line is at 1,448)
FILTER_SHAPES = [(3, 3, 3), (15, 15, 62), (17, 40, 89), (50, 100, 50), (70, 71, 71), (71, 71, 71)]


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("shape", FILTER_SHAPES, ids=str)
def test_filter(shape):
    import top3d_xl_amd as t3x
    print(f"\n[gpu-left-folds] filter {shape}", flush=True)
    g, o = t3x.Problem(np.ones(shape, bool)), Oracle(np.ones(shape, bool))
    src = np.random.default_rng(3).random(o.nE)
    for m in (g, o):
        m.filter_setup(0, 2.5)
    (dg, ig), (do, io) = g.filter(0, src), o.filter(0, src)
    g.close()
    assert ig == io and _rel(dg, do) < 1e-10


@pytest.mark.parametrize("shape", [(4, 4, 4), (14, 14, 60), (16, 16, 272)], ids=str)  # p.q of 1, 16 and 276 tiles
def test_pcg(shape):
    import top3d_xl_amd as t3x
    print(f"\n[gpu-left-folds] PCG {shape}", flush=True)
    vox = np.ones(shape, bool)
    g, o, m = t3x.Problem(vox), Oracle(vox), t3x.Problem(vox, precision=2, vcycle=1, omega=0.4, coarsestControl=0)
    E = 0.5 + np.random.default_rng(4).random(o.nE)
    for q in (g, o, m):
        q.set_modulus(E)
        q.assemble()
    b = o.get("F")
    (xg, ig, _), (xo, io, _), (xm, _, res) = g.pcg(b), o.pcg(b), m.pcg(b)
    assert ig == io and _rel(xg, xo) < 1e-4
    # the precision form stops at the same tolerance, which its recursive residual meets to rounding
    assert res < 1e-3 and np.linalg.norm(b - o.apply_K(xm)) < 1.01e-3 * np.linalg.norm(b)
    g.close(), m.close()


def test_filter_of_a_few_cells_at_the_end_of_a_large_grid():
    """20 M nodes, 64 solid cells: few partials, more elements than a block per
    element's 256 threads can take; the same filter on those cells alone."""
    import top3d_xl_amd as t3x
    vox = np.zeros((2000, 4, 2000), bool)
    vox[-4:, :, -4:] = True
    ny, nx, nz = vox.shape
    node = lambda y, x, z: y + (ny + 1) * (x + (nx + 1) * z)  # noqa: E731
    fix = np.array([node(y, 0, z) for z in range(nz - 4, nz + 1) for y in range(ny - 4, ny + 1)])
    load = np.array([node(ny - 2, 4, nz - 2)])
    big = t3x.Problem(vox, (fix, np.ones((fix.size, 3), np.uint8)), (load, np.array([[0.0, 0.0, -1.0]])))
    small = t3x.Problem(np.ones((4, 4, 4), bool))
    try:
        assert big.nE == small.nE == 64
        src = np.random.default_rng(8).random(64)
        out = []
        for m in (big, small):
            m.filter_setup(0, 2.5)
            out.append(m.filter(0, src))
        assert out[0][1] == out[1][1] and _rel(out[0][0], out[1][0]) < 1e-10
    finally:
        big.close(), small.close()
