"""The FP64 V-cycle against the oracle on both sides of the line between the
restriction's two x-z passes (k_restrict_xz_w, k_restrict_xz: 92,160 coarse
nodes).  Bar: 1e-11, as in test_gpu_parity."""
import numpy as np
import pytest

from oracle import Oracle

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("oracle_lib")]


@pytest.mark.parametrize("shape,nodes", [((136, 272, 136), 84_525), ((144, 288, 144), 99_937)], ids=str)
def test_vcycle(shape, nodes):
    import top3d_xl_amd as t3x
    vox = np.ones(shape, bool)
    g, o = t3x.Problem(vox), Oracle(vox)
    try:
        assert g.levels[1]["numNodes"] == nodes
        rng = np.random.default_rng(19)
        E, r = 1e-6 + rng.random(o.nE) ** 3, rng.standard_normal(3 * o.nN)
        for m in (g, o):
            m.set_modulus(E)
            m.assemble()
        print(f"\n[gpu-transfers] {shape}", flush=True)
        z, zo = g.vcycle(r), o.vcycle(r)
        assert np.abs(z - zo).max() < 1e-11 * np.abs(zo).max()
    finally:
        g.close()
