"""How many handles of a process take the one-launch coarsest solve: a launch's
work-groups of four rows count as a quarter of a CU each (t3x_coarse.hip,
chain_share), so SB / 4 groups of 4 x CUs a handle; the next handle gets a launch
per block, with the same bits."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MULTIPROCESSOR_COUNT = 63  # hipDeviceAttributeMultiprocessorCount

# shape: solve block
SHAPES = {(20, 17, 60): 128, (50, 100, 50): 256, (72, 144, 72): 384, (88, 176, 88): 512, (96, 192, 96): 576,
          (104, 208, 104): 640, (128, 256, 128): 960}


@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_handles_that_fit(shape):
    import top3d_xl_amd as t3x
    cus = C.c_int()
    assert t3x.load_library().hipDeviceGetAttribute(C.byref(cus), MULTIPROCESSOR_COUNT, 0) == 0
    slots = 4 * cus.value
    groups = SHAPES[shape] // 4
    fit = 1_000_000 // -(-1_000_000 * groups // slots)  # shares are whole parts per million
    print(f"\n[gpu-coarse-share] {shape}: {fit} handles", flush=True)
    ms = [t3x.Problem(np.ones(shape, bool)) for _ in range(fit + 1)]
    try:
        assert [m.one_launch_coarse for m in ms] == fit * [True] + [False]
        rng = np.random.default_rng(11)
        E, r = 1e-6 + rng.random(ms[0].nE) ** 3, rng.standard_normal(3 * ms[0].nN)
        z = []
        for m in (ms[0], ms[-2], ms[-1]):
            m.set_modulus(E)
            m.assemble()
            z.append(m.vcycle(r))
        assert np.array_equal(z[0], z[1]) and np.array_equal(z[0], z[2])
    finally:
        for m in ms:
            m.close()
