"""The coarsest direct solve (t3x_coarse.hip) at the edges of its launch forms.

Against the FP64 oracle: the V-cycle bar of test_gpu_parity, 1e-11 (two
factorisations of the same matrix with different roundings).  One launch for
all blocks against a launch per block: bit for bit."""
import numpy as np
import pytest

from oracle import Oracle

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("oracle_lib")]

# coarsest order n and solve block SB of the padded cuboid
SHAPES = {
    (5, 9, 5): "n 36 in one block of 64",
    (12, 24, 12): "n 108, SB 64: two blocks, the second one partly identity",
    (20, 17, 60): "n 432, SB 128, four blocks",
    (50, 100, 50): "SB 256: the last size with 4 chunks per row",
    (72, 144, 72): "SB 384: 8 chunks, everything in one launch",
    (104, 208, 104): "SB 640: own terms apart, a launch per direction",
}


def _outputs(shape):
    import top3d_xl_amd as t3x
    m = t3x.Problem(np.ones(shape, bool))
    try:
        rng = np.random.default_rng(5)
        m.set_modulus(1e-6 + rng.random(m.nE) ** 3)
        m.assemble()
        r = rng.standard_normal(3 * m.nN)
        return m.one_launch_coarse, m.vcycle(r), m.vcycle(2 * r), m.vcycle(r)
    finally:
        m.close()


@pytest.mark.parametrize("shape", [s for s in SHAPES if np.prod(s) < 1_000_000], ids=str)
def test_vcycle_against_oracle(shape):
    print(f"\n[gpu-coarse] {shape}: {SHAPES[shape]}", flush=True)
    one, z, z2, z3 = _outputs(shape)
    assert one
    o = Oracle(np.ones(shape, bool))
    rng = np.random.default_rng(5)
    o.set_modulus(1e-6 + rng.random(o.nE) ** 3)
    o.assemble()
    zo = o.vcycle(rng.standard_normal(3 * o.nN))
    assert np.abs(z - zo).max() < 1e-11 * np.abs(zo).max()
    assert np.array_equal(z, z3) and np.array_equal(2 * z, z2)  # a launch's words never serve the next one


def test_one_launch_equals_a_launch_per_block():
    import top3d_xl_amd as t3x
    print("\n[gpu-coarse] one launch", flush=True)
    got = {s: _outputs(s) for s in SHAPES}
    assert all(g[0] for g in got.values())
    hog = t3x.Problem(np.ones((192, 384, 192), bool))  # holds nearly all of the device's one-launch share
    try:
        assert hog.one_launch_coarse
        for s in list(SHAPES)[2:]:
            print(f"[gpu-coarse] a launch per block {s}", flush=True)
            one, z, _, _ = _outputs(s)
            if not one:  # a small grid may still fit beside it
                assert np.array_equal(z, got[s][1])
        assert not one  # the last, largest one does not
    finally:
        hog.close()


# everything in one launch (SB 128), and a launch per direction with even and odd numbers of blocks
@pytest.mark.parametrize("shape,handles", [((20, 17, 60), 41), ((104, 208, 104), 9), ((96, 192, 96), 9)], ids=str)
def test_handles_on_two_sets_one_set_and_none_agree(shape, handles):
    """Above SB 512 the first handle of a process takes a recurrence's blocks with
    two sets of work-groups in turn, later ones with one set, those beyond the
    device's capacity with a launch per block: the same bits."""
    import top3d_xl_amd as t3x
    ms = [t3x.Problem(np.ones(shape, bool)) for _ in range(handles)]
    try:
        rng = np.random.default_rng(7)
        E = 1e-6 + rng.random(ms[0].nE) ** 3
        r = rng.standard_normal((3, 3 * ms[0].nN))
        r[1, ::7] = 0.0
        first = None
        for m in ms:
            m.set_modulus(E)
            m.assemble()
            z = [m.vcycle(v) for v in r]  # (the words' two places, in turn)
            first = first or z
            assert all(np.array_equal(a, b) for a, b in zip(z, first))
        print(f"\n[gpu-coarse] {shape}: {sum(m.one_launch_coarse for m in ms)} of {handles} in one launch", flush=True)
    finally:
        for m in ms:
            m.close()
