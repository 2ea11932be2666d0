"""The OC bisection by brackets (k_oc_pass / k_oc_fin) against the sequential
loop (TOP3D_XL.m:146-153) written out in numpy: the same number of bisections,
and x from the same final multiplier.

x: each side forms x sqrt(-dc) / sqrt(l) with a few roundings of its own, so
the bar is 4 ulps of the largest unclamped value times the ulp, 1e-15 x 8 =
1e-14 for x <= 1 (values above 1.2 are clamped)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MAX_LEVELS = 256  # the library's limit where no multiplier meets the bound


def sequential(x, xPhys, dc, V0):
    fval = xPhys.mean() - V0
    t = x * np.sqrt(-dc)
    lo, hi = np.maximum(0.0, x - 0.2), np.minimum(1.0, x + 0.2)
    l1, l2, n = 0.0, 1e9, 0
    while (l2 - l1) / (l1 + l2) > 1e-6 and n < MAX_LEVELS:
        lmid = 0.5 * (l2 + l1)
        xn = np.maximum(lo, np.minimum(hi, t * (1.0 / np.sqrt(lmid))))
        if fval + (xn - x).sum() > 0:
            l1 = lmid
        else:
            l2 = lmid
        n += 1
    return xn, np.abs(xn - x).max(), n


def design(n, scale, rng, spread=0.0):
    x = 0.05 + 0.5 * rng.random(n)
    return x, -scale * np.exp(spread * rng.standard_normal(n)) * (0.01 + rng.random(n)) * 3 * x * x


# (cells of the cuboid, sensitivity scale, spread of its logarithm, V0 - mean x)
CASES = {
    "ordinary": ((10, 20, 10), 1.0, 0.0, 0.0),
    "one_cell_row": ((3, 3, 3), 1.0, 0.0, 0.0),
    "spread": ((12, 20, 16), 1.0, 4.0, 0.0),
    "root_above_first_decade": ((8, 16, 8), 3e9, 0.0, 0.0),  # above 2^26: found by midpoints
    "root_below_first_decade": ((8, 16, 8), 1e-13, 0.0, 0.0),  # below 2^-30
    "root_beyond_the_bracket": ((8, 16, 8), 1e14, 0.0, 0.0),  # above 1e9: l1 runs up to it
    "bound_never_met": ((8, 16, 8), 1.0, 0.0, 2e4),  # gt <= 0 throughout: l2 runs down to the limit
    "many_blocks": ((64, 128, 70), 1.0, 1.0, 0.0),  # 573,440 cells: more than 2048 blocks of the padded grid
}


@pytest.mark.parametrize("name", list(CASES))
def test_against_sequential_loop(name):
    import top3d_xl_amd as t3x
    shape, scale, spread, dV = CASES[name]
    print(f"\n[gpu-oc] {name}", flush=True)
    rng = np.random.default_rng(23)
    m = t3x.Problem(np.ones(shape, bool))
    try:
        x, dc = design(m.nE, scale, rng, spread)
        V0 = float(x.mean()) + dV
        xg, ch, nb = m.oc(x, x, dc, V0)
    finally:
        m.close()
    xs, chs, ns = sequential(x, x, dc, V0)
    assert nb == ns
    assert np.abs(xg - xs).max() <= 1e-14 and abs(ch - chs) <= 1e-14
