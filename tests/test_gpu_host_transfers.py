"""Host arrays through the pinned ring: a start vector that goes up and comes
back after a solve of no iterations, its bits unchanged.

The sizes put the copy below one chunk, at a chunk's and the smallest ring's
remainder, across several rounds of the ring, and on each number of threads;
values include NaN, infinities, denormals and signed zeros."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (cells, what the 24 bytes per node of a vector make of the copy)
SHAPES = {
    "part_of_a_chunk": (4, 6, 4),
    "one_chunk_and_a_bit": (27, 27, 28),
    "two_mb_ring_twice": (39, 79, 39),
    "threads_one_ring": (60, 121, 80),
    "threads_several_rounds": (83, 167, 83),
    "most_threads": (110, 223, 110),
}


@pytest.mark.parametrize("name", list(SHAPES))
def test_vector_up_and_back(name):
    import top3d_xl_amd.t3x as t3x
    p = t3x.Problem(np.ones(SHAPES[name], bool))
    p.set_modulus(np.ones(p.nE))
    p.assemble()
    b = p.load_vector()
    rng = np.random.default_rng(len(name))
    x0 = rng.standard_normal(3 * p.nN)
    x0[:6] = [np.nan, np.inf, -np.inf, 5e-324, -0.0, 1.0]
    x0[-1] = 2.0
    for _ in range(3):  # the ring's chunks are used again
        x, its, _ = p.pcg(b, x0=x0, maxit=0)
        assert its == 0 and np.array_equal(x.view(np.int64), x0.view(np.int64))
        x0 = np.roll(x0, 12345)
    p.close()


def test_pinned_and_strided_arrays():
    import ctypes as C
    import top3d_xl_amd.t3x as t3x
    p = t3x.Problem(np.ones((39, 79, 39), bool))
    p.set_modulus(np.ones(p.nE))
    u = np.random.default_rng(5).standard_normal(3 * p.nN)
    mem = C.c_void_p()
    assert p.L.hipHostMalloc(C.byref(mem), C.c_size_t(u.nbytes), C.c_uint(0)) == 0
    pinned = np.ctypeslib.as_array(C.cast(mem, C.POINTER(C.c_double)), u.shape)
    pinned[:] = u
    assert np.array_equal(p.apply_K(u), p.apply_K(pinned))
    assert np.array_equal(p.apply_K(u), p.apply_K(np.repeat(u, 2)[::2]))
    assert p.L.hipHostFree(mem) == 0
    x = 0.1 + 0.3 * np.random.default_rng(6).random(p.nE)
    dc = -x ** 2
    whole, strided = p.oc(x, x, dc, 0.2), p.oc(np.repeat(x, 3)[::3], x, dc, 0.2)
    assert np.array_equal(whole[0], strided[0]) and whole[1:] == strided[1:]
    p.close()


def test_zero_start_is_the_zero_vector():
    import top3d_xl_amd.t3x as t3x
    p = t3x.Problem(np.ones((12, 24, 12), bool))
    p.set_modulus(np.ones(p.nE))
    p.assemble()
    b = p.load_vector()
    a, c = p.pcg(b), p.pcg(b, x0=np.zeros(3 * p.nN))
    assert a[1] == c[1] and a[2] == c[2] and np.array_equal(a[0], c[0])
    p.close()


def test_an_earlier_error_of_the_thread_is_not_the_transfer_s():
    import top3d_xl_amd.t3x as t3x
    p = t3x.Problem(np.ones((6, 8, 6), bool))
    p.set_modulus(np.ones(p.nE))
    u = np.random.default_rng(2).standard_normal(3 * p.nN)
    y = p.apply_K(u)
    assert p.L.hipSetDevice(4096) != 0  # refused by the runtime, and remembered as the thread's last error
    try:
        assert np.array_equal(p.apply_K(u), y)
    finally:
        p.L.hipGetLastError()  # forget it: later calls in this process look at it
        p.close()
