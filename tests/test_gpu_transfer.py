"""Fields to the device and back (kh_set_field / kh_get_field, kh_set_fluid /
kh_get_fluid): the rows come back as they went in, bit for bit in FP64 and
rounded once to FP32 in a mixed run, with the real fields' padding columns
zero. Sizes with one chunk, with a last chunk of a few rows and with several
worker threads; and the same without the pinned staging."""
import concurrent.futures

import numpy as np
import pytest

from kapsel3_amd._abi import FP64, MIXED, Params

import interposed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n", [(8, 8, 8), (24, 12, 48), (64, 96, 24), (96, 128, 192)])
def test_fields_round_trip(gpu, n, precision):
    import kapsel3_amd
    print(f"transfer {n} precision {precision}", flush=True)
    rng = np.random.default_rng(7)
    stored = (lambda a: a) if precision == FP64 else (lambda a: a.astype(np.float32).astype(np.float64))
    with kapsel3_amd.Run(Params(n, a=1.0, a_xi=1.0, precision=precision), 0) as r:
        z = [rng.standard_normal(r.shape) for _ in range(3)]
        r.set_fluid(z[0], z[1], [1.0, 2.0, 3.0])
        r.set_field("u1", z[2])
        for _ in range(2):  # the staging of the first transfer serves the second
            z0, z1, uk = r.get_fluid()
            assert np.array_equal(z0, stored(z[0])) and np.array_equal(z1, stored(z[1]))
            assert np.array_equal(uk, [1.0, 2.0, 3.0])
            u = r.get_field("u1")
            assert np.array_equal(u[..., :n[2]], stored(z[2])[..., :n[2]])
            assert not u[..., n[2]:].any()


def test_threads_read_one_run(gpu):
    """Several threads at once, fluid and fields of different sizes of staging:
    each gets what a single thread gets."""
    n = (64, 64, 96)
    print(f"transfer {n}, four threads", flush=True)
    rng = np.random.default_rng(8)
    with gpu.Run(Params(n, a=1.0, a_xi=1.0), 0) as r:
        z = [rng.standard_normal(r.shape) for _ in range(4)]
        r.set_fluid(z[0], z[1], [1.0, 2.0, 3.0])
        r.set_field("u1", z[2])
        r.set_field("u2", z[3])

        def read(k):
            for _ in range(6):
                if k % 2:
                    z0, z1, uk = r.get_fluid()
                    assert np.array_equal(z0, z[0]) and np.array_equal(z1, z[1]) and np.array_equal(uk, [1.0, 2.0, 3.0])
                else:
                    u = r.get_field("u%d" % (1 + k // 2))[..., :n[2]]
                    assert np.array_equal(u, z[2 + k // 2][..., :n[2]])
            return True

        with concurrent.futures.ThreadPoolExecutor(4) as ex:
            assert list(ex.map(read, range(4))) == 4 * [True]


# hipHostMalloc that fails (hipErrorOutOfMemory) beyond `limit` bytes
NO_PINNED = """
size_t limit = 0;
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    *p = NULL;
    if (n > limit) return 2;
    return ((int (*)(void **, size_t, unsigned))hip("hipHostMalloc"))(p, n, flags);
}
"""

ROUND_TRIP = """
limit = ctypes.c_size_t.in_dll(fake, "limit")
import numpy as np
import kapsel3_amd
from kapsel3_amd._abi import FP64, MIXED, Params
rng = np.random.default_rng(7)
for limit.value in (0, 5 << 20):
    for precision in (FP64, MIXED):
        n = (64, 96, 48)
        stored = (lambda a: a) if precision == FP64 else (lambda a: a.astype(np.float32).astype(np.float64))
        with kapsel3_amd.Run(Params(n, a=1.0, a_xi=1.0, precision=precision), 0) as r:
            z = [rng.standard_normal(r.shape) for _ in range(3)]
            for _ in range(2):
                r.set_fluid(z[0], z[1], [1.0, 2.0, 3.0])
                r.set_field("u1", z[2])
                z0, z1, uk = r.get_fluid()
                u = r.get_field("u1")
                assert np.array_equal(z0, stored(z[0])) and np.array_equal(z1, stored(z[1]))
                assert np.array_equal(u[..., :n[2]], stored(z[2])[..., :n[2]]) and not u[..., n[2]:].any()
                r.step(1)  # the failed allocation is not a later launch's error
                r.sync()
        print("same")
"""


def test_without_pinned_memory(gpu, tmp_path):
    """The transfers where the pinned staging cannot be allocated, and where
    only one worker's two slots of it can."""
    print("transfers without pinned memory", flush=True)
    assert interposed.run(tmp_path, NO_PINNED, ROUND_TRIP).splitlines() == 4 * ["same"]
