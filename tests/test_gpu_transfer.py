"""Fields to the device and back (kh_set_field / kh_get_field, kh_set_fluid /
kh_get_fluid): the rows come back as they went in, bit for bit in FP64 and
rounded once to FP32 in a mixed run, with the real fields' padding columns
zero. Sizes with one chunk, with a last chunk of a few rows and with several
worker threads; and the same without the pinned staging."""
import os
import subprocess
import sys

import numpy as np
import pytest

from kapsel3_amd._abi import FP64, MIXED, Params

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


NO_PINNED = """
#include <dlfcn.h>
#include <stddef.h>
#include <stdlib.h>
/* hipHostMalloc that fails (hipErrorOutOfMemory) beyond LIMIT bytes */
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    *p = NULL;
    if (n > (size_t)atoll(getenv("LIMIT"))) return 2;
    void *h = dlopen("libamdhip64.so.7", RTLD_LAZY);
    return ((int (*)(void **, size_t, unsigned))dlsym(h, "hipHostMalloc"))(p, n, flags);
}
"""

ROUND_TRIP = """
import ctypes, os, sys
ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)  # before the library, whose calls bind to it
import numpy as np
import kapsel3_amd
from kapsel3_amd._abi import FP64, MIXED, Params
rng = np.random.default_rng(7)
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


@pytest.mark.parametrize("limit", [0, 5 << 20], ids=["none", "one worker's"])
def test_without_pinned_memory(gpu, tmp_path, limit):
    """The transfers where the pinned staging cannot be allocated, or only one
    worker's two slots of it."""
    print(f"transfer with {limit} bytes of pinned memory", flush=True)
    src, so = tmp_path / "nopinned.c", tmp_path / "nopinned.so"
    src.write_text(NO_PINNED)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(gpu.__file__)))
    p = subprocess.run([sys.executable, "-c", ROUND_TRIP, str(so)], cwd=root, capture_output=True, text=True,
                       timeout=100, env={**os.environ, "LIMIT": str(limit)})
    assert p.returncode == 0 and p.stdout.strip() == "same", p.stdout + p.stderr
