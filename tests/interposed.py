"""Runs a script in a process whose libkapsel_hip.so finds some HIP calls in a
small C library first (allocations that fail or are counted)."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# hipMallocAsync that fails (hipErrorOutOfMemory) at its call number fail_at, and the number of live allocations
COUNTED = """
int fail_at = -1, calls = 0, live = 0;
int hipMallocAsync(void **p, size_t n, void *s) {
    if (++calls == fail_at) return 2;
    int e = ((int (*)(void **, size_t, void *))hip("hipMallocAsync"))(p, n, s);
    live += e == 0;
    return e;
}
int hipFreeAsync(void *p, void *s) {
    live--;
    return ((int (*)(void *, void *))hip("hipFreeAsync"))(p, s);
}
"""


def run(tmp_path, source, script):
    """The script's standard output; it finds the C library as `fake`."""
    src, so = tmp_path / "fake.c", tmp_path / "fake.so"
    src.write_text('#include <dlfcn.h>\n#include <stddef.h>\n'
                   'static void *hip(const char *f) { return dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), f); }\n'
                   + source)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src), "-ldl"], check=True)
    # loaded before the library, whose calls bind to it
    pre = "import ctypes, sys\nfake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)\n"
    p = subprocess.run([sys.executable, "-c", pre + script, str(so)], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert p.returncode == 0, p.stdout + p.stderr
    return p.stdout
