"""Contexts and batches whose resident memory is not to be had: they are created all the same and run their
solves as launches.  The allocations are made to fail by a hipMalloc that stands before the runtime's in a
process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

INTERPOSER = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = (size_t)-1;
int refused = 0;
void refuse_from(size_t n) { limit = n; }
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (n >= limit) {
        ++refused;
        *p = NULL;
        return 2; /* hipErrorOutOfMemory */
    }
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipMalloc");
    return real(p, n);
}
"""

PROGRAM = r"""
import ctypes as C, sys
import numpy as np
stand_in = C.CDLL(sys.argv[1], C.RTLD_GLOBAL)
stand_in.refuse_from.argtypes = [C.c_size_t]
import cnv
NEVER = 2 ** 64 - 1

def run(kind, limit):
    stand_in.refuse_from(limit)
    kw = dict(Re=400.0, dt=1e-5, tol=1e-4, itmax=100000)
    if kind.startswith("batch"):
        ps = [cnv.default_params(64, precision=int(kind == "batch_refined"), **kw) for _ in range(16)]
        with cnv.Batch(ps) as b:
            stand_in.refuse_from(NEVER)
            st = [s for row in b.step(2) for s in row]
            fields = [b.get_state(i) for i in range(len(ps))]
    else:
        with cnv.Cavity(cnv.default_params(1024, precision=int(kind == "refined"), **kw)) as cav:
            stand_in.refuse_from(NEVER)
            st, fields = cav.step(2), [cav.get_state()]
    return [(s.status, s.k, s.sweeps, s.outer) for s in st], fields

for kind, limit in (("fp64", 20 << 20), ("refined", 12 << 20), ("batch", 1 << 20), ("batch_refined", 1 << 20)):
    want = run(kind, NEVER)
    before = C.c_int.in_dll(stand_in, "refused").value
    got = run(kind, limit)
    assert C.c_int.in_dll(stand_in, "refused").value > before, kind
    assert got[0] == want[0], kind
    for a, b in zip(got[1], want[1]):
        assert all(np.array_equal(a[k], b[k]) for k in ("w", "psi", "u", "v")), kind
    print(kind, "ok", flush=True)
"""


def test_created_without_resident_memory(tmp_path):
    c, so = tmp_path / "stand_in.c", tmp_path / "stand_in.so"
    c.write_text(INTERPOSER)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(c), "-ldl"], check=True)
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "fluid-dynamics1_amd"))
    out = subprocess.run([sys.executable, "-c", PROGRAM, str(so)], env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split()[::2] == ["fp64", "refined", "batch", "batch_refined"]
