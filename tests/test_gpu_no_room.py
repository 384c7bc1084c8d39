"""What is allocated for speed alone must not be what a call fails for: with no
room for the lattice tables of matrix-free CG (an allocation function that
refuses, loaded before the library in a process of its own), the solve takes its
general form and gives the same answer."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static int left = -1, asked = 0;
void room_for(int n) { left = n; asked = 0; }   /* allocations that succeed from now on (-1: all) */
int refused(void) { return asked; }
int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))dlsym(dlopen("libamdhip64.so", RTLD_NOW), "hipMalloc");
    if (left == 0) { asked++; *p = 0; return 2; }   /* hipErrorOutOfMemory */
    if (left > 0) left--;
    return real(p, n);
}
"""

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path[:0] = sys.argv[2:5]
import numpy as np, mastg as M, pyoracle as O
from helpers import ctx_from_oracle
P = O.Problem(O.CANTILEVER, 12, 7, 5, seed=4, lo=0.1, hi=1.0)
opts = dict(solver=M.SOLVER_MATFREE, rtol=1e-10)
answers = []
for room in (-1, 0, 2, 5):
    ctx = ctx_from_oracle(M, P)
    R, _ = ctx.assemble()
    ctx.solve(-R, solver=M.SOLVER_CG_JACOBI, max_iters=3, raise_on_error=False)   # (everything else is allocated)
    shim.room_for(room)
    x, st = ctx.solve(-R, **opts)
    refused = shim.refused()
    y, sy = ctx.solve(-R, **opts)      # and again
    shim.room_for(-1)
    assert (refused > 0) == (room >= 0), (room, refused)
    assert np.array_equal(x, y) and st["rel_res"] <= 1.5e-10
    answers.append((x, st["iters"]))
    ctx.close()
for x, it in answers[1:]:
    assert np.array_equal(x, answers[1][0]) and it == answers[1][1]
    assert np.abs(x - answers[0][0]).max() <= 1e-8 * np.abs(x).max()
print("OK")
"""


def test_matrix_free_cg_without_room_for_its_tables(oracle, mastg, tmp_path):
    print("[no room] matrix-free CG, hex8 12x7x5", flush=True)
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", str(so), str(src), "-ldl"], check=True)
    p = subprocess.run([sys.executable, "-c", CHILD, str(so)] + [os.path.join(ROOT, *d) for d in
                       (("mast-multiphysics_amd", "python"), ("oracle",), ("tests",))],
                       capture_output=True, text=True, timeout=100)
    assert p.returncode == 0 and p.stdout.strip() == "OK", p.stdout + p.stderr
