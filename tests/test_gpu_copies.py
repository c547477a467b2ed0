"""Copies between device and host memory: the bytes at the sizes where their
route changes, and where no pinned memory is to be had."""
import os
import subprocess
import sys

import numpy as np
import pytest

import modalcmb
from conftest import ROOT

pytestmark = pytest.mark.gpu

MIB = 1 << 20
SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
/* the device's allocation of pinned memory, failing from 4 MiB on */
int refused = 0;
int hipHostMalloc(void** p, size_t n, unsigned flags)
{
    static int (*real)(void**, size_t, unsigned);
    if (!real) *(void**)&real = dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), "hipHostMalloc");
    if (n >= 4u << 20) {
        ++refused;
        *p = 0;
        return 2; /* hipErrorOutOfMemory */
    }
    return real(p, n, flags);
}
"""
USER = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import modalcmb
rng = np.random.default_rng(1)
with modalcmb.Context(0) as ctx:
    n = 1100                                   # 9.7 MB: staged in and out, were there pinned memory
    A = rng.standard_normal((n, n))
    G = A @ A.T + n * np.eye(n)
    ortho, lam, norm = ctx.orthonormalise(G)
    F = np.tril(ortho)
    assert np.abs(F @ F.T - G).max() < 1e-11 * np.abs(G).max()
    assert np.abs(np.tril(lam) @ F - np.eye(n)).max() < 1e-9
    n = 2100                                   # 35 MB: the larger staging
    G = np.diag(np.arange(1.0, n + 1))
    ortho, lam, norm = ctx.orthonormalise(G)
    # (i / (sqrt i sqrt i), its root and the product with sqrt i each round once)
    assert np.allclose(ortho, np.diag(np.sqrt(np.arange(1.0, n + 1))), rtol=1e-15, atol=0)
refused = ctypes.c_int.in_dll(shim, "refused").value
assert refused >= 2, refused
print("ok")
"""


# bytes at and next to the sizes from which copies are staged in (4 MiB) and out
# (8 MiB) and from which they take the larger staging (32 MiB): chunks of 2 MiB
# in four slots, of 4 MiB in eight; a short last chunk, fewer chunks than slots
@pytest.mark.parametrize("nbytes", [4 * MIB - 8, 4 * MIB, 4 * MIB + 8, 6 * MIB, 8 * MIB - 8, 8 * MIB, 8 * MIB + 8,
                                    10 * MIB + 520, 32 * MIB - 8, 32 * MIB, 32 * MIB + 8, 45 * MIB + 136])
def test_bytes_in_and_out(ctx, nbytes):
    # a solve with the unit matrix returns its right-hand sides: in and out again
    rhs = np.random.default_rng(nbytes).standard_normal((nbytes // 8, 1))
    got = ctx.cholesky_solve(np.eye(1), rhs.T)
    assert np.array_equal(got.ravel(), rhs.ravel())
    # out alone, to an offset address
    dev = ctx.device_alloc(nbytes)
    try:
        out = [np.zeros(nbytes // 8 + 1) for _ in range(2)]
        ctx.device_to_host(dev, out[0][1:])
        os.environ["MCMB_HOST_COPY"] = "direct"
        try:
            ctx.device_to_host(dev, out[1][1:])
        finally:
            del os.environ["MCMB_HOST_COPY"]
    finally:
        ctx.device_free(dev)
    assert np.array_equal(out[0].view(np.int64), out[1].view(np.int64))


def test_copies_without_pinned_memory(tmp_path):
    (tmp_path / "shim.c").write_text(SHIM)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "shim.c"), "-ldl"], check=True, timeout=60)
    env = dict(os.environ)
    env["PYTHONPATH"] = os.pathsep.join([os.path.join(ROOT, "modal-cmb_amd"), env.get("PYTHONPATH", "")])
    r = subprocess.run([sys.executable, "-c", USER, so], capture_output=True, text=True, env=env, timeout=100)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout + r.stderr
