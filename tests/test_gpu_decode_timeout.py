"""A cached step that reports a lost exchange is not taken: the next one, at the same position,
gives what it would have given. The report is put into the error word as the host reads it
back (the kernel itself ran to its end and moved its position), by a hipMemcpyAsync of this
test's own in front of the runtime's, in a process of its own."""
import shutil
import subprocess
import sys

import pytest

from conftest import REPO

pytestmark = pytest.mark.gpu

HOOK = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
int armed = 0;
int hipMemcpyAsync(void* dst, const void* src, size_t bytes, int kind, void* stream) {
  static int (*copy)(void*, const void*, size_t, int, void*) = 0;
  static int (*wait)(void*) = 0;
  if (!copy) {
    void* rt = dlopen("libamdhip64.so", RTLD_LAZY | RTLD_NOLOAD);
    if (!rt) rt = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    if (!rt) return 1;
    copy = (int (*)(void*, const void*, size_t, int, void*))dlsym(rt, "hipMemcpyAsync");
    wait = (int (*)(void*))dlsym(rt, "hipStreamSynchronize");
  }
  int rc = copy(dst, src, bytes, kind, stream);
  if (armed && rc == 0 && kind == 2 && bytes == sizeof(int)) {  /* the error word, to the host */
    rc = wait(stream);
    *(int*)dst |= 4;
    armed = 0;
  }
  return rc;
}
"""

SCRIPT = r"""
import ctypes as C, sys
hook = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
import numpy as np
import nimbleml_amd as nm
from nimbleml_amd import _native as N
from oracle.weights import GPTConfig, make_weights, random_ids

cfg = GPTConfig(512, 1024, 16, 1, 64)
m = nm.GPT.from_arrays(make_weights(cfg, seed=2, dtype=np.float32), cfg.vocab_size, cfg.d_model, cfg.num_heads,
                       cfg.num_layers, cfg.max_seq_len, dtype=np.float32)
h = m._device_model()
ids = N.DeviceArray.from_host(random_ids((1, 9), cfg.vocab_size, seed=3))

def run(lose):
    cache, out, n = C.c_void_p(), N.DeviceArray((1, cfg.vocab_size), np.float32), C.c_size_t()
    N.check(N.lib.nml_cache_create(h, 1, C.byref(cache)))
    N.check(N.lib.nml_model_forward_cached(h, cache, ids.ptr, 1, 4, out.ptr, 1))
    got = []
    for t in range(4, 9):
        if t == 6 and lose:
            C.c_int.in_dll(hook, "armed").value = 1
            assert N.lib.nml_model_forward_cached(h, cache, ids.ptr + 8 * t, 1, 1, out.ptr, 0) != 0
            assert C.c_int.in_dll(hook, "armed").value == 0
            assert b"timed out" in N.lib.nml_last_error()
        N.check(N.lib.nml_model_forward_cached(h, cache, ids.ptr + 8 * t, 1, 1, out.ptr, 0))
        N.check(N.lib.nml_cache_length(cache, C.byref(n)))
        assert n.value == t + 1
        got.append(out.numpy())
    N.check(N.lib.nml_cache_destroy(cache))
    return got

for a, b in zip(run(False), run(True)):
    assert np.array_equal(a, b)
print("same")
"""


def test_step_after_a_lost_exchange(gpu, tmp_path):
    cc = shutil.which("gcc")
    if not cc:
        pytest.skip("no C compiler")
    src, lib = tmp_path / "hook.c", tmp_path / "libhook.so"
    src.write_text(HOOK)
    subprocess.run([cc, "-shared", "-fPIC", "-O1", "-o", str(lib), str(src), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", SCRIPT, str(lib)], cwd=REPO, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "same" in r.stdout, r.stdout + r.stderr
