"""Input rows of a prefill in pageable memory, which cross in pieces of 64 through pinned memory from 97 rows on: the same rows in
pageable, pinned and device memory leave the same residual stream and cache rows, bit for bit, at the edges of a piece and of that rule, with a
longer prompt and a shorter one behind it, and the caller's buffer is free behind the call.  And where that pinned memory cannot be had, the
same rows cross without it."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

import hipsupport as H
import vtsupport as S

pytestmark = pytest.mark.gpu

ROWS = [96, 97, 128, 129, 300, 2048, 2049, 200]


def test_rows_from_any_memory():
    hip = H.Hip(kv_max=2100)
    libhip = C.CDLL("libamdhip64.so")
    try:
        hip.upload_decoder([S.Layer(11)], S.norm_weight(S.DIM, 98), 1)
        for n in ROWS:
            print(f"prefill of {n} rows", flush=True)
            e = S.f32_normal((n, S.DIM), 60 + n)
            pinned = C.c_void_p()
            assert libhip.hipHostMalloc(C.byref(pinned), C.c_size_t(e.nbytes), C.c_uint(0)) == 0
            C.memmove(pinned, e.ctypes.data, e.nbytes)
            dev = H.DevBuf.from_numpy(hip.lib, e)
            got = []
            for ptr in (e.ctypes.data, pinned.value, dev.ptr):
                x = np.zeros_like(e)
                hip.lib.tts_hip_llm_prefill_out(ptr, n, 0, x.ctypes.data)
                if ptr == e.ctypes.data:
                    e[:] = np.nan
                hip.check()
                k, v = hip.kv()
                got.append((x, k[0, :n].copy(), v[0, :n].copy()))
            assert np.isfinite(got[0][0]).all()
            for other in got[1:]:
                for a, b in zip(got[0], other):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), n
            dev.free()
            assert libhip.hipHostFree(pinned) == 0
    finally:
        hip.close()


# Stands in front of the runtime's function where it is loaded first: no pinned block of more than 1 MB
REFUSE = r"""
#include <dlfcn.h>
#include <stddef.h>
int refused = 0;
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    if (n > (1u << 20)) { refused++; *p = NULL; return 2; }
    return ((int (*)(void **, size_t, unsigned))dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipHostMalloc"))(p, n, flags);
}
"""

# prefills of rows in pageable memory, in a process of their own; saves the residual streams
PREFILLS = """
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
refuse = C.CDLL(sys.argv[3], mode=C.RTLD_GLOBAL) if len(sys.argv) > 3 else None
import numpy as np
import hipsupport as H, vtsupport as S
hip = H.Hip(kv_max=600)
assert refuse is None or C.c_int.in_dll(refuse, "refused").value > 0
hip.upload_decoder([S.Layer(12)], S.norm_weight(S.DIM, 97), 1)
out = {}
for n in (97, 300, 600):
    print("prefill of", n, "rows", flush=True)
    hip.pos = 0
    out[str(n)] = hip.llm_prefill(S.f32_normal((n, S.DIM), 70 + n), want_x=True)
assert hip.lib.tts_hip_error_count() == 0
hip.close()
np.savez(sys.argv[2], **out)
"""


def test_without_pinned_rows(tmp_path):
    src, lib = tmp_path / "refuse.c", tmp_path / "librefuse.so"
    src.write_text(REFUSE)
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"])
    got = []
    for i, extra in enumerate(([], [str(lib)])):
        npz = str(tmp_path / f"{i}.npz")
        subprocess.check_call([sys.executable, "-c", PREFILLS, os.path.dirname(os.path.abspath(__file__)), npz] + extra, timeout=100)
        got.append(np.load(npz))
    for n in got[0].files:
        assert np.isfinite(got[0][n]).all()
        assert np.array_equal(got[0][n].view(np.uint32), got[1][n].view(np.uint32)), n
