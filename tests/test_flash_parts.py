"""The row parts of the flash backward (evk_amd/csrc/flash_parts.h, host
rules) without a GPU: built with g++ and called through ctypes."""
import ctypes as C
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "flash_parts.h"
using namespace evkhip;
extern "C" void plan(int dh, int B, int N, int H, int causal, int64_t* out) {
    const BwdKvPlan p = bwd_kv_plan(dh, B, N, H, causal != 0);
    out[0] = p.part_log2;
    out[1] = p.per_batch;
    out[2] = (int64_t)p.bytes;
}
extern "C" int chunks(int kb, int N, int H, int causal) { return bwd_kv_chunks(kb, N, H, causal != 0); }
"""


@pytest.fixture(scope="module")
def parts(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("parts")
    (d / "shim.cpp").write_text(SHIM)
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + os.path.join(ROOT, "evk_amd", "csrc"),
                        str(d / "shim.cpp"), "-o", str(d / "shim.so")], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    return C.CDLL(str(d / "shim.so"))


def _plan(parts, dh, B, N, H, causal):
    out = (C.c_int64 * 3)()
    parts.plan(dh, B, N, H, int(causal), out)
    return tuple(out)


# dh, B, N, H: one batch of Q below 2 GiB, the largest within 1 %
LONG = [(128, 2, 32768, 8), (128, 1, 65536, 16), (128, 1, 131072, 32), (128, 1, 131072, 63), (128, 64, 16384, 8),
        (128, 1, 8000000, 1), (128, 2, 16384, 8), (64, 1, 65536, 16), (64, 1, 131072, 120), (64, 32, 8192, 8),
        (32, 1, 131072, 250), (32, 4, 65536, 32)]


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dh,B,N,H", LONG)
def test_partials_do_not_grow_with_the_rows(parts, dh, B, N, H, causal):
    """The fp32 partials stay within 5120 slots (a key block's dK and dV: 1 KB
    times the head size) however long the sequence is, while there are still
    enough parts for every CU several times over."""
    assert N * H * dh * 2 < 2**31
    log2, per_batch, nbytes = _plan(parts, dh, B, N, H, causal)
    assert nbytes <= 5120 * dh * 1024
    nkb = -(-N // 128)
    # every chunk of a key block lies in one of its parts
    count = sum(-(-parts.chunks(kb, N, H, int(causal)) // (1 << log2)) for kb in range(nkb))
    assert per_batch == count >= nkb
    assert nbytes == (0 if per_batch == nkb else B * per_batch * dh * 1024)
    assert B * per_batch >= 1024


@pytest.mark.parametrize("dh,B,N,H,causal,log2", [
    (64, 4, 1024, 8, True, 4), (64, 16, 160, 4, True, 2), (32, 1, 888, 1, True, 2), (128, 2, 2000, 8, True, 6),
    (128, 16, 160, 4, True, 2), (128, 1, 130, 2, True, 2), (128, 4, 4096, 8, True, 6), (128, 1, 8, 1, False, 2)])
def test_part_length_of_ordinary_calls(parts, dh, B, N, H, causal, log2):
    assert _plan(parts, dh, B, N, H, causal)[0] == log2
