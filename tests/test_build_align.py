"""The kernels' vector accesses claim no more alignment than a tensor's element
type has: a pointer that promises 16 bytes for memory that only its element
type aligns is undefined behaviour, whatever instructions one compiler makes
of it.  hipcc's front end finds those (-Walign-mismatch); the build refuses
them.  Needs hipcc, no GPU.
"""

import os
import subprocess

import pytest

from luma_amd import build as B

try:
    HIPCC = B.hipcc()
except RuntimeError:
    HIPCC = None

needs_hipcc = pytest.mark.skipif(HIPCC is None, reason="hipcc not installed")


def _check(source, *more):
    return subprocess.run([HIPCC, *B.FLAGS, *more, "-I", os.path.join(B.HERE, "csrc"),
                           "--cuda-device-only", "-fsyntax-only", source],
                          capture_output=True, text=True, timeout=110)


@needs_hipcc
@pytest.mark.parametrize("source,unit", [(s, u) for s, units in B.SOURCES for u in units])
def test_no_access_claims_more_alignment_than_its_pointer(source, unit):
    res = _check(source, f"-DLUMA_UNIT={unit}")
    assert res.returncode == 0, res.stderr
    assert "-Walign-mismatch" not in res.stderr


@needs_hipcc
def test_build_refuses_an_alignment_lost_in_a_template(tmp_path):
    """The form that the flag is there for: the deduced vector type has lost
    the alignment that the pointer was declared with."""
    src = tmp_path / "lost.hip"
    src.write_text(
        "#include <hip/hip_runtime.h>\n"
        "typedef unsigned v4u __attribute__((ext_vector_type(4), aligned(2)));\n"
        "template <typename V> __device__ V get(const V *p) {"
        " return __builtin_nontemporal_load(p); }\n"
        "__global__ void k(const short *a, v4u *o) { *o = get((const v4u *)a); }\n")
    res = _check(str(src))
    assert res.returncode != 0 and "align-mismatch" in res.stderr
