"""The order of the row-split kernel's memory requests, read from the assembly the build's own command line gives: a decode GEMM lives
10-20 us, and a request that the compiler moves behind a hundred instructions costs 1-3 % of it while every result stays the same."""
import importlib.util
import os
import re
import shutil
import subprocess

import pytest

_PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hf-rocm-kernels_amd")


def _instances(tmp_path):
    """(template arguments, instructions and labels) of every instance of the kernel on row-major weights in 4-row units."""
    spec = importlib.util.spec_from_file_location("hfrk_build", os.path.join(_PACKAGE, "build.py"))
    build = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(build)
    hipcc = shutil.which("hipcc") or os.path.join(build.ROCM, "bin", "hipcc")
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc here")
    out = os.path.join(tmp_path, "rows.s")
    subprocess.run([hipcc] + build.HIPCC_FLAGS + ["--offload-device-only", "-S", os.path.join(build.CSRC, "skinny_gemm_rows.hip"), "-o", out],
                   check=True, capture_output=True)
    found, body = {}, None
    for line in open(out):
        start = re.match(r"_ZN4hfrk\d+skinny_gemm_rows_kernelI(\S+?)EEEv", line)
        if start:
            body = found.setdefault(start[1], [])
        elif line.startswith(".Lfunc_end"):
            body = None
        elif body is not None:
            text = line.split(";")[0].strip() + (" ; loop header" if "Loop Header" in line else "")
            if text and (not text.startswith(".") or text.startswith(".LBB")):
                body.append(text)
    return found


def test_requests_stay_where_the_kernel_makes_them(tmp_path):
    instances = _instances(tmp_path)
    assert len(instances) == 20
    for name, body in instances.items():
        first = next(i for i, x in enumerate(body) if x.startswith("buffer_load_dwordx4") and " nt" in x)
        scale = next(i for i, x in enumerate(body) if x.startswith("global_load_dword "))
        assert 0 < scale - first < 60, (name, "the activation scales are requested with the first chunk", scale - first)
        multiply = next(i for i, x in enumerate(body) if x.startswith("v_mfma"))
        loop = max(i for i, x in enumerate(body[:multiply]) if "loop header" in x)
        turn = body[loop:multiply]
        request = next(i for i, x in enumerate(turn) if x.startswith("buffer_load_dwordx4") and " nt" in x)
        copied = max(i for i, x in enumerate(turn[:request]) if x.startswith("ds_write_b128"))
        branches = sum(x.startswith(("s_cbranch", "s_branch")) for x in turn[copied:request])
        assert branches <= 1 and request - copied < 30, (name, "the next chunk is requested behind the copy of this one", branches, request - copied)
