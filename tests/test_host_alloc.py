"""Calls that run out of device memory, and the calls after them (CPU only:
the library's host code is compiled with g++ against a stand-in for the HIP
runtime, tests/host/alloc_failures.cpp, in which no kernel runs)."""
import pathlib
import shutil
import subprocess

import pytest

from conftest import PKG_DIR, REPO

ROCM = pathlib.Path("/opt/rocm/include")

HIPCUB = """#pragma once
#include <hip/hip_runtime.h>
namespace hipcub {
struct DeviceRadixSort {
  template <class... A>
  static hipError_t SortPairs(void*, size_t& bytes, A...) { return bytes = 0, hipSuccess; }
};
}
"""


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if shutil.which("g++") is None or not (ROCM / "hip" / "hip_runtime.h").exists():
        pytest.skip("needs g++ and the HIP headers")
    d = tmp_path_factory.mktemp("host")
    (d / "hipcub").mkdir()
    (d / "hipcub" / "hipcub.hpp").write_text(HIPCUB)
    flags = ["-std=c++17", "-O1", "-x", "c++", "-w", "-D__HIP_PLATFORM_AMD__", "-D__align__(x)=",
             "-DHIP_SYMBOL(x)=((const void*)&(x))", f"-I{d}", f"-I{ROCM}", f"-I{REPO / 'include'}",
             f"-I{PKG_DIR / 'csrc'}"]
    objs = []
    for src in (PKG_DIR / "csrc" / "psdns_api.hip", PKG_DIR / "csrc" / "sgs_api.hip",
                REPO / "tests" / "host" / "alloc_failures.cpp"):
        objs.append(d / (src.name + ".o"))
        subprocess.run(["g++", *flags, "-c", str(src), "-o", str(objs[-1])], check=True)
    # the launchers that the harness does not define do nothing
    syms = subprocess.run(["nm", *map(str, objs)], capture_output=True, text=True, check=True).stdout.split("\n")
    defined = {l.split()[-1] for l in syms if len(l.split()) == 3}
    missing = {l.split()[-1] for l in syms if " U _ZN5psdns" in l} - defined
    stubs = d / "stubs.c"
    stubs.write_text("".join(f"long {m}(void) {{ return 0; }}\n" for m in sorted(missing)))
    exe = d / "alloc_failures"
    subprocess.run(["gcc", "-c", str(stubs), "-o", str(d / "stubs.o")], check=True)
    subprocess.run(["g++", *map(str, objs), str(d / "stubs.o"), "-o", str(exe)], check=True)
    return exe


@pytest.mark.parametrize("case", ["features", "force_list"])
def test_call_after_a_failed_allocation(harness, case):
    r = subprocess.run([str(harness), case], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
