"""Host builds of pieces of the product's C++ that are checked more closely on the CPU than a
GPU run could: tests/native/*.cpp, compiled here with the sources under jieyu_amd/csrc."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "jieyu_amd", "csrc")
NATIVE = os.path.join(ROOT, "tests", "native")


def compile_native(out, *args):
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-I", CSRC, *args, "-o", str(out)],
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout


@pytest.fixture(scope="module")
def gemm_offsets(tmp_path_factory):
    so = tmp_path_factory.mktemp("native") / "gemm_offsets.so"
    compile_native(so, "-shared", "-fPIC", os.path.join(NATIVE, "gemm_offsets.cpp"))
    lib = C.CDLL(str(so))
    lib.gemm_offsets_bad.restype = C.c_longlong
    return lib.gemm_offsets_bad


# rows that end inside a 16-, 32-, 128- and 256-column tile (waves past the last column tile:
# 1152 in 256-column tiles), block counts that leave 0, 1, 2 or 3 blocks of a step of four, one
# block alone, K slices that begin and end inside a step
@pytest.mark.parametrize("nt", [1, 2])
@pytest.mark.parametrize("slices", [1, 3, 8])
def test_prompt_gemm_weight_loads_stay_inside(gemm_offsets, nt, slices):
    """no weight or scale load of any wave, step and prefetch outside the matrix's copy"""
    for rows in (1, 16, 17, 32, 77, 130, 896, 1152, 4112, 4608):
        for cols in (32, 64, 96, 128, 160, 896, 4864, 14336):
            assert gemm_offsets(rows, cols, nt, slices) == 0, (rows, cols)


@pytest.fixture(scope="module")
def stage(tmp_path_factory):
    exe = tmp_path_factory.mktemp("native") / "stage"
    compile_native(exe, "-pthread", "-I", os.path.join(NATIVE, "hip_stub"), os.path.join(NATIVE, "stage.cpp"),
                   os.path.join(CSRC, "jy_stage.cpp"))
    return exe


# no_host_allocation: jyhip_forward_cached_noalloc's transfers, of any size
@pytest.mark.parametrize("case", ["made_when_needed", "round_trip", "no_host_allocation", "after_an_error"])
def test_pinned_ring(stage, case):
    r = subprocess.run([str(stage), case], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_plain_epilogues(tmp_path):
    """the launches of plain products (store, bias, residual) refuse the other epilogues"""
    src = tmp_path / "epi.cpp"
    src.write_text("""
#include "jy_epi.h"
using namespace jy;
static bool refused(Epi e) {
    try { return plain_epi(e) != e; } catch (const std::exception&) { return true; }
}
int main() {
    for (Epi e : {EPI_STORE, EPI_BIAS, EPI_RESID}) if (refused(e)) return 1;
    for (Epi e : {EPI_SWIGLU, EPI_ROPE, EPI_ARGMAX}) if (!refused(e)) return 2;
    return 0;
}
""")
    compile_native(tmp_path / "epi", str(src))
    assert subprocess.run([str(tmp_path / "epi")]).returncode == 0
    # every one of them goes through that check
    for f, n in (("jy_kernels.hip", 1), ("jy_gemm_exact.hip", 2), ("jy_quant.hip", 1)):
        assert open(os.path.join(CSRC, f)).read().count("plain_epi(epi)") == n, f
