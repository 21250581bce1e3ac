"""Kernel shape options without a GPU: every shape that the library accepts
compiles for gfx950 within the 160 KB of LDS, and the rest is refused with a
message of the library's, not the compiler's."""
import shutil
import subprocess
from pathlib import Path

import pytest

from mifem import problems
from test_codegen_cpu import _READELF, _describe, _kernels

ROOT = Path(__file__).resolve().parent.parent


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    build = ROOT / "cuda-dolfinx_amd" / "_build"
    objs = [build / f"{n}.o" for n in ("codegen", "runtime", "owner_kernel", "hex_kernel",
                                       "dg_kernel", "sparsity", "util_kernels", "matrix")]
    if not shutil.which("hipcc") or not _READELF.exists() or not all(o.exists() for o in objs):
        pytest.skip("hipcc / llvm-readelf / library objects not available")
    d = tmp_path_factory.mktemp("shapes")
    subprocess.run(["hipcc", "-c", "--offload-arch=gfx950", "-fPIC", "-std=c++17", "-O1",
                    f"-I{ROOT / 'cuda-dolfinx_amd' / 'csrc'}", f"-I{ROOT / 'include'}",
                    str(ROOT / "tests" / "shape_check.cpp"), "-o", str(d / "check.o")], check=True)
    subprocess.run(["hipcc", str(d / "check.o"), *map(str, objs), "-lhiprtc", "-o", str(d / "check")],
                   check=True)

    def run(form, **options):
        """(kernels of the code object or None, message)"""
        _describe(form, d / "form.txt")
        r = subprocess.run([str(d / "check"), str(d / "form.txt"), str(d / "form.co"),
                            *[f"{k}={v}" for k, v in options.items()]],
                           stdout=subprocess.PIPE, stderr=subprocess.DEVNULL, text=True, timeout=300)
        return (_kernels(d / "form.co") if r.stdout.startswith("OK") else None), r.stdout

    return run


@pytest.mark.parametrize("options", [
    {}, {"hex_block": 64}, {"chunk_rows": 255}, {"chunk_rows": 256}, {"chunk_rows": 600, "hex_block": 512},
    {"chunk_rows": 2000}, {"hex_block": 64, "owner_nb": 70, "owner_lds": 160000},
    {"chunk_values": 343}, {"hex_block": 1024}])
def test_hexahedral_shapes_compile(driver, options):
    K, msg = driver(problems.helmholtz_q3(2).a, **options)
    assert K is not None, msg[:2000]
    for k in ("mf_howner64_cell_0", "mf_howner32_cell_0", "mf_howner16_cell_0"):
        assert K[k][2] <= 160 * 1024


@pytest.mark.parametrize("block", [0, 32, 100, 1088])
def test_hexahedral_block_of_whole_waves(driver, block):
    K, msg = driver(problems.helmholtz_q3(2).a, hex_block=block)
    assert K is None and "hex_block" in msg and "error:" not in msg


def _stiffness(degree):
    from mifem import forms
    from mifem.fem import Function, functionspace
    from mifem.mesh import create_unit_cube
    m = create_unit_cube(2)
    return forms.stiffness(functionspace(m, ("P", degree)), Function(functionspace(m, ("DG", 0))))


@pytest.mark.parametrize("degree,options,fits", [
    (3, {"chunk_values": 4096, "owner_pairs": 256}, True),               # 58,960 bytes of 65,536
    (3, {"chunk_values": 4904, "owner_pairs": 256}, True),               # 65,424
    (3, {"chunk_values": 4936, "owner_pairs": 256}, False),              # 65,680
    (3, {"chunk_values": 8214, "owner_pairs": 256, "owner_lds": 160 * 1024}, True),
    (3, {"chunk_values": 8192, "owner_pairs": 256, "owner_lds": 160 * 1024}, True),
    (2, {"chunk_values": 6144, "owner_pairs": 384}, True),
    (1, {"chunk_values": 7168, "owner_pairs": 384}, True),
    (0, {"chunk_values": 6400, "owner_pairs": 128}, True),               # vector P2: its 16 or 32 gradients
    (0, {"chunk_values": 4608, "owner_pairs": 384}, True),
])
def test_owner_shapes_that_fit_the_budget(driver, degree, options, fits):
    """The LDS that the host counts is the LDS of the compiled kernel: a shape is
    taken exactly when the kernel fits owner_lds, and a store-wave variant that does
    not fit a CU is left out."""
    K, msg = driver(_stiffness(degree) if degree else problems.elasticity_p2(2).a, **options)
    if not fits:
        assert K is None and "LDS budget" in msg
        return
    assert K is not None, msg[:1000]
    lds = K["mf_owner_cell_0"][2]
    assert lds <= options.get("owner_lds", 64 * 1024)
    assert K.get("mf_ownerp_cell_0", (0, 0, 0))[2] <= 160 * 1024
    short, msg = driver(_stiffness(degree) if degree else problems.elasticity_p2(2).a, **{**options, "owner_lds": lds - 1})
    assert short is None and "LDS budget" in msg


def test_allocation_that_may_fail(tmp_path):
    """DevArray::try_alloc of a petabyte (or without a device, of anything): false and
    no exception; with a device, no error left that the next call would report."""
    if not shutil.which("hipcc"):
        pytest.skip("hipcc not available")
    (tmp_path / "t.cpp").write_text('''#include "mf_internal.h"
int main() {
  mf::DevArray<double> d;
  if (d.try_alloc(int64_t(1) << 47) || d.ptr || d.n) return 1;
  if (!d.try_alloc(0) || d.ptr) return 2;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return 0;
  return hipGetLastError() == hipSuccess ? 0 : 3;
}
''')
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-std=c++17", "-O1", f"-I{ROOT / 'cuda-dolfinx_amd' / 'csrc'}",
                    f"-I{ROOT / 'include'}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    assert subprocess.run([str(tmp_path / "t")], timeout=60).returncode == 0
