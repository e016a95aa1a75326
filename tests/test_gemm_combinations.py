"""A matrix product with a combination of transposes and epilogue that has no
kernel does not compile (gemm, csrc/nn.h): it would launch nothing and leave
its output as it was."""
import os
import shutil
import subprocess

import pytest

from libclsph_amd import build

pytestmark = pytest.mark.skipif(not shutil.which(build.HIPCC), reason="needs hipcc")


@pytest.mark.parametrize("combination,built", [
    ("false, false, nn::kEpiEdgeSilu", True), ("true, true, nn::kEpiAdd", True),
    ("false, true, nn::kEpiDsilu", True), ("false, true, nn::kEpiSilu", False),
    ("true, false, nn::kEpiCast", False), ("false, false, nn::kEpiDsilu", False)])
def test_only_built_combinations_compile(tmp_path, combination, built):
    src = tmp_path / "call.hip"
    src.write_text(f'#include "{os.path.join(build.CSRC, "nn.h")}"\n'
                   "using namespace clsph;\n"
                   "void call(hipStream_t s, const nn::GemmArgs& g) "
                   f"{{ nn::gemm<{combination}>(s, g); }}\n")
    r = subprocess.run([build.HIPCC, "--offload-arch=" + build.ARCH, "-std=c++17",
                        "-fsyntax-only", str(src)], capture_output=True, text=True)
    assert (r.returncode == 0) == built, r.stderr
    assert built or "no such matrix product" in r.stderr
