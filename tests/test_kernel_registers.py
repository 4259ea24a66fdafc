"""What the compiler made of the kernels that run the large products and 3x3 convolutions: the registers that decide how many of their workgroups a
compute unit takes at once. The launches are cut into slices on the assumption that eight do."""
import os
import re
import subprocess

import pytest

import neoml_amd

LLVM = "/opt/rocm/llvm/bin"
OBJECT = os.path.join(os.path.dirname(neoml_amd.LIB_PATH), "gemm_mfma.o")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(OBJECT) or not os.path.exists(os.path.join(LLVM, "clang-offload-bundler")):
        pytest.skip("no object file of a build, or no tools to look into it")
    at = tmp_path_factory.mktemp("code")
    bundle, code = str(at / "bundle"), str(at / "code")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + bundle, OBJECT, os.devnull], check=True)
    subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + bundle,
                    "--output=" + code], check=True)
    notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", code], check=True, stdout=subprocess.PIPE, text=True).stdout
    found = {}
    for part in notes.split(".name:")[1:]:
        values = dict(re.findall(r"\.(vgpr_count|vgpr_spill_count|agpr_count):\s+(\d+)", part))
        # ( arguments have names too; a kernel's is followed by its counts )
        if "vgpr_count" in values:
            found.setdefault(part.split()[0], values)
    return found


# rows times rows, 3x3 convolutions, each with one and two groups of wavefronts, without and with a residual
@pytest.mark.parametrize("mode", [0, 6])
@pytest.mark.parametrize("groups", [1, 2])
@pytest.mark.parametrize("kernel", ["matMulKernel", "matMulResidualKernel"])
def test_eight_workgroups_fit(kernels, mode, groups, kernel):
    # 64 x 64 tiles by 2 x 2 wavefronts, vector loads
    name = "%sILi64ELi64ELi2ELi2ELi%dELi0ELb1ELi%dEE" % (kernel, mode, groups)
    of = [v for k, v in kernels.items() if name in k]
    assert len(of) == 1, name
    # 512 registers to a SIMD's lane: eight wavefronts of 64
    assert int(of[0]["vgpr_count"]) <= 64 and int(of[0]["vgpr_spill_count"]) == 0, of
