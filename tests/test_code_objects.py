"""Properties of the compiled gfx950 kernels that no result shows, read from the built library's own
code objects on the CPU."""
import re
import shutil
import subprocess

import pytest

LLVM = "/opt/rocm/llvm/bin/"


@pytest.fixture(scope="module")
def code_objects(mh, tmp_path_factory):
    folder = tmp_path_factory.mktemp("code_objects")
    library = shutil.copy(mh.LIB_PATH, folder)
    subprocess.run([LLVM + "llvm-objdump", "--offloading", library], cwd=folder, check=True, capture_output=True)
    files = sorted(folder.glob("*gfx950"))
    assert files
    return files


def kernel_registers(code_objects):
    """Vector registers of each kernel, by its mangled name."""
    count = {}
    for file in code_objects:
        notes = subprocess.run([LLVM + "llvm-readelf", "--notes", str(file)], check=True, capture_output=True,
                               text=True).stdout
        for name, registers in re.findall(r"\.name: +(_Z\w+).*?\.vgpr_count: +(\d+)", notes, re.S):
            count[name] = int(registers)
    return count


def test_rope_of_whole_sums_keeps_eight_waves_in_flight(code_objects):
    """muyo_rope_split_append_f16kv takes whole sums: its kernel does not carry the registers of the
    eight-part one. A SIMD holds eight waves of at most 64 registers."""
    count = kernel_registers(code_objects)
    assert min(v for k, v in count.items() if "RopeSplitAppendQuadKernel" in k) <= 64
