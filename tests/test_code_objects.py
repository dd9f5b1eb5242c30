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


def test_direct_lds_loads_carry_their_wait_states(code_objects):
    """A load to LDS written as assembly is outside the compiler's hazard pass. Its scalar base may come
    from a vector instruction right before it, which a vector memory instruction may not read for
    five wait states, and m0 needs one: every such load must bring along a scalar move of its base
    between the two. Nothing else may hold a value in m0 across them."""
    loads = 0
    for file in code_objects:
        text = subprocess.run([LLVM + "llvm-objdump", "-d", "--no-show-raw-insn", str(file)], check=True,
                              capture_output=True, text=True).stdout
        code = [line.split("//")[0].split() for line in text.splitlines() if line.startswith("\t")]
        for i, words in enumerate(code):
            if words[0].startswith("global_load_lds"):
                loads += 1
                assert code[i - 2][:2] == ["s_add_u32", "m0,"], code[i - 2]
                assert code[i - 1][0] == "s_mov_b64" and code[i - 1][1].rstrip(",") == words[2], code[i - 1:i + 1]
            elif "m0" in words or "m0," in words:
                assert words[:2] == ["s_add_u32", "m0,"] and code[i + 2][0].startswith("global_load_lds"), words
    assert loads > 0
