"""The gfx950 code that the compiler made of the Q8_0 kernels of few positions, read back from the built code object: what
their comments say of it - every load of a turn is asked for before the first is waited for, and nothing is spilled to
memory - is decided by the compiler, shows in no result and costs a third of such a product's time."""
import os
import re
import subprocess

import pytest

HSACO = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "loadngo_amd", "lng_kernels.hsaco")
TOOLS = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")


def tool(name, *args):
    return subprocess.run([os.path.join(TOOLS, name), *args], stdout=subprocess.PIPE, text=True, check=True).stdout


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Instructions (without addresses) and scratch bytes by kernel name."""
    elf = str(tmp_path_factory.mktemp("code") / "kernels.elf")
    tool("clang-offload-bundler", "--unbundle", "--type=o", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + HSACO, "--output=" + elf)
    code = {}
    for part in re.split(r"^[0-9a-f]+ <", tool("llvm-objdump", "-d", "--no-show-raw-insn", elf), flags=re.M)[1:]:
        name, body = part.split(">:", 1)
        code[name] = [re.sub(r"\s*//.*", "", line).strip() for line in body.splitlines() if line.strip()]
    scratch = {}
    for entry in tool("llvm-readelf", "--notes", elf).split(".agpr_count")[1:]:
        scratch[re.search(r"\.symbol:\s+'?(\w+)\.kd", entry).group(1)] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", entry).group(1))
    return code, scratch


def test_products_of_few_positions_ask_for_all_before_they_wait(kernels):
    code, scratch = kernels
    names = [n for n in code if re.fullmatch(r"lng_q8_(few|one)\w*", n)]
    assert len(names) >= 6
    for name in names:
        loads = [i for i, line in enumerate(code[name]) if line.startswith("global_load_dwordx4")]
        # (the last load of a turn may stand right before the wait)
        waited = [i for i in loads if re.match(r"s_waitcnt vmcnt\(0\)", code[name][i + 1])]
        assert len(loads) >= 8 and len(waited) <= 1, "%s waits for %d of its %d loads of 16 bytes one by one" % (name, len(waited), len(loads))
        # (the preparation of attention looks its item up in a table first)
        early = [] if "prepare" in name else [line for line in code[name][:loads[7]] if re.match(r"s_waitcnt.*vmcnt", line)]
        assert not early, "%s waits for memory before it has asked for its first eight loads of 16 bytes" % name
        assert scratch[name] == 0, "%s keeps %d bytes a lane in memory" % (name, scratch[name])


def test_products_of_one_position_and_many_rows(kernels):
    """lng_q8_tall*, which ask for fewer at once and for the next tile's before the sums of one."""
    code, scratch = kernels
    names = [n for n in code if re.fullmatch(r"lng_q8_tall\w*", n)]
    assert sorted(names) == ["lng_q8_tall", "lng_q8_tall_bf16"]
    for name in names:
        loads = [i for i, line in enumerate(code[name]) if line.startswith("global_load_dwordx4")]
        waited = [i for i in loads if re.match(r"s_waitcnt vmcnt\(0\)", code[name][i + 1])]
        assert len(loads) >= 24 and len(waited) <= 1, "%s waits for %d of its %d loads of 16 bytes one by one" % (name, len(waited), len(loads))
        assert scratch[name] == 0, "%s keeps %d bytes a lane in memory" % (name, scratch[name])
