"""What the compiled kernels take of a lane's registers and scratch memory, from the metadata of the built library's code."""
import os
import re
import shutil
import subprocess

import pytest

from trips_amd import build

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled name: {key: value}} of every kernel of the library."""
    if not shutil.which(f"{LLVM}/llvm-objdump"):
        pytest.skip("needs LLVM's tools")
    if not os.path.exists(build.LIB):
        build.build()
    at = tmp_path_factory.mktemp("code")
    shutil.copy(build.LIB, at / "lib.so")
    subprocess.check_call([f"{LLVM}/llvm-objdump", "--offloading", "lib.so"], cwd=at, stdout=subprocess.DEVNULL)
    found = {}
    for part in sorted(at.glob("lib.so.*gfx950")):
        notes = subprocess.run([f"{LLVM}/llvm-readelf", "--notes", str(part)], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            name = re.search(r"^ {4}\.name: +(\S+)$", kernel, re.M).group(1)
            found[name] = {k: int(v) for k, v in re.findall(r"^ {4}\.(\w+): +(\d+)$", kernel, re.M)}
    names = subprocess.run(["c++filt"], input="\n".join(found), check=True, capture_output=True, text=True).stdout.split("\n")
    return dict(zip(names, found.values()))


def test_weight_gradient_without_scratch_where_it_has_a_cu_to_itself(kernels):
    """The weight gradient of 32 inputs x 64 pre-activations does not fit the 128 registers that two workgroups on a CU leave a
    lane: per kind of image and with and without bias gradients there is an instance that is not held to them, for launches of one
    workgroup a CU, and none that spills more than the 22 registers with which two were still the faster."""
    kinds = {}
    for name, info in kernels.items():
        m = re.search(r"conv_bwd_weight_kernel<32, 64, (true|false), (\d+), (true|false)", name)
        if m:
            kinds.setdefault(m.groups(), []).append(info)
    assert sorted((int(c), f) for _, c, f in kinds) == sorted([(4, "true"), (4, "false"), (8, "false"), (16, "false")] * 2)
    for kind, instances in kinds.items():
        assert min(i["private_segment_fixed_size"] for i in instances) == 0, kind
        assert max(i["vgpr_spill_count"] for i in instances) <= 22, kind
