"""What the compiler says of the kernels in the built library, by the notes of its code objects: kernels whose registers are the limit of
what they do at a time keep nothing in scratch memory."""
import os
import re
import struct
import subprocess

import pytest

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


@pytest.fixture(scope="module")
def scratch_bytes(tmp_path_factory):
    """{demangled kernel: bytes of scratch memory a lane}"""
    from dcnv4_amd import _lib
    if not os.path.exists(READELF):
        pytest.skip("no " + READELF)
    data, path, found = open(_lib.LIB_PATH, "rb").read(), tmp_path_factory.mktemp("code") / "kernels.co", {}
    for bundle in re.finditer(BUNDLE, data):
        at = bundle.start() + len(BUNDLE)
        entries, = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(entries):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" not in target or size == 0:
                continue
            path.write_bytes(data[bundle.start() + offset:bundle.start() + offset + size])
            notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
            for kernel in notes.split(".agpr_count:")[1:]:
                name = re.search(r"\.name:\s+(\S+)", kernel).group(1)
                found[name] = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel).group(1))
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.splitlines()
    return dict(zip((re.sub(r"dcn::|\(anonymous namespace\)::", "", n) for n in names), found.values()))


# kernels by what their names hold, and how many instances there are
@pytest.mark.parametrize("kernel,instances", [(r"dcnv4_grad_value_kernel<\w+, 9, 16, 2, \d+, (true|false)>", 12),
                                              (r"linear_rows_kernel<\w+, [1-8], (true|false)>", 32), (r"mlp_kernel<\w+, [2-7], (true|false)>", 24),
                                              (r"fda_grad_value_kernel<\w+, [248], [48]>", 9), (r"sampled_linear_kernel<\w+>", 2)])
def test_kernels_without_scratch_memory(scratch_bytes, kernel, instances):
    found = {name: size for name, size in scratch_bytes.items() if re.search(kernel, name)}
    assert len(found) == instances, sorted(found)
    assert not any(found.values()), {name: size for name, size in found.items() if size}
