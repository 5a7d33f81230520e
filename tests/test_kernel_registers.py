"""What the compiled kernels need, as their code objects in libmsd_hip.so state it: registers for the wavefronts per SIMD that
the launch rules count on, no registers in memory beyond one known instance, no instance that no dispatch reaches."""
import os
import re
import shutil
import struct
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(REPO, "mobile-stable-diffusion_amd", "csrc", "libmsd_hip.so")
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, pos - 8)[0]):
            offset, size, name_size = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + name_size]
            pos += 24 + name_size
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not os.path.exists(LIB) or not os.path.exists(READELF) or shutil.which("c++filt") is None:
        pytest.skip("no built library, or no tools to read it")
    with open(LIB, "rb") as f:
        objects = list(_code_objects(f.read()))
    found = []
    for i, obj in enumerate(objects):
        path = tmp_path_factory.mktemp("co") / ("%d.o" % i)
        path.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for part in re.split(r"\n  - ", notes):
            name = re.search(r"\.name:\s+(_Z\S+)", part)
            if name:
                found.append((name.group(1), int(re.search(r"\.vgpr_count:\s+(\d+)", part).group(1)),
                              int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", part).group(1))))
    names = subprocess.run(["c++filt"], input="\n".join(n for n, _, _ in found), capture_output=True, text=True, check=True)
    plain = [re.sub(r"\(.*", "", n.split("(anonymous namespace)::", 1)[-1]) for n in names.stdout.splitlines()]
    return {n: found[i][1:] for i, n in enumerate(plain)}


def test_short_groupnorm_slices_leave_room_for_eight_wavefronts_per_simd(kernels):
    seen = 0
    for name, (registers, _) in kernels.items():
        m = re.match(r"gn_slice_kernel<(float|__half), (\d+), ", name)
        if m and int(m.group(2)) <= (6 if m.group(1) == "__half" else 5):
            assert registers <= 64, name
            seen += 1
    assert seen == 8 * (6 + 5) + 2 * 5  # (float slices exist in two orders of requests)


def test_no_kernel_keeps_registers_in_memory(kernels):
    known = {"gn_tokens_kernel<__half, 16>": 64}  # (the longest slices of the token norm)
    for name, (_, private) in kernels.items():
        assert private <= known.get(name, 0), name


def test_token_norms_of_float_end_at_ten_vectors_per_lane(kernels):
    assert any(n.startswith("gn_tokens_kernel<float, 10") for n in kernels)
    for name in kernels:
        m = re.match(r"gn_tokens(?:_unit)?_kernel<float, (\d+)", name)
        assert m is None or int(m.group(1)) <= 10, name
