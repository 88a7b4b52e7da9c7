"""Registers of the kernels in the built library, from the metadata the compiler leaves in it: what decides how many wavefronts share a compute
unit, and whether a loop keeps its values in registers."""
import re
import struct
import subprocess

import pytest

import vdnn_implementation_amd.backend as be

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def code_objects(blob):
    """The gfx950 code objects of the bundles in the library (one bundle per source file)."""
    at = blob.find(MAGIC)
    while at >= 0:
        count, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(count):
            offset, size, name_size = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + name_size].decode()
            p += 24 + name_size
            if "gfx950" in name and size:
                yield blob[at + offset:at + offset + size]
        at = blob.find(MAGIC, at + 1)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{demangled name: {vgpr, agpr, spill}}"""
    found = {}
    for i, elf in enumerate(code_objects(open(be.LIB_PATH, "rb").read())):
        path = tmp_path_factory.mktemp("objects") / ("%d.co" % i)
        path.write_bytes(elf)
        notes = subprocess.run([READELF, "--notes", str(path)], capture_output=True, text=True, check=True).stdout
        for part in re.split(r"\n\s+- \.agpr_count:", notes)[1:]:
            number = lambda key: int(re.search(r"\.%s:\s+(\d+)" % key, part).group(1))
            found[re.search(r"\n\s+\.name:\s+(\S+)", part).group(1)] = {"agpr": int(part.split()[0]), "vgpr": number("vgpr_count"), "spill": number("vgpr_spill_count")}
    names = subprocess.run(["c++filt"], input="\n".join(found), capture_output=True, text=True, check=True).stdout.split("\n")
    return dict(zip((n.split("(")[0].replace("vdnn::", "").replace("void ", "") for n in names), found.values()))


def test_tile_engine_keeps_its_loop_in_registers(kernels):
    """The float tile engine's kernels spill nothing: what they spill they spill once a slice."""
    engine = {n: k for n, k in kernels.items() if re.match(r"igemm(64)?_kernel<|igemm_classes_kernel<", n)}
    assert len(engine) > 50
    assert not {n: k for n, k in engine.items() if k["spill"]}


def test_products_that_add_up_no_splits_leave_room_for_six_wavefronts(kernels):
    """A SIMD has 512 registers a lane: the convolutions' instances of the 64x64 tile with one slice ahead and no split sums are for grids that
    fill the chip."""
    lean = {n: k for n, k in kernels.items() if re.match(r"igemm64_kernel<.*Im2col.*, 1, false>|igemm_classes_kernel<.*, 1>", n) and "StoreFilterTap" not in n}
    assert len(lean) > 20
    assert not {n: k for n, k in lean.items() if k["vgpr"] > 512 // 6 // 8 * 8}
