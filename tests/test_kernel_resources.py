"""Registers and scratch of the built kernels, from the metadata of the code
objects in libftl.so: what the class table says of them."""
import os
import re
import struct

import pytest

from barbu_amd import _ffi, build

msgpack = pytest.importorskip("msgpack")

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _kernels(elf):
    """The kernels of an AMDGPU code object: its amdhsa metadata note."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 24)
        end = off + size
        while off < end:
            nn, nd, nt = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (nn + 3) // 4 * 4
            if nt == 32 and elf[off + 12:off + 12 + nn].rstrip(b"\0") == b"AMDGPU":
                return msgpack.unpackb(elf[desc:desc + nd])["amdhsa.kernels"]
            off = desc + (nd + 3) // 4 * 4
    return []


def code_objects(path):
    """The kernels of each translation unit, in link order."""
    data = open(path, "rb").read()
    out, at = [], data.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n].decode()
            p += 24 + n
            if "amdgcn" in name and size:
                out.append(_kernels(data[at + off:at + off + size]))
        at = data.find(BUNDLE, at + 1)
    return out


@pytest.fixture(scope="module")
def units():
    if not os.path.exists(_ffi.LIB_PATH):
        pytest.skip("libftl.so is not built")
    return code_objects(_ffi.LIB_PATH)


def _classes():
    src = open(os.path.join(build.CSRC, "ftl_classes.h")).read()
    rows = re.findall(r"X\((\d+), (\d+), (\d+), (true|false), (\d+), (\d+)\)", src)
    return [(int(r[0]), int(r[4])) for r in rows]


def test_step_kernels_use_no_scratch(units):
    step = [k for u in units for k in u if re.search(r"ftl_(plain|tiles|wide)", k[".name"])]
    assert len(step) > 2 * build.NCLASSES
    assert {k[".name"]: k[".private_segment_fixed_size"] for k in step if k[".private_segment_fixed_size"]} == {}


@pytest.mark.parametrize("cls,waves", _classes())
def test_class_waves_per_simd(units, cls, waves):
    """The registers of a class's kernels leave the waves per SIMD its row
    targets, or as many as its LDS does (512 vector registers a SIMD lane, in
    blocks of eight; 160 KB of LDS for a CU's four SIMDs)."""
    kernels = units[cls]
    assert any("ftl_plain_kernel" in k[".name"] for k in kernels)
    for k in kernels:
        regs = max(8, -(-k[".vgpr_count"] // 8) * 8)  # accumulation registers counted
        groups = 160 * 1024 // max(1, k[".group_segment_fixed_size"])
        by_lds = groups * k[".max_flat_workgroup_size"] // 64 // 4
        assert 512 // regs >= min(waves, by_lds), (k[".name"], k[".vgpr_count"])


@pytest.mark.parametrize("cls", [11, 12])
def test_guarded_one_lane_classes_write_back(units, cls):
    """The guarded classes of 5 to 16 points on one lane exist with the default
    use of the caches only (FtlCache 0): partial lines merge in the L2."""
    uses = {m for k in units[cls] for m in re.findall(r"FtlCache(\d)", k[".name"])}
    assert uses == {"0"}


def test_wide_forms_built(units):
    """The wide kernels that a launch can name: (points per lane, lanes) of
    launches smaller than the chip written through only and never in a tile
    list of their own; those of launches that fill it in every use of the
    caches."""
    src = open(os.path.join(build.CSRC, "ftl_classes.h")).read()

    def forms(kind):
        rows = re.findall(r"#define FTL_%s_FORMS_\d+\(X\)(.*)" % kind, src)
        return {tuple(map(int, f)) for r in rows for f in re.findall(r"X\((\d+), (\d+)\)", r)}

    def built(kernel):
        names = [k[".name"] for u in units for k in u]
        found = [re.search(kernel + r"ILi(\d+)ELi(\d+)EL\w*FtlCache(\d)E", n) for n in names]
        return {tuple(map(int, f.groups())) for f in found if f}

    assert len(forms("LEVEL")) == 12 and len(forms("DEFAULT")) == 14
    tiles = {f + (c,) for f in forms("DEFAULT") for c in range(3)}
    assert built("ftl_wide_tiles_kernel") == tiles
    assert built("ftl_wide_kernel") == tiles | {f + (1,) for f in forms("LEVEL")}
