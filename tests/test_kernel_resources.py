"""Registers of the built kernels, from the metadata notes of the library's gfx950 code objects: the launches are sized to
the waves per SIMD that a kernel's registers leave (512 VGPRs a lane, in blocks of 8), which no output shows."""
import os
import struct
import subprocess

import pytest

msgpack = pytest.importorskip("msgpack")


@pytest.fixture(scope="module")
def kernels():
    """{kernel name without arguments: metadata} of every kernel in libgfl_moe.so."""
    import _native
    if not os.path.exists(_native.LIB_PATH):
        pytest.skip("library not built")
    data = open(_native.LIB_PATH, "rb").read()
    found, at = [], data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            off, size, name = struct.unpack_from("<QQQ", data, entry)
            target, entry = data[entry + 24:entry + 24 + name], entry + 24 + name
            if target.endswith(b"gfx950"):
                found += _elf_kernels(data[at + off:at + off + size])
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 1)
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in found), capture_output=True, text=True,
                           check=True).stdout.split("\n")
    return {n.split("(")[0].replace("void ", "").replace("gfl::", ""): k for n, k in zip(names, found)}


def _elf_kernels(elf):
    shoff = struct.unpack_from("<Q", elf, 40)[0]
    entry, count = struct.unpack_from("<HH", elf, 58)
    for k in range(count):
        kind = struct.unpack_from("<I", elf, shoff + k * entry + 4)[0]
        at = struct.unpack_from("<Q", elf, shoff + k * entry + 24)[0]
        if kind == 7:   # SHT_NOTE
            name, size = struct.unpack_from("<II", elf, at)
            at += 12 + (name + 3) // 4 * 4
            return msgpack.unpackb(elf[at:at + size])["amdhsa.kernels"]
    return []


def _waves(k):
    return min(8, 512 // ((k[".vgpr_count"] + k[".agpr_count"] + 7) // 8 * 8))


@pytest.mark.parametrize("K", [2, 3, 4, 5])
def test_one_wave_relay_launches_fit_their_waves(kernels, K):
    """At M = 4 gate|up puts 6 waves on a SIMD: with 5 resident the sixth runs alone, and the call is slower than with 4."""
    for name in ("gu_relay_kernel", "dn_relay_kernel"):
        k = kernels["%s<%d, 1>" % (name, K)]
        assert _waves(k) >= (5 if K == 5 else 6) and k[".vgpr_spill_count"] == 0, (name, k[".vgpr_count"])


@pytest.mark.parametrize("K", [2, 3, 4, 5])
@pytest.mark.parametrize("slots,waves", [(16, 8), (32, 6), (64, 4)])
def test_chain_gemm_fits_without_spills(kernels, K, slots, waves):
    """The chain GEMM's loops are bound by issue: a register spilled is a scratch reload in every tile row."""
    k = kernels["xg_gemm_kernel<%d, %d>" % (K, slots)]
    assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0 and _waves(k) >= waves
