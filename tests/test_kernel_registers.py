"""Registers of M2L and P2P kernels in the built library (their code objects' metadata):
a SIMD holds 512 vector registers a lane, so a kernel's count decides its waves."""

from __future__ import annotations

import re
import struct
import subprocess

import pytest

from jaccpot_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
EM_AMDGPU = 224


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Mangled kernel name -> (vector registers, scratch bytes)."""
    lib = build.LIB.read_bytes()
    out = {}
    for at in (m.start() for m in re.finditer(b"\x7fELF", lib)):
        if struct.unpack_from("<H", lib, at + 18)[0] != EM_AMDGPU:
            continue
        obj = tmp_path_factory.mktemp("obj") / "code.o"
        end = lib.find(b"__CLANG_OFFLOAD_BUNDLE__", at)
        obj.write_bytes(lib[at:end if end > 0 else None])
        notes = subprocess.run([READELF, "--notes", obj], capture_output=True, text=True, check=True).stdout
        for block in re.split(r"\n  - \.agpr_count", notes)[1:]:
            name = re.search(r"^    \.name:\s+(\S+)", block, re.M).group(1)
            vgpr = int(re.search(r"\.vgpr_count:\s+(\d+)", block).group(1))
            scratch = int(re.search(r"\.private_segment_fixed_size:\s+(\d+)", block).group(1))
            out[name] = (vgpr, scratch)
    return out


# (type, order, most registers): the cascade of the wave-per-target kernel at three
# waves a SIMD (orders 6 and 7) and two (order 8); float64 only has to hold its state
@pytest.mark.parametrize("t,order,most", (("f", 6, 168), ("f", 7, 168), ("f", 8, 256), ("d", 6, 512), ("d", 7, 512),
                                          ("d", 8, 512)))
def test_m2l_cascade_registers(kernels, t, order, most):
    head = f"m2l_kernelI{t}Li{order}ELi{order}ELb"
    found = {n: v for n, v in kernels.items() if head in n and "ELb0EEE" in n}  # the VALU engine
    assert len(found) == 2, sorted(found)  # storing and adding
    for name, (vgpr, scratch) in found.items():
        print(name, vgpr, scratch)
        assert vgpr <= most and scratch == 0, name


# order 5 where the cascade's waves are worth more than the direct form's instructions:
# flat at seven waves a SIMD (float32) and four (float64), by target at four and two
@pytest.mark.parametrize("kernel,t,most", (("m2l_flat_kernel", "f", 72), ("m2l_flat_kernel", "d", 128),
                                           ("m2l_kernel", "f", 128), ("m2l_kernel", "d", 256)))
def test_m2l_order_5_registers(kernels, kernel, t, most):
    valu = "ELb0ELb[01]EEE" if kernel == "m2l_flat_kernel" else "ELb[01]ELb0EEE"  # (engine, weights), (adding, engine)
    found = {n: v for n, v in kernels.items() if re.search(f"{kernel}I{t}Li5ELi5{valu}", n)}
    assert len(found) == 2, sorted(found)
    for name, (vgpr, scratch) in found.items():
        print(name, vgpr, scratch)
        assert vgpr <= most and scratch == 0, name


def test_p2p_any_registers(kernels):
    """Every instance runs the five waves a SIMD that its LDS admits."""
    found = {n: v for n, v in kernels.items() if "p2p_any_kernel" in n}
    assert len(found) == 16
    for name, (vgpr, scratch) in found.items():
        assert vgpr <= 96 and scratch == 0, (name, vgpr, scratch)
