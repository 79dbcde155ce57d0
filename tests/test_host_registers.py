"""Registers of kernels whose waves wait for weights, from the metadata of the built library: how many
workgroups a CU holds."""
import os
import re
import struct

import msgpack
import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def registers():
    """Kernel name -> vector registers of a lane, in the steps of eight that the hardware allots."""
    path = os.path.join(ROOT, "ponyexl3_amd", "libexl3_hip.so")
    if not os.path.exists(path):
        from ponyexl3_amd import build

        build.build()
    data, out = open(path, "rb").read(), {}
    for m in re.finditer(rb"AMDGPU\0\0", data):  # ELF notes: name size, description size, type, name, description
        if m.start() < 12:
            continue
        namesz, descsz, kind = struct.unpack_from("<III", data, m.start() - 12)
        if namesz == 7 and kind == 32 and m.end() + descsz <= len(data):
            for k in msgpack.unpackb(data[m.end():m.end() + descsz])["amdhsa.kernels"]:
                out[k[".name"]] = (k[".vgpr_count"] + 7) // 8 * 8
    return out


def _workgroups_of_eight(registers, kernel, *args):
    pattern = re.compile(kernel + "I" + "".join(f"L[ib]{a}E" for a in args) + "E")
    found = [v for n, v in registers.items() if pattern.search(n)]
    assert len(found) == 1, (kernel, args, found)
    return 512 // found[0] // 2  # two of a workgroup's waves on each SIMD


@pytest.mark.parametrize("half", [0, 1])
@pytest.mark.parametrize("cb", [0, 1])
@pytest.mark.parametrize("k", range(1, 9))
def test_moe_gate_up_workgroups_of_a_cu(registers, k, cb, half):
    """Scales and choices that are held over the weights had cost a workgroup of three or four: blocks of a few
    tokens took 2 to 6 % longer at K = 6 and 7."""
    least = {0: (4, 4, 3, 3, 3, 3, 3, 2), 1: (4, 4, 4, 4, 3, 3, 3, 3)}[cb][k - 1]
    if cb == 1 and half:
        least = 4 if k <= 7 else 3
    assert _workgroups_of_eight(registers, "moe_gateup_pair_kernel", k, cb, half) >= least


@pytest.mark.parametrize("k", range(1, 9))
def test_moe_grouped_down_workgroups_of_a_cu(registers, k):
    """20 tokens of 9 slots, 65 experts of 2048 x 512 at K = 8: 71.4 us with four workgroups to a CU, 73.2 with three."""
    assert _workgroups_of_eight(registers, "moe_down_grouped_kernel", k, 0, 8, 0) >= 4


@pytest.mark.parametrize("cb", [0, 1, 2])
@pytest.mark.parametrize("k", range(1, 9))
def test_rows_kernel_workgroups_of_a_cu(registers, k, cb):
    """Up to 32 rows: three, which is what their LDS allows up to K = 4."""
    assert _workgroups_of_eight(registers, "linear_rows_kernel", k, cb, 1, 4) >= 3
