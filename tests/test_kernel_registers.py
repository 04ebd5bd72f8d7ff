"""Kernels that rely on several waves a SIMD stay within the registers that allow them, and one that is all latency requests its
operands behind a single fetch of its arguments.

From the metadata and the disassembly of the library's own gfx950 code objects; no GPU."""
import functools
import re
import subprocess

import pytest

from test_mfma_wait_states import code_objects, kernels

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
GENERIC, RELU, FUSED, LINEAR, CLAMPQ, F32, POOL = 0, 2, 3, 4, 5, 7, 8  # EPI_KIND_*
LANES = 1  # ADDR_LANES


@functools.lru_cache(None)
def resources(directory):
    """mangled name -> (vector registers, bytes of scratch a lane)"""
    found = {}
    for i, image in enumerate(code_objects()):
        path = directory / ("%d.elf" % i)
        path.write_bytes(image)
        notes = subprocess.run([READELF, "--notes", str(path)], stdout=subprocess.PIPE, check=True, text=True).stdout
        for kernel in notes.split("  - .agpr_count:")[1:]:
            value = {k: re.search(r"\.%s:\s+(\S+)" % k, kernel).group(1) for k in ("symbol", "vgpr_count", "private_segment_fixed_size")}
            found[value["symbol"]] = int(value["vgpr_count"]), int(value["private_segment_fixed_size"])
    return found


def instances(name, *parameters):
    """fragment of a mangled name: a template's integer (Li) and boolean (Lb) arguments"""
    return name + "I" + "".join("L%c%dE" % ("b" if isinstance(p, bool) else "i", p) for p in parameters) + "E"


CASES = (
    # workgroups of 512 threads, two waves a SIMD: two of them share a CU
    [("conv_ksplit_kernel", (4, 2, LANES, epi), 4) for epi in (GENERIC, RELU, FUSED, LINEAR, F32, POOL)]
    + [("conv_ksplit_kernel", (4, 2, 0, epi), 4) for epi in (RELU, FUSED, LINEAR, F32, POOL)]
    # a wave pays one trip to memory, which other waves cover
    + [("conv_stream_kernel", p + (GENERIC,), waves) for p, waves in (((1, 2), 7), ((1, 4), 6), ((1, 8), 6), ((2, 2), 5), ((2, 4), 4), ((2, 8), 4))]
    # 16 pixels x 64 features to a wave: what covers its waits is other waves
    + [("conv_bdir_kernel", (64, 1, 1, False, epi), 4) for epi in (RELU, FUSED, LINEAR, F32, POOL)]
    # the same with K split over four groups: 16 waves in 128 registers
    + [("conv_bdir_kernel", (64, 1, 4, False, epi), 4) for epi in (GENERIC, RELU, FUSED, LINEAR, F32, POOL)]
    # large planes are bound by memory
    + [("conv_dw_rows_kernel", (taps, blocks, epi), waves) for taps, blocks, waves in ((3, 2, 4), (5, 2, 4), (5, 3, 3)) for epi in (RELU, LINEAR, CLAMPQ)]
)


@pytest.mark.parametrize("name,parameters,waves", CASES, ids=lambda v: "_".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_registers_leave_the_waves_that_the_kernel_relies_on(tmp_path_factory, name, parameters, waves):
    table = resources(tmp_path_factory.getbasetemp())
    found = [v for k, v in table.items() if instances(name, *parameters) in k]
    assert len(found) == 1, "%d kernels" % len(found)
    registers, scratch = found[0]
    assert 512 // (-(-registers // 8) * 8) >= waves and scratch == 0, "%d registers, %d bytes of scratch" % (registers, scratch)


@pytest.mark.parametrize("epi", [RELU, LINEAR])
def test_depthwise_requests_wait_for_the_arguments_once(tmp_path, epi):
    wanted, found = instances("conv_dw3x3_kernel", epi), []
    for i, image in enumerate(code_objects()):
        if wanted.encode() in image:
            path = tmp_path / ("%d.elf" % i)
            path.write_bytes(image)
            found += [code for name, code in kernels(str(path)).items() if wanted in name]
    assert len(found) == 1, "%d kernels" % len(found)
    waits = 0
    for op, operands, _ in found[0]:
        if op.startswith("global_load"):
            break
        waits += op == "s_waitcnt" and "lgkmcnt" in operands
    assert waits == 1
