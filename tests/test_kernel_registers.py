"""Scratch memory (register spills) and waves per SIMD of the built kernels, from the metadata that the compiler wrote into the
library: the staged, row, patch and binning kernels run from registers, apart from the forms named here, whose state is two query
rows or rows of 256 elements in 128 registers (16 waves a workgroup)."""
import os
import re
import subprocess

import pytest

from ops import _native

READELF = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-readelf")
# bytes a lane; fwd_slot_kernel<storage, D, elements a lane, row blocks>
SPILLED = {"fwd_slot_kernel<BF16, 64, 8, 2>": 80, "fwd_slot_kernel<BF16, 256, 16, 1>": 8, "fwd_slot_kernel<F32, 256, 16, 1>": 52,
           "fwd_slot_kernel<F32, 64, 8, 1>": 8}
# the coordinate gradient in bf16: outside the loop of the samples, and 3 % faster than with the taps held apart for fewer registers
SPILLED.update({f"bwd_dq_slot_kernel<BF16, {d}, 8, true, 1, false>": 20 for d in (16, 32, 64, 128)})


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    if not (os.path.exists(_native.LIB_PATH) and os.path.exists(READELF)):
        pytest.skip("no built library, or no llvm-readelf")
    blob, out = open(_native.LIB_PATH, "rb").read(), {}
    for m in re.finditer(rb"\x7fELF\x02\x01\x01\x40", blob):           # (64: the AMD GPU ABI)
        part = tmp_path_factory.mktemp("co") / "code.o"
        part.write_bytes(blob[m.start():])
        notes = subprocess.run([READELF, "--notes", str(part)], capture_output=True, text=True).stdout
        for entry in notes.split("- .agpr_count:")[1:]:
            field = lambda name: re.search(r"\." + name + r":\s+(\S+)", entry).group(1)
            out[field("name")] = (int(field("private_segment_fixed_size")), int(field("vgpr_count")))
    names = subprocess.run(["c++filt"], input="\n".join(out), capture_output=True, text=True).stdout.splitlines()
    short = lambda n: re.sub(r"\(.*", "", n.replace("dsdpa::", "").replace("void ", "")).strip()
    return {short(n): v for n, v in zip(names, out.values())}


def test_main_kernels_do_not_spill(kernels):
    ours = {n: v for n, v in kernels.items() if re.match(r"(fwd_slot|bwd_dq_slot|fwd_rows|bwd_dq_rows|bwd_dkdv_patch|bin_)", n)}
    assert len(ours) > 100
    over = {n: v[0] for n, v in ours.items() if v[0] > SPILLED.get(n, 0)}
    assert not over, over


def test_row_dq_keeps_the_waves_that_its_rules_count_on(kernels):
    """bwd_dq_rows_kernel<storage, D, elements a lane, coordinate gradient, samples a step, bins>: registers for six waves a SIMD
    (80 of 512) in fp32 with one sample a step, for five (96) with the coordinate gradient, in fp16 where it does not bin."""
    name = r"bwd_dq_rows_kernel<(\w+), (\d+), \d+, (true|false), (\d), (true|false)>"
    over, seen = {}, 0
    for n, (_, regs) in kernels.items():
        m = re.match(name, n)
        if not m:
            continue
        storage, D, coords, step, bins = m[1], int(m[2]), m[3] == "true", int(m[4]), m[5] == "true"
        most = 128
        if storage == "F32" and not coords and step == 1 and (D <= 128 or not bins):
            most = 80
        elif coords and not bins and ((storage == "F32" and D <= 128) or (storage == "F16" and D >= 32)):
            most = 96
        seen += most < 128
        if regs > most:
            over[n] = regs
    assert not over and seen == 4 + 5 + 4 + 4, (seen, over)


def test_row_kernels_keep_four_waves_a_simd(kernels):
    over = {n: v[1] for n, v in kernels.items() if re.match(r"(fwd_rows|bwd_dq_rows)", n) and v[1] > 128}
    assert not over, over
