"""What the grouped GEMM's hand-written copies rely on, read from its assembly (no GPU).

M0 holds the copies' LDS address.  It is a reserved register, which an asm statement cannot declare as
clobbered, so the compiler itself must have no use for it in these kernels.

The first stage of a block ends in a wait that leaves the block's last four 16-byte weight copies in
flight.  Only 16-byte LDS copies are relied on to complete in order, so between the barrier before
and this wait nothing that the next stage reads may come by a 4-byte copy: the only ones allowed
are Q4_K's two pieces of the next block's weights, which a later wait for all covers."""
import re
import subprocess

import pytest

from mnemocuda_amd import build as mbuild


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    out = tmp_path_factory.mktemp("asm") / "gemm_grouped.s"
    subprocess.run([str(mbuild.ROCM / "bin" / "hipcc"), *mbuild.HIPCC_FLAGS, "-S", "--offload-device-only",
                    str(mbuild.CSRC / "gemm_grouped.hip"), "-o", str(out)], check=True, capture_output=True)
    return out.read_text().splitlines()


def counted_waits(lines, type_id):
    """For each counted wait of the kernels of a type: the LDS copies and register loads since the
    last barrier, in the order of the text."""
    kernel, ops, asm = "", [], False
    for line in lines:
        m = re.match(r"(_Z\w*gemm_grouped_kernel\w*):", line)
        if m:
            kernel, ops = m.group(1), []
        if f"ILi{type_id}E" not in kernel:
            continue
        asm = (asm or "ASMSTART" in line) and "ASMEND" not in line
        m = re.match(r"\s+((?:global|buffer|flat|scratch)_\w+)", line)
        if m:
            ops.append(m.group(1))
        elif asm and re.search(r"s_waitcnt vmcnt\([1-9]", line):
            yield list(ops), int(re.search(r"vmcnt\((\d+)\)", line).group(1))
        if "s_barrier" in line:
            ops = []


@pytest.mark.parametrize("type_id,weights4,kernels", [(12, 2, 2), (14, 0, 1)])
def test_counted_wait_covers_16_byte_copies_only(assembly, type_id, weights4, kernels):
    waits = list(counted_waits(assembly, type_id))
    assert len(waits) >= 6 * kernels  # one per count of token columns (the compiler may split a path)
    for ops, left in waits:
        copies = [o for o in ops if o.startswith("global_load_lds")]
        assert copies[-left:] == ["global_load_lds_dwordx4"] * left, ops
        assert copies[:-left].count("global_load_lds_dword") == weights4, ops
        assert "global_load_lds_dwordx4" in copies[:-left], ops


def test_compiler_leaves_m0_alone(assembly):
    asm, own = False, 0
    for line in assembly:
        asm = (asm or "ASMSTART" in line) and "ASMEND" not in line
        if re.search(r"\bm0\b", line.split(";")[0]):
            assert asm, line
            own += 1
    assert own
