"""Machine code of the buffer-store row writer: the instruction after a 16-byte store must not write the registers the
store takes its data from.  The compiler keeps that distance only for stores without a scalar offset register."""
import os
import re
import subprocess

import pytest

from teletron_amd import build as B

SOURCE = """
#include "norm_device.h"
using namespace ttn;
// twelve pieces, each formed from the one before it, hence in its registers
__global__ void rows(float *out, const float *x, const float *w) {
    const int l = threadIdx.x & 63;
    u32x4 piece = load16(reinterpret_cast<const u32x4 *>(x) + l);
    const u32x4 add = load16(reinterpret_cast<const u32x4 *>(w) + l);
    const RowWriter<WRITER> o(out, l * 16);
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        o.put(k * 64, piece);
#pragma unroll
        for (int j = 0; j < 4; ++j) piece[j] = as_u32(as_f32(piece[j]) * as_f32(add[j]));
    }
}
"""


def _registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"v(\d+)$", operand)
    return {int(m[1])} if m else set()


@pytest.mark.parametrize("writer", [1])
def test_store_data_is_not_overwritten_by_the_next_instruction(tmp_path, writer):
    (tmp_path / "rows.hip").write_text(SOURCE)
    asm = tmp_path / "rows.s"
    subprocess.run([B.HIPCC, *B.HIP_FLAGS, "-w", f"-DWRITER={writer}", "-I" + B.CSRC, "--cuda-device-only", "-S",
                    str(tmp_path / "rows.hip"), "-o", str(asm)], check=True, capture_output=True)
    lines = [t for t in (l.split(";")[0].strip() for l in asm.read_text().splitlines()) if t and not t.startswith(".")]
    stores = 0
    for this, after in zip(lines, lines[1:]):
        op, _, args = this.partition("\t") if "\t" in this else this.partition(" ")
        if op != "buffer_store_dwordx4":
            continue
        stores += 1
        data = _registers(args.split(",")[0].strip())
        next_op, _, next_args = after.partition("\t") if "\t" in after else after.partition(" ")
        if next_op.startswith("v_"):
            assert not data & _registers(next_args.split(",")[0].strip()), (this, after)
    assert stores == 12
