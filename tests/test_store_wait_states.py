"""Machine code of the 16-byte buffer-store writers: the registers a store takes its data from must not be written within
two wait states of it.  The compiler keeps that distance only for stores without a scalar offset register."""
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
    const WRITER;
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        o.put(k * 64, piece);
#pragma unroll
        for (int j = 0; j < 4; ++j) piece[j] = as_u32(as_f32(piece[j]) * as_f32(add[j]));
    }
}
"""
WAIT_STATES = 2


def _registers(operand):
    m = re.match(r"v\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"v(\d+)$", operand)
    return {int(m[1])} if m else set()


def _split(line):
    op, _, args = line.replace("\t", " ").partition(" ")
    return op, [a.strip() for a in args.split(",")]


def overwritten(lines):
    """(number of 16-byte buffer stores, those whose data an instruction within the wait states overwrites)."""
    stores, bad = 0, []
    for i, line in enumerate(lines):
        op, args = _split(line)
        if op != "buffer_store_dwordx4":
            continue
        stores += 1
        data, passed = _registers(args[0]), 0
        for after in lines[i + 1:]:
            if passed >= WAIT_STATES or after.endswith(":"):
                break
            next_op, next_args = _split(after)
            if next_op.startswith("v_") and data & _registers(next_args[0]):
                bad.append((line, after))
            passed += int(next_args[0]) + 1 if next_op == "s_nop" else 1
    return stores, bad


def _assembly(tmp_path, writer):
    (tmp_path / "rows.hip").write_text(SOURCE.replace("WRITER", writer))
    asm = tmp_path / "rows.s"
    subprocess.run([B.HIPCC, *B.HIP_FLAGS, "-w", "-I" + B.CSRC, "--cuda-device-only", "-S",
                    str(tmp_path / "rows.hip"), "-o", str(asm)], check=True, capture_output=True)
    lines = (l.split(";")[0].strip() for l in asm.read_text().splitlines())
    return [t for t in lines if t and not t.startswith(".")]


@pytest.mark.parametrize("writer", ["RowWriter<1> o(out, l * 16)", "BoundedRow<18> o(out, 12 * 1024, l)",
                                    "BoundedRow<2> o(out, 12 * 1024, l)"])
def test_store_data_is_not_overwritten_within_the_wait_states(tmp_path, writer):
    stores, bad = overwritten(_assembly(tmp_path, writer))
    assert stores == 12 and not bad


@pytest.mark.parametrize("between,clean", [([], False), (["s_nop 0"], False), (["s_nop 1"], True), (["v_mov_b32 v9, v8"], False),
                                           (["s_waitcnt vmcnt(0)", "s_nop 0"], True)])
def test_the_check_sees_an_early_overwrite(between, clean):
    lines = ["buffer_store_dwordx4 v[0:3], v4, s[0:3], 0 offen"] + between + ["v_mul_f32 v2, v2, v6", "s_endpgm"]
    assert overwritten(lines) == (1, [] if clean else [(lines[0], "v_mul_f32 v2, v2, v6")])
