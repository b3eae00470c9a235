"""Decoded weights on their way to the matrix unit, in the assembly that hipcc makes of the decode.

Between a vector instruction that writes a register and a matrix instruction that reads it as an operand there are at least two other
instructions or an s_nop of that length: the compiler sees to that for its own instructions, not for ones written in an asm statement.
"""
import re
import subprocess

import pytest

from htr_amd import build

KERNEL = """
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "../../include/htr_gfx950.h"
#include "decode.hpp"
template <int K> __global__ void k(const uint32_t* p, const h8* x, f4* y) {
  StreamRegs<K> r;
  for (int i = 0; i < K; ++i) r.d[i] = p[threadIdx.x * K + i];
  Window<K> win;
  win.build(r, p[threadIdx.x]);
  const h8 b = x[threadIdx.x];
  f4 acc = y[threadIdx.x];
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.template group8<0>(), b, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(win.template group8<24>(), b, acc, 0, 0, 0);
  y[threadIdx.x] = acc;
}
#define I(K) template __global__ void k<K>(const uint32_t*, const h8*, f4*);
I(2) I(3) I(4) I(5) I(6) I(7) I(8)
"""


def _registers(operand):
    """Numbers of the vector registers that an operand names."""
    m = re.match(r"v\[(\d+):(\d+)\]$|v(\d+)$", operand.strip())
    if not m:
        return range(0)
    return range(int(m[1]), int(m[2]) + 1) if m[1] else range(int(m[3]), int(m[3]) + 1)


def _shortest_waits(assembly):
    """Matrix instructions, and for each the fewest wait states since one of its A or B registers was written by a vector instruction."""
    written, now, found = {}, 0, []
    for line in assembly.splitlines():
        code = line.split(";")[0].strip()
        if not code or code.startswith((".", "#")) or code.endswith(":"):
            continue
        op, _, rest = code.partition(" ")
        args = rest.split(",")
        if op.startswith("v_mfma"):
            waits = [now - written[r] - 1 for a in args[1:3] for r in _registers(a) if r in written]
            found.append((code, min(waits, default=99)))
            for r in _registers(args[0]):
                written.pop(r, None)
        elif op.startswith("v_"):
            for r in _registers(args[0]):
                written[r] = now
        now += int(args[0]) + 1 if op == "s_nop" else 1
    return found


def test_matrix_instructions_wait_for_decoded_weights(tmp_path):
    source, out = tmp_path / "decode.hip", tmp_path / "decode.s"
    source.write_text(KERNEL)
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-Wall")]
    done = subprocess.run([build.hipcc(), *flags, "-w", "-S", "--cuda-device-only", "-I", build.CSRC, str(source), "-o", str(out)], capture_output=True, text=True)
    assert done.returncode == 0, done.stderr[-2000:]
    found = _shortest_waits(out.read_text())
    assert len(found) == 14                                           # two for every K
    assert all(wait >= 2 for _, wait in found), [f for f in found if f[1] < 2]


@pytest.mark.parametrize("between,wait", [("", 0), ("\ts_nop 0\n", 1), ("\ts_nop 1\n", 2), ("\tv_mov_b32_e32 v40, 0\n\ts_nop 0\n", 2)])
def test_wait_states_as_counted(between, wait):
    text = "\tv_sad_hi_u8 v3, v9, 0, v3\n" + between + "\tv_mfma_f32_16x16x32_f16 v[20:23], v[0:3], v[4:7], v[20:23]\n"
    assert _shortest_waits(text)[0][1] == wait
