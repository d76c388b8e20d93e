"""The multi-instruction multiply-add blocks of csrc/common.hpp in the compiler's gfx950 output: no multiply of a
block reads a register that an earlier one of the block has written as its sum. The kernels here give the register
allocator every reason to share one: factors that are halves of a sum's start value, or zero like it. (The CPU
emulation replaces the blocks by C and cannot see this.)"""
import re
import shutil
import subprocess

import pytest

from sdpvibe_amd import build

SOURCE = """
#include "common.hpp"
#define IN(i) p[threadIdx.x + 64 * (i)]
__global__ void chain(u32* p, u64* q) {
    u32 a[4] = {IN(0), IN(1), IN(2), IN(3)}, b[4] = {IN(4), IN(5), IN(6), IN(7)};
    u64 acc = a[3] | ((u64)b[2] << 32);
    u32 ov = b[1];
    SDPV_MAC96_CHAIN4(acc, ov, a, b);
    q[threadIdx.x] = acc;
    IN(0) = ov;
}
__global__ void columns(u32* p, u64* q) {
    u32 x = IN(0), y[4] = {IN(1), IN(2), IN(3), IN(4)};
    u64 acc[4] = {y[3] | ((u64)x << 32), IN(5), IN(6), IN(7)};
    u32 ov[4] = {0, 0, 0, 0};
    SDPV_MAC96_COLS4(acc, ov, x, y);
    for (int i = 0; i < 4; i++) { q[threadIdx.x + 64 * i] = acc[i]; IN(i) = ov[i]; }
}
__global__ void zeros(u32* p, u64* q) {
    u32 x = IN(0), y[4] = {IN(1), 0, 0, 0};
    u64 acc[4] = {0, 0, 0, 0};
    u32 ov[4] = {0, 0, 0, 0};
    SDPV_MAC96_COLS4(acc, ov, x, y);
    for (int i = 0; i < 4; i++) { q[threadIdx.x + 64 * i] = acc[i]; IN(i) = ov[i]; }
}
__global__ void one(u32* p, u64* q) {
    u32 x = IN(0), y = IN(1), ov = y;
    u64 acc = x | ((u64)y << 32);
    SDPV_MAC96(acc, ov, x, y);
    q[threadIdx.x] = acc;
    IN(0) = ov;
}
"""
MAD = re.compile(r"v_mad_u64_u32 v\[(\d+):(\d+)\], s\[\d+:\d+\], v(\d+), v(\d+), v\[\d+:\d+\]")
ADD = re.compile(r"v_addc_co_u32(?:_e64)? v(\d+),")


def test_no_factor_shares_a_sums_register(tmp_path):
    if shutil.which(build.HIPCC) is None:
        pytest.skip("no hipcc")
    src, out = tmp_path / "blocks.hip", tmp_path / "blocks.s"
    src.write_text(SOURCE)
    subprocess.run([build.HIPCC, *build.FLAGS, f"-I{build.CSRC}", "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    blocks = re.findall(r";#ASMSTART\n(.*?);;#ASMEND", out.read_text(), re.S)
    blocks = [b for b in blocks if "v_mad_u64_u32" in b]
    assert len(blocks) == 4
    for block in blocks:
        written = set()
        for line in block.splitlines():
            m = MAD.search(line)
            if m:
                lo, hi, a, b = map(int, m.groups())
                assert not {a, b} & written, block
                written |= {lo, hi}
            m = ADD.search(line)
            if m:
                assert int(m.group(1)) not in written, block
