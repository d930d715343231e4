"""Tables with entries per grid block, at the block numbers where a 32-bit byte offset from their start
would wrap (2^30 int32 entries: block 2^24 of the float form's 64 cells, 2^25 of the double form's 32)."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ziran2020_amd", "csrc")

PROGRAM = """
#include "zmpm_kernels.hpp"
#include <cstdio>
int main()
{
    // addresses only: the table is never read
    int* const table = reinterpret_cast<int*>(uintptr_t(1) << 40);
    const long long blocks[] = { 0, 1, (1 << 24) - 1, 1 << 24, (1 << 25) - 1, 1 << 25, (1 << 26) - 2 };
    for (long long b : blocks) {
        const char* const at[] = { (char*)zmpm::blockRow<64>(table, (int)b), (char*)zmpm::blockRow<32>(table, (int)b),
                                   (char*)zmpm::blockRow<8>(table, (int)b) };
        const int row[] = { 64, 32, 8 };
        for (int k = 0; k < 3; k++)
            if (at[k] - (char*)table != 4 * b * row[k]) return std::printf("block %lld, row of %d\\n", b, row[k]), 1;
    }
}
"""


def test_row_addresses(tmp_path):
    src, exe = tmp_path / "rows.hip", tmp_path / "rows"
    src.write_text(PROGRAM)
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "-x", "hip", "--offload-host-only", "-std=c++17", "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


@pytest.mark.parametrize("table", ("cell_start", "cell_count"))
def test_32_bit_accesses_start_at_a_row(table):
    """ldAt and stAt form a byte offset of 32 bits from their base: a table per cell goes through its block's row."""
    text = open(os.path.join(CSRC, "zmpm_device.hpp")).read()
    assert not re.findall(r"\b(?:ldAt|stAt)\(D\.%s\b[^;]*;" % table, text)
    assert re.search(r"\bldAt\(blockRow<\w+>\(D\.%s, \w+\)" % table, text)
