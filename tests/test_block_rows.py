"""Tables with entries per grid block, at the block numbers where a 32-bit byte offset from their start
would wrap (2^30 int32 entries: block 2^24 of the float form's 64 cells, 2^25 of the double form's 32)."""
import os
import re
import subprocess

import numpy as np
import pytest

from ziran2020_amd import _abi as A, scenes

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


@pytest.mark.gpu
@pytest.mark.parametrize("precision,per_axis", ((A.PREC_FP32, 131), (A.PREC_FP64, 163)))
def test_lone_particles_in_blocks_past_the_wrap(gpu, monkeypatch, precision, per_axis):
    """2.2M (4.3M) particles, each alone in eight blocks of its own: the last blocks are past the wrap, and
    every particle falls as a free one does (the grid takes 130 to 160 GB)."""
    n = per_axis ** 3
    block_nodes = 64 if precision == A.PREC_FP32 else 32
    assert 8 * n * block_nodes > 2 ** 30 + 2 ** 24
    monkeypatch.setenv("ZMPM_BLOCK_CAPACITY", str(8 * n + 1000))
    dx, dt, steps, g = 1 / 64, 1e-3, 3, np.array([0.0, -9.8, 0.0])
    rng = np.random.default_rng(1)
    site = np.stack(np.meshgrid(*[np.arange(per_axis) * 12 + 24] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = (site + 1.5 + rng.uniform(0.1, 0.9, (n, 3))) * dx
    v = rng.uniform(-0.5, 0.5, (n, 3)).astype(np.float32).astype(float)
    sim = A.Simulation(gpu, dx=dx, precision=precision, domain_nodes=2048, gravity=tuple(g))
    sim.set_materials([A.make_material()])
    sim.upload(x, v, np.zeros((n, 9)), scenes.identity_F(n), np.full(n, 1e-3), np.full(n, 1e-6), np.zeros(n, np.int32))
    sim.run(steps, dt)
    out = sim.download()
    sim.close()
    assert np.abs(out["v"] - (v + steps * dt * g)).max() < 1e-5
    fall = dt * (steps * v + steps * (steps + 1) / 2 * dt * g)
    assert np.abs(out["x"] - (x + fall)).max() < 1e-4 * dx
