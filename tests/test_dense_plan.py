"""How the dense kernels split a gate's matrix and the state (dense.h),
checked on the CPU: a host program calls plan_dense for every width, number of
free index bits and column count, and replays which matrix rows each wave of
k_dense_rows takes: every row tile exactly once, none past the matrix, columns
within the kernels' tiles, results in place only where one workgroup holds
all rows and all of the columns."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "dense.h"
using namespace q1t;

int main()
{
    long cases = 0, rows = 0, bad = 0;
    for (size_t elem : {8, 16})
        for (int K = 4; K <= 12; ++K)
            for (int nc = 0; nc <= 3; ++nc)
                for (int n = K + nc; n <= 24; ++n)
                    for (size_t cols : {1, 2, 3, 7, 8, 16, 31, 32, 63, 64, 100, 127, 128, 255, 256, 257, 511, 512, 1000,
                                        1023, 1024, 2048, 4096, 16384, 65535}) {
                        GateOp op;
                        for (int t = 0; t < K; ++t) op.targets.push_back(t);
                        for (int c = 0; c < nc; ++c) op.ctrl_mask |= uint64_t(1) << (K + c);
                        const DensePlan p = plan_dense(op, n, cols, elem);
                        const int free_bits = n - nc - K, tiles = (1 << K) / 16;
                        bool ok = p.K == K && p.log_cols <= free_bits &&
                                  p.nblocks == uint64_t(1) << (free_bits - p.log_cols);
                        ++cases;
                        if (!p.tiles) {
                            ++rows;
                            std::vector<int> taken(size_t(tiles), 0);
                            for (uint32_t y = 0; y < p.splits; ++y)
                                for (int wave = 0; wave < 4; ++wave) {
                                    const int rt0 = (int(y) * 4 + wave) * p.rtw;
                                    if (rt0 >= tiles) continue;
                                    for (int t = 0; t < p.rtw; ++t) {
                                        if (rt0 + t >= tiles) ok = false;
                                        else taken[size_t(rt0 + t)] += 1;
                                    }
                                }
                            for (int x : taken) ok = ok && x == 1;
                            ok = ok && p.log_cols <= 3 && p.log_slice <= K && p.chunk >= 1 &&
                                 (elem << (p.log_slice + p.log_cols)) <= (size_t(64) << 10);
                            ok = ok && (p.scratch_bytes != 0) == (p.splits > 1 || p.log_slice < K);
                            if (!p.scratch_bytes) ok = ok && p.chunk == p.nblocks * cols;
                            else ok = ok && p.scratch_bytes == p.chunk * (elem << (K + p.log_cols));
                        }
                        if (!ok && ++bad <= 10)
                            std::printf("elem %zu K %d controls %d n %d columns %zu: tiles %d rtw %d splits %u slice %d\n",
                                        elem, K, nc, n, cols, int(p.tiles), p.rtw, p.splits, p.log_slice);
                    }
    std::printf("%ld cases, %ld by rows, %ld bad\n", cases, rows, bad);
    return bad || !rows || rows == cases;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="needs a host compiler")
def test_every_matrix_row_is_taken_once(tmp_path):
    from q1tsim_amd import _lib
    _lib.lib()   # built
    pkg = os.path.join(ROOT, "q1tsim_amd")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    "-I", os.path.join(pkg, "csrc"), str(src), "-L", pkg, "-l:libq1tsim.so",
                    "-Wl,-rpath," + pkg, "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
