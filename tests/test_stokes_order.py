"""Host side of the Stokes sweeps: the chunks of csrc/rbfx_stokes_order.h. A small C++ driver checks that they take
every row once, level by level, and that their packed entries follow one another without overlap, also
past 2^31 of them."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r'''
#include <cstdio>
#include "rbfx_stokes_order.h"
int main() {
    int bad = 0;
    for (long long N : {1LL, 63LL, 1000LL, 34000000LL}) {  // 34e6 rows of 63 entries, padded to 64: 2.18e9
        const int n_lev = N > 100 ? 2 : 1;
        std::vector<int32_t> lev(N);
        for (long long r = 0; r < N; r++) lev[r] = n_lev > 1 && r % 1000 == 7;
        HostSide D;
        order_side(lev, n_lev, [](int r) { return r % 5 ? 63 : 62; }, D);
        size_t ent = 0;
        long long rows = 0;
        for (const SweepChunk& C : D.chunks) {
            bad += C.base < 0 || (size_t)C.base * SWEEP_BLK != ent || C.t0 != rows || C.nr < 1 || C.nr > SWEEP_ROWS || C.nblk != 8;
            ent += (size_t)C.nblk * SWEEP_BLK * C.nr;
            rows += C.nr;
        }
        bad += rows != N || ent != D.n_ent;
        for (long long t = 0; t < N; t++) {
            const int r = D.rows[t], c = D.chunk_of[r];
            bad += D.task[r] != t || t < D.chunks[c].t0 || t >= D.chunks[c].t0 + D.chunks[c].nr;
            bad += t > 0 && lev[D.rows[t - 1]] > lev[r];
        }
        std::printf("N %lld: %zu chunks, %zu entries, %d bad\n", N, D.chunks.size(), ent, bad);
    }
    return bad != 0;
}
'''


def test_sweep_order(tmp_path):
    src, exe = tmp_path / "order_driver.cpp", tmp_path / "order_driver"
    src.write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "rbffd_gpu_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(p.stdout)
    assert p.returncode == 0, p.stdout + p.stderr
