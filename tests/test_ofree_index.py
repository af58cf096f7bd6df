"""Where k_sx_ofree reads, on the CPU (rbm-nqs_amd/csrc/ofree_index.hpp as the
kernel compiles it): for every machine that of_ok admits, every lane and every
pair,

  * a place read of a staged row is a tanh value or the 1 behind them, so inside
    the row and the block's LDS, and written before it is read;
  * for the machine's own parameters it is the right unit with the right spins."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <initializer_list>
#include "ofree_index.hpp"
using namespace rbmgpu;
int main() {
    long machines = 0, bad = 0;
    for (int rsize = 4; rsize <= 8; rsize += 4)
        for (int N = 2; N <= 64; N += 2)
            for (int M = 2; M <= 128; M += 2)
                for (int npf = 0; npf <= 4 * N * N; npf += npf ? 4 * N : 4) {
                    const int P_rbm = N + M + N * M, P = P_rbm + npf, ld = P + (P & 1);
                    if (ld > 128 * 24) break;
                    // the instance that launch_sx takes
                    int zm = 24, waves = ld <= 128 * 4 ? 16 : 4;
                    for (int z : {18, 12, 8, 4, 2})
                        if (ld <= 128 * z) zm = z;
                    if (!of_ok(rsize, N, M, ld, npf, waves)) continue;
                    machines++;
                    const int rows = of_rows(rsize, waves, 128 * zm), pw = npf ? P_rbm : ld;
                    const long xs = of_xs(ld, npf), lds = of_lds(rsize, ld, M, npf, waves) / (2 * rsize);
                    bool ok = rows == of_rows(rsize, waves, ld);
                    auto read = [&](int place) {  // of the last wave's last row
                        const long at = xs + ((long)(waves - 1) * rows + rows - 1) * (M + 1) + place;
                        ok = ok && place >= 0 && place <= M && at < lds;
                    };
                    for (int lane = 0; lane < 64; lane++) {
                        const OfLane o = of_lane(lane, N, M);
                        int u = o.u1, j = o.j1;
                        for (int i = 0; i < zm; i++) {
                            if (i > 1) of_next(u, j, 128 / N, 128 % N, N, M);
                            if (128 * i >= pw) break;
                            ok = ok && 2 * lane + 128 * i + 1 < xs;
                            for (int e = 0; e < 2; e++) {
                                const int place = i ? u : e ? o.e1 : o.e0, spin = (i ? j : o.ej) + e;
                                read(place);
                                ok = ok && spin >= 0 && spin < 64;
                                const int p = 2 * lane + 128 * i + e;
                                if (p >= P_rbm) continue;
                                const bool vis = p < N, bias = !vis && p < N + M;
                                const int q = p - N - M;
                                ok = ok && place == (vis ? M : bias ? p - N : q / N);
                                ok = ok && (bias ? spin >= N : spin == (vis ? p : q % N));
                            }
                        }
                    }
                    if (!ok && bad++ < 8) printf("N=%d M=%d npf=%d real=%d\n", N, M, npf, rsize);
                }
    printf("%ld machines, %ld bad\n", machines, bad);
    return machines == 0 || bad != 0;
}
"""


def test_ofree_reads_in_range(tmp_path):
    src, exe = tmp_path / "ofree.cpp", tmp_path / "ofree"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "rbm-nqs_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
