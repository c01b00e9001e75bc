"""Every address from which the batched K-quant products load activations lies
in the rows that the batch is laid out in: the kernel's own index functions
(csrc/tile_index.hpp, compiled here for the host) walked over every thread,
piece and block of every token tile.  Scales and sums lie behind those rows,
and raw buffer loads do not check their scalar offset, so nothing else keeps a
ragged last tile inside."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include "tile_index.hpp"
int main(int argc, char **argv) {
    const int T = atoi(argv[1]), K = atoi(argv[2]);
    const int64_t end = rh::batch_rows(T) * K;
    for (int nt = 1; nt <= 2; nt++)
        for (int t0 = 0; t0 < T; t0 += 32 * nt)
            for (int tid = 0; tid < 256; tid++)
                for (int j = 0; j < 2 * nt; j++)
                    for (int b = 0; b < K / 256; b++) {
                        const int64_t lo = (int64_t)t0 * K + rh::gemm_x_lane(tid, K) + rh::gemm_x_step(j, b, K);
                        if (lo < 0 || lo + 16 > end) {
                            printf("tokens %d K %d tile of %d at %d: thread %d piece %d block %d reads %lld .. of %lld\n", T,
                                   K, 32 * nt, t0, tid, j, b, (long long)lo, (long long)end);
                            return 1;
                        }
                        const int tok = t0 + tid / 16 + 16 * j, at = 256 * b + 16 * (tid % 16);
                        if (lo != (int64_t)tok * K + at) {
                            printf("token %d element %d at %lld\n", tok, at, (long long)lo);
                            return 1;
                        }
                    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("tile")
    src = d / "walk.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "rustyllm_amd", "csrc"), "-o", d / "walk", src],
                   check=True)
    return str(d / "walk")


@pytest.mark.parametrize("tokens", [1, 2, 15, 16, 17, 31, 32, 33, 37, 48, 49, 63, 64, 65, 100, 511, 513])
@pytest.mark.parametrize("k", [256, 4096, 14336])
def test_activation_loads_stay_in_the_batch(walk, tokens, k):
    r = subprocess.run([walk, str(tokens), str(k)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
