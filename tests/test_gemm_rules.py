"""The rules that choose a product's kernel (csrc/gemm_rules.hpp), compiled for
the host, against products timed with both kernels."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "linear-massiv_amd", "csrc")

PROGRAM = r"""
#include "gemm_rules.hpp"
#include <cstdio>
#include <cstring>
using namespace lmx;
int main() {
    char rule[16];
    int bytes, ta, tb, nn, tile;
    long m, n, k;
    while (scanf("%15s %d %d %d %d %d %ld %ld %ld", rule, &bytes, &ta, &tb, &nn, &tile, &m, &n, &k) == 9)
        printf("%d\n", !strcmp(rule, "bf16")    ? bf16_large_tile(ta, tb, m, n, k) > 0
                       : !strcmp(rule, "split") ? (int)ksplit_is_faster(bytes, ksplit_tile(m, n, false, 1), nn, tb, k)
                                              : (int)direct_is_faster(ta, tb, nn, tile, m, n, k));
}
"""

# type, transposes, row padding, m, n, k, us on 64 x 64 tiles, us split
SPLIT = [
    ("d", "NN", 1, 960, 960, 64, 8.4, 12.5), ("s", "NN", 0, 16000, 64, 48, 5.0, 6.0),
    ("s", "NT", 0, 960, 960, 48, 4.9, 5.9), ("d", "NN", 0, 16000, 64, 48, 6.8, 11.7),
    ("d", "TT", 1, 16000, 64, 48, 7.4, 11.8), ("d", "NN", 0, 1648, 296, 100, 10.0, 11.9),
    ("d", "TT", 0, 108, 7768, 60, 8.5, 11.8), ("d", "NN", 0, 13536, 52, 64, 7.4, 12.3),
    ("d", "NT", 0, 960, 960, 64, 7.7, 14.2), ("s", "NN", 0, 1000, 700, 100, 6.7, 8.7),
    ("s", "NT", 0, 5624, 4, 104, 5.9, 3.7), ("d", "TT", 1, 16, 16000, 256, 20.2, 10.0),
    ("s", "TT", 1, 12211, 1, 366, 19.0, 8.8), ("s", "NN", 1, 16000, 16, 1024, 47.0, 18.4),
    ("s", "NT", 0, 10424, 48, 3016, 90.0, 59.8), ("d", "TN", 1, 16, 16, 8192, 529.5, 30.4),
    ("d", "NT", 1, 3490, 22, 52, 7.2, 3.5), ("d", "NN", 0, 500, 500, 500, 32.1, 10.0),
]
# the same, us on the tiles through LDS, us on the kernel without
DIRECT = [
    ("d", "TN", 1, 6000, 320, 3000, 299.6, 362.1), ("d", "NN", 0, 17713, 6, 242, 24.7, 38.1),
    ("d", "TN", 0, 40000, 64, 256, 39.3, 53.7), ("d", "NN", 1, 16384, 129, 64, 14.4, 17.1),
    ("d", "NN", 0, 27234, 20, 228, 24.8, 38.3), ("d", "NT", 1, 18295, 6, 69, 10.1, 14.6),
    ("d", "NN", 0, 128, 18000, 64, 13.7, 17.1), ("d", "NN", 0, 23225, 1, 2405, 253.6, 316.6),
    ("d", "TN", 0, 40000, 9, 256, 37.2, 51.0), ("d", "TN", 1, 16, 16, 8192, 30.4, 489.0),
    ("d", "TT", 0, 40000, 320, 256, 216.8, 158.6), ("d", "TN", 0, 100000, 96, 64, 72.7, 44.9),
    ("d", "NN", 0, 100000, 9, 64, 59.5, 41.0), ("d", "NT", 1, 4096, 4096, 256, 190.5, 145.5),
    ("d", "TT", 0, 7842, 2258, 264, 286.7, 186.9), ("d", "NN", 1, 3118, 1277, 218, 49.5, 39.3),
    ("d", "NN", 0, 7144, 144, 1664, 144.3, 110.8), ("d", "TN", 0, 668, 1898, 1576, 158.8, 101.5),
    ("d", "NT", 1, 1025, 1100, 300, 34.1, 25.7), ("d", "TN", 0, 1999, 1001, 777, 90.0, 68.8),
]
# BF16, aligned: the same, us with 32 k a step, us on the large tiles
BF16 = [("b", f, 0, *rest) for f, *rest in [
    ("NT", 2048, 2048, 64, 7.0, 8.4), ("NT", 38520, 24, 208, 6.9, 8.6), ("NT", 1048, 29528, 16, 26.7, 32.2),
    ("TN", 408, 22216, 16, 11.5, 13.8), ("NT", 392, 7440, 32, 5.8, 7.7), ("NT", 3344, 416, 136, 5.8, 8.5),
    ("NN", 896, 3512, 24, 5.9, 7.9), ("NT", 8, 34184, 256, 6.6, 8.2), ("TN", 24640, 1976, 24, 38.3, 48.8),
    ("TT", 13216, 40, 8, 3.8, 6.9), ("NN", 2048, 2048, 8, 6.6, 8.4), ("NT", 16384, 64, 256, 6.3, 8.9),
    ("NT", 4096, 4096, 256, 28.3, 20.1), ("TN", 24704, 184, 1224, 64.7, 35.1), ("NT", 136, 30760, 7576, 371.1, 178.9),
    ("TT", 10376, 6696, 1104, 312.6, 243.5), ("NT", 14824, 904, 560, 44.7, 30.6), ("NN", 64, 65536, 256, 17.9, 14.3),
    ("TT", 7280, 1496, 1576, 88.5, 65.5), ("TN", 152, 20272, 552, 25.5, 19.5), ("NN", 8192, 8192, 8192, 2390, 1090)]]


def aligned(t, f, pad, m, n, k):
    """Whether gemm_nn_kernel takes it (gemm.hip: nn_ok)."""
    e = 2 if t == "d" else 4
    lda, ldb = (m if f[0] == "T" else k) + pad, (k if f[1] == "T" else n) + pad
    return f[0] == "N" and lda % e == 0 and ldb % e == 0 and k % e == 0 and (f[1] == "T" or n % e == 0)


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(d / "rules.cpp"), "-o", str(d / "rules")],
                   check=True)

    def run(lines):
        out = subprocess.run([str(d / "rules")], input="\n".join(lines), capture_output=True, text=True, check=True)
        return [int(x) for x in out.stdout.split()]
    return run


@pytest.mark.parametrize("rule,cases", [("split", SPLIT), ("direct", DIRECT), ("bf16", BF16)])
def test_the_faster_kernel_is_chosen(choose, rule, cases):
    lines = []
    for t, f, pad, m, n, k, _, _ in cases:
        nn = aligned(t, f, pad, m, n, k)
        large = -(-m // 128) * -(-n // 128) >= 512
        tile = 1 if not large else 2 if nn else 3
        lines.append(f"{rule} {8 if t == 'd' else 4} {f[0] == 'T':d} {f[1] == 'T':d} {nn:d} {tile} {m} {n} {k}")
    assert choose(lines) == [int(new < old) for *_, old, new in cases]
