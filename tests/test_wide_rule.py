"""Which small-M products take the wide kernel (matmul_wide_wins, m27q_route.h):
the rule is host code without a HIP call, evaluated here for 256 CUs."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mono-qwen27_amd", "csrc")
TYPES = {"Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "Q8_0": 8, "IQ4_XS": 23}
MAIN = """#include <cstdio>
#include "m27q_route.h"
int main() {
    unsigned t;
    int layout, rows, K, M;
    while (scanf("%u %d %d %d %d", &t, &layout, &rows, &K, &M) == 5)
        printf("%d\\n", (int)m27q::matmul_wide_wins(t, layout, (rows + 15) / 16, K, M, 256));
}
"""

# type, layout (1 TILED, 0 GGUF), rows, K, M: measured slower on the wide kernel (the time it took, as a
# multiple of the other kernel's) ...
SLOWER = [
    ("Q8_0", 0, 50000, 2048, 9), ("Q8_0", 0, 50000, 2048, 16),      # 1.54 1.47
    ("Q8_0", 0, 24576, 2048, 9), ("Q8_0", 0, 23629, 992, 12),       # 1.27 1.17
    ("Q8_0", 0, 100000, 2048, 17), ("Q8_0", 0, 100000, 512, 24),    # 1.21 1.05
    ("Q8_0", 0, 2048, 128, 5), ("Q8_0", 0, 17408, 5120, 5),         # 1.27 1.10
    ("IQ4_XS", 0, 24576, 512, 9), ("IQ4_XS", 0, 12288, 256, 9),     # 1.19 1.14
    ("IQ4_XS", 0, 4096, 512, 5), ("IQ4_XS", 0, 1005, 256, 6),       # 1.13 1.19
    ("Q5_K", 1, 6144, 17408, 17), ("Q5_K", 1, 6160, 32768, 20),     # 1.23 1.24
    ("Q5_K", 0, 6144, 17408, 24), ("Q4_K", 1, 7168, 2560, 24),      # 1.07 1.06
    ("Q4_K", 1, 7680, 32768, 17), ("Q4_K", 0, 7168, 32768, 17),     # 1.16 1.20
    ("Q4_K", 0, 6144, 2048, 24), ("Q4_K", 1, 50000, 5120, 17),      # 1.06 1.06
    ("Q8_0", 1, 6144, 2048, 17), ("Q8_0", 1, 8208, 1024, 24),       # 1.16 1.24
    ("Q8_0", 1, 14336, 1024, 32), ("Q8_0", 1, 7168, 1024, 32),      # 1.20 1.16
    ("IQ4_XS", 1, 14336, 1024, 17), ("IQ4_XS", 1, 50000, 17408, 17),  # 1.19 1.19
    ("IQ4_XS", 1, 50000, 5120, 24), ("IQ4_XS", 1, 34816, 17408, 17),  # 1.14 1.13
    ("Q6_K", 0, 13885, 9984, 22), ("Q6_K", 0, 28756, 9984, 17),     # 1.16 1.15
    ("Q6_K", 1, 5120, 17408, 17), ("Q6_K", 0, 5120, 17408, 17),     # 1.07 1.23
]
# ... and faster (the other kernel's time as a multiple of its own)
FASTER = [
    ("Q4_K", 1, 34816, 5120, 64), ("Q6_K", 1, 5120, 17408, 64), ("Q8_0", 0, 12288, 2048, 37),  # 1.7 1.6 3.0
    ("Q4_K", 1, 17408, 5120, 17), ("Q6_K", 1, 17408, 5120, 24), ("Q5_K", 0, 17408, 5120, 32),  # 1.6 1.5 1.5
    ("Q4_K", 1, 1024, 17408, 17), ("Q8_0", 1, 4096, 5120, 17), ("IQ4_XS", 1, 4096, 17408, 24),  # 1.5 1.3 1.4
    ("Q6_K", 1, 8192, 5120, 17), ("Q4_K", 1, 8192, 5120, 32), ("Q5_K", 0, 8192, 512, 17),      # 1.1 1.1 1.2
    ("Q8_0", 1, 10240, 5120, 17), ("IQ4_XS", 1, 17408, 5120, 32), ("IQ4_XS", 1, 16384, 1024, 17),  # 1.3 1.3 1.2
    ("Q6_K", 0, 27960, 8704, 28), ("Q6_K", 0, 10240, 5120, 17), ("Q8_0", 1, 17408, 512, 24),   # 1.3 1.4 1.3
    ("Q8_0", 0, 6144, 6144, 9), ("Q8_0", 0, 1024, 5120, 5), ("Q8_0", 0, 17408, 5120, 9),       # 2.4 2.5 1.4
    ("IQ4_XS", 0, 6144, 6144, 16), ("IQ4_XS", 0, 2048, 2048, 8), ("IQ4_XS", 0, 17408, 17408, 9),  # 2.0 1.2 1.5
    ("Q8_0", 0, 17408, 2048, 24), ("IQ4_XS", 0, 50000, 5120, 17),                              # 1.5 1.2
]


@pytest.fixture(scope="module")
def wins(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(MAIN)
    exe = str(d / "rule")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC,
                    str(d / "rule.cpp"), "-o", exe], check=True)

    def run(cases):
        text = "\n".join("%d %d %d %d %d" % (TYPES[t], layout, rows, K, M) for t, layout, rows, K, M in cases)
        out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True).stdout.split()
        return [x == "1" for x in out]
    return run


def test_gpu_cases_take_the_kernel_they_name(wins):
    """The parity tests' lists: the wide kernel's cases reach it, the others don't."""
    import test_gpu_matmul as g
    order = lambda cases: [(t, layout, rows, K, M) for t, rows, K, M, layout in cases]  # noqa: E731
    assert [c for c, w in zip(g.WIDE, wins(order(g.WIDE))) if not w] == []
    other = g.VALU_SHORT + g.TWO_LAUNCHES
    assert [c for c, w in zip(other, wins(order(other))) if w] == []
    assert wins([("IQ4_XS", 1, 49200, 7424, 32)]) == [False]


def test_products_measured_slower_keep_their_kernel(wins):
    assert [c for c, w in zip(SLOWER, wins(SLOWER)) if w] == []


def test_products_measured_faster_take_the_wide_kernel(wins):
    assert [c for c, w in zip(FASTER, wins(FASTER)) if not w] == []


def test_rows_that_never_and_always_take_it(wins):
    """Up to 4 rows never, up to 16 only GGUF Q8_0 / IQ4_XS (the wide kernel has
    no 16-row instances of the others); past 32 rows always."""
    shapes = [(rows, K) for rows in (1, 100, 4096, 6144, 12345, 14336, 50000, 200000) for K in (256, 2048, 5120, 17408)]
    for t in TYPES:
        for layout in (0, 1):
            gguf8 = layout == 0 and t in ("Q8_0", "IQ4_XS")
            assert not any(wins([(t, layout, r, K, M) for r, K in shapes for M in ((2, 3, 4) if gguf8 else (2, 4, 8, 16))]))
            assert all(wins([(t, layout, r, K, M) for r, K in shapes for M in (33, 48, 64)]))
