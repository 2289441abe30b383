"""Which kernel an fp32 product takes (f32_use_split in vedic_common.hpp): the
rule compiled for the host and asked on the CPU.  With 128 x 128 tiles for
exactly half the CUs the bf16 split kernel is the faster only where the
contraction is also split over workgroups, in slices of at least 384 steps."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include <hip/hip_runtime.h>
#include "logos_amd/csrc/vedic_common.hpp"
#include <stdio.h>
int main() {
    int op, M, N, K, vec, scatter;
    while (scanf("%d %d %d %d %d %d", &op, &M, &N, &K, &vec, &scatter) == 6)
        printf("%d\\n", (int)vedic::f32_use_split(op, M, N, K, vec, scatter, 256));
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    from logos_amd import build

    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("route")
    (d / "route.hip").write_text(SOURCE)
    subprocess.run([cc, "-std=c++17", "--offload-host-only", f"-I{ROOT}", str(d / "route.hip"), "-o", str(d / "route")],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)

    def ask(cases):
        text = "\n".join(" ".join(str(int(x)) for x in c) for c in cases)
        return [int(x) for x in subprocess.run([str(d / "route")], input=text, text=True, check=True,
                                               stdout=subprocess.PIPE).stdout.split()]

    return ask


def test_half_the_cus(route):
    """2048 x 1024 is 128 tiles: half of 256 CUs."""
    cases = [(op, 2048, 1024, K, True, False) for op in range(3) for K in range(4, 2049, 4)]
    got = dict(zip(cases, route(cases)))
    for (op, _, _, K, _, _), split in got.items():
        assert not split or K // 384 >= 2, (op, K)  # never on the split kernel without slices
        if K <= 640:
            assert not split, (op, K)
        if K >= 1024:
            assert split, (op, K)
    assert route([(0, 2048, 1024, K, True, True) for K in (512, 1024, 4096)]) == [0, 0, 0]  # scattered: no slices


def test_more_fewer_and_unaligned(route):
    assert route([(0, 2049, 1024, 4, True, False), (1, 8192, 8192, 64, True, True), (2, 4096, 1024, 8, True, False)]) == [1] * 3
    assert route([(0, 1920, 1024, 8192, True, False), (1, 8192, 64, 8192, True, False), (2, 512, 1024, 1024, True, False)]) == [0] * 3
    assert route([(0, 2048, 1024, 16, False, False), (1, 100, 60, 7, False, False)]) == [1] * 2
