"""Which batches the ragged kernels take (ragged_pages, ztcp_ragged.h), against
measured times of both kernel families (256 CUs), on the CPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "vlx-tee_amd" / "csrc"
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

LAYOUT_WORDS = 40  # at least what a Layout and its index take
# direction, payload bytes, pages, us with the payloads in LDS, us with the layout-agnostic kernels
MEASURED = [
    ("ingress", 2988, 30, 75, 136), ("ingress", 2988, 20000, 727, 822), ("ingress", 10708, 20000, 1670, 3136),
    ("ingress", 15120, 20000, 2444, 3163), ("ingress", 19440, 20000, 3866, 4152),
    ("ingress", 23760, 6144, 1748, 1896), ("ingress", 23760, 8000, 2391, 2304), ("ingress", 23760, 20000, 5797, 4939),
    ("ingress", 32400, 2560, 1391, 1512), ("ingress", 32400, 8000, 4417, 3168), ("ingress", 32400, 20000, 10930, 6683),
    ("ingress", 36720, 20000, 12575, 8075), ("ingress", 49680, 700, 1249, 1483), ("ingress", 49680, 768, 1251, 1510),
    ("ingress", 49680, 1024, 1652, 1618), ("ingress", 49680, 2000, 3264, 2166), ("ingress", 66960, 300, 1130, 1754),
    ("ingress", 66960, 3000, 6559, 3603), ("ingress", 66960, 20000, 42850, 13817),
    ("ingress", 32400, 3072, 1668, 1696), ("ingress", 77760, 900, 2525, 3278),
    ("egress", 10708, 20000, 1224, 9650), ("egress", 66960, 20000, 22670, 30050), ("egress", 77760, 40000, 51480, 64650),
    ("egress", 84240, 2304, 6165, 6383), ("egress", 84240, 4000, 10931, 9261), ("egress", 105840, 1000, 3453, 5733),
    ("egress", 105840, 8000, 27420, 20747), ("egress", 118800, 2304, 8655, 8844), ("egress", 118800, 2560, 9609, 9446),
    ("egress", 153360, 20000, 97500, 63060), ("egress", 157680, 2304, 11473, 12525), ("egress", 157680, 2560, 12755, 13345),
]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text("""
#include <cstdio>
#include <cstdlib>
#include "ztcp_ragged.h"
int main(int argc, char** argv) {
    for (int i = 1; i + 3 < argc; i += 4) {
        const bool in = argv[i][0] == 'i';
        const size_t b = ztcp::ragged_page_bytes((uint32_t)atol(argv[i + 1]), in, %d);
        const int n = ztcp::ragged_pages(atoll(argv[i + 2]), b, in, atoi(argv[i + 3]));
        printf("%%d %%d\\n", n, (size_t)n * b <= ztcp::kRaggedRoom);
    }
}""" % LAYOUT_WORDS)
    exe = d / "rule"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", str(CSRC), str(d / "rule.cpp"), "-o", str(exe)], check=True)

    def run(calls):
        out = subprocess.run([str(exe), *(str(x) for c in calls for x in c)], check=True, capture_output=True, text=True)
        return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]

    return run


def test_no_measured_batch_takes_the_slower_kernels(rule):
    got = rule([(w, p, n, 256) for w, p, n, _, _ in MEASURED])
    for (w, p, n, lds, other), (pages, _) in zip(MEASURED, got):
        taken, best = (lds if pages else other), min(lds, other)
        # 3 %: at a line the two families cross, and the layout-agnostic kernels' times differ
        # by up to a third between blob strides (50 KB and 78 KB pages, four rounds, above)
        assert taken <= 1.03 * best, (w, p, n, pages, lds, other)


@pytest.mark.parametrize("cus", [1, 64, 256, 304])
def test_workgroups_fit_the_lds(rule, cus):
    calls = [(w, p, n, cus) for w in ("ingress", "egress") for p in (10, 64, 2988, 10708, 40000, 81000, 83000, 160000, 163712, 163713, 200000)
             for n in (1, 7, 1023, 1025, 5000, 100000, 1 << 30, (1 << 30) + 1)]
    for c, (pages, fits) in zip(calls, rule(calls)):
        assert 0 <= pages <= 32 and fits, c
        if c[1] > 163712 or c[2] > 1 << 30 or (c[0] == "ingress" and c[1] > 81792):
            assert pages == 0, c
        if c[2] <= cus and c[1] <= (80000 if c[0] == "ingress" else 160000):
            assert pages == 1, c  # one round, one page a workgroup
