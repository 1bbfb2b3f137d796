"""Which passes take the shared expert's tiles along in the routed launches (csrc/shared_along.h), compiled with the host compiler, at
sizes on either side of each of the rule's lines.  256 compute units, three narrow workgroups each."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llmxabe_amd", "csrc")

PROGRAM = r"""
#include <stdio.h>
#include "shared_along.h"
int main() {
  size_t v[6];
  while (scanf("%zu %zu %zu %zu %zu %zu", v, v + 1, v + 2, v + 3, v + 4, v + 5) == 6)
    printf("%d\n", xabe::shared_along(v[0], v[1], v[2], v[3], v[4], v[5], 768));
}
"""

# tokens, tokens the buffers hold, experts per token, experts, hidden, expert width; along
CASES = [
    ((64, 64, 8, 256, 2048, 512), True), ((512, 512, 8, 256, 2048, 512), True),
    ((1024, 1024, 8, 256, 2048, 512), True), ((1025, 1025, 8, 256, 2048, 512), False),      # a share of 32 rows, and more
    ((512, 3072, 8, 256, 2048, 512), True), ((512, 3073, 8, 256, 2048, 512), False),        # the buffers
    ((300, 8192, 8, 256, 2048, 512), False), ((512, 4096, 8, 512, 2048, 512), False),
    ((512, 8192, 8, 256, 7168, 2048), True), ((200, 8192, 8, 128, 4096, 1536), True),       # long routed launches in large buffers
    ((128, 4, 1, 4, 2048, 512), True), ((256, 256, 4, 32, 1024, 512), True), ((256, 8192, 4, 32, 1024, 512), True),  # little work
    ((64, 64, 6, 64, 2048, 1280), True), ((65, 65, 6, 64, 2048, 1280), False),              # 7.9 and 15.7 million weights
    ((256, 256, 8, 128, 2048, 768), True), ((256, 256, 8, 127, 2048, 768), False),          # two rounds of gate/up items, and fewer
    ((256, 256, 8, 96, 2048, 1024), True), ((256, 256, 8, 96, 1920, 1024), False),          # two rounds of down items, and fewer
    ((64, 2048, 2, 8, 4096, 14336), False), ((128, 2048, 2, 16, 4096, 6400), False), ((200, 200, 2, 32, 4096, 2048), False),
    ((100, 100, 6, 64, 2048, 1536), False), ((64, 64, 2, 8, 8192, 2048), False), ((256, 256, 2, 16, 7168, 2048), False),
]


@pytest.fixture(scope="module")
def along(tmp_path_factory):
    d = tmp_path_factory.mktemp("along")
    (d / "along.cpp").write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-I", CSRC, str(d / "along.cpp"), "-o", str(d / "along")])
    lines = "\n".join(" ".join(map(str, sizes)) for sizes, _ in CASES)
    out = subprocess.run([str(d / "along")], input=lines, capture_output=True, text=True, check=True).stdout.split()
    return [o == "1" for o in out]


@pytest.mark.parametrize("i", range(len(CASES)), ids=["-".join(map(str, sizes)) for sizes, _ in CASES])
def test_rule(along, i):
    assert along[i] == CASES[i][1]
