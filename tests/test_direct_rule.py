"""The host's rule for the small jobs' binning, compiled on its own: which jobs
k_tile_bin bins, and which of those with 1024 threads a tile. It goes by the
scenes' triangles and tiles, not by how many draws or scenes bring them."""
import os
import re
import subprocess

import pytest

from rusterizer_amd import build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    text = open(os.path.join(build.CSRC, "rz_api.hip")).read()
    a = text.index("constexpr uint64_t DIRECT_WORK")
    b = text.index("};", text.index("struct DirectRule")) + 2
    header = open(os.path.join(build.CSRC, "rz_kernels.h")).read()
    tris = re.search(r"constexpr uint32_t DIRECT_TRIS = \d+;", header).group(0)
    d = tmp_path_factory.mktemp("rule")
    src = d / "rule.cpp"
    src.write_text("#include <algorithm>\n#include <cstdint>\n#include <cstdio>\n" + tris + "\n" + text[a:b] + """
int main() {
    unsigned n_cu, scenes, w, h, t;
    DirectRule r;
    if (scanf("%u %u", &n_cu, &scenes) != 2) return 1;
    while (scenes-- && scanf("%u %u %u", &w, &h, &t) == 3) r.scene(w, h, t);
    printf("%d %d\\n", (int)r.direct(), (int)r.wide(n_cu));
}
""")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", str(src), "-o", str(d / "rule")], check=True)

    def ask(scenes, n_cu=256):
        text = f"{n_cu} {len(scenes)}\n" + "".join("%d %d %d\n" % s for s in scenes)
        out = subprocess.run([str(d / "rule")], input=text, capture_output=True, text=True, check=True).stdout.split()
        return tuple(map(int, out))

    return ask


@pytest.mark.parametrize("scenes,n_cu,want", [
    ([(64, 64, 10)] * 16, 256, (1, 0)),            # 16 chunks of triangles, hardly any in each
    ([(32, 32, 200)] * 256, 256, (1, 0)),
    ([(512, 512, 3840)], 256, (1, 0)),
    ([(512, 512, 3841)], 256, (1, 1)),
    ([(513, 512, 3841)], 256, (1, 0)),             # a tile more than CUs
    ([(512, 512, 3841)], 255, (1, 0)),
    ([(64, 64, 10)] * 15 + [(64, 64, 9000)], 256, (1, 1)),
    ([(512, 512, 16384)], 256, (1, 1)),
    ([(512, 512, 16385)], 256, (0, 0)),            # beyond a scene's bit masks
    ([(4096, 4096, 3)], 256, (0, 0)),              # too many tiles
])
def test_rule(rule, scenes, n_cu, want):
    assert rule(scenes, n_cu) == want
