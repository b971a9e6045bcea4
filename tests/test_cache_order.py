"""Which token a workgroup of the cache-writing kernels takes (csrc/cache_order.h, compiled for the host): every token once,
neighbours on one XCD."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cpm.cu_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_token_once(tmp_path):
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text('#define __device__\n#include "cache_order.h"\n#include <cstdio>\n#include <cstdlib>\n'
                   "int main(int n, char** v) { for (int i = 1; i < n; ++i) { const int t = atoi(v[i]);\n"
                   'for (int w = 0; w < t; ++w) printf("%d ", cache_order(w, t)); puts(""); } }\n')
    subprocess.run(["g++", "-O1", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    counts = list(range(1, 700)) + [1023, 1024, 1025, 1087, 1088, 2048, 2395, 4097, 32768]
    lines = subprocess.run([str(exe)] + [str(n) for n in counts], check=True, capture_output=True, text=True).stdout.splitlines()
    assert len(lines) == len(counts)
    for n, line in zip(counts, lines):
        order = [int(t) for t in line.split()]
        assert sorted(order) == list(range(n)), n
        # 8 neighbouring tokens, whose values share lines of the cache, go to workgroups of one XCD (up to the last 63 tokens)
        place = {t: w for w, t in enumerate(order)}
        for t in range(0, n & ~63, 8):
            assert len({place[t + i] % 8 for i in range(8)}) == 1, (n, t)
