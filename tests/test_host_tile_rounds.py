"""Host test of the block order of unsplit traversal launches: xcd_round_block deals chunks of
consecutive blocks to the 8 XCDs round by round. It has to be a bijection of [0, n) for every n, and in
every full round each XCD's blocks have to be consecutive. Compiles the functions' own source text."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HARNESS = r"""
#include <cstdint>
#include <cstdio>
#include <vector>
#define __device__
#define __forceinline__ inline
%s
%s
static int check(int64_t n, int64_t chunk) {
    std::vector<int> seen(n, 0);
    for (int64_t b = 0; b < n; ++b) {
        const int64_t t = xcd_round_block(b, n, chunk);
        if (t < 0 || t >= n || seen[t]++) return 1;
        const int64_t first = b / (8 * chunk) * (8 * chunk);
        if (first + 8 * chunk <= n && t != first + b %% 8 * chunk + (b - first) / 8) return 2;
        if (t < first || t >= first + 8 * chunk) return 3;
    }
    return 0;
}
int main() {
    const int64_t chunks[] = {1, 3, 4, %d, 64};
    for (int64_t c : chunks)
        for (int64_t n = 1; n <= 1100; ++n)
            if (int e = check(n, c)) { std::printf("n=%%lld chunk=%%lld error %%d\n", (long long)n, (long long)c, e); return 1; }
    return check(8100, %d) || check(3907, %d);
}
"""


def test_xcd_round_block_is_a_bijection(tmp_path):
    src = open(os.path.join(ROOT, "smallupbp_amd", "csrc", "traverse.hip")).read()
    fns = [re.search(r"__device__ __forceinline__ int64_t %s\(.*?\n\}" % f, src, re.S).group(0)
           for f in ("xcd_block", "xcd_round_block")]
    chunk = int(re.search(r"constexpr int64_t kXcdChunk = (\d+);", src).group(1))
    cpp = tmp_path / "rounds.cpp"
    cpp.write_text(HARNESS % (fns[0], fns[1], chunk, chunk, chunk))
    exe = tmp_path / "rounds"
    try:
        subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", str(cpp), "-o", str(exe)])
    except (OSError, subprocess.CalledProcessError) as e:
        pytest.fail("host build of xcd_round_block failed: %s" % e)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
