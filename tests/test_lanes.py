"""Which search lanes are taken (csrc/lanes.h), on the CPU with simulated
measurements: every lane whose hardware queue no earlier lane has, whatever
measurements a stalled host lengthens."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <vector>
#include "lanes.h"

// Lane l runs on queue queues[l]; kernels of one queue run one after the other.
// Measurement number `stalled` takes 20 kernels' time longer and the one after it
// 7, `failing` fails.
static int pick(const std::vector<int>& queues, int stalled, int failing, int* use, int* calls) {
    *calls = 0;
    return jhq::pick_lanes((int)queues.size(), use, [&](const int* ls, int m, bool brief, float* ms) {
        int most = 0;
        for (int i = 0; i < m; i++) {
            int n = 0;
            for (int j = 0; j < m; j++) n += queues[ls[j]] == queues[ls[i]];
            if (n > most) most = n;
        }
        *ms = (brief ? 0.001f : 0.27f) * most + 0.02f;
        if (*calls == stalled) *ms += 5.4f;
        if (stalled >= 0 && *calls == stalled + 1) *ms += 1.9f;
        return (*calls)++ != failing;
    });
}

int main() {
    const std::vector<std::vector<int>> maps = {
        {0, 1, 2, 3, 0, 1}, {0, 0, 1, 1, 2, 3}, {0, 0, 0, 0, 0, 0}, {0, 1, 2, 3, 4, 5}, {0}};
    for (const auto& q : maps) {
        std::vector<int> want;
        for (int l = 0; l < (int)q.size(); l++) {
            bool own = true;
            for (int w : want) own = own && q[w] != q[l];
            if (own) want.push_back(l);
        }
        int use[8], calls = 1;
        for (int stalled = -1; stalled < calls; stalled++) {
            const int n = pick(q, stalled, -1, use, &calls);
            if (std::vector<int>(use, use + n) != want) {
                std::printf("stalled %d: %d lanes of %zu\n", stalled, n, want.size());
                return 1;
            }
        }
        const int total = calls;
        for (int failing = 0; failing < total; failing++)
            if (pick(q, -1, failing, use, &calls) != (failing < calls ? 0 : (int)want.size())) return 2;
    }
    std::printf("lanes ok\n");
    return 0;
}
"""


def test_stalled_measurements_cost_no_lane(tmp_path):
    src, exe = tmp_path / "lanes.cpp", str(tmp_path / "lanes")
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fsanitize=address,undefined", "-I",
                    os.path.join(ROOT, "jhq_gpu_amd", "csrc"), str(src), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "lanes ok" in r.stdout, r.stdout + r.stderr
