"""The step order of the flow head's residual GEMM (csrc/flow_steps.h, which its kernel and this test share) on the
host: every 32-k step of a K slice is worked once, in order, from a register set that holds it, and nothing past the
slice is loaded -- for every K that the rule accepts up to the widest feed-forward, and every tile."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "ming-tts-serve_amd", "csrc", "flow_steps.h")

PROGRAM = """
#include "%s"
#include <cstdio>
#include <vector>
using namespace ming;

template <int CH>
int run(int K) {
    const int S = K / k_slices(K) / 32;
    int held[2] = {-1, -1}, bad = 0;
    std::vector<int> order;
    auto load = [&](int set, int s) {
        bad += s < 0 || s + CH > S;
        held[set] = s;
    };
    auto work = [&](int set) {
        for (int k = 0; k < CH; k++) order.push_back(held[set] + k);
    };
    flow_first<CH>(S, load);
    flow_turns<CH>(S, load, work);
    bad += (int)order.size() != S;
    for (int i = 0; i < (int)order.size(); i++) bad += order[i] != i;
    return bad;
}

int main() {
    const int tiles[5][2] = {{1, 1}, {2, 1}, {3, 1}, {2, 2}, {3, 2}};
    for (int K = 64; K <= 4096; K += 64) {
        if (!flow_k_fits(K)) continue;
        int bad = 0;
        for (auto& t : tiles) bad += flow_set_steps(t[0], t[1]) == 8 ? run<8>(K) : (flow_set_steps(t[0], t[1]) == 4 ? run<4>(K) : 1);
        printf("%%d %%d\\n", K, bad);
    }
}
"""


def test_every_step_once(tmp_path):
    src, exe = tmp_path / "steps.cpp", tmp_path / "steps"
    src.write_text(PROGRAM % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas", str(src), "-o", str(exe)], check=True, timeout=120)
    got = [tuple(map(int, l.split())) for l in subprocess.run([str(exe)], capture_output=True, text=True, check=True,
                                                              timeout=60).stdout.splitlines()]
    assert [k for k, _ in got] == [256, 512, 768, 1024, 1536, 2048, 3072, 4096]
    assert [k for k, bad in got if bad] == []
