"""The tickets that hand a queue's entries to a launch's waves (FeedPlace,
csrc/ljx_feed.h): whichever wave comes next, every chunk of 64 entries is
handed out exactly once, an exhausted wave's place lies at or past the queue's
end, and a ticket stays within one run.  Grids below, at and above the number
of feeds and no multiples of it, ragged queues up to the longest, tickets of 1
to 16 chunks.  Host code built with hipcc from the device header; no GPU
needed."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "lajolla_public_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROG = r"""
#include "ljx_feed.h"
#include <cstdio>
#include <random>
#include <set>
#include <vector>
using namespace ljx;
int main() {
    std::mt19937 rng(7);
    const int grids[] = {1, 3, 7, 8, 9, 17, 64, 250, 2048};
    const int tails[] = {0, 1, 63, 64, 65, 1000};
    std::set<int> spans;
    long long checked = 0, bad = 0;
    for (int blocks : grids)
        for (int wpb : {1, 4})
            for (int tickets : {0, 1, kFeedTickets})
                for (int f = 0; f < 9; f++)
                    for (int tail : tails) {
                        // queues around the lengths where a ticket's span doubles, and short ones
                        long long len = f == 0 ? tail : 64ll * (2ll << (f - 1)) * (tickets ? tickets : 1) * blocks * wpb / 4 + tail - 64;
                        if (f == 8 && blocks == 2048 && tail == 0) len = kMaxQueue;
                        else if (len < 0 || len > (1ll << 22)) continue;
                        const int n = int(len), chunks = (n + 63) / 64;
                        for (int greedy = 0; greedy < 2; greedy++) {
                            std::vector<FeedPlace> w;
                            std::vector<int> counter(kFeeds, 0), seen(chunks, 0);
                            for (int b = 0; b < blocks; b++)
                                for (int k = 0; k < wpb; k++) {
                                    FeedPlace p;
                                    p.place(b, blocks, k, wpb, n, tickets);
                                    w.push_back(p);
                                }
                            if (kFeedRun % w[0].span || (tickets == 0 && w[0].span != 1)) bad++;
                            spans.insert(w[0].span);
                            std::vector<int> live(w.size());
                            for (size_t i = 0; i < live.size(); i++) live[i] = int(i);
                            while (!live.empty()) {
                                // greedy: one wave takes all it can before the next moves
                                const size_t at = greedy ? live.size() - 1 : rng() % live.size();
                                FeedPlace &p = w[live[at]];
                                const int base = p.base();
                                checked++;
                                if (base < 0 || base % 64) bad++;
                                if (base >= n) {
                                    p.advance([&] { return counter[p.feed]++; });
                                    if (p.sub == 0 && p.base() < n) bad++;  // nothing after the end
                                    live[at] = live.back();
                                    live.pop_back();
                                    continue;
                                }
                                seen[base / 64]++;
                                p.advance([&] { return counter[p.feed]++; });
                            }
                            for (int c : seen) bad += c != 1;
                        }
                    }
    for (int s : {1, 2, 4, 8, 16})
        if (!spans.count(s)) bad++;
    std::printf("checked %lld bad %lld\n", checked, bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(not shutil.which(HIPCC) and not os.path.exists(HIPCC), reason="hipcc not installed")
def test_every_chunk_is_handed_out_once(tmp_path):
    src = tmp_path / "feed.hip"
    src.write_text(PROG)
    exe = tmp_path / "feed"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-w", "-I" + CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
