"""The loop that moves large results in pieces (csrc/sfg_pieces.h), on the CPU:
every piece arrives once, and a transfer that fails anywhere is reported."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "seisfem_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <mutex>
#include <vector>
#include "sfg_pieces.h"

// pieces "arrive" when they are waited for; call number `fail` of kind `what` fails
struct Port : sfg::PiecePort {
    std::mutex mu;
    char what = '-';
    int fail = -1, count = 0, open_now = 0;
    std::vector<int> taken;
    long queued[16][2], arrived[16][2];
    int step(char k) { std::lock_guard<std::mutex> lk(mu); return k == what && count++ == fail ? 7 : 0; }
    int open(int q) override
    {
        for (int b = 0; b < 2; ++b) queued[q][b] = arrived[q][b] = -1;
        { std::lock_guard<std::mutex> lk(mu); ++open_now; }
        return step('o');
    }
    int issue(int q, int b, size_t p) override { queued[q][b] = (long)p; return step('i'); }
    int wait(int q, int b) override { arrived[q][b] = queued[q][b]; return step('w'); }
    void take(int q, int b, size_t p) override
    {
        std::lock_guard<std::mutex> lk(mu);
        if (arrived[q][b] == (long)p) ++taken[p];
    }
    void close(int) override { std::lock_guard<std::mutex> lk(mu); --open_now; }
};

int main()
{
    int bad = 0;
    for (int threads : {1, 2, 8})
        for (int pieces : {0, 1, 2, 3, 6, 40})
            for (char what : {'-', 'o', 'i', 'w'})
                for (int fail = 0; fail < (what == '-' ? 1 : what == 'o' ? threads : pieces); ++fail) {
                    Port port;
                    port.what = what;
                    port.fail = fail;
                    port.taken.assign(pieces, 0);
                    const int e = sfg::deliver(port, pieces, threads);
                    bool all = true;
                    for (int t : port.taken) all = all && t == 1;
                    // the call that was to fail may not have come to pass only if every piece arrived
                    const bool hit = port.count > fail && what != '-';
                    if (port.open_now != 0 || (hit ? e != 7 : e != 0 || !all)) {
                        std::printf("threads %d pieces %d %c%d: error %d, all %d\n", threads, pieces, what, fail, e, all);
                        ++bad;
                    }
                }
    return bad ? 1 : 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no C++ compiler")
def test_every_piece_arrives_or_the_error_is_reported(tmp_path):
    src, exe = tmp_path / "pieces.cpp", tmp_path / "pieces"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
