"""The comparisons behind the group sweeps' barrier (group_steps.hpp), on the
host.  The meeting before a launch's first step: a word that no launch has
refreshed must not count as reached, however many steps other launches have
made since.  Its steps: words that lie within the launch compare right wherever
the 32-bit count wraps.  A smoothing call of any number of sweeps is split so that
no launch has more steps than those comparisons hold for."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <initializer_list>
#include "group_steps.hpp"
using namespace unap_hip;
using U64 = unsigned long long;
int main() {
    const U64 epochs[] = {0ull, 1ull, 0x7fffffffull, 0x80000000ull, 0x80000001ull, 0xffffff00ull, 0xffffffffull,
                          0x100000000ull, 0x100000200ull, 0x1ffffffffull, 1ull << 52};
    const U64 stale[] = {0ull, 1ull, 511ull, 0x7fffffffull, 0xffffffffull, 0x100000001ull};
    const U64 steps[] = {1, 2, 3, 511, 512, 65537, 1 << 20, 0x7ffffffe};
    int bad = 0;
    for (U64 e : epochs) {
        const GroupStep s = e + 1;  // the meeting of a launch that starts at e
        bad += !groupReached(s, s) || !groupReached(s + 1, s) || groupReached((GroupStep)e, s);
        for (U64 w : stale) bad += w <= e && groupReached((GroupStep)w, s);
        for (U64 k : steps)
            for (U64 w : {e, e + 1, e + k - 1, e + k, e + k + 1})
                bad += groupReached((unsigned)w, (unsigned)(e + k)) != (w >= e + k);
    }
    // sweeps are split so that a launch's steps stay countable
    for (long long nl : {1, 2, 3, 60, 511, 512, 1 << 20, 0x7fffffff})
        for (long long left : {1, 2, 100, 2048, 2049, 1 << 20, 0x7fffffff}) {
            const long long k = groupSweeps((int)nl, (int)left);
            bad += k < 1 || k > left || (k > 1 && k * nl > (1 << 20)) || (k < left && (k + 1) * nl <= (1 << 20));
        }
    std::printf("%d\\n", bad);
}
"""


def test_stale_and_wrapped_words(tmp_path):
    src, exe = tmp_path / "steps.cpp", tmp_path / "steps"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "unap_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True)
    assert int(subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout) == 0
