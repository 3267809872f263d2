"""sq_exp_above (sqaod_amd/csrc/sq_expf.h): the least float x with sq_expf(x) > u,
by which the team sweep decides `expf(-dE*beta) > u`
(CPUDenseGraphAnnealer.cpp:262) as a comparison with x."""
import subprocess

SOURCE = r"""
#include "sq_expf.h"
#include <cstdio>
#include <thread>
#include <vector>
#include <atomic>
static float asFloat(uint32_t u) { union { uint32_t u; float f; } v; v.u = u; return v.f; }
template <class F> static long count(uint32_t lo, uint32_t hi, F bad) {
    std::atomic<long> n{0};
    std::vector<std::thread> th;
    const int T = 8;
    for (int t = 0; t < T; ++t)
        th.emplace_back([&, t] {
            long c = 0;
            for (uint64_t i = lo + (uint64_t)(hi - lo) * t / T; i < lo + (uint64_t)(hi - lo) * (t + 1) / T; ++i)
                c += bad((uint32_t)i);
            n += c;
        });
    for (auto &x : th) x.join();
    return n;
}
int main() {
    /* every float from -0 down to -104, in order */
    const long rising = count(0x80000000u, 0xc2d10000u, [](uint32_t b) { return !(sq_expf(asFloat(b + 1)) <= sq_expf(asFloat(b))); });
    /* every u in [2^-33, 1): all uniforms of a 32-bit word but 0 */
    const long wrong = count(0x2f000000u, 0x3f800000u, [](uint32_t b) {
        const float u = asFloat(b), x = sq_exp_above(u, sq_exp2_tab32);
        return !(x < 0.f && sq_expf(x) > u && !(sq_expf(asFloat(sq_f2u(x) + 1)) > u));
    });
    const float x0 = sq_exp_above(0.f, sq_exp2_tab32), x1 = sq_exp_above(1.f, sq_exp2_tab32);
    const int ends = sq_expf(x0) > 0.f && !(sq_expf(asFloat(sq_f2u(x0) + 1)) > 0.f) && x1 != x1;
    std::printf("%ld %ld %d\n", rising, wrong, ends);
}
"""


def test_least_accepted_exponent_for_every_uniform(tmp_path):
    import os
    csrc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sqaod_amd", "csrc")
    src, exe = tmp_path / "above.cpp", tmp_path / "above"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-march=native", "-ffp-contract=off", "-pthread", "-I" + csrc,
                           str(src), "-o", str(exe)])
    assert subprocess.check_output([str(exe)], text=True).split() == ["0", "0", "1"]
