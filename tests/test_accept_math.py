"""CPU checks of the acceptance weights' float64 arithmetic (accept_math.h):
the header compiled for the host, against 80-bit long double."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "yuuka_amd" / "csrc"

PROGRAM = r"""
#include "accept_math.h"
#include <cstdio>
#include <random>

using namespace yk;

int main() {
    std::mt19937_64 rng(7);
    auto uniform = [&](double lo, double hi) { return lo + (hi - lo) * ((rng() >> 11) * 0x1p-53); };
    // exp: relative error in units of the last place (normal results), and in
    // units of the smallest denormal below them
    double worst = 0, low = 0;
    for (int i = 0; i < 2000000; i++) {
        double x = i % 4 == 0 ? -uniform(0, 0.1) : i % 4 == 1 ? -std::exp(uniform(-40, 6.5)) : -uniform(0, 708);
        if (i % 16 == 3) x = -uniform(708, 760);
        if (i < 800) x = -i * (0.0433216987849966 / 2);  // the table's ends and middles
        if (x < -1000) continue;
        const long double want = expl((long double)x), got = exp_nonpos(x, kExpTab);
        if (want >= 0x1p-1022L) {
            int e;
            frexpl(want, &e);
            worst = std::fmax(worst, (double)(fabsl(got - want) / ldexpl(1, e - 53)));
        } else {
            low = std::fmax(low, (double)(fabsl(got - want) / 0x1p-1074L));
        }
    }
    printf("exp %.4f %.4f\n", worst, low);
    printf("ends %d %d %d\n", exp_nonpos(0.0, kExpTab) == 1.0, exp_nonpos(-1000.0, kExpTab) == 0.0,
           std::isnan(exp_nonpos(NAN, kExpTab)));
    // the exponent: the correctly rounded quotient, at temperatures from the
    // smallest to the largest float
    long bad = 0;
    for (int i = 0; i < 2000000; i++) {
        const float temperature = i % 3 ? (float)uniform(0.05, 5) : (float)std::exp2(uniform(-148, 127.9));
        const float mx = (float)uniform(-40, 40), l = (float)(mx - std::exp(uniform(-20, 5)));
        const double a = (double)(l - mx), want = a / (double)temperature;
        const double got = exponent_of(l, mx, make_temp(temperature));
        if (want < -1000.0 ? !(got <= -999.9 && got >= -1000.1) : got != want && std::fabs(want) > 1e-290) bad++;
    }
    printf("quotient %ld\n", bad);
    const float big = 3e38f;
    printf("overflow %d %d %d\n", exp_nonpos(exponent_of(-big, big, make_temp(1e38f)), kExpTab) == 0.0,
           exp_nonpos(exponent_of(-big, big, make_temp(1e-45f)), kExpTab) == 0.0,
           std::isnan(exp_nonpos(exponent_of(-big, big, make_temp(INFINITY)), kExpTab)));
    // tie groups against one addition after the other
    bad = 0;
    long longest = 0;
    for (int i = 0; i < 60000; i++) {
        uint32_t ties = 1 + (uint32_t)std::exp(uniform(0, i % 100 ? 7 : 12));
        double w = i % 3 ? std::exp(-uniform(0, 12)) : 1.0, before = i % 2 ? 0.0 : uniform(0, 2) * w * ties;
        double total = (before + w * ties) * (i % 5 ? 1 + uniform(0, 1) : 1.0), p = (float)uniform(0.01, 1);
        if (i % 7 == 0) p = 0.25 * (1 + i % 3);
        if (i % 11 == 0) total = std::exp2(std::ceil(std::log2(total)));
        // shares halfway between two multiples of a sum's last place
        if (i % 13 == 0) w = std::ldexp(2 * (double)(rng() % 1000) + 1, -(int)(50 + rng() % 6)), total = 1.0, before = uniform(0, 1);
        if (i % 17 == 0) w *= 1e-17;
        uint32_t want = ties;
        double cum = before / total;
        for (uint32_t k = 1; k < ties; k++) {
            cum += w / total;
            if (cum >= p) {
                want = k;
                break;
            }
        }
        if (tie_members(before, w, total, p, ties) != want) bad++;
        if (want < ties && want > longest) longest = want;
    }
    printf("ties %ld %ld\n", bad, longest);
    printf("flat %d\n", exp_nonpos(exponent_of(-big, 0.f, make_temp(INFINITY)), kExpTab) == 1.0);
}
"""


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("accept_math")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-D__device__=", "-D__forceinline__=inline",
                    "-D__constant__=static const", f"-I{CSRC}", "-o", d / "t", d / "t.cpp"], check=True)
    out = subprocess.run([d / "t"], capture_output=True, text=True, check=True, timeout=100).stdout
    return {line.split()[0]: line.split()[1:] for line in out.splitlines()}


def test_exponential_within_its_stated_error(report):
    """0.58 ulp; below the normal range a second rounding, together under one denormal step."""
    worst, low = map(float, report["exp"])
    assert 0.5 <= worst <= 0.58 and low <= 1.0
    assert report["ends"] == ["1", "1", "1"]


def test_exponent_is_the_correctly_rounded_quotient(report):
    assert report["quotient"] == ["0"]


def test_overflowed_differences_weigh_nothing(report):
    assert report["overflow"] == ["1", "1", "1"] and report["flat"] == ["1"]


def test_tie_group_as_one_addition_after_the_other(report):
    assert report["ties"][0] == "0" and int(report["ties"][1]) > 50000
