"""The row passes' scalar arithmetic, swept on the CPU from the header the kernels include."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "d3d_amd" / "csrc"


def _run(tmp_path, source):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    src, exe = tmp_path / "sweep.cpp", tmp_path / "sweep"
    src.write_text(source)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-D__device__=", "-D__forceinline__=inline",
                    f"-I{CSRC}", str(src), "-o", str(exe)], check=True, capture_output=True, text=True)
    return subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()


EXP = r"""
#include <cmath>
#include <cstdio>
#include <cstring>
#include "scalar_math.hpp"
static float red(float d) {
    return d3d::exp_reduced(d, [](float f) { return (float)std::exp2((double)f); },
                            [](float p, int n) { return std::ldexp(p, n); });
}
int main() {
    double worst = 0, sum = 0;
    long count = 0;
    unsigned s = 1;
    const float lo[] = {-1e-4f, -0.6931f, -4.f, -32.f, -87.f};
    for (float l : lo) {
        double sq = 0;
        const int n = 400000;
        for (int i = 0; i < n; ++i) {
            s = s * 1664525u + 1013904223u;
            const float d = l * ((s >> 8) * (1.f / 16777216.f));
            const double t = std::exp((double)d);
            int e;
            std::frexp(t, &e);
            const double u = (red(d) - t) / std::ldexp(1.0, e - 24);
            worst = std::fmax(worst, std::fabs(u));
            sq += u * u;
        }
        std::printf("%.4f ", std::sqrt(sq / n));
    }
    std::printf("%.4f %d %d %d", worst, red(0.f) == 1.f, red(-104.f) < 1e-44f, red(NAN) != red(NAN));
}
"""


def test_reduced_exponential(tmp_path):
    *rms, worst, one, small, nan = map(float, _run(tmp_path, EXP))
    # exp2's rounding (half a unit at most, 0.289 rms) and the reduced argument's
    # (2^-26 of it times ln 2: up to 0.18 units).  The unreduced form rounds
    # twice more: 1.0 and 0.41.
    assert worst < 0.7 and max(rms) < 0.31
    assert one and small and nan


QUOTIENT = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include "scalar_math.hpp"
template <bool DIRECT>
static void sweep(float T, const d3d::Quotient& q) {
    double off = 0;
    long bad = 0;
    for (uint32_t m = 0; m < (1u << 23); ++m) {
        const uint32_t u = 0x3f800000u | m;
        float x;
        std::memcpy(&x, &u, 4);
        const double exact = (double)x / (double)T;
        const double unit = std::ldexp(1.0, std::ilogb(exact) - 23);
        off = std::fmax(off, std::fabs(q.first<DIRECT>(x) - exact) / unit);
        bad += q.of<DIRECT>(x) != x / T;
    }
    std::printf("%.6f %ld ", off, bad);
}
int main(int argc, char** argv) {
    const float ts[] = {TEMPERATURES};
    for (float T : ts) {
        const d3d::Quotient q(T);
        if (q.direct) sweep<true>(T, q);
        sweep<false>(T, q);
    }
}
"""


@pytest.mark.parametrize("ts", ["0.7f, 0.8f, 1.3f, 0.9f", "1.7f, 1.95f, 0.95f, 0.487f",
                                "0x1.fffff8p0f, 0x1.fffffcp0f, 0x1.000002p0f, 0x1.000004p0f"])
def test_quotients_round_as_the_division(ts, tmp_path):
    """Every mantissa of x at temperatures of either kind and next to powers of
    two (the worst 1 / T): q within the unit that the theorem asks for, and the
    division's bits.  q = x * inv alone is up to 1.5 units off."""
    out = _run(tmp_path, QUOTIENT.replace("TEMPERATURES", ts))
    assert len(out) >= 8
    for off, bad in zip(out[::2], out[1::2]):
        assert float(off) <= 1.0 and int(bad) == 0
