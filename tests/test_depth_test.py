"""The linear-depth rejection's decision without divisions (taa-star_amd/csrc/taa_depth_test.hpp), compiled for
the host: wherever it decides, it decides as the two IEEE single-precision divisions of the FP32 path do --
for random depths, for depths within a few ulp of the threshold, for coincident, extreme and non-finite ones --
with the factor thr / |n f| off by the few ulp of a hardware reciprocal; and on ordinary frames it decides almost always."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "taa-star_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PROGRAM = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include "taa_depth_test.hpp"
static long long checked = 0, wrong = 0, open_cases = 0;
static void check(float hd, float d, float n, float f, float thr) {
    const float nf = n * f, q1 = f + hd * (n - f), q2 = f + d * (n - f);
    const bool want = std::fabs(nf / q1 - nf / q2) > thr;
    const float k = thr * (1.0f / std::fabs(nf));
    const float ks[] = {k, k * (1.0f + 0x1p-22f), k * (1.0f - 0x1p-22f)};
    for (float kk : ks) {
        const int r = taastar::linear_depth_decided(q1, q2, kk);
        ++checked;
        if (r < 0) ++open_cases;
        else if ((r != 0) != want) ++wrong;
    }
}
int main() {
    std::mt19937_64 g(1);
    const float planes[][2] = {{0.1f, 100.0f}, {0.01f, 1000.0f}, {1.0f, 50.0f}, {0.5f, 1e6f}, {-0.1f, 100.0f}};
    const float thrs[] = {0.01f, 1e-4f, 1.0f, 1e-7f};
    std::uniform_real_distribution<float> u(0.0f, 1.0f);
    for (auto& p : planes)
        for (float thr : thrs) {
            const float n = p[0], f = p[1];
            for (int i = 0; i < 200000; ++i) {
                const float d = i & 1 ? u(g) : 1.0f - u(g) * u(g) * 0.01f;
                check(d, u(g), n, f, thr);
                check(d, d, n, f, thr);
                // the depth whose linear depth is thr away, and its neighbours
                const double L = (double)n * f / (f + (double)d * (n - f));
                for (double s : {-1.0, 1.0}) {
                    const double e = ((double)n * f / (L + s * thr) - f) / ((double)n - f);
                    float h = (float)e;
                    for (int k = -3; k <= 3; ++k) {
                        float x = h;
                        for (int j = 0; j < std::abs(k); ++j) x = std::nextafterf(x, k < 0 ? -1e30f : 1e30f);
                        check(x, d, n, f, thr);
                    }
                }
            }
            const float odd[] = {0.0f, -0.0f, 1.0f, f / (f - n), INFINITY, -INFINITY, NAN, 1e30f, -1e30f, 1e-40f, 2.0f, -1.0f};
            for (float a : odd)
                for (float b : odd) check(a, b, n, f, thr);
        }
    printf("%lld %lld\n", checked, wrong);
    checked = wrong = open_cases = 0;
    for (int i = 0; i < 1000000; ++i) check(u(g), u(g), 0.1f, 100.0f, 0.01f);
    printf("%lld %lld %lld\n", checked, wrong, open_cases);
    return 0;
}
"""


def test_decisions_equal_the_divisions(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    src = tmp_path / "depth.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "depth"
    subprocess.run([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-D__HIP_PLATFORM_AMD__", "-I" + CSRC,
                    "-I" + os.path.join(ROCM, "include"), str(src), "-o", str(exe)], check=True)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    checked, wrong = map(int, lines[0].split())
    assert checked > 10_000_000 and wrong == 0
    checked, wrong, undecided = map(int, lines[1].split())
    assert wrong == 0 and undecided < checked // 1000
