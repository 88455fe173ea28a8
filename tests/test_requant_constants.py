"""The constants of every form of the requantisation (epilogue.h, modes 1 to 6) against the reference's literal sequence, on the host:
the library's own search, its results evaluated with the device's instructions written out in plain C++ (a fused multiply-add is fmaf, the
conversion to an unsigned byte rounds to even and saturates), on both sides of every step of the output, around them, at the ends of the
accumulators' range and on random ones. Mode 5, the sums that start as floats, among them: within 2^22 its sums are whole floats, beyond
it only their order counts. Every scale for which there is a threshold table has at least one form."""
import os
import subprocess

import pytest

import megcc_amd

CLANG = "/opt/rocm/llvm/bin/clang++"
LIB = os.path.join(os.path.dirname(megcc_amd.__file__), "libmegcc_gfx950.so")

PROGRAM = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <random>
#include <vector>
namespace mg {
struct RequantPack { float s1, s2, c, d; int mode; };
struct RequantAffine { float c, d; };
RequantPack requant_pack_for(int, float, float, float, bool);
RequantPack requant_shifted_for(int, float, float, float);
RequantPack requant_started_for(int, float, float, float, bool);
}
using namespace mg;
enum { IDENTITY, RELU, H_SWISH };
static int literal(int act, int a, float s, float f, float d) {
    float v = (float)a * s * f / d;
    if (act == RELU) v = v > 0 ? v : 0;
    if (act == H_SWISH) { float t = v + 3; t = t > 0 ? t : 0; t = t > 6 ? 6 : t; v = v * t * (1.f / 6.f); }
    const float r = roundf(v);
    return r > 127 ? 127 : r < -128 ? -128 : (int)r;
}
static int clamp8(float t) { return t > 127 ? 127 : t < -128 ? -128 : (int)t; }
static int byte_of(int act, float y) {
    const float r = nearbyintf(y);
    const int u = r < 0 ? 0 : r > 255 ? 255 : (int)r;
    return act == IDENTITY ? u - 128 : u >> 1;
}
static const float HALF = 0x1.fffffep-2f;
static int form(int act, int a, const RequantPack& q) {
    float x = (float)a;
    switch (q.mode) {
        case 1: return byte_of(act, fmaf(x, q.c, q.d));
        case 2: return byte_of(act, fmaf(x * q.s1 * q.s2, q.c, q.d));
        case 3: {
            x = x * q.s1 * q.s2;
            float v = fmaf(x, q.c, x * q.d);
            if (act == IDENTITY) return clamp8(truncf(v + copysignf(HALF, v)));
            if (act == H_SWISH) v = v * std::min(std::max(v + 3, 0.f), 6.f) * (2.f * (1.f / 6.f));
            return byte_of(act, v + HALF);
        }
        case 4: return clamp8(floorf(fmaf(x, q.c, q.d)));
        case 5: {
            // (as requant_bias() starts the sums; the rest of the sum is 0 here)
            int bits, start = a > 1 << 29 ? 1 << 29 : a < -(1 << 29) ? -(1 << 29) : a;
            memcpy(&bits, &q.s1, 4);
            bits += start;
            memcpy(&x, &bits, 4);
            return byte_of(act, fmaf(x, q.c, q.d));
        }
        case 6: x = x * q.s1 * q.s2; return clamp8(truncf(fmaf(x, q.c, copysignf(q.d, x))));
    }
    return 1000;
}
int main() {
    std::mt19937 r(5);
    std::uniform_real_distribution<float> near1(0.8f, 1.2f), small(-7.f, 1.f);
    const float grid[] = {0.5f, 0.25f, 0.1f, 0.05f, 0.02f, 0.01f, 1.f / 127, 0.003f};
    long modes[7] = {}, shifted = 0, none = 0;
    for (int i = 0; i < 900; ++i) {
        float s, f, d;
        if (i % 3 == 0) {  // calibrated layers of 9 to 8192 products
            s = 0.02f * near1(r), f = 0.01f * near1(r), d = s * f * 150.f * sqrtf(9.f * powf(2.f, (float)(i / 3 % 11))) * near1(r);
        } else if (i % 3 == 1) {  // ties
            s = grid[r() % 8], f = grid[r() % 8], d = grid[r() % 8];
        } else {  // ratios down to the smallest that a table is built for
            const float c = std::max(powf(10.f, small(r)), 4.8e-7f);
            s = powf(10.f, small(r) / 2), f = powf(10.f, small(r) / 2), d = s * f / c;
        }
        for (int act : {IDENTITY, RELU, H_SWISH}) {
            const RequantPack forms[] = {requant_pack_for(act, s, f, d, true), requant_pack_for(act, s, f, d, false), requant_shifted_for(act, s, f, d),
                                         requant_started_for(act, s, f, d, true)};
            none += !forms[0].mode + !forms[1].mode + !forms[3].mode;
            if (!forms[1].mode)
                printf("no form: act %d %a %a %a\n", act, s, f, d);
            if (forms[1].mode && forms[1].mode != 3)
                return printf("mode %d without multiply-adds\n", forms[1].mode), 1;
            shifted += forms[2].mode == 5;
            const double c = (double)s * f / d;
            std::vector<int> acc = {INT32_MIN, INT32_MAX, 0, 1, -1, (1 << 29) + 1, -(1 << 29) - 1};
            auto add = [&](double a) { if (a > -2147483648. && a < 2147483647.) acc.push_back((int)a); };
            for (int k = -129; k <= 129; ++k) {
                double v = k - 0.5;
                if (act == H_SWISH && v > 0 && v < 3) v = 0.5 * (sqrt(9 + 24 * v) - 3);
                for (int e = -3; e <= 3; ++e) add(floor(v / c) + e);
                add(floor((v + 5e-6 * v) / c)), add(floor((v - 5e-6 * v) / c));
            }
            for (int e = 0; e < 200; ++e) add((double)(int)r() / (1 << r() % 20));
            for (const RequantPack& q : forms) {
                if (!q.mode) continue;
                ++modes[q.mode];
                for (int a : acc) {
                    const double scaled = fabs((double)a * c);
                    if (scaled >= 2147483648.) continue;  // (the reference's conversion is undefined)
                    if (form(act, a, q) != literal(act, a, s, f, d))
                        return printf("mode %d act %d scales %a %a %a accumulator %d: %d, not %d\n", q.mode, act, s, f, d, a, form(act, a, q),
                                      literal(act, a, s, f, d)), 1;
                }
            }
        }
    }
    printf("none %ld shifted %ld modes", none, shifted);
    for (int m = 1; m < 7; ++m) printf(" %ld", modes[m]);
    printf("\n");
    return 0;
}
"""


@pytest.fixture(scope="module")
def result(tmp_path_factory):
    if not os.path.exists(CLANG) or not os.path.exists(LIB):
        pytest.skip("needs ROCm's clang++ and the built library")
    folder = tmp_path_factory.mktemp("requant")
    src, exe = folder / "constants.cpp", str(folder / "constants")
    src.write_text(PROGRAM)
    subprocess.check_call([CLANG, "-std=c++17", "-O2", "-ffp-contract=off", str(src), "-o", exe, LIB, "-Wl,-rpath," + os.path.dirname(LIB)])
    return subprocess.run([exe], capture_output=True, text=True, timeout=600)


def test_every_form_gives_the_reference_s_outputs(result):
    assert result.returncode == 0, result.stdout[-500:] + result.stderr[-500:]
    counts = [int(n) for n in result.stdout.split("modes")[1].split()]
    assert all(n >= 40 for n in counts), result.stdout[-200:]  # (each form met)


def test_every_scale_with_a_table_has_a_form(result):
    assert " ".join(result.stdout.splitlines()[-1].split()[:2]) == "none 0", result.stdout[:500]
