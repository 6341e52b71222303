"""What the list count pass decides about a lane's sixteen products, on the
host: csrc/sph_count.h is compiled with the host compiler and run over
destinations and candidates with a NaN of either sign or an infinity in each
component, particles clamped into the grid, radii that are NaN or far above the
reach, ordinary pairs on and beside the radius, and cells from 2^-200 to 2^200 (in
single precision where its squares under- and overflow).  The hits must be the
predicate's for the candidates that exist, and none for the others."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pysph_amd",
                    "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <random>
#include "sph_count.h"

struct P { double x, y, z; };
static uint32_t word(float f) { uint32_t r; memcpy(&r, &f, 4); return r; }

// the kernel's preparation (a cell of size cs around the origin) and tile of one
// destination and sixteen candidates, `left` of which exist
template <typename T = double>
static int wrong(P d, double radius, const P *c, int left, int reach, double cs = 1.0)
{
    const double inv_cs = nn_cell_size(cs) ? 1.0 / cs : NAN, rr = radius * inv_cs;
    const float inv = (float)inv_cs;
    const float lim = (float)reach + 0.75f, band = NN_BAND * (float)((reach + 1) * (reach + 1));
    const float x = (float)d.x * inv, y = (float)d.y * inv, z = (float)d.z * inv;
    const bool odd = !nn_regular(x, y, z, (float)rr, lim);
    float B[4] = {-2.0f * x, -2.0f * y, -2.0f * z, 1.0f};
    float C = (float)((double)x * x + (double)y * y + (double)z * z - rr * rr);
    if (odd) B[0] = B[1] = B[2] = C = 0.0f;
    bool far = false;
    float D[4][4], near = NN_FAR;
    uint32_t bits = 0;
    for (int e = 15; e >= 0; --e) {
        float A[4] = {0.0f, 0.0f, 0.0f, NN_FAR};
        if (e < left) {
            A[0] = (float)c[e].x * inv, A[1] = (float)c[e].y * inv, A[2] = (float)c[e].z * inv;
            far |= !nn_inside(A[0], A[1], A[2], lim);
            A[3] = fmaf(A[0], A[0], fmaf(A[1], A[1], A[2] * A[2]));
        }
        float s = C;
        for (int k = 0; k < 4; ++k) s = fmaf(A[k], B[k], s);
        D[e >> 2][e & 3] = s;
        bits = bits << 1 | word(s) >> 31;
        near = fminf(near, fabsf(s));
    }
    const bool all = odd || far;
    auto hit = [&](int e) {
        const T ex = T(c[e].x) - T(d.x), ey = T(c[e].y) - T(d.y), ez = T(c[e].z) - T(d.z);
        return ex * ex + ey * ey + ez * ez < T(radius) * T(radius);
    };
    if (all || near < band) bits = nn_decide(bits, D, band, all, C == NN_FAR, left, hit);
    uint32_t want = 0;
    for (int e = 0; e < left; ++e) want |= (uint32_t)hit(e) << e;
    return bits != want;
}

int main()
{
    std::mt19937 rng(3);
    std::uniform_real_distribution<double> in(-0.5, 0.5), around(-1.5, 1.5);
    std::uniform_int_distribution<int> some(0, 16), grid(-96, 96);
    const double bad[] = {NAN, -NAN, INFINITY, -INFINITY, 50.0, -1e30, 1e200};
    const double radii[] = {NAN, -NAN, INFINITY, 1e17, 1e200, 0.0, -0.5};
    const int powers[] = {-200, -150, -131, -127, -61, -60, 59, 60, 127, 131, 150, 200};
    int w[6] = {0, 0, 0, 0, 0, 0};
    for (int it = 0; it < 4000; ++it) {
        P c[16];
        for (P &p : c) p = {around(rng), around(rng), around(rng)};
        const P d = {in(rng), in(rng), in(rng)};
        const int left = some(rng);
        w[0] += wrong(d, 1.0, c, left, 1);
        for (double v : bad)
            for (int k = 1; k < 8; ++k) {  // every choice of components
                P q = d;
                if (k & 1) q.x = v;
                if (k & 2) q.y = v;
                if (k & 4) q.z = v;
                w[1] += wrong(q, 1.0, c, left, 1);
                P s[16];
                memcpy(s, c, sizeof(s));
                if (k & 1) s[it % 16].x = v;
                if (k & 2) s[it % 16].y = v;
                if (k & 4) s[it % 16].z = v;
                w[2] += wrong(d, 1.0, s, left, 1);
            }
        for (double r : radii) w[3] += wrong(d, r, c, left, 1);
        for (int k : powers) {
            const double cs = ldexp(1.37, k);
            P s[16];
            for (int e = 0; e < 16; ++e) s[e] = {c[e].x * cs, c[e].y * cs, c[e].z * cs};
            w[4] += wrong({d.x * cs, d.y * cs, d.z * cs}, cs, s, left, 1, cs);
        }
        for (int k : {-75, -70, -66, -61, -60, 59, 60, 63, 66}) {
            const double cs = (float)ldexp(1.37, k);
            auto f = [&](double v) { return (double)(float)(v * cs); };
            P s[16];
            for (int e = 0; e < 16; ++e) s[e] = {f(c[e].x), f(c[e].y), f(c[e].z)};
            w[5] += wrong<float>({f(d.x), f(d.y), f(d.z)}, cs, s, left, 1, cs);
        }
        for (P &p : c) p = {grid(rng) / 64.0, grid(rng) / 64.0, 0.0};  // many at the radius
        w[0] += wrong({it % 64 / 64.0 - 0.5, 0.0, 0.0}, 1.0, c, left, 1);
    }
    for (int k : w) printf("%d ", k);
    return 0;
}
"""


def test_hits_are_the_predicates_and_only_of_candidates_that_exist(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "count.cpp", tmp_path / "count"
    src.write_text(PROGRAM)
    subprocess.check_call([gxx, "-std=c++17", "-O1", "-ffp-contract=off", "-Wno-unknown-pragmas",
                           "-D__host__=", "-D__device__=", "-D__forceinline__=inline", "-I", CSRC,
                           str(src), "-o", str(exe)])
    wrong = subprocess.check_output([str(exe)], text=True).split()
    # ordinary pairs; destinations outside; candidates outside; radii; cell sizes,
    # in double and in single precision
    assert wrong == ["0"] * 6
