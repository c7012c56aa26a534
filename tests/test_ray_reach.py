"""The bound by which ray walks drop stacked nodes, against the leaf test itself: compiled for
the host from the kernels' own header."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include "qr_geom.h"
#include <cstdio>
#include <random>
using namespace qr;
int main() {
    std::mt19937 g(1);
    auto U = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(g); };
    long hits = 0, beyond = 0, slack = 0;
    for (long i = 0; i < 4000000; ++i) {
        const double size = i % 2 ? 1000.0 : 30.0, flat = 1e-4;  // grazing: triangles nearly along the ray
        const double cx = U(-size, size), cy = U(-size, size), cz = U(-size, size);
        auto V = [&] { return V3{float(cx + U(-1, 1)), float(cy + U(-1, 1)), float(cz + flat * U(-1, 1))}; };
        Tri t;
        t.a = V();
        t.b = V();
        t.c = V();
        const float w = float(U(0, 1)), u = float(U(0, 1 - w));
        const V3 h = add(t.a, add(scale(sub(t.b, t.a), w), scale(sub(t.c, t.a), u)));
        Ray r;
        r.origin = {float(U(-2 * size, 2 * size)), float(U(-2 * size, 2 * size)), float(h.z + flat * U(-1, 1))};
        r.dir = sub(h, r.origin);
        r.dir = scale(r.dir, 1.0f / sqrtf(dot(r.dir, r.dir)));
        r.tMin = 1e-6f;
        r.tMax = kInf;
        float hit, enter;
        if (!rayTri(r, t, hit) || !rayBoxPre(rayPrepare(r), triBounds(t), kInf, enter)) continue;
        ++hits;
        beyond += enter > rayReach(hit);
        slack += enter > hit * (1.0f + 1e-6f) + 1e-6f;
    }
    std::printf("%ld %ld %ld\n", hits, beyond, slack);
}
"""


def test_hits_lie_within_reach_of_their_box(tmp_path):
    """A hit the leaf test takes is never behind a box entry beyond rayReach(hit): a node with
    such an entry may still hold the hit, or an equal one with a smaller index."""
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "reach.hip", tmp_path / "reach"
    src.write_text(PROGRAM)
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "quarry-gpu_amd", "csrc"), "-x", "hip", str(src), "-o", str(exe)],
                   check=True, capture_output=True, timeout=120)
    hits, beyond, slack = map(int, subprocess.run([str(exe)], check=True, capture_output=True, text=True,
                                                  timeout=120).stdout.split())
    assert hits > 2_000_000
    assert beyond == 0
    assert slack > 0  # (a single slack, as the walks once used, is too short)
