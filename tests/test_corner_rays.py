"""Host-side test of the corner rays by which the 3D forward bounds a workgroup's samples
(curadon_amd/csrc/geometry3d.hpp, line_on_planes): the header is compiled with the host C++ compiler,
and for blocks of 16 x 16 panel pixels, at sources near and far, every FP32 sample position must lie
between the four corner rays' FP32 crossings of its slice, a quarter of the staged boxes' margin of
1/16 voxel aside."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "curadon_amd", "csrc")

PROGRAM = r"""
#include "geometry3d.hpp"
#include <algorithm>
#include <cstdio>
#include <vector>
using namespace cmi::cone3d;
int main() {
    const double PAD = 2.0;
    double worst = 0.0, wnear = 0.0;
    long checked = 0;
    const double sources[] = {1.3, 3.0, 1e3, 4e3, 1e4, 1.7e4, 1e6};   // in volume edges
    for (double far : sources)
        for (int t = 0; t < 6; ++t) {
            Desc g{};
            const int n = 256, U = 384;
            g.nx = n, g.ny = n, g.nz = n, g.nu = U, g.nv = U;
            g.sx = g.sy = g.sz = 1.0, g.du = g.dv = 1.0;
            g.dso = far * n, g.dsd = g.dso * 1.5;
            if (far > 100.0) g.dsd = g.dso + 300.0;
            const FwdGeom a = fwd_angle(g, 0.3 + 1.1 * t, 0.05 * t, 0.02 * t);
            for (int iv0 = 0; iv0 < U; iv0 += 48)
                for (int iu0 = 0; iu0 < U; iu0 += 48) {
                    double dir[3] = {0, 0, 0};
                    for (int c = 0; c < 4; ++c)
                        for (int d = 0; d < 3; ++d)
                            dir[d] += a.org[d] + (iu0 + 15 * (c & 1)) * a.du[d] +
                                      (iv0 + 15 * (c >> 1)) * a.dv[d] - a.src[d];
                    int K = 0;
                    for (int d = 1; d < 3; ++d)
                        if (std::fabs(dir[d]) > std::fabs(dir[K])) K = d;
                    const double c0 = (n + 4) / 2;   // centre of the padded volume
                    float at[4][3], slope[4][3];
                    for (int c = 0; c < 4; ++c)
                        for (int d = 0; d < 3; ++d) {
                            if (d == K) continue;
                            double p, s;
                            line_on_planes(a, iu0 + 15 * (c & 1), iv0 + 15 * (c >> 1), K, d,
                                           c0 - PAD, p, s);
                            at[c][d] = (float)(p + PAD - c0), slope[c][d] = (float)s;
                        }
                    for (int r = 0; r < 256; r += 5) {
                        const Ray3 q = setup_ray3(a, n, n, n, iu0 + r / 16, iv0 + r % 16);
                        if (!q.hit) continue;
                        const int64_t im = q.nst / 2;
                        const double tm = q.tmin + (double)im * q.dt;
                        float m[3], st[3];
                        for (int d = 0; d < 3; ++d) {
                            m[d] = (float)(q.s[d] + tm * q.d[d] + PAD - c0);
                            st[d] = (float)(q.dt * q.d[d]);
                        }
                        for (int e = 0; e <= 8; ++e) {
                            const float j = (float)(-im + q.nst * e / 8);
                            const float k = std::fma(j, st[K], m[K]);
                            for (int d = 0; d < 3; ++d) {
                                if (d == K) continue;
                                const float p = std::fma(j, st[d], m[d]);
                                float lo = INFINITY, hi = -INFINITY;
                                for (int c = 0; c < 4; ++c) {
                                    const float x = std::fma(k, slope[c][d], at[c][d]);
                                    lo = std::min(lo, x), hi = std::max(hi, x);
                                }
                                const double out = std::max(lo - p, p - hi);
                                worst = std::max(worst, out);
                                if (far < 100.0) wnear = std::max(wnear, out);
                                ++checked;
                            }
                        }
                    }
                }
        }
    std::printf("checked %ld worst %.3g (near sources %.3g)\n", checked, worst, wnear);
    return !(checked > 100000 && worst < 0.0625 / 4);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_samples_between_corner_rays(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "t"
    subprocess.run(["g++", "-std=c++17", "-O2", "-w", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I", CSRC, "-isystem", "/opt/rocm/include", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
