"""The exchange that gives the 16 lanes of a droplet the heights of its stencil
(hg_stencil.hpp), run on the host with lanes that are an array: whatever the
lanes loaded, all of them must go on with the same four heights, the sums of
rock and dirt that lanes 0-7 loaded."""
from __future__ import annotations

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#define __device__
#define __forceinline__ inline
#include "hg_stencil.hpp"
struct V {
    float l[16];
};
V operator+(const V& a, const V& b) {
    V c;
    for (int g = 0; g < 16; ++g) c.l[g] = a.l[g] + b.l[g];
    return c;
}
struct Lanes {
    static V other_layer(const V& v) {
        V r;
        for (int g = 0; g < 16; ++g) r.l[g] = v.l[g ^ 1];
        return r;
    }
    template <int L>
    static V lane(const V& v) {
        V r;
        for (int g = 0; g < 16; ++g) r.l[g] = v.l[L];
        return r;
    }
};
int main() {
    // powers of two: a sum says which lanes it is of; the second copies of the
    // cells (lanes 8-15) were loaded with them, or after a change
    for (int changed = 0; changed < 2; ++changed) {
        V v, h[4];
        for (int g = 0; g < 16; ++g) v.l[g] = float(1 << (changed ? g : g & 7));
        hgk::corner_heights<Lanes>(v, h[0], h[1], h[2], h[3]);
        for (int c = 0; c < 4; ++c)
            for (int g = 0; g < 16; ++g)
                if (h[c].l[g] != float(3 << (2 * c))) {
                    std::printf("lane %d of corner %d: %g\n", g, c, h[c].l[g]);
                    return 1;
                }
    }
    return 0;
}
"""


def test_lanes_of_a_droplet_share_their_heights(tmp_path):
    src, exe = tmp_path / "stencil.cpp", tmp_path / "stencil"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "hydro-gen_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0, p.stdout
