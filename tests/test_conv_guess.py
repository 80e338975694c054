"""The implicit fp32 convolution's scale guess reads inside its pixel.

vla.simd_amd/csrc/convgeom.h holds the offset that the kernel uses; here a host
program walks every output pixel and channel lane of small convolutions (both
slab widths, maps whose last pixel is a patch's centre) and checks each offset:
four channels of the centre pixel, or none.
"""

import os
import shutil
import subprocess

import pytest

from helpers import ROOT

PROGRAM = r"""
#include "convgeom.h"
#include <cstdio>
#include <initializer_list>
using namespace vla::hip;
int main() {
    long reads = 0, last = 0;
    for (int cin : {32, 64, 96, 128}) for (int slab : {32, 64}) for (int k : {1, 3, 5}) for (int stride : {1, 2, 3})
    for (int pad = 0; pad <= k / 2; pad++) for (int h = k; h < 14; h++) for (int w = k; w < 14; w++) {
        const int wo = (w + 2 * pad - k) / stride + 1, ho = (h + 2 * pad - k) / stride + 1;
        const ConvGeom cg{h, w, cin, k, stride, pad, wo};
        for (int m = 0; m < ho * wo; m++) for (int kq = 0; kq < slab; kq += 4) {
            const int iy = m / wo * stride, ix = m % wo * stride;  // patch origin + pad
            const int o = guess_offset(cg, iy, ix, kq);
            if (o < 0) continue;
            reads++;
            if (o + 4 > h * w * cin) { std::printf("past the map: %d of %d\n", o, h * w * cin); return 1; }
            if (o / cin != iy * w + ix || (o + 3) / cin != iy * w + ix) { std::puts("another pixel"); return 1; }
            last += o + 4 == h * w * cin;
        }
    }
    std::printf("%ld %ld\n", reads, last);
    return reads > 0 && last > 0 ? 0 : 1;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_guess_stays_in_its_pixel(tmp_path):
    src = tmp_path / "guess.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "guess"
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{os.path.join(ROOT, 'vla.simd_amd', 'csrc')}", str(src), "-o", str(exe)],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
