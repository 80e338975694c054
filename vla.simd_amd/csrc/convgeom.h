// convgeom.h - index arithmetic of the implicit fp32 convolution, shared with
// host code that checks it.
#pragma once

#ifdef __HIPCC__
#define VLA_HOST_DEVICE __host__ __device__
#else
#define VLA_HOST_DEVICE
#endif

namespace vla {
namespace hip {

// an NHWC map [H, Wd, Cin], its k x k patches and the output's width
struct ConvGeom {
    int H, Wd, Cin, k, stride, pad, Wout;
};

// Where in the map a thread reads its four values of pixel (iy, ix) for the
// guess of a row's scale, kq (a multiple of 4) channels in; -1: nowhere. A slab
// may be wider than a pixel (64 channels on maps of 32).
VLA_HOST_DEVICE inline int guess_offset(const ConvGeom& cg, int iy, int ix, int kq) {
    return kq < cg.Cin && iy >= 0 && iy < cg.H && ix >= 0 && ix < cg.Wd ? (iy * cg.Wd + ix) * cg.Cin + kq : -1;
}

}  // namespace hip
}  // namespace vla
