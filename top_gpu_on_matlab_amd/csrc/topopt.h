// Device objects of the optimisation layer (see topopt.hip).
#pragma once

#include "kernels.h"
#include "model.h"
#include "pcg.h"

namespace tg {

// Nodal Helmholtz (PDE) density filter on the finest grid.
struct Filter {
    const tg_model &m;
    hipStream_t st;
    Grid g{};
    int64_t Ne = 0;
    double kd[4] = {};           // the element matrix: entries between corners 0, 1, 2 and 3 edges apart
    DevBuf<double> inv, y, parts;  // the preconditioner per set of solid elements around a node; the iterate; partial sums
    DevBuf<uint8_t> code;        // the solid elements around each node
    DevBuf<int32_t> eleFwd, eleFull0;
    int ty = 0, tx = 0, tyn = 0, tiles = 0, chunk = 0, chunks = 0, np = 0;  // k_filter_step's tiles; partials of a sum
    PcgWork pw;
    Filter(const tg_model &mm, double rMin, hipStream_t s);
    void apply(const double *src, double *tar, double tol, int maxIT, int *its, double *res);
};

// imfilter density filter of super-element mode on the num-times refined voxel grid.
struct ConvFilter {
    int num, X = 0, Y = 0, Z = 0, GY = 0, GX = 0, GZ = 0, hr = 0;
    hipStream_t st;
    DevBuf<double> hd, Hs;       // weights (one octant), their sums on the grid
    DevBuf<int32_t> lim;         // last dy with a weight, per (dx, dz)
    int LY = 0, LX = 0, pitch = 0;  // lanes along y and x of k_conv's workgroups, LDS column stride (LY = 0: another form)
    ConvFilter(int nelx, int nely, int nelz, double r, int n, hipStream_t s);
    void forward(const double *x, double *out);
    void adjoint(const double *dc, double *out);
    template <int MODE>
    void convolve(const double *src, double *out);
};

}  // namespace tg

struct tg_filter {
    tg::Filter *f = nullptr;
};

struct tg_convfilter {
    tg::ConvFilter *f = nullptr;
};
