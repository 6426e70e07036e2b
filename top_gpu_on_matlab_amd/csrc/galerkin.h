// Galerkin coarse-stiffness core of the MEX entry points:
//   Kout = sum_s  B_s^T * Kch_s * B_s      (24 x 24, FP32/FP64)
// One workgroup per coarse element, its children dealt to its WAVES wavefronts in turn and their sums added in
// wavefront order; lane t of a wavefront owns the 3x3 block (rows 3*(t%8).., cols 3*(t/8)..) of a product.  B
// (row-major) and Kch (column-major), then T = Kch*B (row-major), are the wavefront's own LDS, so it never
// waits for the others.  Every product runs over k = 0..23 in order.  Bound by a child's chain of loads and two
// products out of LDS where there are few elements (1,024 of 8 children: 31 us, from 51 with one wavefront for all of
// them), by LDS reads where there are many.
#pragma once

#include <hip/hip_runtime.h>

namespace tg {

// LDS written by this wavefront is read by it: the hardware keeps one wavefront's LDS accesses in order, this
// keeps the compiler's.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T, int WAVES>
struct GalerkinLds {
    T B[WAVES][576], K[WAVES][576];
};

// Src must provide:
//   __device__ int child(int s) const;              // < 0: skip child s
//   __device__ void kch(int f, int t, T (&k)[9]) const;  // entries 64 j + t (= r + 24c) of the child's matrix
// ADD: to what Kout holds.
template <bool ADD, int WAVES, typename T, class Src>
__device__ inline void galerkin_block(T *__restrict__ Kout, const Src &src, int nCh, const T *__restrict__ P,
                                      GalerkinLds<T, WAVES> &lds) {
    const int t = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rb = 3 * (t & 7), cb = 3 * (t >> 3);
    T *sB = lds.B[w], *sK = lds.K[w];
    T acc[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) acc[i] = (T)0;
    // this wavefront's children: every WAVES-th of those there are, looked up 64 at a time
    int turn = 0, s0 = -64, mine = -1;
    unsigned long long left = 0;
    auto next = [&](int &s, int &f) {
        for (;;) {
            while (left == 0) {
                s0 += 64;
                if (s0 >= nCh) return false;
                mine = s0 + t < nCh ? src.child(s0 + t) : -1;
                left = __ballot(mine >= 0);
            }
            const int l = __ffsll(left) - 1;
            left &= left - 1;
            if (turn++ % WAVES != w) continue;
            s = s0 + l;
            f = __builtin_amdgcn_readlane(mine, l);
            return true;
        }
    };
    T pv[9], kv[9];  // the next child's B and Kch, in flight while this one's products run
    auto fetch = [&](int s, int f) {
#pragma unroll
        for (int k = 0; k < 9; ++k) pv[k] = P[(size_t)s * 576 + 64 * k + t];
        src.kch(f, t, kv);
    };
    int s, f;
    bool more = next(s, f);
    if (more) fetch(s, f);
    while (more) {  // uniform over the wavefront
        wave_sync();  // the last child's B and T have been read
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const int i = 64 * k + t, r = i % 24, c = i / 24;
            sB[r * 24 + c] = pv[k];
            sK[i] = kv[k];
        }
        more = next(s, f);
        if (more) fetch(s, f);
        wave_sync();
        T tb[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) tb[i] = (T)0;
#pragma unroll
        for (int k = 0; k < 24; ++k) {
            const T k0 = sK[rb + 0 + 24 * k], k1 = sK[rb + 1 + 24 * k], k2 = sK[rb + 2 + 24 * k];
            const T b0 = sB[k * 24 + cb + 0], b1 = sB[k * 24 + cb + 1], b2 = sB[k * 24 + cb + 2];
            tb[0] += k0 * b0; tb[1] += k0 * b1; tb[2] += k0 * b2;
            tb[3] += k1 * b0; tb[4] += k1 * b1; tb[5] += k1 * b2;
            tb[6] += k2 * b0; tb[7] += k2 * b1; tb[8] += k2 * b2;
        }
        wave_sync();  // Kch has been read: T takes its place
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) sK[(rb + i) * 24 + cb + j] = tb[3 * i + j];
        wave_sync();
        T ub[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) ub[i] = (T)0;
#pragma unroll
        for (int k = 0; k < 24; ++k) {
            const T b0 = sB[k * 24 + rb + 0], b1 = sB[k * 24 + rb + 1], b2 = sB[k * 24 + rb + 2];
            const T t0 = sK[k * 24 + cb + 0], t1 = sK[k * 24 + cb + 1], t2 = sK[k * 24 + cb + 2];
            ub[0] += b0 * t0; ub[1] += b0 * t1; ub[2] += b0 * t2;
            ub[3] += b1 * t0; ub[4] += b1 * t1; ub[5] += b1 * t2;
            ub[6] += b2 * t0; ub[7] += b2 * t1; ub[8] += b2 * t2;
        }
#pragma unroll
        for (int i = 0; i < 9; ++i) acc[i] += ub[i];
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < 9; ++i) sK[64 * i + t] = acc[i];
    __syncthreads();
    for (int o = threadIdx.x; o < 576; o += 64 * WAVES) {  // entry r + 24 c
        const int r = o % 24, c = o / 24, at = 64 * (3 * (r % 3) + c % 3) + r / 3 + 8 * (c / 3);
        T v = lds.K[0][at];
        for (int k = 1; k < WAVES; ++k) v += lds.K[k][at];
        Kout[o] = ADD ? Kout[o] + v : v;
    }
}

}  // namespace tg
