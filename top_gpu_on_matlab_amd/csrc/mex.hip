// The six MEX entry points of the reference as C functions (mexFunction calling convention).
//
// Argument order, in-place contracts, class/shape checks and error identifiers follow the
// reference gateways; the kernels are this library's own deterministic gfx950 kernels:
//   * gather: one lane per element, coalesced column writes;
//   * scatter / scatter_accum3: a stable radix sort of (target row, entry) pairs, kept per
//     connectivity as a CSR incidence, then one lane per target row sums its entries in ascending
//     entry order (no floating-point atomics);
//   * Galerkin assembly: one workgroup per coarse element (galerkin.h); the FP64 level-2 entry uses the
//     product's linearity in the children moduli (a GEMM on the matrix cores) and recomputes only the
//     children that carry boundary matrices.
#include <cstring>
#include <memory>
#include <mutex>

#include "galerkin.h"
#include "kernels.h"
#include "scatter.h"
#include "scratch.h"

namespace tg {
namespace {

// ---- gather ----------------------------------------------------------------------------
template <typename T, typename IDX>
__global__ void k_gather(T *__restrict__ uMat, const T *__restrict__ u, const IDX *__restrict__ eNod, int64_t Ne,
                         int64_t Nn) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= Ne) return;
    int64_t node[8];
#pragma unroll
    for (int n = 0; n < 8; ++n) node[n] = (int64_t)eNod[e + Ne * n] - 1;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int n = 0; n < 8; ++n) {
            const bool ok = node[n] >= 0 && node[n] < Nn;
            uMat[e + Ne * (3 * n + c)] = ok ? u[node[n] + Nn * c] : (T)0;
        }
}

// Row pointers of a sorted key array: rowptr[r] = first position with key >= r, r = 0..M.
__global__ void k_rowptr(const uint32_t *__restrict__ skeys, int64_t N, int64_t M, uint32_t *__restrict__ rowptr) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > M) return;
    rowptr[r] = (uint32_t)lower_bound_u32(skeys, N, (uint32_t)r);
}

// The scatter kernels: a thread per row, which adds its entries in ascending order.  Bound by reading the entries'
// values; a row's chain is its bounds, its entry numbers and their values, so both are loaded in batches (past
// the row's end its last entry again: no branch between the loads).  Consecutive rows stay on one XCD, where they
// share the lines of their neighbours' entries.  ok (optional): nothing is added unless it holds 1 (k_hash_check).
// 14.2 million entries of 8 columns in FP64 98 us (447 MB, 4.5 TB/s; entry by entry 108), 3.5 million of a list in FP32
// 33 (38).

// Y(r, c) += sum of uMat(e, c + 3j) over the entries 8e + j of row r, CSR form.
template <typename T>
__global__ __launch_bounds__(256) void k_csr_scatter_enod(T *__restrict__ Y, int64_t M, const uint32_t *__restrict__ rowptr,
                                                          const uint32_t *__restrict__ ent, const T *__restrict__ uMat,
                                                          int64_t Ne, const uint32_t *__restrict__ ok) {
    constexpr int BATCH = 8;
    if (ok && *ok != 1) return;
    const int64_t r = (int64_t)xcd_contiguous((int)blockIdx.x, (int)gridDim.x) * 256 + threadIdx.x;
    if (r >= M) return;
    const uint32_t lo = rowptr[r], hi = rowptr[r + 1];
    if (hi == lo) return;
    T a0 = 0, a1 = 0, a2 = 0;
    for (uint32_t k0 = lo; k0 < hi; k0 += BATCH) {
        uint32_t en[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) en[k] = ent[min(k0 + k, hi - 1)];
        T v0[BATCH], v1[BATCH], v2[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            const T *u = uMat + (en[k] >> 3) + Ne * 3 * (en[k] & 7);
            v0[k] = u[0];
            v1[k] = u[Ne];
            v2[k] = u[2 * Ne];
        }
#pragma unroll
        for (int k = 0; k < BATCH; ++k)
            if (k0 + k < hi) {
                a0 += v0[k];
                a1 += v1[k];
                a2 += v2[k];
            }
    }
    Y[r] += a0;
    Y[r + M] += a1;
    Y[r + 2 * M] += a2;
}

// xF(r, c) += sum of Tmp(i, c) over the entries i of row r, CSR form.
template <typename T>
__global__ __launch_bounds__(256) void k_csr_scatter_list(T *__restrict__ xF, int64_t M, const uint32_t *__restrict__ rowptr,
                                                          const uint32_t *__restrict__ ent, int64_t N,
                                                          const T *__restrict__ Tmp, const uint32_t *__restrict__ ok) {
    constexpr int BATCH = 4;
    if (ok && *ok != 1) return;
    const int64_t r = (int64_t)xcd_contiguous((int)blockIdx.x, (int)gridDim.x) * 256 + threadIdx.x;
    if (r >= M) return;
    const uint32_t lo = rowptr[r], hi = rowptr[r + 1];
    if (hi == lo) return;
    T a0 = 0, a1 = 0, a2 = 0;
    for (uint32_t k0 = lo; k0 < hi; k0 += BATCH) {
        uint32_t en[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) en[k] = ent[min(k0 + k, hi - 1)];
        T v0[BATCH], v1[BATCH], v2[BATCH];
#pragma unroll
        for (int k = 0; k < BATCH; ++k) {
            v0[k] = Tmp[en[k]];
            v1[k] = Tmp[en[k] + N];
            v2[k] = Tmp[en[k] + 2 * N];
        }
#pragma unroll
        for (int k = 0; k < BATCH; ++k)
            if (k0 + k < hi) {
                a0 += v0[k];
                a1 += v1[k];
                a2 += v2[k];
            }
    }
    xF[r] += a0;
    xF[r + M] += a1;
    xF[r + 2 * M] += a2;
}

// Content hash of an int32 array, four entries at a time: the sum over the groups i of the folded 128-bit product of their
// two 64-bit words, each under a key of its own place (integer adds, so no order matters).  One multiply-fold and
// two keys a group, three loads in flight: bound by reading the array: 14.2 million
// entries 18 us, where a mixed multiplier an entry took 43.
constexpr int HASH_BLOCKS = 2048;  // partial sums, in a call's working memory
static_assert(HASH_BLOCKS + 16 <= SCRATCH_DOUBLES, "the hash's partial sums");

template <bool WIDE>  // WIDE: the array is aligned to 16 bytes
__global__ __launch_bounds__(256) void k_hash_i32(const int32_t *__restrict__ a, int64_t n,
                                                  unsigned long long *__restrict__ parts) {
    __shared__ unsigned long long part[256];
    const int64_t groups = (n + 3) / 4, stride = (int64_t)gridDim.x * 256;
    auto get = [&](int64_t i) {
        if (WIDE && 4 * i + 4 <= n) return ((const int4 *)a)[i];
        int4 v;
        v.x = 4 * i < n ? a[4 * i] : 0;
        v.y = 4 * i + 1 < n ? a[4 * i + 1] : 0;
        v.z = 4 * i + 2 < n ? a[4 * i + 2] : 0;
        v.w = 4 * i + 3 < n ? a[4 * i + 3] : 0;
        return v;
    };
    auto fold = [&](int64_t i, const int4 &v) {
        const uint64_t x = ((uint64_t)i + 1) * 0x9E3779B97F4A7C15ull, y = ((uint64_t)i + 1) * 0xBF58476D1CE4E5B9ull + (uint64_t)n;
        const uint64_t p = ((uint64_t)(uint32_t)v.x | (uint64_t)(uint32_t)v.y << 32) ^ x ^ (x >> 31);
        const uint64_t q = ((uint64_t)(uint32_t)v.z | (uint64_t)(uint32_t)v.w << 32) ^ y ^ (y >> 29);
        return (p * q) ^ __umul64hi(p, q);
    };
    unsigned long long h = 0;
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    for (; i + 2 * stride < groups; i += 3 * stride) {
        const int4 v0 = get(i), v1 = get(i + stride), v2 = get(i + 2 * stride);
        h += fold(i, v0) + fold(i + stride, v1) + fold(i + 2 * stride, v2);
    }
    for (; i < groups; i += stride) h += fold(i, get(i));
    part[threadIdx.x] = h;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) parts[blockIdx.x] = part[0];
}

// The sum of the partial hashes to the host, and whether it is the expected one to the kernels behind.
__global__ __launch_bounds__(256) void k_hash_check(const unsigned long long *__restrict__ parts, int nb,
                                                    unsigned long long expected, uint32_t *__restrict__ ok,
                                                    unsigned long long *__restrict__ host, unsigned long long *seq_ptr,
                                                    unsigned long long seq) {
    __shared__ unsigned long long part[256];
    unsigned long long h = 0;
    for (int i = threadIdx.x; i < nb; i += 256) h += parts[i];
    part[threadIdx.x] = h;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *ok = part[0] == expected ? 1 : 0;
        *host = part[0];
        __hip_atomic_store(seq_ptr, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---- cached node-owned incidence ------------------------------------------------------------
// The reference's scatter entry points are called with the same connectivity many times (every K*u,
// restriction and prolongation of TOP_GPU.m).  The (row, entry) incidence of a connectivity is
// sorted once and kept as CSR; a later call reuses it when the device, pointer, dims and a content
// hash of the index array all match (the hash is recomputed on every call, so an array rewritten in
// place is sorted again).  The hash is compared on the device: a call that finds an incidence of the same array
// launches its scatter behind the comparison, which lets it through or not, and waits for the stream once; the host
// looks at the hash afterwards and, had the array changed, builds the incidence and scatters then.
struct Incidence {
    int dev = -1;
    const void *src = nullptr;
    int kind = 0;  // 0 = eNodMat (entries 8e + j), 1 = key list (entries i)
    int64_t n = 0, m = 0;
    unsigned long long hash = 0;
    uint64_t used = 0;
    DevBuf<uint32_t> rowptr, ent;
};
typedef std::shared_ptr<Incidence> IncidenceRef;  // a call keeps what it uses while another thread replaces it

struct IncidenceCache {
    std::mutex mu;
    std::vector<IncidenceRef> items;
    uint64_t tick = 0;
};

IncidenceCache &inc_cache() {
    static IncidenceCache c;
    return c;
}

constexpr size_t INC_CACHE_MAX = 8;

// The incidence of `idx` kept for these dims, whatever its content was; hash: with this content only.
IncidenceRef find_incidence(int dev, const int32_t *idx, int kind, int64_t N, int64_t M, const unsigned long long *hash) {
    IncidenceCache &C = inc_cache();
    std::lock_guard<std::mutex> lock(C.mu);
    for (auto &it : C.items)
        if (it->dev == dev && it->src == idx && it->kind == kind && it->n == N && it->m == M && (!hash || it->hash == *hash)) {
            it->used = ++C.tick;
            return it;
        }
    return nullptr;
}

// Sorts `idx` (eNodMat [Ne x 8] when kind == 0, keys [N] when kind == 1; content hash h) into the incidence with
// rows 0..M-1, entries of out-of-range ids left out, and keeps it.
IncidenceRef build_incidence(int dev, const int32_t *idx, int kind, int64_t Ne_or_N, int64_t M, unsigned long long h,
                             hipStream_t st, const char *id) {
    const int64_t N = kind == 0 ? 8 * Ne_or_N : Ne_or_N;
    IncidenceRef inc(new Incidence);
    {
        DevBuf<uint32_t> k0(N), k1(N), v0(N), v1(N);
        if (kind == 0) k_make_keys_enod<<<grid_for(N, 256), 256, 0, st>>>(idx, Ne_or_N, M, k0, v0);
        else k_make_keys_list<<<grid_for(N, 256), 256, 0, st>>>(idx, N, M, k0, v0);
        TG_LAUNCH_CHECK(id);
        hipcub::DoubleBuffer<uint32_t> kb(k0.p, k1.p), vb(v0.p, v1.p);
        size_t tmp = 0;
        sort_pairs_db(kb, vb, N, M, nullptr, tmp, st, id);
        DevBuf<char> t(tmp ? tmp : 1);
        sort_pairs_db(kb, vb, N, M, t.p, tmp, st, id);
        inc->rowptr.alloc(M + 1);
        k_rowptr<<<grid_for(M + 1, 256), 256, 0, st>>>(kb.Current(), N, M, inc->rowptr);
        TG_LAUNCH_CHECK(id);
        inc->ent.alloc(N);
        TG_HIP(hipMemcpyAsync(inc->ent.p, vb.Current(), N * sizeof(uint32_t), hipMemcpyDeviceToDevice, st), id);
        TG_HIP(hipStreamSynchronize(st), id);  // the temporaries are freed on leaving the scope
    }
    inc->dev = dev;
    inc->src = idx;
    inc->kind = kind;
    inc->n = N;
    inc->m = M;
    inc->hash = h;
    IncidenceCache &C = inc_cache();
    std::lock_guard<std::mutex> lock(C.mu);
    inc->used = ++C.tick;
    // replace a stale entry of the same array, else the least recently used one when full
    size_t slot = C.items.size();
    for (size_t i = 0; i < C.items.size(); ++i)
        if (C.items[i]->dev == dev && C.items[i]->src == idx && C.items[i]->kind == kind) slot = i;
    if (slot == C.items.size() && C.items.size() >= INC_CACHE_MAX) {
        slot = 0;
        for (size_t i = 1; i < C.items.size(); ++i)
            if (C.items[i]->used < C.items[slot]->used) slot = i;
    }
    if (slot == C.items.size()) C.items.push_back(inc);
    else C.items[slot] = inc;
    return inc;
}

// launch(incidence, ok) adds the scatter's entries on st with the incidence of idx; done when this returns.
template <class Launch>
void scatter_by_incidence(const int32_t *idx, int kind, int64_t Ne_or_N, int64_t M, hipStream_t st, const char *id,
                          Launch launch) {
    const int64_t N = kind == 0 ? 8 * Ne_or_N : Ne_or_N;
    check_items(N, id);
    int dev = 0;
    TG_HIP(hipGetDevice(&dev), id);
    IncidenceRef inc = find_incidence(dev, idx, kind, N, M, nullptr);  // outlives the scratch: its kernels use it
    Scratch sc(st);
    unsigned long long *parts = (unsigned long long *)sc.dbl();
    uint32_t *ok = (uint32_t *)(parts + HASH_BLOCKS);
    const int nb = (int)std::min<int64_t>(std::max<int64_t>((N + 1023) / 1024, 1), HASH_BLOCKS);
    if ((uintptr_t)idx % 16 == 0) k_hash_i32<true><<<nb, 256, 0, st>>>(idx, N, parts);
    else k_hash_i32<false><<<nb, 256, 0, st>>>(idx, N, parts);
    k_hash_check<<<1, 256, 0, st>>>(parts, nb, inc ? inc->hash : 0ull, ok, (unsigned long long *)sc.host(), sc.seq_ptr(),
                                    sc.next());
    TG_LAUNCH_CHECK(id);
    if (inc) {
        launch(*inc, ok);
        TG_LAUNCH_CHECK(id);
        TG_HIP(hipStreamSynchronize(st), id);
    }
    unsigned long long h;
    std::memcpy(&h, sc.wait(id), sizeof h);
    if (inc && inc->hash == h) return;
    inc = find_incidence(dev, idx, kind, N, M, &h);  // another thread may have built it since
    if (!inc) inc = build_incidence(dev, idx, kind, Ne_or_N, M, h, st, id);
    launch(*inc, nullptr);
    TG_LAUNCH_CHECK(id);
    TG_HIP(hipStreamSynchronize(st), id);
}

bool is_device_ptr(const void *p) {
    if (!p) return false;
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return at.type == hipMemoryTypeDevice || at.type == hipMemoryTypeManaged;
}

// ---- Galerkin sources (reference layouts: Ks column-major per element, 1-based maps) ----
template <typename T>
struct SrcLevel2 {
    const int32_t *up;
    int64_t Ne;
    int e;
    const T *E, *K0, *uf, *ux;
    const int32_t *mapU;
    bool hasFixed;
    int64_t nFine, nU;
    __device__ int child(int s) const {
        const int32_t f = up[e + Ne * s];
        return (f > 0 && f <= nFine) ? f - 1 : -1;
    }
    __device__ void kch(int f, int t, T (&k)[9]) const {
        const T mod = E[f];
        int32_t uid = hasFixed ? mapU[f] - 1 : -1;
        if (uid >= nU) uid = -1;
        if (uid >= 0) unique(uid, mod, t, k);
        else
#pragma unroll
            for (int j = 0; j < 9; ++j) k[j] = K0[64 * j + t] * mod;
    }
    __device__ void unique(int32_t uid, T mod, int t, T (&k)[9]) const {
#pragma unroll
        for (int j = 0; j < 9; ++j) k[j] = uf[(size_t)uid * 576 + 64 * j + t] * mod + ux[(size_t)uid * 576 + 64 * j + t];
    }
};

template <typename T>
struct SrcHigher {
    const int32_t *up;
    int64_t Ne;
    int e;
    const T *prev;
    int64_t nFine;
    __device__ int child(int s) const {
        const int32_t f = up[e + Ne * s];
        return (f > 0 && f <= nFine) ? f - 1 : -1;
    }
    __device__ void kch(int f, int t, T (&k)[9]) const {
#pragma unroll
        for (int j = 0; j < 9; ++j) k[j] = prev[(size_t)f * 576 + 64 * j + t];
    }
};

template <typename T>
struct SrcSuper {
    const int32_t *up;
    int64_t Ne;
    int e;
    const T *Ks0, *E, *uf, *ux;
    const int32_t *mapU;
    bool hasFixed;
    int64_t nFine, nU;
    __device__ int child(int s) const {
        const int32_t f = up[e + Ne * s];
        return (f > 0 && f <= nFine) ? f - 1 : -1;
    }
    __device__ void kch(int f, int t, T (&k)[9]) const {
        int32_t uid1 = hasFixed ? mapU[f] : 0;
        if (uid1 > nU) uid1 = 0;
        if (uid1 > 0) {
            const T *u = uf + (size_t)(uid1 - 1) * 576 * 64 + t, *mod = E + (size_t)f * 64;
#pragma unroll
            for (int j = 0; j < 9; ++j) k[j] = 0;
            for (int q = 0; q < 64; ++q)
#pragma unroll
                for (int j = 0; j < 9; ++j) k[j] += u[(size_t)q * 576 + 64 * j] * mod[q];
#pragma unroll
            for (int j = 0; j < 9; ++j) k[j] += ux[(size_t)(uid1 - 1) * 576 + 64 * j + t];
        } else {
#pragma unroll
            for (int j = 0; j < 9; ++j) k[j] = Ks0[(size_t)f * 576 + 64 * j + t];
        }
    }
};

template <typename T, int MODE, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_galerkin_mex(T *__restrict__ Ks, const int32_t *__restrict__ up, int64_t Ne,
                                                             int nCh, const T *__restrict__ P,
                                                             const T *a0, const T *a1, const T *a2, const T *a3,
                                                             const int32_t *mapU, int hasFixed, int64_t nFine,
                                                             int64_t nU) {
    __shared__ GalerkinLds<T, WAVES> lds;
    const int e = blockIdx.x;
    T *out = Ks + (size_t)e * 576;
    if (MODE == 0) {
        SrcLevel2<T> src{up, Ne, e, a0, a1, a2, a3, mapU, hasFixed != 0, nFine, nU};
        galerkin_block<false, WAVES>(out, src, nCh, P, lds);
    } else if (MODE == 1) {
        SrcHigher<T> src{up, Ne, e, a0, nFine};
        galerkin_block<false, WAVES>(out, src, nCh, P, lds);
    } else {
        SrcSuper<T> src{up, Ne, e, a0, a1, a2, a3, mapU, hasFixed != 0, nFine, nU};
        galerkin_block<false, WAVES>(out, src, nCh, P, lds);
    }
}

// Wavefronts per element.  With few elements the chain of one element's children is what bounds a call, and four
// wavefronts share it; with many the chip is full of elements, and wavefronts whose share of the children is uneven or
// empty only take LDS from others.  Measured, us, with 1, 2, 4 wavefronts: single, level 2 of 8 children: 200 elements
// 40, 32, 28; 2,500 58, 54, 60; 20,000 260, 239, 310; of 64: 157, 101, 63; 284, 248, 272; 1704, 1676, 2065; double, the
// levels above, 8 children: 40, 31, 28; 87, 90, 85; 504, 475, 489; 3 children, 20,000: 201, 220, 243.  Super-elements in
// double, whose children's sums over 64 sub-voxels fill the registers: 207, 142, 41; 334, 302, 90; 655, 658, 486.
template <typename T, int MODE>
int galerkin_waves(int64_t Ne, int nCh) {
    if (nCh == 1) return 1;
    if (Ne <= 2048 || (MODE == 2 && sizeof(T) == 8)) return 4;
    return nCh < 4 ? 1 : 2;
}
template <typename T, int MODE>
void launch_galerkin(hipStream_t st, void *Ks, const void *up, int64_t Ne, int nCh, const void *P, const void *a0,
                     const void *a1 = nullptr, const void *a2 = nullptr, const void *a3 = nullptr,
                     const void *mapU = nullptr, int hasFixed = 0, int64_t nFine = 0, int64_t nU = 0) {
    auto go = [&](auto kernel, int waves) {
        kernel<<<(unsigned)Ne, 64 * waves, 0, st>>>((T *)Ks, (const int32_t *)up, Ne, nCh, (const T *)P, (const T *)a0, (const T *)a1,
                                                    (const T *)a2, (const T *)a3, (const int32_t *)mapU, hasFixed, nFine, nU);
    };
    switch (galerkin_waves<T, MODE>(Ne, nCh)) {
        case 1: go(k_galerkin_mex<T, MODE, 1>, 1); break;
        case 2: go(k_galerkin_mex<T, MODE, 2>, 2); break;
        default: go(k_galerkin_mex<T, MODE, 4>, 4);
    }
}

// ---- level-2 Galerkin through its linearity (FP64) ---------------------------------------------------
// Ks_e = sum_s Pch_s' Kch_s Pch_s with Kch_s = E_f K0 for children without boundary matrices is linear in
// the children moduli: Ks_e = sum_s E_s G_s, G_s = Pch_s' K0 Pch_s.  G is formed per call from the
// caller's Pch and K0, the sum is one GEMM on the matrix cores, and the children with boundary matrices
// (mapUnique > 0) are added exactly, child by child (galerkin_block).

// G[s * 576 + r + 24 c] = (Pch_s' K0 Pch_s)(r, c), one workgroup per child
__global__ __launch_bounds__(256) void k_mex_gmat(const double *__restrict__ P, const double *__restrict__ K0,
                                                  double *__restrict__ G) {
    __shared__ double sP[576], sK[576], sT[576];
    const int s = blockIdx.x, t = threadIdx.x;
    for (int i = t; i < 576; i += 256) {
        sP[i] = P[(size_t)s * 576 + i];
        sK[i] = K0[i];
    }
    __syncthreads();
    for (int i = t; i < 576; i += 256) {  // T = K0 P_s
        const int a = i % 24, c = i / 24;
        double v = 0.0;
        for (int b = 0; b < 24; ++b) v += sK[a + 24 * b] * sP[b + 24 * c];
        sT[i] = v;
    }
    __syncthreads();
    for (int i = t; i < 576; i += 256) {  // G = P_s' T
        const int r = i % 24, c = i / 24;
        double v = 0.0;
        for (int a = 0; a < 24; ++a) v += sP[a + 24 * r] * sT[a + 24 * c];
        G[(size_t)s * 576 + i] = v;
    }
}

// Ech[e + Ne s] = modulus of child s of coarse element e, 0 for void children and children with boundary
// matrices (those are added by k_mex_galerkin_bnd); bnd[e]: whether e has any.  A workgroup has 64 elements, its
// wavefronts every eighth child of theirs.
__global__ __launch_bounds__(512) void k_mex_ech(const int32_t *__restrict__ up, const double *__restrict__ E,
                                                 const int32_t *__restrict__ mapU, int hasFixed, int64_t nFine,
                                                 int64_t nU, int64_t Ne, int nCh, double *__restrict__ Ech,
                                                 int32_t *__restrict__ bnd) {
    __shared__ int32_t any[8][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t e = (int64_t)blockIdx.x * 64 + lane;
    int32_t has = 0;
    if (e < Ne)
#pragma unroll 8
        for (int s = w; s < nCh; s += 8) {
            const int32_t f1 = up[e + Ne * s];
            double v = 0.0;
            if (f1 > 0 && f1 <= nFine) {
                const int32_t u1 = hasFixed ? mapU[f1 - 1] : 0;
                if (u1 > 0 && u1 <= nU) has = 1;
                else v = E[f1 - 1];
            }
            Ech[e + Ne * s] = v;
        }
    any[w][lane] = has;
    __syncthreads();
    if (w == 0 && e < Ne) {
#pragma unroll
        for (int k = 1; k < 8; ++k) has |= any[k][lane];
        bnd[e] = has;
    }
}

// Ks[e * 576 + i] = sum_k Ech[e + Ne k] G[k * 576 + i] on MFMA f64 16x16x4 (lane l holds A(l % 16, l / 16),
// B(l / 16, l % 16), result register r at (4 r + l / 16, l % 16)): A = 16 elements x 4 children of Ech,
// B = 4 children x 16 entries of G, so every store row is 16 consecutive entries of one element's page.
// A wavefront owns 16 NG elements and `tiles` of the 36 tiles of entries (blockIdx.y: which), a serial chain of
// 2.5 us a tile, so that few elements are shared out over more wavefronts; elements past Ne read zero moduli and store
// nothing.  8,192 elements of 64 children: 26 us, all tiles in one wavefront 102.
typedef double tg_mdbl4 __attribute__((ext_vector_type(4)));
template <int KS, int NG>
__global__ __launch_bounds__(256) void k_mex_galerkin_gemm(const double *__restrict__ Ech, const double *__restrict__ G,
                                                           double *__restrict__ Ks, int64_t Ne, int tiles) {
    const int t0 = blockIdx.y * tiles, t1 = min(t0 + tiles, 36);
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int64_t e0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * (16 * NG);
    if (e0 >= Ne) return;
    double a[NG][KS];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        const int64_t e = e0 + 16 * g + li;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) a[g][kk] = e < Ne ? Ech[e + Ne * (lk + 4 * kk)] : 0.0;
    }
    const double *gp = G + (int64_t)lk * 576 + li;
    for (int t = t0; t < t1; ++t) {
        tg_mdbl4 acc[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) acc[g] = tg_mdbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            const double b = gp[(int64_t)4 * kk * 576 + 16 * t];
#pragma unroll
            for (int g = 0; g < NG; ++g) acc[g] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[g][kk], b, acc[g], 0, 0, 0);
        }
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t e = e0 + 16 * g + 4 * r + lk;
                if (e < Ne) Ks[e * 576 + 16 * t + li] = acc[g][r];
            }
    }
}

// Children with boundary matrices only (child() skips the others), added to the GEMM's result.  k_mex_ech has
// marked the elements that have any, so that the other workgroups end at once: 8,192 elements, 256 of them with 16
// such children, 40 us, where one wavefront an element that looked through its children singly took 190.
struct SrcLevel2Bnd : SrcLevel2<double> {
    __device__ int child(int s) const {
        const int f = SrcLevel2<double>::child(s);
        if (f < 0 || !hasFixed) return -1;
        const int32_t u1 = mapU[f];
        return (u1 > 0 && u1 <= nU) ? f : -1;
    }
    __device__ void kch(int f, int t, double (&k)[9]) const { unique(mapU[f] - 1, E[f], t, k); }
};

constexpr int GB_WAVES = 4;
__global__ __launch_bounds__(64 * GB_WAVES) void k_mex_galerkin_bnd(double *__restrict__ Ks, const int32_t *__restrict__ up,
                                                                 int64_t Ne, int nCh, const double *__restrict__ P,
                                                                 const double *E, const double *K0, const double *uf,
                                                                 const double *ux, const int32_t *mapU, int64_t nFine,
                                                                 int64_t nU, const int32_t *__restrict__ bnd) {
    __shared__ GalerkinLds<double, GB_WAVES> lds;
    const int e = blockIdx.x;
    if (!bnd[e]) return;
    SrcLevel2Bnd src;
    src.up = up;
    src.Ne = Ne;
    src.e = e;
    src.E = E;
    src.K0 = K0;
    src.uf = uf;
    src.ux = ux;
    src.mapU = mapU;
    src.hasFixed = true;
    src.nFine = nFine;
    src.nU = nU;
    galerkin_block<true, GB_WAVES>(Ks + (size_t)e * 576, src, nCh, P, lds);
}

}  // namespace
}  // namespace tg

using namespace tg;

extern "C" {

int Gathering_inplace(int nlhs, tg_array *, int nrhs, const tg_array *prhs, void *stream) {
    return guard("Gathering_inplace:Args", [&] {
        const char *A = "Gathering_inplace:Args", *Ty = "Gathering_inplace:Type", *Sh = "Gathering_inplace:Shape";
        if (nrhs != 3 || !prhs) fail(TG_ERR_ARGS, A, "Usage: Gathering_inplace(gUMat, gU, gE)");
        if (nlhs != 0) fail(TG_ERR_ARGS, A, "This function returns no outputs. gUMat is modified in-place.");
        Arr out = arr(&prhs[0]), u = arr(&prhs[1]), e = arr(&prhs[2]);
        if (!is_float(u.cls)) fail(TG_ERR_TYPE, Ty, "gU must be single or double gpuArray.");
        if (out.cls != u.cls) fail(TG_ERR_TYPE, Ty, "gUMat precision must match gU.");
        if (!(e.cls == TG_INT32 || e.cls == TG_UINT32)) fail(TG_ERR_TYPE, Ty, "gE must be int32 or uint32 gpuArray.");
        if (u.nd != 2 || u.d[1] != 3) fail(TG_ERR_SHAPE, Sh, "gU must be (numNodes x 3).");
        if (e.nd != 2 || e.d[1] != 8) fail(TG_ERR_SHAPE, Sh, "gE must be (nElem x 8).");
        const int64_t Ne = e.d[0], Nn = u.d[0];
        if (out.nd != 2 || out.d[0] != Ne || out.d[1] != 24) fail(TG_ERR_SHAPE, Sh, "gUMat must be (nElem x 24).");
        if (Ne == 0) return;
        const unsigned g = grid_for(Ne, 256);
        if (u.cls == TG_DOUBLE) {
            if (e.cls == TG_INT32) k_gather<double, int32_t><<<g, 256, 0, S(stream)>>>((double *)out.p, (const double *)u.p, (const int32_t *)e.p, Ne, Nn);
            else k_gather<double, uint32_t><<<g, 256, 0, S(stream)>>>((double *)out.p, (const double *)u.p, (const uint32_t *)e.p, Ne, Nn);
        } else {
            if (e.cls == TG_INT32) k_gather<float, int32_t><<<g, 256, 0, S(stream)>>>((float *)out.p, (const float *)u.p, (const int32_t *)e.p, Ne, Nn);
            else k_gather<float, uint32_t><<<g, 256, 0, S(stream)>>>((float *)out.p, (const float *)u.p, (const uint32_t *)e.p, Ne, Nn);
        }
        TG_LAUNCH_CHECK("Gathering_inplace:CUDA");
    });
}

int Scattering_inplace(int, tg_array *, int nrhs, const tg_array *prhs, void *stream) {
    return guard("Scattering_inplace:arity", [&] {
        const char *Cu = "Scattering_inplace:cuda";
        const ScatterArgs a = scatter_args(nrhs, prhs);
        hipStream_t st = S(stream);
        if (a.Ne > 0 && a.Nn > 0) {
            scatter_by_incidence((const int32_t *)a.en.p, 0, a.Ne, a.Nn, st, Cu, [&](const Incidence &inc, const uint32_t *ok) {
                if (a.Y.cls == TG_DOUBLE)
                    k_csr_scatter_enod<double><<<grid_for(a.Nn, 256), 256, 0, st>>>((double *)a.Y.p, a.Nn, inc.rowptr, inc.ent,
                                                                                   (const double *)a.um.p, a.Ne, ok);
                else
                    k_csr_scatter_enod<float><<<grid_for(a.Nn, 256), 256, 0, st>>>((float *)a.Y.p, a.Nn, inc.rowptr, inc.ent,
                                                                                  (const float *)a.um.p, a.Ne, ok);
            });
            return;
        }
        TG_HIP(hipStreamSynchronize(st), Cu);
    });
}

int scatter_accum3_inplace(int nlhs, tg_array *, int nrhs, const tg_array *prhs, void *stream) {
    return guard("scatter_accum3:args", [&] {
        const char *Sh = "scatter_accum3:shape", *Ty = "scatter_accum3:type", *Cu = "scatter_accum3:cuda";
        if (nrhs != 3 || !prhs)
            fail(TG_ERR_ARGS, "scatter_accum3:args", "Usage: scatter_accum3_inplace(transferMatGPU[int32], TmpGPU[Nx3], xFinerGPU[Mx3]).");
        if (nlhs != 0) fail(TG_ERR_ARGS, "scatter_accum3:nlhs", "No output. xFiner is updated in-place.");
        Arr keys = arr(&prhs[0]), tmp = arr(&prhs[1]), xf = arr(&prhs[2]);
        for (int i = 0; i < 3; ++i) {
            Arr a = arr(&prhs[i]);
            if (a.numel > 0 && !is_device_ptr(a.p)) fail(TG_ERR_ARGS, "scatter_accum3:gpu", "All inputs must be gpuArray.");
        }
        if (tmp.nd != 2 || tmp.d[1] != 3) fail(TG_ERR_SHAPE, Sh, "`Tmp` must be [N x 3] gpuArray.");
        const int64_t N = tmp.d[0];
        if (xf.nd != 2 || xf.d[1] != 3) fail(TG_ERR_SHAPE, Sh, "`xFiner` must be [M x 3] gpuArray.");
        const int64_t M = xf.d[0];
        if (keys.cls != TG_INT32) fail(TG_ERR_TYPE, Ty, "`transferMat` must be int32 gpuArray.");
        if (tmp.cls != xf.cls) fail(TG_ERR_TYPE, Ty, "`Tmp` and `xFiner` must have the same class (single/double).");
        if (!is_float(tmp.cls)) fail(TG_ERR_TYPE, Ty, "Only single or double supported for `Tmp`/`xFiner`.");
        if (keys.numel != N) fail(TG_ERR_SHAPE, Sh, "`transferMat` must hold exactly N = size(Tmp,1) keys.");
        check_items(N, Sh);
        if (N == 0 || M == 0) return;
        hipStream_t st = S(stream);
        scatter_by_incidence((const int32_t *)keys.p, 1, N, M, st, Cu, [&](const Incidence &inc, const uint32_t *ok) {
            if (xf.cls == TG_DOUBLE)
                k_csr_scatter_list<double><<<grid_for(M, 256), 256, 0, st>>>((double *)xf.p, M, inc.rowptr, inc.ent, N,
                                                                             (const double *)tmp.p, ok);
            else
                k_csr_scatter_list<float><<<grid_for(M, 256), 256, 0, st>>>((float *)xf.p, M, inc.rowptr, inc.ent, N,
                                                                            (const float *)tmp.p, ok);
        });
    });
}

int assembleKs_level2_inplace(int nlhs, tg_array *plhs, int nrhs, const tg_array *prhs, void *stream) {
    return guard("assembleKs_level2_inplace:Input", [&] {
        const char *In = "assembleKs_level2_inplace:Input", *Ty = "assembleKs_level2_inplace:Type",
                   *Sh = "assembleKs_level2_inplace:Shape", *Cu = "assembleKs_level2_inplace:CUDA";
        if (nrhs != 8 || !prhs) fail(TG_ERR_ARGS, In, "Expected 8 inputs.");
        Arr Ks = arr(&prhs[0]), up = arr(&prhs[1]), em = arr(&prhs[2]), k0 = arr(&prhs[3]), pch = arr(&prhs[4]),
            mu = arr(&prhs[5]), uf = arr(&prhs[6]), ux = arr(&prhs[7]);
        const int cls = Ks.cls;
        if (!is_float(cls)) fail(TG_ERR_TYPE, Ty, "d_Ks must be single/double gpuArray.");
        if (up.cls != TG_INT32 || mu.cls != TG_INT32) fail(TG_ERR_TYPE, Ty, "d_upMap and d_mapUnique must be int32 gpuArray.");
        if (Ks.d[0] != 24 || Ks.d[1] != 24 || Ks.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_Ks must be [24 x 24 x nElem].");
        const int64_t Ne = Ks.d[2];
        if (up.nd != 2 || up.d[0] != Ne) fail(TG_ERR_SHAPE, Sh, "d_upMap must be [nElem x nCh].");
        const int nCh = (int)up.d[1];
        if (pch.d[0] != 24 || pch.d[1] != 24 || pch.d[2] != nCh || pch.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_Pch must be [24 x 24 x nCh].");
        if (k0.nd != 2 || k0.d[0] * k0.d[1] != 576) fail(TG_ERR_SHAPE, Sh, "d_K_0 must contain 576 elements.");
        int64_t nU = 0;
        if (uf.numel > 0) {
            if (uf.nd != 2 || uf.d[0] != 576) fail(TG_ERR_SHAPE, Sh, "d_uniqueFree must be [576 x nUnique] or empty.");
            nU = uf.d[1];
        }
        if (ux.numel > 0 && (ux.nd != 2 || ux.d[0] != 576 || ux.d[1] != nU))
            fail(TG_ERR_SHAPE, Sh, "d_uniqueFixed must be [576 x nUnique] matching d_uniqueFree.");
        if (em.cls != cls || k0.cls != cls || pch.cls != cls) fail(TG_ERR_TYPE, Ty, "d_eleModulus/d_K_0/d_Pch must match d_Ks class.");
        if (uf.numel > 0 && uf.cls != cls) fail(TG_ERR_TYPE, Ty, "d_uniqueFree class must match d_Ks.");
        if (ux.numel > 0 && ux.cls != cls) fail(TG_ERR_TYPE, Ty, "d_uniqueFixed class must match d_Ks.");
        const int hasFixed = (nU > 0 && mu.p && uf.p && ux.numel > 0 && ux.p) ? 1 : 0;
        const int64_t nFine = hasFixed ? std::min(em.numel, mu.numel) : em.numel;
        hipStream_t st = S(stream);
        if (Ne > 0) {
            if (cls == TG_DOUBLE && (nCh == 64 || nCh == 8)) {
                // one allocation: G, the children's moduli, the flags of the elements with boundary matrices
                const size_t nG = (size_t)nCh * 576, nE = (size_t)Ne * nCh;
                DevBuf<double> buf(nG + nE + ((size_t)Ne + 1) / 2);
                double *G = buf.p, *Ech = G + nG;
                int32_t *bnd = (int32_t *)(Ech + nE);
                k_mex_gmat<<<nCh, 256, 0, st>>>((const double *)pch.p, (const double *)k0.p, G);
                k_mex_ech<<<grid_for(Ne, 64), 512, 0, st>>>((const int32_t *)up.p, (const double *)em.p, (const int32_t *)mu.p,
                                                            hasFixed, nFine, nU, Ne, nCh, Ech, bnd);
                // 64 elements per wavefront; the entry tiles shared out until there are 512 workgroups
                const unsigned gg = grid_for(Ne, 256);
                const int tiles = (int)std::max<int64_t>(1, std::min<int64_t>(36, 36 * (int64_t)gg / 512));
                const dim3 gt(gg, (36 + tiles - 1) / tiles);
                if (nCh == 64) k_mex_galerkin_gemm<16, 4><<<gt, 256, 0, st>>>(Ech, G, (double *)Ks.p, Ne, tiles);
                else k_mex_galerkin_gemm<2, 4><<<gt, 256, 0, st>>>(Ech, G, (double *)Ks.p, Ne, tiles);
                if (hasFixed)
                    k_mex_galerkin_bnd<<<(unsigned)Ne, 64 * GB_WAVES, 0, st>>>((double *)Ks.p, (const int32_t *)up.p, Ne, nCh,
                        (const double *)pch.p, (const double *)em.p, (const double *)k0.p, (const double *)uf.p,
                        (const double *)ux.p, (const int32_t *)mu.p, nFine, nU, bnd);
                TG_LAUNCH_CHECK(Cu);
                TG_HIP(hipStreamSynchronize(st), Cu);  // buf is released on leaving the scope
            } else if (cls == TG_DOUBLE)
                launch_galerkin<double, 0>(st, Ks.p, up.p, Ne, nCh, pch.p, em.p, k0.p, uf.p, ux.p, mu.p, hasFixed, nFine, nU);
            else
                launch_galerkin<float, 0>(st, Ks.p, up.p, Ne, nCh, pch.p, em.p, k0.p, uf.p, ux.p, mu.p, hasFixed, nFine, nU);
            TG_LAUNCH_CHECK(Cu);
        }
        TG_HIP(hipStreamSynchronize(st), Cu);
        if (nlhs > 0 && plhs) plhs[0] = prhs[0];
    });
}

int assembleKs_higherLevel_inplace(int nlhs, tg_array *plhs, int nrhs, const tg_array *prhs, void *stream) {
    return guard("assembleKs_higherLevel_inplace:Input", [&] {
        const char *In = "assembleKs_higherLevel_inplace:Input", *Ty = "assembleKs_higherLevel_inplace:Type",
                   *Sh = "assembleKs_higherLevel_inplace:Shape", *Cu = "assembleKs_higherLevel_inplace:CUDA";
        if (nrhs != 4 || !prhs) fail(TG_ERR_ARGS, In, "Expected 4 inputs: (d_Ks, d_upMap, d_KsPrev, d_Psub).");
        Arr Ks = arr(&prhs[0]), up = arr(&prhs[1]), prev = arr(&prhs[2]), ps = arr(&prhs[3]);
        const int cls = Ks.cls;
        if (!is_float(cls)) fail(TG_ERR_TYPE, Ty, "d_Ks must be single/double gpuArray.");
        if (up.cls != TG_INT32) fail(TG_ERR_TYPE, Ty, "d_upMap must be int32 gpuArray.");
        if (prev.cls != cls || ps.cls != cls) fail(TG_ERR_TYPE, Ty, "d_KsPrev and d_Psub must match d_Ks class.");
        if (Ks.d[0] != 24 || Ks.d[1] != 24 || Ks.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_Ks must be [24 x 24 x nElem].");
        const int64_t Ne = Ks.d[2];
        if (up.nd != 2 || up.d[0] != Ne) fail(TG_ERR_SHAPE, Sh, "d_upMap must be [nElem x nSub].");
        const int nSub = (int)up.d[1];
        if (prev.d[0] != 24 || prev.d[1] != 24 || prev.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_KsPrev must be [24 x 24 x nFinElem].");
        if (ps.d[0] != 24 || ps.d[1] != 24 || ps.d[2] != nSub || ps.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_Psub must be [24 x 24 x nSub].");
        const int64_t nFine = prev.d[2];
        hipStream_t st = S(stream);
        if (Ne > 0) {
            if (cls == TG_DOUBLE)
                launch_galerkin<double, 1>(st, Ks.p, up.p, Ne, nSub, ps.p, prev.p, nullptr, nullptr, nullptr, nullptr, 0, nFine, 0);
            else
                launch_galerkin<float, 1>(st, Ks.p, up.p, Ne, nSub, ps.p, prev.p, nullptr, nullptr, nullptr, nullptr, 0, nFine, 0);
            TG_LAUNCH_CHECK(Cu);
        }
        TG_HIP(hipStreamSynchronize(st), Cu);
        if (nlhs > 0 && plhs) plhs[0] = prhs[0];
    });
}

int assembleKs_level2_superEle_inplace(int nlhs, tg_array *plhs, int nrhs, const tg_array *prhs, void *stream) {
    return guard("assembleKs_level2_superEle_inplace:Input", [&] {
        const char *In = "assembleKs_level2_superEle_inplace:Input", *Ty = "assembleKs_level2_superEle_inplace:Type",
                   *Sh = "assembleKs_level2_superEle_inplace:Shape", *Cu = "assembleKs_level2_superEle_inplace:CUDA";
        if (nrhs != 8 || !prhs)
            fail(TG_ERR_ARGS, In, "Expected 8 inputs: d_Ks, d_upMap, d_Ks0, d_Psub, d_mapUnique, d_eleModulus, d_uniqueFree, d_uniqueFixed.");
        Arr Ks = arr(&prhs[0]), up = arr(&prhs[1]), ks0 = arr(&prhs[2]), ps = arr(&prhs[3]), mu = arr(&prhs[4]),
            em = arr(&prhs[5]), uf = arr(&prhs[6]), ux = arr(&prhs[7]);
        const int cls = Ks.cls;
        if (!is_float(cls)) fail(TG_ERR_TYPE, Ty, "d_Ks must be single/double gpuArray.");
        if (up.cls != TG_INT32 || mu.cls != TG_INT32) fail(TG_ERR_TYPE, Ty, "d_upMap and d_mapUnique must be int32 gpuArray.");
        if (ks0.cls != cls || ps.cls != cls || em.cls != cls) fail(TG_ERR_TYPE, Ty, "d_Ks0, d_Psub, d_eleModulus must match d_Ks class.");
        if (uf.numel > 0 && uf.cls != cls) fail(TG_ERR_TYPE, Ty, "d_uniqueFree class must match d_Ks.");
        if (ux.numel > 0 && ux.cls != cls) fail(TG_ERR_TYPE, Ty, "d_uniqueFixed class must match d_Ks.");
        if (Ks.d[0] != 24 || Ks.d[1] != 24 || Ks.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_Ks must be [24 x 24 x nElem].");
        const int64_t Ne = Ks.d[2];
        if (up.nd != 2 || up.d[0] != Ne) fail(TG_ERR_SHAPE, Sh, "d_upMap must be [nElem x nSub].");
        const int nSub = (int)up.d[1];
        if (ks0.numel % 576 != 0) fail(TG_ERR_SHAPE, Sh, "d_Ks0 total elements must be a multiple of 576.");
        if (ps.d[0] != 24 || ps.d[1] != 24 || ps.d[2] != nSub || ps.d[3] != 1) fail(TG_ERR_SHAPE, Sh, "d_Psub must be [24 x 24 x nSub].");
        if (em.numel % 64 != 0) fail(TG_ERR_SHAPE, Sh, "d_eleModulus total elements must be a multiple of 64.");
        int64_t nU = 0;
        if (uf.numel > 0) {
            if (uf.nd == 3) {
                if (uf.d[0] != 576 || uf.d[1] != 64) fail(TG_ERR_SHAPE, Sh, "d_uniqueFree must be [576 x 64 x nUnique].");
                nU = uf.d[2];
            } else if (uf.nd == 2) {
                if (uf.d[0] != 576 * 64) fail(TG_ERR_SHAPE, Sh, "d_uniqueFree must be [576*64 x nUnique] or [576 x 64 x nUnique].");
                nU = uf.d[1];
            } else {
                fail(TG_ERR_SHAPE, Sh, "d_uniqueFree must be 2-D or 3-D.");
            }
        }
        if (ux.numel > 0 && (ux.nd != 2 || ux.d[0] != 576 || ux.d[1] != nU))
            fail(TG_ERR_SHAPE, Sh, "d_uniqueFixed must be [576 x nUnique] matching d_uniqueFree.");
        const int hasFixed = (nU > 0 && mu.p && uf.p && ux.numel > 0 && ux.p) ? 1 : 0;
        int64_t nFine = std::min(ks0.numel / 576, em.numel / 64);
        if (hasFixed) nFine = std::min(nFine, mu.numel);
        hipStream_t st = S(stream);
        if (Ne > 0) {
            if (cls == TG_DOUBLE)
                launch_galerkin<double, 2>(st, Ks.p, up.p, Ne, nSub, ps.p, ks0.p, em.p, uf.p, ux.p, mu.p, hasFixed, nFine, nU);
            else
                launch_galerkin<float, 2>(st, Ks.p, up.p, Ne, nSub, ps.p, ks0.p, em.p, uf.p, ux.p, mu.p, hasFixed, nFine, nU);
            TG_LAUNCH_CHECK(Cu);
        }
        TG_HIP(hipStreamSynchronize(st), Cu);
        if (nlhs > 0 && plhs) plhs[0] = prhs[0];
    });
}

}  // extern "C"
