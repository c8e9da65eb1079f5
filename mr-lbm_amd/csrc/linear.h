// Fields in groups of four nodes: the map between x-fastest order and the
// block layout, and the storage words of a group of one moment plane.
#pragma once

#include "context.h"

namespace mrlbm {

typedef float __attribute__((ext_vector_type(4))) f32x4;
typedef double __attribute__((ext_vector_type(4))) f64x4;

// x-fastest order in groups of four nodes along x (every tile is a multiple
// of four nodes wide, so a group is one 16- or 8-byte run of a moment plane)
// and the block layout. Tile extents are powers of two.
struct Linear {
    FastDiv by_nx4, by_ny;
    uint32_t nx4, ny, ntx, nty, T;
    uint32_t groups;  // per plane
    int lx, ly, lz;   // log2 of the tile extents
    float scale[10], rscale[10];
    // element of moment 0 of node (x, y, z); moment m lies m T further
    __device__ __forceinline__ size_t at(uint32_t x, uint32_t y, uint32_t z) const {
        const uint32_t tile = (x >> lx) + ntx * ((y >> ly) + nty * (z >> lz));
        const uint32_t t = (x & ((1u << lx) - 1)) + ((y & ((1u << ly) - 1)) << lx) + ((z & ((1u << lz) - 1)) << (lx + ly));
        return (size_t)tile * 10 * T + t;
    }
    // the same of a group's first node
    __device__ __forceinline__ size_t node(uint32_t group) const {
        const uint32_t row = by_nx4.div(group), z = by_ny.div(row);
        return at(4 * (group - row * nx4), row - z * ny, z);
    }
};

inline int log2_of(int v) {
    int l = 0;
    while ((1 << l) < v) l++;
    return l;
}

inline Linear linear_of(const mrlbm_ctx* c) {
    Linear L{};
    L.nx4 = (uint32_t)c->p.nx / 4;
    L.ny = (uint32_t)c->p.ny;
    L.by_nx4 = make_fastdiv(L.nx4);
    L.by_ny = make_fastdiv(L.ny);
    L.ntx = (uint32_t)c->ntx;
    L.nty = (uint32_t)c->nty;
    L.T = (uint32_t)c->T;
    L.groups = (uint32_t)(c->N / 4);
    L.lx = log2_of(c->bx);
    L.ly = log2_of(c->by);
    L.lz = log2_of(c->bz);
    for (int m = 0; m < 10; m++) {
        L.scale[m] = c->mscale[m];
        L.rscale[m] = c->mrscale[m];
    }
    return L;
}

// Storage word of a stored moment, rounded to nearest even (through FP32),
// and back, as the host encodes single values (to_half, to_bf16).
template <int S> struct Word;
template <> struct Word<0> {
    using T = uint32_t;
    typedef uint32_t __attribute__((ext_vector_type(4))) V;
    __device__ static float dec(uint32_t w, float) { return __uint_as_float(w); }
    __device__ static uint32_t enc(double v, float s) { return __float_as_uint((float)(v * (double)s)); }
};
template <> struct Word<1> {
    using T = uint16_t;
    typedef uint16_t __attribute__((ext_vector_type(4))) V;
    __device__ static float dec(uint16_t w, float rs) { return (float)__builtin_bit_cast(_Float16, w) * rs; }
    __device__ static uint16_t enc(double v, float s) {
        return __builtin_bit_cast(uint16_t, (_Float16)(float)(v * (double)s));
    }
};
template <> struct Word<2> {
    using T = uint16_t;
    typedef uint16_t __attribute__((ext_vector_type(4))) V;
    __device__ static float dec(uint16_t w, float) { return __uint_as_float((uint32_t)w << 16); }
    __device__ static uint16_t enc(double v, float s) {
        uint32_t u = __float_as_uint((float)(v * (double)s));
        u += 0x7FFFu + ((u >> 16) & 1u);
        return (uint16_t)(u >> 16);
    }
};

// Four consecutive nodes of a moment plane, decoded (element e a multiple of
// four: one 16- or 8-byte load; non-temporal, each value is read once).
template <int S>
__device__ __forceinline__ f32x4 load_group(const void* mom, size_t e, float rscale) {
    using W = Word<S>;
    const auto w = __builtin_nontemporal_load((const typename W::V*)((const typename W::T*)mom + e));
    return f32x4{W::dec(w.x, rscale), W::dec(w.y, rscale), W::dec(w.z, rscale), W::dec(w.w, rscale)};
}

// Groups of a field taken patch by patch: a wave covers w4 groups along x
// times 64 / w4 rows, so that it reads whole lines of a moment plane (the
// rows of a tile lie together) and runs of up to 256 bytes of an x-fastest
// FP64 field. Along one row alone a wave reads 16 bytes (FP16, 8-wide tiles)
// of 32 different tiles.
struct Patches {
    FastDiv by_px, by_ny;
    uint32_t px;     // patches along x
    uint32_t lw;     // log2 w4, the largest of 2, 4, 8 groups that divide a row
    uint32_t rows;   // ny nz
    uint32_t n;      // lanes of all patches (the last rows' may be idle)
    // node coordinates of lane i and its group in x-fastest order
    __device__ __forceinline__ bool at(uint32_t i, const Linear& L, uint32_t& x, uint32_t& y, uint32_t& z,
                                       size_t& group) const {
        const uint32_t p = i / 64, lane = i % 64;
        const uint32_t pr = by_px.div(p);
        const uint32_t x4 = ((p - pr * px) << lw) + (lane & ((1u << lw) - 1));
        const uint32_t row = pr * (64u >> lw) + (lane >> lw);
        z = by_ny.div(row);
        y = row - z * L.ny;
        x = 4 * x4;
        group = (size_t)row * L.nx4 + x4;
        return i < n && row < rows;
    }
};
inline Patches patches_of(const mrlbm_ctx* c) {
    Patches P{};
    const uint32_t nx4 = (uint32_t)c->p.nx / 4;
    P.lw = nx4 % 8 == 0 ? 3 : (nx4 % 4 == 0 ? 2 : 1);  // nx is a multiple of 8
    P.px = nx4 >> P.lw;
    P.rows = (uint32_t)c->p.ny * (uint32_t)c->p.nz;
    P.by_px = make_fastdiv(P.px);
    P.by_ny = make_fastdiv((uint32_t)c->p.ny);
    const uint32_t r = 64u >> P.lw;
    P.n = 64 * P.px * ((P.rows + r - 1) / r);
    return P;
}

// Groups in the block layout's own order (any order does for a sum): group i
// of the lattice starts at element index(i) of moment 0.
struct BlockGroups {
    uint32_t n;  // groups of the lattice
    int lg;      // log2 of the groups per tile
    uint32_t T;
    __device__ __forceinline__ size_t index(uint32_t i) const {
        return (size_t)(i >> lg) * 10 * T + 4 * (i & ((1u << lg) - 1));
    }
};
inline BlockGroups block_groups(size_t ntiles, int T) {
    return BlockGroups{(uint32_t)(ntiles * (size_t)T / 4), log2_of(T / 4), (uint32_t)T};
}

// Workgroups of a sum over n groups: enough to fill the chip, no more than
// there are groups, at most RED_BLOCKS_MAX (the partial-sum buffers).
constexpr int RED_THREADS = 256;
constexpr int RED_BLOCKS_MAX = 1024;
inline int red_blocks(uint32_t n) {
    const uint32_t b = (n + RED_THREADS - 1) / RED_THREADS;
    return (int)(b < 1 ? 1 : (b > RED_BLOCKS_MAX ? RED_BLOCKS_MAX : b));
}

// Sums of K values over a workgroup in a fixed order (lanes by halving
// distances, then the waves); the result is in thread 0.
template <int K>
__device__ __forceinline__ void block_sum(double (&v)[K]) {
    __shared__ double w[RED_THREADS / 64][K];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1)
        for (int k = 0; k < K; k++) v[k] += __shfl_down(v[k], d);
    if (threadIdx.x % 64 == 0)
        for (int k = 0; k < K; k++) w[threadIdx.x / 64][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (int k = 0; k < K; k++)
            for (int j = 1; j < RED_THREADS / 64; j++) v[k] += w[j][k];
}

// x / 3 for x of a 32-bit value: a product with 1/3 and one correction (an FP64
// division takes several times as many instructions). For an infinite x the
// correction would be inf - inf; the product is the quotient then.
__host__ __device__ __forceinline__ double third(double x) {
    const double q = x * (1.0 / 3.0);
    const double r = __builtin_fma(__builtin_fma(-3.0, q, x), 1.0 / 3.0, q);
    return __builtin_isinf(x) ? q : r;
}

// Fold n partial records of K sums (record b at partial[K b]) in a fixed
// order into out[0..K), sum k divided by div[k] (reduce.hip).
template <int K>
struct Divisors {
    double d[K];
};
template <int K>
hipError_t launch_fold(const double* partial, int n, double* out, const Divisors<K>& div, hipStream_t s);

}  // namespace mrlbm
