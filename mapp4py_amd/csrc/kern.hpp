// kern.hpp -- device helpers shared by the HIP translation units: launch
// geometry (wave64, 8 XCDs), deterministic block reductions, cell helpers.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace mapp {
namespace {

constexpr int kBlock = 256;
constexpr int kXcd = 8;
constexpr int kPartW = 8;  // doubles per partial-sum row

// number of workgroups, rounded up so the XCD remap below is a bijection
inline int grid_for(int n) { int b = (n + kBlock - 1) / kBlock; return ((b + kXcd - 1) / kXcd) * kXcd; }

// Workgroups are dealt to the 8 XCDs round-robin; give XCD x the contiguous
// block range [x*q, (x+1)*q) so neighbor gathers stay in that XCD's L2.
__device__ inline int xcd_block()
{
    const int nb = gridDim.x;
    const int q = nb / kXcd;
    return (blockIdx.x % kXcd) * q + blockIdx.x / kXcd;
}

// The walk of persistent workgroups (see the LDS passes of the EAM force
// field): an XCD's workgroups stride side by side through a contiguous eighth
// of the chunks.
struct ChunkWalk {
    int c, end, step;
};
// chunks of `size` atoms
__device__ inline ChunkWalk chunk_walk(int n, int size)
{
    const int nchunks = (n + size - 1) / size;
    const int per = (nchunks + kXcd - 1) / kXcd;
    const int x = blockIdx.x % kXcd;
    ChunkWalk w;
    w.c = x * per + (int)blockIdx.x / kXcd;
    w.end = min((x + 1) * per, nchunks);
    w.step = gridDim.x / kXcd;
    return w;
}

// P sums (a power of two) over the 64 lanes of a wave, in a fixed order: lanes
// a bit apart each keep half of the values and give the other half away, until
// one is left, so 8 values take 4 + 2 + 1 + 3 exchanges instead of 48. Lane l
// (l < P) ends with the sum of value lane_value<P>(l) in v[0].
template <int P, class T>
__device__ inline void wave_sums(T (&v)[P])
{
    const int lane = threadIdx.x & 63;
    int off = 1;
#pragma unroll
    for (int half = P / 2; half > 0; half /= 2, off *= 2) {
        const bool up = (lane & off) != 0;
#pragma unroll
        for (int k = 0; k < half; ++k) {
            const T a = v[k], b = v[k + half];
            const T keep = up ? b : a, give = up ? a : b;
            v[k] = keep + __shfl_xor(give, off, 64);
        }
    }
#pragma unroll
    for (; off < 64; off *= 2) v[0] += __shfl_xor(v[0], off, 64);
}
template <int P>
__device__ inline int lane_value(int l)
{
    int k = 0;
#pragma unroll
    for (int half = P / 2, off = 1; half > 0; half /= 2, off *= 2) k += (l & off) ? half : 0;
    return k;
}

// wave_sums of K (at most 8) values that start at v[O], to row[O ..]
template <int O, int K, int N>
__device__ inline void wave_sums_to(const double (&v)[N], double* row)
{
    constexpr int P = K <= 1 ? 1 : K <= 2 ? 2 : K <= 4 ? 4 : 8;
    double t[P];
#pragma unroll
    for (int k = 0; k < P; ++k) t[k] = v[O + (k < K ? k : 0)];
    wave_sums<P>(t);
    const int lane = threadIdx.x & 63, k = lane_value<P>(lane);
    if (lane < P && k < K) row[O + k] = t[0];
}

// K FP64 sums over a workgroup of NT threads: thread k < K returns the k-th
// (the others 0)
template <int K, int NT = kBlock>
__device__ inline double block_sums(const double (&v)[K])
{
    __shared__ double sh[NT / 64][K];
    double* row = sh[threadIdx.x >> 6];
    wave_sums_to<0, (K < 8 ? K : 8)>(v, row);
    if constexpr (K > 8) wave_sums_to<8, K - 8>(v, row);
    __syncthreads();
    double s = 0.0;
    if ((int)threadIdx.x < K)
        for (int q = 0; q < NT / 64; ++q) s += sh[q][threadIdx.x];
    return s;
}

// the same, written as one row of kPartW (zeros past K, so that any column
// count can be reduced)
template <int K, int NT = kBlock>
__device__ inline void block_sum_store(const double (&v)[K], double* out)
{
    const double s = block_sums<K, NT>(v);
    if (threadIdx.x < kPartW) out[threadIdx.x] = s;
}

// Fixed-order reduction of rows of partial sums: out[k] = sum_r part[r*W + k].
// Block b sums rows [b*chunk, (b+1)*chunk) and writes row b of out, so a
// launch over G blocks followed by one over a single block is a fixed-order
// (deterministic) two-level reduction.
__global__ __launch_bounds__(kBlock) void k_reduce_rows(int nrows, int ncols, const double* __restrict__ part,
                                                        double* __restrict__ out, int chunk)
{
    __shared__ double sh[kBlock][kPartW];
    double acc[kPartW];
    for (int k = 0; k < kPartW; ++k) acc[k] = 0.0;
    const int r0 = blockIdx.x * chunk;
    const int r1 = min(nrows, r0 + chunk);
    for (int r = r0 + threadIdx.x; r < r1; r += kBlock)
        for (int k = 0; k < ncols; ++k) acc[k] += part[(size_t)r * kPartW + k];
    out += (size_t)blockIdx.x * (gridDim.x > 1 ? kPartW : 0);
    for (int k = 0; k < kPartW; ++k) sh[threadIdx.x][k] = acc[k];
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int k = 0; k < kPartW; ++k) sh[threadIdx.x][k] += sh[threadIdx.x + s][k];
        __syncthreads();
    }
    if ((int)threadIdx.x < ncols) out[threadIdx.x] = sh[0][threadIdx.x];
}



// Lanes sharing an atom (or a site): 2^lg neighboring lanes take the batches
// of its row in turn and meet in a butterfly, so that a small system still
// fills the chip (one lane an atom leaves most CUs without work below 262,144
// atoms). Every lane of the group ends with the same sum.
template <class T>
__device__ inline T lane_sum(T v, int lg)
{
    for (int o = 1; o < (1 << lg); o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// The lanes take the entries in blocks of 4 whatever the batch length B is, so
// the sums do not depend on it: entry after k0's batch of a lane.
template <int B>
__device__ inline int next_batch(int k0, int lg)
{
    return k0 + B + (B >= 4 || ((k0 + B) & 3) == 0 ? (4 << lg) - 4 : 0);
}

// workgroups of kBlock threads for n items of 2^lg lanes each
inline int grid_lanes(int n, int lg) { return (int)((((long)n << lg) + kXcd * kBlock - 1) / (kXcd * kBlock)) * kXcd; }

__device__ inline int cell_coord(double s, int nc)
{
    int c = (int)(s * (double)nc);
    return c < nc - 1 ? c : nc - 1;
}

__device__ inline int floordiv(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

// r = sqrt(rsq) to ~1e-14 relative: FP32 root and one FP64 Newton step
__device__ inline double root64(double rsq)
{
    const float rf = __builtin_sqrtf((float)rsq);
    const double r0 = (double)rf;
    const double e = fma(-r0, r0, rsq);
    return fma(e, (double)(0.5f / rf), r0);
}

// r = sqrt(x) and 1 / r to an ulp or so: the hardware's reciprocal root
// (about 24 bits), one third-order step for the inverse, one for the root.
// The steps multiply 0 by infinity at x = 0 and x = infinity, which are their
// own roots and have the hardware's inverses: a caller's comparison takes such
// a distance as it takes sqrt's.
__device__ inline void root_inv(double x, double& r, double& r_inv)
{
    const double y0 = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * y0), y0, 1.0);
    const double y = fma(y0 * e, fma(0.375, e, 0.5), y0);
    const double t = x * y;
    const bool inside = e < 1.0;  // not for 0, infinity and NaN
    r = inside ? fma(fma(-t, t, x), 0.5 * y, t) : x;
    r_inv = inside ? y : y0;
}

// A cubic from its end values and slopes (per unit offset) at offset p: the
// basis, shared by the functions of an interval, and the value. In FP64 y0
// comes last, so that only one rounding is of its size, as in the Horner scheme
// of a coefficient row (the same rms error; 1.73 times it with y0 first; 1% of a
// DMD gradient's time).
template <class F>
struct HermiteBasis {
    F h1, h2, h3;
};
template <class F>
__device__ inline HermiteBasis<F> hermite_basis(double p)
{
    const F q = (F)p, q1 = (F)1 - q, q2 = q * q;
    return HermiteBasis<F>{q2 * ((F)3 - (F)2 * q), q * q1 * q1, -q2 * q1};
}
template <class F>
__device__ inline F hermite_eval(F y0, F s0, F y1, F s1, const HermiteBasis<F>& h)
{
    if constexpr (sizeof(F) == sizeof(double))
        return y0 + ((y1 - y0) * h.h1 + s0 * h.h2 + s1 * h.h3);
    else
        return y0 + (y1 - y0) * h.h1 + s0 * h.h2 + s1 * h.h3;
}

inline uint32_t morton3(uint32_t a, uint32_t b, uint32_t c)
{
    auto spread = [](uint32_t v) {
        v &= 0x3ff;
        v = (v | (v << 16)) & 0x030000FF;
        v = (v | (v << 8)) & 0x0300F00F;
        v = (v | (v << 4)) & 0x030C30C3;
        v = (v | (v << 2)) & 0x09249249;
        return v;
    };
    return spread(a) | (spread(b) << 1) | (spread(c) << 2);
}

}  // namespace
}  // namespace mapp
