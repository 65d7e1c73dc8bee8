// md_nst.hip -- MDNST on the GPU: velocity Verlet under a Nose-Hoover chain
// with a box that follows a target stress (src/md_nst.cpp). The per-atom work
// (the exponential velocity and position updates, the kinetic tensor) runs in
// two streaming kernels; the 3x3 box algebra, both thermostats and the
// box-velocity kicks run on one workgroup between them, so that steps are
// launched ahead of the host. The neighbor list survives box changes: the
// image shifts follow the new box every step and the list is rebuilt only when
// an atom has moved half the skin (DynamicMD::update with a changed box,
// src/dynamic_md.h:38-56).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <limits>
#include <vector>

#include "kern.hpp"
#include "md.hpp"

namespace mapp {
namespace {

// lower-triangular 3x3 matrices packed by rows: 00, 10, 11, 20, 21, 22
struct Lt6 {
    double m[6];
};

__device__ inline Lt6 pack_lt(const double (&M)[3][3])
{
    return Lt6{{M[0][0], M[1][0], M[1][1], M[2][0], M[2][1], M[2][2]}};
}

// row vector times lower-triangular matrix: o_j = sum_{i >= j} a_i M_ij
__device__ inline void row_lt(const Lt6& M, double a0, double a1, double a2, double& o0, double& o1,
                                       double& o2)
{
    o0 = a0 * M.m[0] + a1 * M.m[1] + a2 * M.m[3];
    o1 = a1 * M.m[2] + a2 * M.m[4];
    o2 = a2 * M.m[5];
}

// What an NST run keeps on the device between its steps.
struct NstState {
    double H[3][3], B_ref[3][3], vol_ref;
    double VH[3][3];                 // box velocity, lower triangle
    double S_pe[3][3];               // potential stress, lower triangle
    double eta_p[3], eta_b[3];       // the chains of the atoms and of the box
    double T_part, T_baro, mvv[6];   // mvv: sum of m v (x) v, voigt of the lower triangle
    double xi;                       // factor the velocities are due
    double com[3];                   // centre-of-mass displacement of the step
    double e[7];                     // energy and virial of the last forces
    Lt6 E, F0, F1, V;                // the step's update matrices and V_H
};
static_assert(sizeof(NstState) % sizeof(double) == 0);

struct NstArgs {
    double dt, dt2, kB, T, ndof, s_hyd, vol0, inv_q;
    double freq_p, freq_b;           // squared frequencies of the chains
    double S_dev[3][3], tau[3][3], prefac[3][3];
    int sdof[3][3], ndof_baro, natms;
};

struct MassInv {
    double m[kMaxElems], inv[kMaxElems];
};

// update_x_d__x__x_d, first half (src/md_nst.cpp:80-153): v <- xi v E +
// f F0 / m, the displacement u = (x V_H + v) F1, x <- x + u - c with the
// centre-of-mass displacement c that the end of the last step made of the sums
// of x, v and f / m; then DynamicMD::decide's skin check against the positions
// of the last build, and the 16-byte position record.
__global__ __launch_bounds__(kBlock) void k_nst_drift(int n, double4* __restrict__ x, double4* __restrict__ v,
                                                      const float4* __restrict__ f, MassInv M,
                                                      const NstState* __restrict__ st, const double4* __restrict__ x0,
                                                      double skin_sq4, int* __restrict__ flags, double inv_q,
                                                      uint4* __restrict__ rec)
{
    const int i = xcd_block() * kBlock + threadIdx.x;
    if (i >= n || flags[FL_HALT]) return;
    double4 xq = x[i];
    double4 vq = v[i];
    const float4 fq = f[i];
    const double4 a = x0[i];
    const double m_inv = M.inv[(int)xq.w], xi = st->xi;
    double a0, a1, a2, b0, b1, b2;
    row_lt(st->E, vq.x, vq.y, vq.z, a0, a1, a2);
    row_lt(st->F0, (double)fq.x, (double)fq.y, (double)fq.z, b0, b1, b2);
    vq.x = xi * a0 + m_inv * b0;
    vq.y = xi * a1 + m_inv * b1;
    vq.z = xi * a2 + m_inv * b2;
    double w0, w1, w2, u0, u1, u2;
    row_lt(st->V, xq.x, xq.y, xq.z, w0, w1, w2);
    w0 += vq.x;
    w1 += vq.y;
    w2 += vq.z;
    row_lt(st->F1, w0, w1, w2, u0, u1, u2);
    xq.x += u0;
    xq.y += u1;
    xq.z += u2;
    xq.x -= st->com[0];
    xq.y -= st->com[1];
    xq.z -= st->com[2];
    x[i] = xq;
    v[i] = vq;
    rec[i] = make_uint4((unsigned)__double2ll_rn(xq.x * inv_q), (unsigned)__double2ll_rn(xq.y * inv_q),
                        (unsigned)__double2ll_rn(xq.z * inv_q), (unsigned)(int)xq.w);
    if (rsq_exact(a.x, a.y, a.z, xq.x, xq.y, xq.z) > skin_sq4) atomicOr(&flags[FL_REBUILD], 1);
}

// entry c of the 128-entry image-shift table of the record grid (refresh_frame)
__device__ inline uint4 image_shift(const unsigned* cH, int c)
{
    uint4 sh = make_uint4(0u, 0u, 0u, 0u);
    if (c < 125) {
        const unsigned n0 = (unsigned)(c % 5 - 2), n1 = (unsigned)(c / 5 % 5 - 2), n2 = (unsigned)(c / 25 - 2);
        sh = make_uint4(n0 * cH[0] + n1 * cH[3] + n2 * cH[6], n1 * cH[4] + n2 * cH[7], n2 * cH[8], 0u);
    }
    return sh;
}

__global__ __launch_bounds__(128) void k_shift_table(Rec16Frame R, uint4* __restrict__ out)
{
    out[threadIdx.x] = image_shift(R.cH, threadIdx.x);
}

// second half (src/md_nst.cpp:133-152): v <- v E + f F0 / m when kick, and
// partial sums of the kinetic tensor m v (x) v, of v, of f / m and of x; a
// column of rows for each, since one workgroup adds them up
constexpr int kNstCols = 15;
__global__ __launch_bounds__(kBlock) void k_nst_kick(int n, const double4* __restrict__ x, double4* __restrict__ v,
                                                     const float4* __restrict__ f, MassInv M,
                                                     const NstState* __restrict__ st, int kick,
                                                     const int* __restrict__ flags, double* __restrict__ part)
{
    if (flags[FL_REBUILD]) return;
    double acc[kNstCols] = {};
    for (ChunkWalk w = chunk_walk(n, kBlock); w.c < w.end; w.c += w.step) {
        const int i = w.c * kBlock + threadIdx.x;
        if (i >= n) continue;
        const double4 xq = x[i];
        double4 vq = v[i];
        const float4 fq = f[i];
        const double m = M.m[(int)xq.w], m_inv = M.inv[(int)xq.w];
        if (kick) {
            double a0, a1, a2, b0, b1, b2;
            row_lt(st->E, vq.x, vq.y, vq.z, a0, a1, a2);
            row_lt(st->F0, (double)fq.x, (double)fq.y, (double)fq.z, b0, b1, b2);
            vq.x = a0 + m_inv * b0;
            vq.y = a1 + m_inv * b1;
            vq.z = a2 + m_inv * b2;
            v[i] = vq;
        }
        acc[0] += vq.x * vq.x * m;
        acc[1] += vq.y * vq.x * m;
        acc[2] += vq.z * vq.x * m;
        acc[3] += vq.y * vq.y * m;
        acc[4] += vq.z * vq.y * m;
        acc[5] += vq.z * vq.z * m;
        acc[6] += vq.x;
        acc[7] += vq.y;
        acc[8] += vq.z;
        acc[9] += (double)fq.x * m_inv;
        acc[10] += (double)fq.y * m_inv;
        acc[11] += (double)fq.z * m_inv;
        acc[12] += xq.x;
        acc[13] += xq.y;
        acc[14] += xq.z;
    }
    const double s = block_sums<kNstCols>(acc);
    if (threadIdx.x < kNstCols) part[(size_t)threadIdx.x * gridDim.x + blockIdx.x] = s;
}

__global__ __launch_bounds__(kBlock) void k_nst_scale_v(int n, double4* __restrict__ v,
                                                        const NstState* __restrict__ st)
{
    const int i = xcd_block() * kBlock + threadIdx.x;
    if (i >= n) return;
    const double s = st->xi;
    double4 q = v[i];
    q.x *= s;
    q.y *= s;
    q.z *= s;
    v[i] = q;
}

// ---------------- box and thermostats ----------------

// phi(x) = (e^x - 1) / x and its first two derivatives, by their Taylor
// series below |x| = 1/64 (MDMath::f, df, ddf, src/md_nst.cpp:843-871)
__device__ inline double phi0(double x)
{
    if (fabs(x) < 0.015625) return 1.0 + x / 2.0 + x * x / 6.0 + x * x * x / 24.0;
    return (exp(x) - 1.0) / x;
}
__device__ inline double phi1(double x)
{
    if (fabs(x) < 0.015625) return 0.5 + x / 3.0 + x * x / 8.0 + x * x * x / 30.0;
    const double e = exp(x);
    return (e - (e - 1.0) / x) / x;
}
__device__ inline double phi2(double x)
{
    if (fabs(x) < 0.015625) return 1.0 / 3.0 + x / 4.0 + x * x / 10.0 + x * x * x / 36.0;
    const double e = exp(x);
    return (e - 2.0 * ((e - (e - 1.0) / x) / x)) / x;
}

constexpr double kSqrtEps = 1.4901161193847656e-08;
constexpr double kEps = 2.220446049250313e-16;

// A function g of a lower-triangular 3x3 matrix Z from its values on the
// diagonal and their divided differences: g(Z)_ii = g(z_i), g(Z)_ij =
// z_ij g[z_i, z_j], g(Z)_20 = z_20 g[z_2, z_0] + z_21 z_10 g[z_0, z_1, z_2].
// Near-coincident nodes take the derivative at their mean (thresholds of
// src/md_nst.cpp:890-901, 960-986).
// is_exp: g = exp, else g = phi.
__device__ inline double tri_fn(bool is_exp, double x) { return is_exp ? exp(x) : phi0(x); }
__device__ inline double tri_d1(bool is_exp, double x, double y, double gx, double gy)
{
    const double m = 0.5 * (x + y);
    const double lim = is_exp ? kSqrtEps : sqrt(kEps * phi0(m) / phi2(m));
    if (fabs(x - y) < lim) return is_exp ? exp(m) : phi1(m);
    return (gx - gy) / (x - y);
}
__device__ inline double tri_d2(bool is_exp, double x, double y, double z, double g_yz, double g_zx, double g_xy)
{
    const double m = (x + y + z) / 3.0;
    const double lim = is_exp ? kSqrtEps : sqrt(kEps * phi0(m) / phi2(m));
    if (fabs(x - z) > lim) return (g_xy - g_yz) / (x - z);
    if (fabs(y - x) > lim) return (g_yz - g_zx) / (y - x);
    if (fabs(z - y) > lim) return (g_zx - g_xy) / (z - y);
    return is_exp ? exp(m) : phi2(m);
}

// ThermostatNHC(dt, t_relax, L = 3, niters = 1)::operator() (src/thermostat.cpp:47-143)
__device__ inline double nhc_step(double* e, double ddt, double freq_sq, double T_r, int ndof)
{
    const double ddt2 = 0.5 * ddt;
    double rescale = 1.0, prev, tmp;
    e[2] += ddt2 * (e[1] * e[1] - freq_sq);
    prev = -e[2];
    e[1] += ddt2 * phi0(prev * ddt2) * (prev * e[1] + e[0] * e[0] - freq_sq);
    prev = -e[1];
    e[0] += ddt2 * phi0(prev * ddt2) * (prev * e[0] + freq_sq * (T_r - 1.0));
    prev = -e[0];
    tmp = exp(ddt * prev);
    rescale *= tmp;
    T_r *= tmp * tmp;
    prev = (T_r - 1.0) * freq_sq;
    e[0] += ddt2 * phi0(-e[1] * ddt2) * (-e[1] * e[0] + prev);
    prev = ndof * e[0] * e[0] - freq_sq;
    e[1] += ddt2 * phi0(-e[2] * ddt2) * (-e[2] * e[1] + prev);
    prev = e[1] * e[1] - freq_sq;
    e[2] += ddt2 * prev;
    return rescale;
}

__host__ __device__ inline int lt_voigt(int i, int j) { return i + j * 3 - j * (j + 1) / 2; }

// MDNST::update_V_H (src/md_nst.cpp:320-351)
__device__ inline void update_VH(NstState& s, const NstArgs& A)
{
    const double vol = s.H[0][0] * (s.H[1][1] * s.H[2][2]);
    double L[3][3] = {}, SL[3][3] = {}, M2[3][3] = {};
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j <= i; ++j)
            for (int k = j; k <= i; ++k) L[i][j] += s.B_ref[i][k] * s.H[k][j];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j < 3; ++j)
            for (int k = 0; k < 3; ++k) SL[i][j] += A.S_dev[i][k] * L[k][j];
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j <= i; ++j)
            for (int k = 0; k < 3; ++k) M2[i][j] += L[k][i] * SL[k][j];
    for (int i = 0; i < 3; ++i)
        if (A.sdof[i][i]) s.VH[i][i] += (A.kB * s.T_part + vol * A.s_hyd) * A.prefac[i][i] * A.dt2;
    s.T_baro = 0.0;
    for (int j = 0; j < 3; ++j)
        for (int i = j; i < 3; ++i) {
            if (!A.sdof[i][j]) continue;
            s.VH[i][j] += (s.vol_ref * M2[i][j] - vol * s.S_pe[i][j] + s.mvv[lt_voigt(i, j)]) * A.prefac[i][j] * A.dt2;
            s.T_baro += s.VH[i][j] * s.VH[i][j] * A.tau[i][j] * A.tau[i][j];
        }
    s.T_baro *= A.ndof * A.T / A.ndof_baro;
}

// The end of an NST step on one workgroup: the sums of the second half and of
// the force passes, the stress, the second half of the box velocity and both
// thermostats; then, unless it was the last step, what the next one needs: its
// thermostats, V_H, the update matrices (MDMath::calc, src/md_nst.cpp:887-1002:
// E = exp(-dt2 (V_H + a I)), F0 = dt2 phi(-dt2 (V_H + a I)), F1 = dt phi(dt
// V_H)), the centre-of-mass displacement, the new box H (I + F1 V_H) and the
// image shifts. start: before the first step. A wave sums a column. The
// algebra is a short serial chain, and what it costs is the fetch of code that
// runs once: so both half-steps go through the same code, the two thermostats
// side by side on two lanes and the nine values of the matrix functions on
// nine (13 us; 23 with all of it inlined on one lane). With the algebra on the
// host, which cost six reductions and two round trips, a step of 260,000 atoms
// took 240 us; with this kernel 157, of which the force passes take 75.
// told: steps done; 1 where the list is to be rebuilt, 2 where the box left
// its bounds.
constexpr int kNstEndThreads = 512;
__global__ __launch_bounds__(kNstEndThreads) void k_nst_end(NstState* __restrict__ st, const double* __restrict__ cols,
                                                            int nc, const double* __restrict__ rows_e, int ne,
                                                            NstArgs A, int start, int last, int reset,
                                                            double* __restrict__ hist, int* __restrict__ flags,
                                                            uint4* __restrict__ shift, volatile int* __restrict__ told)
{
    __shared__ NstState s;
    __shared__ double sum[kNstCols + 7], fac[2], zs[3][3], gs[3][3], ds[3][3];
    __shared__ unsigned cH[9];
    const int t = threadIdx.x, lane = t & 63;
    const int rebuild = flags[FL_REBUILD], halt = flags[FL_HALT];
    constexpr int kWords = sizeof(NstState) / sizeof(double);
    static_assert(kWords <= kNstEndThreads);
    if (t < kWords) reinterpret_cast<double*>(&s)[t] = reinterpret_cast<const double*>(st)[t];
    if (!rebuild)
        for (int c = t >> 6; c < kNstCols + 7; c += kNstEndThreads / 64) {
            const bool kin = c < kNstCols;
            const double* p = kin ? cols + (size_t)c * nc : rows_e + (c - kNstCols);
            const int nr = kin ? nc : ne, ld = kin ? 1 : kPartW;
            double a[1] = {0.0};
#pragma unroll 8
            for (int r = lane; r < nr; r += 64) a[0] += p[(size_t)r * ld];
            wave_sums<1>(a);
            if (lane == 0) sum[c] = a[0];
        }
    __syncthreads();
    if (halt) return;
    if (rebuild) {
        if (t == 0) {
            flags[FL_HALT] = 1;
            told[1] = 1;
        }
        return;
    }
    const double vol = s.H[0][0] * (s.H[1][1] * s.H[2][2]);
    if (t == 0) {
        for (int k = 0; k < 7; ++k) s.e[k] = sum[kNstCols + k];
        for (int k = 0; k < 6; ++k) s.mvv[k] = sum[k];
        s.T_part = (s.mvv[0] + (s.mvv[3] + s.mvv[5])) / (A.ndof * A.kB);
        for (int j = 0; j < 3; ++j)
            for (int i = j; i < 3; ++i) s.S_pe[i][j] = -s.e[1 + lt_voigt(i, j)] / vol;
        s.xi = 1.0;
    }
    __syncthreads();
    // second half: V_H (0), thermostats (1); the next step's first half:
    // thermostats (2), V_H (3)
    bool go = false;
#pragma unroll 1
    for (int phase = start ? 2 : 0; phase < 4; ++phase) {
        if (phase == 2) {
            go = !last && vol > 0.125 * A.vol0 && vol < 8.0 * A.vol0 && isfinite(s.T_part);
            if (t == 0) {
                if (start || reset) {
                    const Box bx = make_box(&s.H[0][0]);
                    for (int i = 0; i < 3; ++i)
                        for (int j = 0; j < 3; ++j) s.B_ref[i][j] = bx.B[i][j];
                    s.vol_ref = vol;
                }
                if (!start) {
                    if (hist) {
                        hist[0] = s.T_part;
                        hist[1] = s.e[0];
                        for (int i = 0, k = 2; i < 3; ++i)
                            for (int j = 0; j <= i; ++j) hist[k++] = s.H[i][j];
                        for (int j = 0; j < 3; ++j)
                            for (int i = j; i < 3; ++i) hist[8 + lt_voigt(i, j)] = s.S_pe[i][j];
                    }
                    told[0] = flags[FL_DONE] += 1;
                }
                if (!last && !go) {
                    flags[FL_HALT] = 1;
                    flags[FL_REBUILD] = 1;
                    told[1] = 2;
                }
            }
            __syncthreads();
            if (!go) break;
        }
        if (phase == 0 || phase == 3) {
            if (t == 0) update_VH(s, A);
        } else {
            if (t < 2)
                fac[t] = nhc_step(t ? s.eta_b : s.eta_p, A.dt2, t ? A.freq_b : A.freq_p,
                                  (t ? s.T_baro : s.T_part) / A.T, t ? A.ndof_baro : (int)A.ndof);
            __syncthreads();
            if (t == 0) {
                const double p2 = fac[0] * fac[0];
                s.xi *= fac[0];
                for (int k = 0; k < 6; ++k) s.mvv[k] *= p2;
                s.T_part *= p2;
                for (int i = 0; i < 3; ++i)
                    for (int j = 0; j <= i; ++j) s.VH[i][j] *= fac[1];
                s.T_baro *= fac[1] * fac[1];
            }
        }
        __syncthreads();
    }
    if (go) {
        // the matrix functions: E, F0 and F1 are g(s_q (V_H + a_q I)) times o_q
        const double a = (s.VH[0][0] + s.VH[1][1] + s.VH[2][2]) / A.ndof;
        const int q = t < 9 ? t / 3 : t < 12 ? t - 9 : 0;
        const double sq = q < 2 ? -A.dt2 : A.dt, aq = q < 2 ? a : 0.0;
        if (t < 9) {
            const int i = t % 3;
            zs[q][i] = sq * (s.VH[i][i] + aq);
            gs[q][i] = tri_fn(q == 0, zs[q][i]);
        }
        __syncthreads();
        if (t < 9) {  // divided differences of z1, z0 (0), z2, z0 (1) and z2, z1 (2)
            const int p = t % 3, i = p == 0 ? 1 : 2, j = p == 2 ? 1 : 0;
            ds[q][p] = s.VH[i][j] != 0.0 ? tri_d1(q == 0, zs[q][i], zs[q][j], gs[q][i], gs[q][j]) : 0.0;
        }
        __syncthreads();
        if (t >= 9 && t < 12) {
            const double oq = q == 0 ? 1.0 : q == 1 ? A.dt2 : A.dt;
            const double(&V)[3][3] = s.VH;
            Lt6 G{{oq * gs[q][0], oq * sq * V[1][0] * ds[q][0], oq * gs[q][1], oq * sq * V[2][0] * ds[q][1],
                   oq * sq * V[2][1] * ds[q][2], oq * gs[q][2]}};
            if (V[1][0] != 0.0 && V[2][1] != 0.0)
                G.m[3] += oq * sq * sq * V[2][1] * V[1][0] *
                          tri_d2(q == 0, zs[q][0], zs[q][1], zs[q][2], ds[q][2], ds[q][1], ds[q][0]);
            (q == 0 ? s.E : q == 1 ? s.F0 : s.F1) = G;
        }
        __syncthreads();
        if (t == 0) {
            s.V = pack_lt(s.VH);
            const double *sv = sum + 6, *sf = sum + 9, *sx = sum + 12;
            double a0, a1, a2, b0, b1, b2, w0, w1, w2;
            row_lt(s.E, sv[0], sv[1], sv[2], a0, a1, a2);
            row_lt(s.F0, sf[0], sf[1], sf[2], b0, b1, b2);
            row_lt(s.V, sx[0], sx[1], sx[2], w0, w1, w2);
            w0 += s.xi * a0 + b0;
            w1 += s.xi * a1 + b1;
            w2 += s.xi * a2 + b2;
            row_lt(s.F1, w0, w1, w2, s.com[0], s.com[1], s.com[2]);
            for (int k = 0; k < 3; ++k) s.com[k] /= (double)A.natms;
            const double* f = s.F1.m;
            const double F1[3][3] = {{f[0], 0.0, 0.0}, {f[1], f[2], 0.0}, {f[3], f[4], f[5]}};
            double G[3][3] = {}, Hn[3][3] = {};
            for (int i = 0; i < 3; ++i)
                for (int j = 0; j <= i; ++j) {
                    for (int k = j; k <= i; ++k) G[i][j] += F1[i][k] * s.VH[k][j];
                    if (i == j) G[i][j] += 1.0;
                }
            for (int i = 0; i < 3; ++i)
                for (int j = 0; j <= i; ++j)
                    for (int k = j; k <= i; ++k) Hn[i][j] += s.H[i][k] * G[k][j];
            for (int i = 0; i < 3; ++i)
                for (int j = 0; j < 3; ++j) {
                    s.H[i][j] = Hn[i][j];
                    cH[3 * i + j] = (unsigned)(unsigned long long)llrint(Hn[i][j] * A.inv_q);
                }
        }
        __syncthreads();
        if (t < 128) shift[t] = image_shift(cH, t);
    }
    if (t < kWords) reinterpret_cast<double*>(st)[t] = reinterpret_cast<const double*>(&s)[t];
}

}  // namespace

// Image shifts of the 16-byte records for the current box (the record grid q
// depends on the cut-off only), made on the device in stream order so that a
// box change costs no host synchronisation: code c = (n0+2) + 5(n1+2) +
// 25(n2+2) shifts by n0 h0 + n1 h1 + n2 h2 on the grid (modulo 2^32); codes
// 125..127 are unused
void MDSystem::refresh_frame()
{
    for (int k = 0; k < 3; ++k)
        for (int d = 0; d < 3; ++d)
            r16_.cH[3 * k + d] = (unsigned)(unsigned long long)std::llrint(box_.H[k][d] * r16_.inv_q);
    shift_.reserve(128);
    hipLaunchKernelGGL(k_shift_table, dim3(1), dim3(128), 0, stream_, r16_, shift_.get());
    r16_.shift = shift_.get();
}

int MDSystem::nst_run(const double* masses, double kB, double T, double dt, const double* S9, const double* tau9,
                      int nreset, int nsteps, MDReport* rep, double* T_part_out, double* H9, double* hist)
{
    MAPP_REQUIRE(nsteps >= 0 && dt > 0.0 && T > 0.0 && kB > 0.0 && nreset >= 0, ERR_ARG, "invalid NST parameters");
    const EamTables& t = ff_->tables();
    MassInv M{};
    for (int a = 0; a < t.ne; ++a) {
        MAPP_REQUIRE(masses[a] > 0.0, ERR_ARG, "masses must be positive");
        M.m[a] = masses[a];
        M.inv[a] = 1.0 / masses[a];
    }
    NstArgs A{};
    A.dt = dt;
    A.dt2 = dt / 2.0;
    A.kB = kB;
    A.T = T;
    A.ndof = 3.0 * n_;
    A.natms = n_;
    A.inv_q = r16_.inv_q;
    A.freq_p = 1.0 / ((100.0 * dt) * (100.0 * dt));
    A.freq_b = 1.0 / ((1000.0 * dt) * (1000.0 * dt));
    A.vol0 = box_.vol;
    // pre_init (src/md_nst.cpp:291-319): free components (NaN) carry no box
    // motion; S_dev keeps the target's lower triangle, less the hydrostatic
    // part on the diagonal
    double S[3][3] = {};
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j <= i; ++j) {
            A.tau[i][j] = tau9 ? tau9[3 * i + j] : 1000.0 * dt;
            MAPP_REQUIRE(A.tau[i][j] > 0.0, ERR_ARG, "tau must be positive");
            if (std::isnan(S9[3 * i + j])) continue;
            A.sdof[i][j] = 1;
            S[i][j] = S9[3 * i + j];
            A.prefac[i][j] = 1.0 / (A.tau[i][j] * A.tau[i][j] * A.ndof * kB * T);
            ++A.ndof_baro;
        }
    MAPP_REQUIRE(A.ndof_baro > 0, ERR_ARG, "at least one stress component must be set (not NaN)");
    A.s_hyd = (S[0][0] + S[1][1] + S[2][2]) / 3.0;
    for (int i = 0; i < 3; ++i)
        for (int j = 0; j <= i; ++j) A.S_dev[i][j] = S[i][j] - (i == j ? A.s_hyd : 0.0);

    const int nb = grid_for(n_), nk = std::min(kStepRows, nb);
    double* cols = part_.get() + (size_t)2 * part_rows() * kPartW;
    nst_.reserve(sizeof(NstState) / sizeof(double));
    NstState* st = reinterpret_cast<NstState*>(nst_.get());
    NstState s{};
    std::memcpy(s.H, box_.H, sizeof s.H);
    MAPP_HIP(hipMemcpyAsync(st, &s, sizeof s, hipMemcpyHostToDevice, stream_));
    MAPP_HIP(hipMemsetAsync(flags_.get() + 1, 0, sizeof(int) * 3, stream_));
    if (hist) hist_.reserve(std::max((size_t)1, (size_t)14 * nsteps));
    const double skin_sq4 = 0.25 * skin_ * skin_;
    const int rebuilds0 = nrebuild_;
    const auto drift = [&]() {
        prof_.begin(K_INTEGRATE, stream_);
        hipLaunchKernelGGL(k_nst_drift, dim3(nb), dim3(kBlock), 0, stream_, n_, x_.get(), v_.get(), f_.get(), M, st,
                           x0_.get(), skin_sq4, flags_.get(), r16_.inv_q, rec_.get());
        prof_.end(stream_);
    };
    // the forces, the second half and the end of a step (-1: before the first)
    const auto finish = [&](int step) {
        force_passes(nullptr, step >= 0, nullptr, nullptr, true, flags_.get() + FL_REBUILD, true);
        const bool deferred = 2 * pass_rows_ <= kStepRows;
        prof_.begin(K_INTEGRATE, stream_);
        hipLaunchKernelGGL(k_nst_kick, dim3(nk), dim3(kBlock), 0, stream_, n_, x_.get(), v_.get(), f_.get(), M, st,
                           step >= 0 ? 1 : 0, flags_.get(), cols);
        hipLaunchKernelGGL(k_nst_end, dim3(1), dim3(kNstEndThreads), 0, stream_, st, cols, nk,
                           deferred ? part_.get() : red_.get(), deferred ? 2 * pass_rows_ : 1, A, step < 0 ? 1 : 0,
                           step + 1 >= nsteps ? 1 : 0, nreset && (step + 1) % nreset == 0 ? 1 : 0,
                           hist ? hist_.get() + (size_t)14 * std::max(0, step) : nullptr, flags_.get(), shift_.get(),
                           told_.get());
        prof_.end(stream_);
    };
    const auto fetch = [&]() {
        MAPP_HIP(hipMemcpyAsync(&s, st, sizeof s, hipMemcpyDeviceToHost, stream_));
        MAPP_HIP(hipStreamSynchronize(stream_));
        box_ = make_box(&s.H[0][0]);
    };
    // groups of steps as in an NVT run: what follows a step that finds the
    // list due does nothing, and the host reads the answers after a group
    volatile int* told = told_.get();
    int interval = 12, since = 0, step = 0, base = 0;
    told[0] = told[1] = 0;
    finish(-1);
    while (step < nsteps) {
        int group = prof_.on ? 1 : std::max(2, std::min(64, interval - 2 - since));
        group = std::min(group, nsteps - step);
        size_t timed = 0;
        for (int k = 0; k < group; ++k) {
            drift();
            timed = prof_.mark();
            finish(step + k);
        }
        MAPP_HIP(hipStreamSynchronize(stream_));
        if (told[1] == 1) prof_.drop(timed);  // its passes returned at once
        prof_.flush();
        const int done = told[0] - base;
        step += done;
        since += done;
        base += done;
        if (!told[1]) continue;
        fetch();
        if (told[1] == 2) {
            refresh_frame();
            throw Error(ERR_STATE, "the box left [vol0 / 8, 8 vol0]: NST run stopped");
        }
        setup_grid();
        rebuild();  // the permute rewrites the records
        interval = since + 1;
        MAPP_HIP(hipMemsetAsync(flags_.get() + 1, 0, sizeof(int) * 3, stream_));
        told[0] = told[1] = 0;
        finish(step);
        ++step;
        since = 0;
        base = 1;
    }
    hipLaunchKernelGGL(k_nst_scale_v, dim3(nb), dim3(kBlock), 0, stream_, n_, v_.get(), st);
    if (hist && nsteps > 0)
        MAPP_HIP(hipMemcpyAsync(hist, hist_.get(), sizeof(double) * 14 * nsteps, hipMemcpyDeviceToHost, stream_));
    fetch();
    refresh_frame();
    prof_.flush();
    MDReport r{};
    std::memcpy(r.e, s.e, sizeof r.e);
    if (rep) *rep = r;
    if (T_part_out) *T_part_out = s.T_part;
    if (H9)
        for (int k = 0; k < 9; ++k) H9[k] = box_.H[k / 3][k % 3];
    return nrebuild_ - rebuilds0;
}

}  // namespace mapp
