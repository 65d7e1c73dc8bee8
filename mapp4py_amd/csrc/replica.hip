// replica.hip -- batched energy minimisation of many small periodic cells.
//
// Reference behaviour restated here, per replica:
//   MinCG::__run (conjugate gradients, Polak-Ribiere)   src/min_cg.h:453-533
//   MinMDHandler::ls_prep / F / F_reset               src/min_cg.h:231-278
//   LineSearchBackTrack::min (init_flag 1)            src/ls.h:711-769
//   ForceFieldEAM::__force_calc / __energy_calc       src/ff_eam.cpp:99-318
//   DynamicMD::decide (skin check, rebuild)           src/dynamic_md.cpp:90-105
//
// Design: a replica's minimisation is sequential, so the parallelism is
// across replicas and, inside one, across its atoms. One wave or a whole
// workgroup of 4 or 16 waves owns a replica for the entire minimisation: its
// full neighbor list (every periodic image, 7-bit image codes), both EAM
// passes in FP64, the inner products and the line search all run inside the
// one persistent launch, with no host round trip per step. The size classes
// are split between the shapes by a rule on the batch (default_waves) or by a
// tuner that times every threshold on a copy of it. All arithmetic is
// FP64 with contraction off, so energies and line-search decisions are the
// reference's to the rounding of the sums.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>

#include "box.hpp"
#include "kern.hpp"
#include "replica.hpp"

#pragma clang fp contract(off)

namespace mapp {

namespace {

// the reference's error codes (src/min.cpp:7-25, src/ls.h)
enum { LS_S = 0, LS_F_DOWNHILL = 1, LS_F_GRAD0 = 2, LS_MIN_ALPHA = 3, MIN_S_TOLERANCE = 4, MIN_F_MAX_ITER = 5 };
enum { FAIL_LIST = 101, FAIL_IMAGE = 102 };

int rep_class_of(int n)
{
    if (n < 256) return 0;
    if (n < 512) return 1;
    if (n < 1024) return 2;
    if (n < 2048) return 3;
    return 4;
}

__device__ inline double hval(const double4 c, double p) { return ((c.w * p + c.z) * p + c.y) * p + c.x; }
__device__ inline double dhval(const double4 c, double p) { return (3.0 * c.w * p + 2.0 * c.z) * p + c.y; }

__device__ inline void spline_at(double v, double inv, int n, int& m, double& p)
{
    p = v * inv;
    int mm = (int)p;
    mm = mm < n - 2 ? mm : n - 2;
    mm = mm > 0 ? mm : 0;
    p -= (double)mm;
    p = p < 1.0 ? p : 1.0;
    m = mm;
}

__device__ inline int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ inline double uni(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
    const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Waves of the workgroup that owns a replica. Where the largest replica's
// chain of steps ends the launch, it gets every wave a CU can hold at 128
// registers a lane. 1024 Ni-H cells of 108 to 4,076 atoms, 20 steps each: 390
// ms with four waves, all-pairs list builds and one entry after another in the
// passes, 59 ms now. In the largest cell a density pass takes 0.31 ms (its
// issue bound, 4 atoms a lane, is about 0.15), a force pass 0.44 and a list
// build 2.3, of 20 steps' 40 density and 20 force passes and 8 builds.
// Where there are more small replicas than CUs, four workgroups of 4 waves a
// CU (wide_workgroup).
constexpr int kWide = 16, kNarrow = 4;
constexpr int kShifts = 125;  // image codes

template <int K>  // waves of the workgroup
struct Shared {
    double red[2][K];             // partial sums, two rows in turn
    double shift[K][kShifts][3];  // n H of every image code: row 0 of a workgroup's replica, row w of a wave's
    int own0[65 * K];             // list build: where each cell's (segment's) atoms start in ord,
    int cand0[65 * K];            // and its candidates; 65 a wave or all for a workgroup
    double cut_sq[kMaxElems * kMaxElems], cutsk_sq[kMaxElems * kMaxElems];
    int next;
};

template <int W>
__device__ inline void group_sync()
{
    if constexpr (W == 1) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

struct Ctx {
    int off, n, maxn, nt, t, w;
    int lg;    // log2 of the lanes that share an atom in the EAM passes
    int flip;  // row of red of the next sum
    long long loff;
    double h[6], b[6], cs[3];
    // the replica's parts of Shared
    double* red;
    double (*shift)[3];
    int *own0, *cand0;
    const double *cut_sq, *cutsk_sq;
};

// sums and maxima over the replica's lanes, in a fixed order, returned alike
// to every lane. A row of partial sums is written again only after the
// barrier of the reduction in between, so one barrier each is enough; it also
// orders the replica's memory, as group_sync does.
template <int W, class Op>
__device__ inline double group_fold(double v, Ctx& C, Op op)
{
    for (int off = 32; off > 0; off >>= 1) v = op(v, __shfl_xor(v, off, 64));
    v = uni(v);
    if constexpr (W == 1) {
        group_sync<1>();
        return v;
    } else {
        double* row = C.red + C.flip * W;
        C.flip ^= 1;
        row[C.w] = v;
        __syncthreads();
        double s = row[0];
        for (int k = 1; k < W; ++k) s = op(s, row[k]);
        return uni(s);
    }
}
template <int W>
__device__ inline double group_sum(double v, Ctx& C)
{
    return group_fold<W>(v, C, [](double a, double b) { return a + b; });
}
template <int W>
__device__ inline double group_max(double v, Ctx& C)
{
    return group_fold<W>(v, C, [](double a, double b) { return fmax(a, b); });
}

// x -> s = x B without the wrap (the positions move freely during a
// minimisation; image codes are taken relative to the current positions)
__device__ inline void to_s(const double* b, const double4& x, double* s)
{
    s[0] = b[0] * x.x + (b[1] * x.y + b[2] * x.z);
    s[1] = b[3] * x.y + b[4] * x.z;
    s[2] = b[5] * x.z;
}

// x_i - (x_j + n H) of an image code
__device__ inline void image_dx(const double (*shift)[3], const double4& xi, const double4& xj, uint32_t code,
                                double& dx, double& dy, double& dz)
{
    const double* sh = shift[code];
    dx = xi.x - (xj.x + sh[0]);
    dy = xi.y - (xj.y + sh[1]);
    dz = xi.z - (xj.z + sh[2]);
}

// The full list of the replica: every (j, image) with |x_i - x_j - n H| below
// r_c + skin, except i itself at the zero image. Returns a failure code (0 ok).
// The atoms are binned into cells at least as wide as the cut-off's extent
// along each box vector (their s wrapped into the box), and the candidates of
// a cell's atoms are the atoms of the 27 cells around it; comparing all pairs
// took 7.5 ms a build at 4,076 atoms, most of the launch (2.3 ms now). Candidates are
// collected in index order (a group of lanes scans all atoms for each cell, a
// segment each), so a row lists its neighbors in the order of (j, image): its
// sums do not depend on when it was built. Rows are worked on in cell order,
// so that the lanes of a wave read the same candidates.
template <int W>
__device__ int build_list(const RepArgs& A, Ctx& C, const RepArrays& R)
{
    constexpr int kCells = 64 * W;  // most cells, and cells times segments
    const int ne = A.ne;
    int *own0 = C.own0, *cand0 = C.cand0;
    int* ord = R.ord + C.off;
    uint32_t* cand = R.cand + 27 * (size_t)C.off;
    int nc[3];
    for (int d = 0; d < 3; ++d) {
        const double k = 1.0 / (C.cs[d] * 1.0000001), most = kCells < 256 ? kCells : 256;
        nc[d] = (int)(k < most ? k : most);
        nc[d] = nc[d] > 1 ? nc[d] : 1;
    }
    while (nc[0] * nc[1] * nc[2] > kCells) {
        const int d = nc[0] >= nc[1] && nc[0] >= nc[2] ? 0 : nc[1] >= nc[2] ? 1 : 2;
        nc[d] = (nc[d] + 1) / 2;
    }
    const int ncell = nc[0] * nc[1] * nc[2];
    int nseg = 1;
    while (2 * nseg * ncell <= C.nt && nseg < 16) nseg *= 2;
    const int seg = (C.n + nseg - 1) / nseg;
    // how many boxes away from the origin the atoms lie, per box vector
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    for (int i = C.t; i < C.n; i += C.nt) {
        double s[3];
        to_s(C.b, R.x[C.off + i], s);
        for (int d = 0; d < 3; ++d) {
            lo[d] = fmin(lo[d], floor(s[d]));
            hi[d] = fmax(hi[d], floor(s[d]));
        }
    }
    // In a box of at least 3 cells along each vector, whose atoms lie in one
    // box or the next, a candidate can be listed at one image only, which its
    // cell gives: the entry of cand then holds the image's code too.
    bool fast = true;
    for (int d = 0; d < 3; ++d) {
        lo[d] = -group_max<W>(-lo[d], C);
        hi[d] = group_max<W>(hi[d], C);
        fast = fast && nc[d] >= 3 && hi[d] - lo[d] <= 1.0;
    }
    // cid: 8 bits of cell per box vector, then one each for lying in the next box
    for (int i = C.t; i < C.n; i += C.nt) {
        const double4 xi = R.x[C.off + i];
        R.xb[C.off + i] = xi;
        double s[3];
        to_s(C.b, xi, s);
        int id = 0;
        for (int d = 0; d < 3; ++d) {
            const double w = floor(s[d]);
            const int c = (int)((s[d] - w) * nc[d]);
            id |= (c < nc[d] - 1 ? c : nc[d] - 1) << (8 * d) | (w > lo[d] ? 1 << (24 + d) : 0);
        }
        R.cid[C.off + i] = id;
    }
    group_sync<W>();
    // 0: own cell, 1: a cell next to it (through the box faces too), 2: neither;
    // the code of the candidate's image
    auto relation = [&](int id, const int* c, uint32_t& code) {
        int rel = 0, step = 1, k = kZeroImage;
        for (int d = 0; d < 3; ++d, step *= 5) {
            const int e = (id >> (8 * d) & 255) - c[d];
            const int r = e == 0 ? 0 : e == 1 || e == -1 || e == nc[d] - 1 || e == 1 - nc[d] ? 1 : 2;
            rel = r > rel ? r : rel;
            k += step * ((e == 1 - nc[d] ? 1 : e == nc[d] - 1 ? -1 : 0) - (id >> (24 + d) & 1));
        }
        code = fast ? (uint32_t)k << kIndexBits : 0u;
        return rel;
    };
    for (int fill = 0; fill < 2; ++fill) {
        for (int u = C.t; u < ncell * nseg; u += C.nt) {
            const int cc = u / nseg;
            const int c[3] = {cc % nc[0], cc / nc[0] % nc[1], cc / (nc[0] * nc[1])};
            const int j0 = (u & (nseg - 1)) * seg, j1 = j0 + seg < C.n ? j0 + seg : C.n;
            int ko = fill ? own0[u] : 0, kc = fill ? cand0[u] : 0;
            for (int jb = j0; jb < j1; jb += 4) {
                int id[4];
                for (int b = 0; b < 4; ++b) id[b] = R.cid[C.off + (jb + b < j1 ? jb + b : jb)];
                for (int b = 0; b < 4; ++b) {
                    const int j = jb + b;
                    uint32_t code = 0u;
                    const int rel = j < j1 ? relation(id[b], c, code) : 2;
                    if (rel < 2 && fill) cand[kc] = (uint32_t)j | code;
                    if (rel == 0 && fill) ord[ko] = j;
                    kc += rel < 2 ? 1 : 0;
                    ko += rel == 0 ? 1 : 0;
                }
            }
            if (!fill) {
                own0[u] = ko;
                cand0[u] = kc;
            }
        }
        group_sync<W>();
        if (!fill && C.t == 0) {
            int ko = 0, kc = 0;
            for (int u = 0; u < ncell * nseg; ++u) {
                const int o = own0[u], k = cand0[u];
                own0[u] = ko;
                cand0[u] = kc;
                ko += o;
                kc += k;
            }
            cand0[ncell * nseg] = kc;
        }
        group_sync<W>();
    }
    // a sphere thinner than half the box along every box vector holds one
    // image of an atom at most, the nearest
    const bool nearest = C.cs[0] < 0.499 && C.cs[1] < 0.499 && C.cs[2] < 0.499;
    double fail = 0.0;
    for (int q = C.t; q < C.n; q += C.nt) {
        const int i = ord[q];
        const int id = R.cid[C.off + i];
        const double4 xi = R.x[C.off + i];
        const int ei = (int)xi.w;
        const int cell = (id & 255) + nc[0] * ((id >> 8 & 255) + nc[1] * (id >> 16 & 255));
        double si[3];
        to_s(C.b, xi, si);
        int cnt = 0;
        auto visit = [&](int j, const double4& xj, uint32_t code) {
            double dx, dy, dz;
            image_dx(C.shift, xi, xj, code, dx, dy, dz);
            const double rsq = dx * dx + (dy * dy + dz * dz);
            if (rsq < C.cutsk_sq[ei * ne + (int)xj.w] && (j != i || code != (uint32_t)kZeroImage)) {
                if (cnt < C.maxn) R.list[C.loff + (long long)cnt * C.n + i] = (uint32_t)j | (code << kIndexBits);
                ++cnt;
            }
        };
        // the next candidate's position and the entry after it are loaded
        // while one is looked at
        const int kb = cand0[cell * nseg], ke = cand0[(cell + 1) * nseg];
        const uint32_t wrap = (uint32_t)((id >> 24 & 1) + 5 * (id >> 25 & 1) + 25 * (id >> 26 & 1));
        uint32_t en = cand[kb], enn = cand[kb + 1 < ke ? kb + 1 : kb];
        double4 xn = R.x[C.off + (int)(en & kIndexMask)];
        for (int k = kb; k < ke; ++k) {
            const uint32_t e = en;
            const int j = (int)(e & kIndexMask);
            const double4 xj = xn;
            en = enn;
            xn = R.x[C.off + (int)(en & kIndexMask)];
            enn = cand[k + 2 < ke ? k + 2 : ke - 1];
            if (fast) {
                visit(j, xj, (e >> kIndexBits) + wrap);
                continue;
            }
            double ds[3];
            to_s(C.b, xj, ds);
            for (int d = 0; d < 3; ++d) ds[d] = si[d] - ds[d];
            if (nearest) {
                const double n0 = rint(ds[0]), n1 = rint(ds[1]), n2 = rint(ds[2]);
                if (fmax(fabs(ds[0] - n0) - C.cs[0], fmax(fabs(ds[1] - n1) - C.cs[1], fabs(ds[2] - n2) - C.cs[2])) > 0.0)
                    continue;
                if (fmax(fabs(n0), fmax(fabs(n1), fabs(n2))) > (double)kRepMaxImages)
                    fail = fmax(fail, (double)FAIL_IMAGE);
                else
                    visit(j, xj, (uint32_t)(int)(n0 + 5.0 * n1 + 25.0 * n2 + (double)kZeroImage));
                continue;
            }
            // the images in reach along every vector, of those that have a code
            double lo[3], hi[3];
            bool any = true, far = false;
            for (int d = 0; d < 3; ++d) {
                const double a = ceil(ds[d] - C.cs[d]), b = floor(ds[d] + C.cs[d]);
                any = any && a <= b;
                far = far || a < -(double)kRepMaxImages || b > (double)kRepMaxImages;
                lo[d] = fmax(a, -(double)kRepMaxImages);
                hi[d] = fmin(b, (double)kRepMaxImages);
            }
            if (any && far) fail = fmax(fail, (double)FAIL_IMAGE);
            if (!any) continue;
            for (double n2 = lo[2]; n2 <= hi[2]; n2 += 1.0)
                for (double n1 = lo[1]; n1 <= hi[1]; n1 += 1.0)
                    for (double n0 = lo[0]; n0 <= hi[0]; n0 += 1.0)
                        visit(j, xj, (uint32_t)(int)(n0 + 5.0 * n1 + 25.0 * n2 + (double)kZeroImage));
        }
        if (cnt > C.maxn) fail = fmax(fail, (double)FAIL_LIST);
        R.nn[C.off + i] = cnt < C.maxn ? cnt : C.maxn;
    }
    return (int)group_max<W>(fail, C);
}

// B list entries k0 .. k0 + B - 1 of atom i with their neighbors' positions,
// all loads in flight together (a pass on its own waits for list, position
// and spline row of one entry after another): entries past the row's end
// repeat its last one and are marked out.
template <int B>
__device__ inline void fetch(const Ctx& C, const RepArrays& R, int i, int cnt, int k0, uint32_t (&e)[B],
                             double4 (&xj)[B])
{
    for (int b = 0; b < B; ++b) {
        const int k = k0 + b < cnt ? k0 + b : cnt - 1;
        e[b] = R.list[C.loff + (long long)k * C.n + i];
    }
    for (int b = 0; b < B; ++b) xj[b] = R.x[C.off + (int)(e[b] & kIndexMask)];
}

// The density pass of ForceFieldEAM: E = sum_i F(rho_i) + 1/2 sum over the
// full list of phi; F extended linearly past rho_max (src/ff_eam.cpp:181-192,
// 313-314); leaves F'(rho_i) in dF. 2^lg lanes share an atom's entries.
template <int W>
__device__ double eam_energy(const RepArgs& A, Ctx& C, const RepArrays& R)
{
    constexpr int B = 4;
    const int ne = A.ne, nr = A.nr, G = 1 << C.lg, g = C.t & (G - 1), units = C.nt >> C.lg;
    double part = 0.0;
    for (int i0 = 0; i0 < C.n; i0 += units) {
        const int i = i0 + (C.t >> C.lg);
        const bool own = i < C.n;
        const double4 xi = R.x[C.off + (own ? i : 0)];
        const int ei = (int)xi.w;
        const int cnt = own ? R.nn[C.off + i] : 0;
        double rho = 0.0, ephi = 0.0;
        for (int k0 = g * B; k0 < cnt; k0 += G * B) {
            uint32_t e[B];
            double4 xj[B], cr[B], cp[B];
            double p[B], ri[B];
            bool in[B];
            fetch<B>(C, R, i, cnt, k0, e, xj);
            for (int b = 0; b < B; ++b) {
                const int ej = (int)xj[b].w;
                double dx, dy, dz, r;
                image_dx(C.shift, xi, xj[b], e[b] >> kIndexBits, dx, dy, dz);
                const double rsq = dx * dx + (dy * dy + dz * dz);
                in[b] = k0 + b < cnt && rsq < C.cut_sq[ei * ne + ej];
                int m;
                root_inv(in[b] ? rsq : 1.0, r, ri[b]);
                spline_at(r, A.dr_inv, nr, m, p[b]);
                cr[b] = A.rho[(size_t)(ej * ne + ei) * nr + m];
                cp[b] = A.phi[(size_t)(ei * ne + ej) * nr + m];
            }
            for (int b = 0; b < B; ++b) {
                rho += in[b] ? hval(cr[b], p[b]) : 0.0;
                ephi += in[b] ? hval(cp[b], p[b]) * ri[b] : 0.0;
            }
        }
        for (int o = 1; o < G; o <<= 1) {
            rho += __shfl_xor(rho, o, 64);
            ephi += __shfl_xor(ephi, o, 64);
        }
        if (own && g == 0) {
            int m;
            double p;
            spline_at(rho, A.drho_inv, A.nrho, m, p);
            const double4 c = A.F[(size_t)ei * A.nrho + m];
            double Fi = hval(c, p);
            const double dFi = dhval(c, p) * A.drho_inv;
            if (rho > A.rho_max) Fi += dFi * (rho - A.rho_max);
            R.dF[C.off + i] = dFi;
            part += Fi + 0.5 * ephi;
        }
    }
    return group_sum<W>(part, C);
}

// The force pass at the positions of the last density pass.
template <int W>
__device__ void eam_force(const RepArgs& A, Ctx& C, const RepArrays& R)
{
    constexpr int B = 2;
    const int ne = A.ne, nr = A.nr, G = 1 << C.lg, g = C.t & (G - 1), units = C.nt >> C.lg;
    for (int i0 = 0; i0 < C.n; i0 += units) {
        const int i = i0 + (C.t >> C.lg);
        const bool own = i < C.n;
        const double4 xi = R.x[C.off + (own ? i : 0)];
        const int ei = (int)xi.w;
        const double dFi = R.dF[C.off + (own ? i : 0)];
        const int cnt = own ? R.nn[C.off + i] : 0;
        double fx = 0.0, fy = 0.0, fz = 0.0;
        for (int k0 = g * B; k0 < cnt; k0 += G * B) {
            uint32_t e[B];
            double4 xj[B], cz[B], ca[B], cb[B];
            double dx[B], dy[B], dz[B], p[B], ri[B], dFj[B];
            bool in[B];
            fetch<B>(C, R, i, cnt, k0, e, xj);
            for (int b = 0; b < B; ++b) {
                const int ej = (int)xj[b].w;
                double r;
                dFj[b] = R.dF[C.off + (int)(e[b] & kIndexMask)];
                image_dx(C.shift, xi, xj[b], e[b] >> kIndexBits, dx[b], dy[b], dz[b]);
                const double rsq = dx[b] * dx[b] + (dy[b] * dy[b] + dz[b] * dz[b]);
                in[b] = k0 + b < cnt && rsq < C.cut_sq[ei * ne + ej];
                int m;
                root_inv(in[b] ? rsq : 1.0, r, ri[b]);
                spline_at(r, A.dr_inv, nr, m, p[b]);
                cz[b] = A.phi[(size_t)(ei * ne + ej) * nr + m];
                ca[b] = A.rho[(size_t)(ej * ne + ei) * nr + m];
                cb[b] = A.rho[(size_t)(ei * ne + ej) * nr + m];
            }
            for (int b = 0; b < B; ++b) {
                const double phi = hval(cz[b], p[b]) * ri[b];
                const double dphi = (dhval(cz[b], p[b]) * A.dr_inv - phi) * ri[b];
                const double drho_ji = dhval(ca[b], p[b]) * A.dr_inv;
                const double drho_ij = dhval(cb[b], p[b]) * A.dr_inv;
                const double u = -(dphi + dFi * drho_ji + dFj[b] * drho_ij) * ri[b];
                fx += in[b] ? u * dx[b] : 0.0;
                fy += in[b] ? u * dy[b] : 0.0;
                fz += in[b] ? u * dz[b] : 0.0;
            }
        }
        for (int o = 1; o < G; o <<= 1) {
            fx += __shfl_xor(fx, o, 64);
            fy += __shfl_xor(fy, o, 64);
            fz += __shfl_xor(fz, o, 64);
        }
        if (own && g == 0) R.f[C.off + i] = make_double4(fx, fy, fz, 0.0);
    }
    group_sync<W>();
}

// MinMDHandler::F(alpha) / F_reset: x = x0 + alpha h, the skin check of
// DynamicMD::update (a rebuild when any atom moved more than skin / 2 since
// the last build), then the energy
template <int W>
__device__ double trial(const RepArgs& A, Ctx& C, const RepArrays& R, double alpha, bool energy, int& builds, int& fail)
{
    double moved = 0.0;
    for (int i = C.t; i < C.n; i += C.nt) {
        const double4 a = R.x0[C.off + i], hh = R.h[C.off + i];
        const double4 x = make_double4(a.x + alpha * hh.x, a.y + alpha * hh.y, a.z + alpha * hh.z, a.w);
        R.x[C.off + i] = x;
        const double4 b = R.xb[C.off + i];
        const double d0 = x.x - b.x, d1 = x.y - b.y, d2 = x.z - b.z;
        moved = fmax(moved, d0 * d0 + (d1 * d1 + d2 * d2));
    }
    moved = group_max<W>(moved, C);
    if (moved > A.skin_sq4) {
        fail = build_list<W>(A, C, R);
        ++builds;
    }
    if (!energy || fail) return 0.0;
    return eam_energy<W>(A, C, R);
}

// One replica, the whole MinCG::__run on W waves (w = this wave's index in
// the group). Control flow is uniform over the replica's lanes: every branch
// condition derives from the header (read through readfirstlane) or from
// group sums that every lane receives alike, and every lane stores the
// results alike.
template <int W, int K>
__device__ void run_rep(const RepArgs& A, RepCell* __restrict__ cells, int r, const RepArrays& R, Shared<K>& S, int w,
                        int lane)
{
    Ctx C;
    {
        const RepCell hd = cells[r];
        C.off = uni(hd.off);
        C.n = uni(hd.n);
        C.maxn = uni(hd.maxn);
        const unsigned long long lo = (unsigned long long)hd.loff;
        C.loff = (long long)(((unsigned long long)(unsigned)uni((int)(lo >> 32)) << 32) |
                             (unsigned)uni((int)(lo & 0xffffffffull)));
        for (int k = 0; k < 6; ++k) {
            C.h[k] = uni(hd.h[k]);
            C.b[k] = uni(hd.b[k]);
        }
        for (int d = 0; d < 3; ++d) C.cs[d] = uni(hd.cs[d]);
    }
    C.nt = 64 * W;
    C.w = w;
    C.t = W == 1 ? lane : w * 64 + lane;
    C.flip = 0;
    C.red = &S.red[0][0];
    C.shift = S.shift[W == 1 ? w : 0];
    C.own0 = S.own0 + (W == 1 ? 65 * w : 0);
    C.cand0 = S.cand0 + (W == 1 ? 65 * w : 0);
    C.cut_sq = S.cut_sq;
    C.cutsk_sq = S.cutsk_sq;
    // lanes per atom: the fewest rounds of a pass over about 70 entries in
    // batches of 4, with the constant work of a round (its loads and sums)
    // taken as 8 entries
    C.lg = 0;
    for (int lg = 1, best = ((C.n + C.nt - 1) / C.nt) * 80; lg <= 4; ++lg) {
        const int cost = (((C.n << lg) + C.nt - 1) / C.nt) * (((72 >> lg) + 3) / 4 * 4 + 8 + 2 * lg);
        if (cost < best) {
            best = cost;
            C.lg = lg;
        }
    }
    for (int c = C.t; c < kShifts; c += C.nt) {
        const int n2 = c / 25 - 2, n1 = c % 25 / 5 - 2, n0 = c % 5 - 2;
        double* sh = C.shift[c];
        sh[0] = C.h[0] * n0 + C.h[1] * n1 + C.h[2] * n2;
        sh[1] = C.h[3] * n1 + C.h[4] * n2;
        sh[2] = C.h[5] * n2;
    }
    int builds = 1, evals = 0;
    int fail = build_list<W>(A, C, R);
    double e_curr = 0.0, e0 = 0.0;
    int err = LS_S, istep = 0;
    if (!fail) {
        e_curr = eam_energy<W>(A, C, R);
        eam_force<W>(A, C, R);
        ++evals;
        e0 = e_curr;
        double ff = 0.0;
        for (int i = C.t; i < C.n; i += C.nt) {
            const double4 f = R.f[C.off + i];
            R.h[C.off + i] = f;
            ff += f.x * f.x + (f.y * f.y + f.z * f.z);
        }
        double f0_f0 = group_sum<W>(ff, C);
        err = A.max_nsteps == 0 ? MIN_F_MAX_ITER : LS_S;
        double prev_val = -1.0;  // LineSearchBackTrack's memory (init_flag 1)
        while (err == LS_S) {
            if (f0_f0 == 0.0) {
                err = LS_F_GRAD0;
                ++istep;
                continue;
            }
            double fh = 0.0;
            for (int i = C.t; i < C.n; i += C.nt) {
                const double4 x = R.x[C.off + i], f = R.f[C.off + i], hh = R.h[C.off + i];
                R.x0[C.off + i] = x;
                R.f0[C.off + i] = f;
                fh += f.x * hh.x + (f.y * hh.y + f.z * hh.z);
            }
            const double e_prev = e_curr;
            double f_h = group_sum<W>(fh, C);
            if (f_h < 0.0) {
                for (int i = C.t; i < C.n; i += C.nt) R.h[C.off + i] = R.f[C.off + i];
                f_h = f0_f0;
                group_sync<W>();
            }
            // LineSearchBackTrack::min with MinMDHandler::ls_prep
            double hh2 = 0.0, hmax = 0.0;
            for (int i = C.t; i < C.n; i += C.nt) {
                const double4 hh = R.h[C.off + i];
                hh2 += hh.x * hh.x + (hh.y * hh.y + hh.z * hh.z);
                hmax = fmax(hmax, fmax(fabs(hh.x), fmax(fabs(hh.y), fabs(hh.z))));
            }
            const double h_norm = group_sum<W>(hh2, C);
            hmax = group_max<W>(hmax, C);
            double dfa = -f_h, max_a;
            if (h_norm == 0.0) {
                dfa = 0.0;
                max_a = 0.0;
            } else if (dfa >= 0.0) {
                dfa = 1.0;
                max_a = 0.0;
            } else {
                max_a = fabs(A.max_dx / hmax);
            }
            if (dfa == 0.0) {
                err = LS_F_GRAD0;
            } else if (max_a == 0.0) {
                err = LS_MIN_ALPHA;
            } else if (dfa >= 0.0) {
                err = LS_F_DOWNHILL;
            } else {
                if (prev_val > 0.0 && dfa < 0.0) max_a = fmin(max_a, -prev_val / dfa);
                prev_val = -dfa;
                if (max_a <= A.ls_min_alpha) {
                    err = LS_MIN_ALPHA;
                } else {
                    double alpha = max_a;
                    while (true) {
                        const double ideal = e_curr + alpha * A.ls_c * dfa;
                        const double cur = trial<W>(A, C, R, alpha, true, builds, fail);
                        ++evals;
                        if (fail) break;
                        if (cur <= ideal) {
                            prev_val *= alpha;
                            e_curr = cur;
                            break;
                        }
                        alpha *= A.ls_rho;
                        if (alpha <= A.ls_min_alpha || alpha != alpha) {
                            trial<W>(A, C, R, 0.0, false, builds, fail);  // F_reset
                            err = LS_MIN_ALPHA;
                            break;
                        }
                    }
                }
            }
            if (fail) break;
            if (err != LS_S) continue;
            // force_calc at the accepted point, whose density pass was the trial's
            eam_force<W>(A, C, R);
            ++evals;
            if (e_prev - e_curr < A.e_tol) err = MIN_S_TOLERANCE;
            if (istep + 1 == A.max_nsteps) err = MIN_F_MAX_ITER;
            if (err) {
                ++istep;
                continue;
            }
            double s_ff = 0.0, s_ff0 = 0.0;
            for (int i = C.t; i < C.n; i += C.nt) {
                const double4 f = R.f[C.off + i], g = R.f0[C.off + i];
                s_ff += f.x * f.x + (f.y * f.y + f.z * f.z);
                s_ff0 += f.x * g.x + (f.y * g.y + f.z * g.z);
            }
            const double f_f = group_sum<W>(s_ff, C);
            const double f_f0 = group_sum<W>(s_ff0, C);
            const double ratio = (f_f - f_f0) / f0_f0;
            for (int i = C.t; i < C.n; i += C.nt) {
                const double4 hh = R.h[C.off + i], f = R.f[C.off + i];
                R.h[C.off + i] = make_double4(ratio * hh.x + f.x, ratio * hh.y + f.y, ratio * hh.z + f.z, 0.0);
            }
            group_sync<W>();
            f0_f0 = f_f;
            ++istep;
        }
    }
    double fm = 0.0;
    if (!fail)
        for (int i = C.t; i < C.n; i += C.nt) {
            const double4 f = R.f[C.off + i];
            fm = fmax(fm, fmax(fabs(f.x), fmax(fabs(f.y), fabs(f.z))));
        }
    fm = group_max<W>(fm, C);
    if (w == 0 || W == 1) {
        RepCell& o = cells[r];
        o.status = fail ? fail : err;
        o.steps = istep;
        o.evals = evals;
        o.builds = builds;
        o.e0 = e0;
        o.e = e_curr;
        o.fmax = fm;
    }
}

// Persistent launch: workgroups first take the replicas that a whole
// workgroup owns (largest first) from queue[0]; then each wave takes one-wave
// replicas from queue[1] on its own. Every lane of a wave joins the queue
// atomic (lane 0 adds 1, the others 0) and the ticket is read from the first
// lane, so the replica index is wave-uniform. Only the first w1 waves of a
// workgroup take one-wave replicas, w1 as few as spread them over all
// workgroups.
template <int K>
__global__ __launch_bounds__(64 * K, 4) void k_replica_cg(RepArgs A, RepCell* cells, const int* __restrict__ q4,
                                                          int n4, const int* __restrict__ q1, int n1, int w1,
                                                          int* queue, RepArrays R)
{
    __shared__ Shared<K> S;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int k = threadIdx.x; k < A.ne * A.ne; k += 64 * K) {
        S.cut_sq[k] = A.cut_sq[k];
        S.cutsk_sq[k] = A.cutsk_sq[k];
    }
    while (true) {
        if (w == 0) {
            const int t = __builtin_amdgcn_readfirstlane(atomicAdd(&queue[0], lane == 0 ? 1 : 0));
            S.next = t;
        }
        __syncthreads();
        const int t = __builtin_amdgcn_readfirstlane(S.next);
        __syncthreads();
        if (t >= n4) break;
        run_rep<K>(A, cells, q4[t], R, S, w, lane);
        __syncthreads();
    }
    while (w < w1) {
        const int t = __builtin_amdgcn_readfirstlane(atomicAdd(&queue[1], lane == 0 ? 1 : 0));
        if (t >= n1) break;
        run_rep<1>(A, cells, q1[t], R, S, w, lane);
    }
}

// the queue counters cleared by a kernel (a graph replays it)
__global__ void k_replica_reset(int* queue)
{
    if (threadIdx.x < 2) queue[threadIdx.x] = 0;
}

}  // namespace

ReplicaBatch::ReplicaBatch(std::shared_ptr<EamForceField> ff, int nrep, const int* natms, const double* H,
                           const double* x, const uint8_t* elem, double skin)
    : ff_(std::move(ff)), nr_(nrep)
{
    const EamTables& tb = ff_->tables();
    MAPP_REQUIRE(!tb.dmd, ERR_ARG, "replica minimisation needs a plain (non-DMD) EAM force field");
    MAPP_REQUIRE(nrep > 0, ERR_ARG, "at least one replica is required");
    MAPP_REQUIRE(skin >= 0.0, ERR_ARG, "skin must be non-negative");
    const int ne = tb.ne;
    RepArgs& A = A0_;
    A.ne = ne;
    A.nr = tb.nr;
    A.nrho = tb.nrho;
    A.dr_inv = 1.0 / tb.dr;
    A.drho_inv = 1.0 / tb.drho;
    A.rho_max = (double)tb.nrho * tb.drho;
    double max_cut = 0.0;
    for (int i = 0; i < ne * ne; ++i) {
        A.cut_sq[i] = tb.rc[i] * tb.rc[i];
        A.cutsk_sq[i] = (tb.rc[i] + skin) * (tb.rc[i] + skin);
        max_cut = std::max(max_cut, tb.rc[i] + skin);
    }
    A.skin_sq4 = 0.25 * skin * skin;
    {
        std::vector<double4> ph((size_t)ne * ne * tb.nr), rh((size_t)ne * ne * tb.nr), fh((size_t)ne * tb.nrho);
        for (int a = 0; a < ne; ++a)
            for (int b = 0; b < ne; ++b)
                for (int k = 0; k < tb.nr; ++k) {
                    const double* p = tb.rphi_at(a, b) + 4 * k;
                    const double* r = tb.rho_at(a, b) + 4 * k;
                    ph[((size_t)a * ne + b) * tb.nr + k] = make_double4(p[0], p[1], p[2], p[3]);
                    rh[((size_t)a * ne + b) * tb.nr + k] = make_double4(r[0], r[1], r[2], r[3]);
                }
        for (int a = 0; a < ne; ++a)
            for (int k = 0; k < tb.nrho; ++k) {
                const double* f = tb.F_at(a) + (size_t)tb.nf() * k;
                fh[(size_t)a * tb.nrho + k] = make_double4(f[0], f[1], f[2], f[3]);
            }
        phi_.reserve(ph.size());
        rho4_.reserve(rh.size());
        F4_.reserve(fh.size());
        MAPP_HIP(hipMemcpy(phi_.get(), ph.data(), ph.size() * sizeof(double4), hipMemcpyHostToDevice));
        MAPP_HIP(hipMemcpy(rho4_.get(), rh.data(), rh.size() * sizeof(double4), hipMemcpyHostToDevice));
        MAPP_HIP(hipMemcpy(F4_.get(), fh.data(), fh.size() * sizeof(double4), hipMemcpyHostToDevice));
        A.phi = phi_.get();
        A.rho = rho4_.get();
        A.F = F4_.get();
    }
    host_cells_.resize(nrep);
    size_t off = 0, loff = 0;
    for (int r = 0; r < nrep; ++r) {
        MAPP_REQUIRE(natms[r] >= 1, ERR_ARG, "every replica needs at least one atom");
        RepCell& c = host_cells_[r];
        std::memset(&c, 0, sizeof c);
        const Box bx = make_box(H + 9 * (size_t)r);
        MAPP_REQUIRE(bx.H[0][0] > 0.0 && bx.H[1][1] > 0.0 && bx.H[2][2] > 0.0 && H[9 * r + 1] == 0.0 &&
                         H[9 * r + 2] == 0.0 && H[9 * r + 5] == 0.0,
                     ERR_ARG, "H must be lower triangular with a positive diagonal");
        c.off = (int)off;
        c.n = natms[r];
        c.loff = (long long)loff;
        c.cls = rep_class_of(natms[r]);
        for (int k = 0; k < 6; ++k) {
            c.h[k] = bx.h[k];
            c.b[k] = bx.b[k];
        }
        for (int i = 0; i < 3; ++i) {
            double t = 0.0;
            for (int j = i; j < 3; ++j) t += bx.B[j][i] * bx.B[j][i];
            c.cs[i] = std::sqrt(t) * max_cut;
            // every list image within -2..2 while atoms stay within one box
            // length of where they started
            MAPP_REQUIRE(c.cs[i] <= 1.0, ERR_CAPACITY,
                         "replica " + std::to_string(r) + " is thinner than r_c + skin along a box vector");
        }
        const double dens = natms[r] / bx.vol;
        const double sphere = 4.0 / 3.0 * M_PI * max_cut * max_cut * max_cut;
        c.maxn = (int)(1.5 * dens * sphere) + 32;
        off += natms[r];
        loff += (size_t)natms[r] * c.maxn;
    }
    natot_ = off;
    ltot_ = loff;
    st_.cells.reserve(nrep);
    st_.x.reserve(natot_);
    x0_.reserve(natot_);
    xb_.reserve(natot_);
    h_.reserve(natot_);
    f_.reserve(natot_);
    f0_.reserve(natot_);
    dF_.reserve(natot_);
    nn_.reserve(natot_);
    cid_.reserve(natot_);
    ord_.reserve(natot_);
    cand_.reserve(27 * natot_);
    list_.reserve(ltot_);
    queue_.reserve(2);
    {
        // positions wrapped into the box as a rebuild wraps them (x2s, s2x)
        std::vector<double4> xe(natot_);
        size_t src = 0;
        for (int r = 0; r < nrep; ++r) {
            const RepCell& c = host_cells_[r];
            for (int i = 0; i < c.n; ++i, ++src) {
                MAPP_REQUIRE(elem[src] < ne, ERR_ARG, "element index out of range");
                double s0, s1, s2, x0, x1, x2;
                x_to_s(c.b, x[3 * src], x[3 * src + 1], x[3 * src + 2], s0, s1, s2);
                s_to_x(c.h, s0, s1, s2, x0, x1, x2);
                xe[c.off + i] = make_double4(x0, x1, x2, (double)elem[src]);
            }
        }
        MAPP_HIP(hipMemcpy(st_.x.get(), xe.data(), natot_ * sizeof(double4), hipMemcpyHostToDevice));
        MAPP_HIP(hipMemcpy(st_.cells.get(), host_cells_.data(), nrep * sizeof(RepCell), hipMemcpyHostToDevice));
    }
    MAPP_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    int dev = 0, per[2] = {0, 0};
    MAPP_HIP(hipGetDevice(&dev));
    MAPP_HIP(hipDeviceGetAttribute(&ncu_, hipDeviceAttributeMultiprocessorCount, dev));
    MAPP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[0], k_replica_cg<kNarrow>, 64 * kNarrow, 0));
    MAPP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per[1], k_replica_cg<kWide>, 64 * kWide, 0));
    for (int k = 0; k < 2; ++k) grid_[k] = std::max(1, ncu_ * std::max(1, per[k]));
    default_waves();
}

ReplicaBatch::~ReplicaBatch()
{
    if (graph_) (void)hipGraphExecDestroy(graph_);
    if (stream_) {
        (void)hipStreamSynchronize(stream_);
        (void)hipStreamDestroy(stream_);
    }
}

RepArgs ReplicaBatch::args(int max_nsteps, double e_tol, double max_dx, double c, double rho, double min_alpha) const
{
    MAPP_REQUIRE(max_nsteps >= 0, ERR_ARG, "max_nsteps must be non-negative");
    MAPP_REQUIRE(max_dx > 0.0, ERR_ARG, "max_dx must be positive");
    MAPP_REQUIRE(c > 0.0 && c < 1.0 && rho > 0.0 && rho < 1.0 && min_alpha >= 0.0, ERR_ARG,
                 "the back-tracking search needs 0 < c < 1, 0 < rho < 1 and min_alpha >= 0");
    RepArgs A = A0_;
    A.max_nsteps = max_nsteps;
    A.e_tol = e_tol;
    A.max_dx = max_dx;
    A.ls_c = c;
    A.ls_rho = rho;
    A.ls_min_alpha = min_alpha;
    return A;
}

// Whether workgroups of 16 waves take the num replicas of which the largest has
// nmax atoms. A small replica leaves most of 16 waves waiting at barriers; a
// large one's chain is twice as long on 4. 10 steps, 4 waves and 16:
//   384 cells of 108 atoms  3.0 and 4.8 ms, of 256  3.6 and  5.5, of 500 10.1 and 10.6
// 1,024 cells of 108 atoms  3.7 and 9.8 ms, of 256  5.8 and 10.9, of 500 16.5 and 21.0
//   256 cells of 108 atoms  2.6 and 2.7 ms, of 500  8.6 and  6.1
//   864 atoms: 512 cells 26.9 and 24.4, 768 32.7 and 34.7; 1,372 atoms: 768 45.7 and 41.7, 1,024 54.3 and 55.3
bool ReplicaBatch::wide_workgroup(int num, int nmax) const
{
    return !(nmax < 512 ? num > ncu_ : nmax < 1024 && num >= 3 * ncu_);
}

// The shapes until set_waves or tune: workgroups, except for small cells in
// numbers beside large ones, which hold the workgroups at 16 waves (10 steps,
// one wave and 16 waves a cell: 1,024 cells of 108 atoms 6.0 and 9.8 ms, of 256
// 11.5 and 10.9; 2,048 of 256 14.6 and 20.9, of 400 32 and 33, of 500 45 and 41)
void ReplicaBatch::default_waves()
{
    int cnt[5] = {0, 0, 0, 0, 0};
    for (const RepCell& c : host_cells_) ++cnt[c.cls];
    std::fill(waves_, waves_ + 5, 4);
    if (cnt[2] + cnt[3] + cnt[4] == 0) return;
    if (cnt[0] >= 4 * ncu_) waves_[0] = 1;
    if (cnt[1] >= 8 * ncu_) waves_[1] = 1;
}

void ReplicaBatch::build_queues(const int* waves, DevBuf<int>& q4, int& n4, DevBuf<int>& q1, int& n1, bool& wide) const
{
    std::vector<int> order(nr_);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(),
                     [&](int a, int b) { return host_cells_[a].n > host_cells_[b].n; });
    std::vector<int> v4, v1;
    for (int r : order) (waves[host_cells_[r].cls] == 4 ? v4 : v1).push_back(r);
    n4 = (int)v4.size();
    n1 = (int)v1.size();
    wide = wide_workgroup(n4, n4 ? host_cells_[v4[0]].n : 0);
    q4.reserve(std::max(1, n4));
    q1.reserve(std::max(1, n1));
    if (n4) MAPP_HIP(hipMemcpy(q4.get(), v4.data(), n4 * sizeof(int), hipMemcpyHostToDevice));
    if (n1) MAPP_HIP(hipMemcpy(q1.get(), v1.data(), n1 * sizeof(int), hipMemcpyHostToDevice));
}

void ReplicaBatch::launch(State& st, const RepArgs& A, const int* q4, int n4, const int* q1, int n1, bool wide)
{
    RepArrays R{st.x.get(), x0_.get(), xb_.get(), h_.get(), f_.get(), f0_.get(), dF_.get(), list_.get(), nn_.get(),
                cid_.get(), ord_.get(), cand_.get()};
    k_replica_reset<<<1, 64, 0, stream_>>>(queue_.get());
    const auto run = wide ? k_replica_cg<kWide> : k_replica_cg<kNarrow>;
    const int K = wide ? kWide : kNarrow;
    // one workgroup per replica up to what the chip holds at once, of either shape
    const int blocks = std::max(1, std::min(grid_[wide], std::max(n4, n1)));
    const int w1 = std::min(K, (n1 + blocks - 1) / blocks);
    run<<<blocks, 64 * K, 0, stream_>>>(A, st.cells.get(), q4, n4, q1, n1, w1, queue_.get(), R);
    MAPP_HIP(hipGetLastError());
}

void ReplicaBatch::set_waves(const int* waves)
{
    for (int k = 0; k < 5; ++k) MAPP_REQUIRE(waves[k] == 1 || waves[k] == 4, ERR_ARG, "waves must be 1 or 4");
    std::copy(waves, waves + 5, waves_);
    queues_dirty_ = true;
}

void ReplicaBatch::use_graph(bool on)
{
    graph_on_ = on;
    if (!on && graph_) {
        (void)hipGraphExecDestroy(graph_);
        graph_ = nullptr;
    }
}

void ReplicaBatch::min_cg(int max_nsteps, double e_tol, double max_dx, double c, double rho, double min_alpha,
                          int* steps, int* status, double* e0, double* e, int* evals)
{
    const RepArgs A = args(max_nsteps, e_tol, max_dx, c, rho, min_alpha);
    if (queues_dirty_) {
        build_queues(waves_, q4_, n4_, q1_, n1_, wide_);
        queues_dirty_ = false;
        if (graph_) {
            (void)hipGraphExecDestroy(graph_);
            graph_ = nullptr;
        }
    }
    prof_.begin(K_REPLICA, stream_);
    if (graph_on_) {
        if (!graph_ || std::memcmp(&graph_args_, &A, sizeof A) != 0) {
            if (graph_) (void)hipGraphExecDestroy(graph_);
            graph_ = nullptr;
            hipGraph_t g;
            MAPP_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
            launch(st_, A, q4_.get(), n4_, q1_.get(), n1_, wide_);
            MAPP_HIP(hipStreamEndCapture(stream_, &g));
            MAPP_HIP(hipGraphInstantiate(&graph_, g, nullptr, nullptr, 0));
            MAPP_HIP(hipGraphDestroy(g));
            graph_args_ = A;
        }
        MAPP_HIP(hipGraphLaunch(graph_, stream_));
    } else {
        launch(st_, A, q4_.get(), n4_, q1_.get(), n1_, wide_);
    }
    prof_.end(stream_);
    MAPP_HIP(hipStreamSynchronize(stream_));
    prof_.flush();
    std::vector<RepCell> hc(nr_);
    MAPP_HIP(hipMemcpy(hc.data(), st_.cells.get(), nr_ * sizeof(RepCell), hipMemcpyDeviceToHost));
    for (int r = 0; r < nr_; ++r) {
        if (steps) steps[r] = hc[r].steps;
        if (status) status[r] = hc[r].status;
        if (e0) e0[r] = hc[r].e0;
        if (e) e[r] = hc[r].e;
        if (evals) evals[r] = hc[r].evals;
    }
    for (int r = 0; r < nr_; ++r) {
        MAPP_REQUIRE(hc[r].status != FAIL_LIST, ERR_CAPACITY,
                     "replica " + std::to_string(r) + ": a neighbor list row exceeded its capacity");
        MAPP_REQUIRE(hc[r].status != FAIL_IMAGE, ERR_STATE,
                     "replica " + std::to_string(r) + ": an atom moved more than a box length");
    }
}

// Tile tuner: one wave per replica for the size classes below a threshold,
// a workgroup from there up. Every threshold is timed on a copy of the batch (the
// production positions are not moved) and the fastest is kept.
RepTuneReport ReplicaBatch::tune(int max_nsteps, double e_tol, double max_dx, double c, double rho, double min_alpha)
{
    const RepArgs A = args(max_nsteps, e_tol, max_dx, c, rho, min_alpha);
    RepTuneReport rep{};
    hipEvent_t e0, e1;
    MAPP_HIP(hipEventCreate(&e0));
    MAPP_HIP(hipEventCreate(&e1));
    scratch_.cells.reserve(nr_);
    scratch_.x.reserve(natot_);
    double best = 1e300;
    int best_t = 5;
    // one untimed launch first (code objects, caches), then the best of two
    // timed launches per threshold
    for (int th = -1; th <= 5; ++th) {
        int wv[5];
        for (int k = 0; k < 5; ++k) wv[k] = k < th ? 1 : 4;
        DevBuf<int> d4, d1;
        int n4 = 0, n1 = 0;
        bool wide = true;
        build_queues(wv, d4, n4, d1, n1, wide);
        float ms = 1e30f;
        for (int k = 0; k < (th < 0 ? 1 : 2); ++k) {
            MAPP_HIP(hipMemcpyAsync(scratch_.cells.get(), st_.cells.get(), nr_ * sizeof(RepCell),
                                    hipMemcpyDeviceToDevice, stream_));
            MAPP_HIP(hipMemcpyAsync(scratch_.x.get(), st_.x.get(), natot_ * sizeof(double4), hipMemcpyDeviceToDevice,
                                    stream_));
            MAPP_HIP(hipEventRecord(e0, stream_));
            launch(scratch_, A, d4.get(), n4, d1.get(), n1, wide);
            MAPP_HIP(hipEventRecord(e1, stream_));
            MAPP_HIP(hipEventSynchronize(e1));
            float t = 0.f;
            MAPP_HIP(hipEventElapsedTime(&t, e0, e1));
            ms = std::min(ms, t);
        }
        if (th < 0) continue;
        rep.ms[th] = ms;
        if (ms < best) {
            best = ms;
            best_t = th;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    for (int k = 0; k < 5; ++k) rep.waves[k] = k < best_t ? 1 : 4;
    set_waves(rep.waves);
    return rep;
}

void ReplicaBatch::get(int r, double* x)
{
    MAPP_REQUIRE(r >= 0 && r < nr_, ERR_ARG, "replica index out of range");
    const RepCell& c = host_cells_[r];
    std::vector<double4> b(c.n);
    MAPP_HIP(hipMemcpy(b.data(), st_.x.get() + c.off, c.n * sizeof(double4), hipMemcpyDeviceToHost));
    for (int i = 0; i < c.n; ++i) {
        x[3 * i] = b[i].x;
        x[3 * i + 1] = b[i].y;
        x[3 * i + 2] = b[i].z;
    }
}

}  // namespace mapp
