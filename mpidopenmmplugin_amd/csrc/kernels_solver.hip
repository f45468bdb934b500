// The mutual-polarization solver's kernels: the operator A = I - S T S on the
// polarisable sites, the conjugate-gradient update and the residual norms.
//
// The solver's vectors (b, x, r, p, A p) hold the polarisable sites only, in
// the order of their sorted index (t-th entry: atom idx[t]); a site without
// polarisability has S = 0 and a zero entry in every one of them.  The
// operator's input mu = S p is stored by atom, with zeros elsewhere, for the
// spreading and the neighbour lists.
//
// A solver iteration is a chain of short dependent kernels, so its time on
// small systems is their number times the 4-6 us a dependent dispatch takes.
// The chain is therefore kept short: the operator's kernel gathers the
// reciprocal field, adds the real-space field, applies S and leaves the
// partial sums of p.Ap; the update kernels fold the reductions in (every
// workgroup sums the previous kernel's partials in the same order, so the
// result is the same in each and from run to run).
#include "pair_math.h"
#include "pme_math.h"

#include <algorithm>

namespace mpid {

typedef V3<double> D3;

__device__ __forceinline__ D3 sym_mul6(const double* S, D3 v) {
    return mk(S[0] * v.x + S[1] * v.y + S[2] * v.z, S[1] * v.x + S[3] * v.y + S[4] * v.z,
              S[2] * v.x + S[4] * v.y + S[5] * v.z);
}
__device__ __forceinline__ D3 load3(const double* a, size_t t) { return mk(a[3 * t], a[3 * t + 1], a[3 * t + 2]); }
__device__ __forceinline__ void store3(double* a, size_t t, D3 v) {
    a[3 * t] = v.x;
    a[3 * t + 1] = v.y;
    a[3 * t + 2] = v.z;
}
template <class R> __device__ __forceinline__ void store_mu(R* mu, size_t i, D3 v) {
    mu[3 * i] = (R)v.x;
    mu[3 * i + 1] = (R)v.y;
    mu[3 * i + 2] = (R)v.z;
}

// Sums over a workgroup of THREADS threads in a fixed order, the result in
// every thread; sh: THREADS / 64 * K words.
template <int THREADS, int K> __device__ __forceinline__ void group_sum(double (&v)[K], double* sh) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1)
#pragma unroll
        for (int k = 0; k < K; k++) v[k] += __shfl_xor(v[k], off);
    constexpr int kWaves = THREADS / 64;
    if constexpr (kWaves > 1) {
        __syncthreads();  // sh may still be read from a previous sum
        if ((threadIdx.x & 63) == 0)
#pragma unroll
            for (int k = 0; k < K; k++) sh[(threadIdx.x >> 6) * K + k] = v[k];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; k++) {
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < kWaves; w++) s += sh[w * K + k];
            v[k] = s;
        }
    }
}
// The same over `count` partials of each of K sums, stored one sum after the
// other at a stride of kMaxPartials.
template <int THREADS, int K>
__device__ __forceinline__ void sum_partials(const double* __restrict__ partial, int count, double (&v)[K], double* sh) {
#pragma unroll
    for (int k = 0; k < K; k++) {
        v[k] = 0.0;
        for (int i = threadIdx.x; i < count; i += THREADS) v[k] += partial[k * kMaxPartials + i];
    }
    group_sum<THREADS, K>(v, sh);
}

// ---------------------------------------------------------------------------
// operator
// ---------------------------------------------------------------------------
// Av_t = v_t - S (E_rec + E_real + selfc mu) at polarisable site t, and with
// `partial` one partial sum of v.Av per workgroup.
template <class R>
__device__ __forceinline__ double operator_row(const SolverSites& st, int t, int i, D3 e, const R* __restrict__ mu,
                                               double selfc, const double* __restrict__ v, double* Av) {
    e.x += selfc * (double)mu[3 * (size_t)i];
    e.y += selfc * (double)mu[3 * (size_t)i + 1];
    e.z += selfc * (double)mu[3 * (size_t)i + 2];
    const D3 w = sym_mul6(st.S + 6 * (size_t)i, e);
    const D3 pv = load3(v, t);
    const D3 a = pv - w;
    store3(Av, t, a);
    return dot(pv, a);
}

// The parts of a site's field (reciprocal, listed neighbours, covalent partners)
// are formed in R and meet in FP64: a partner's field can be far smaller than
// the list's sum.
//
// Everything after the inverse transform in one kernel, 32 lanes per site:
// the site's splines (lanes 0-2, one axis each, through LDS), the stencil's
// points over the lanes, the neighbours over the lanes, the covalent partners.
// For systems whose kernels do not fill the chip (kFusedSites): there the
// list of a site is walked in 3 steps instead of the 18-24 of four lanes, and
// five dispatches become one.
constexpr int kOpLanes = 32;
constexpr int kOpSites = 256 / kOpLanes;  // sites per workgroup
template <class R>
__global__ __launch_bounds__(256) void k_operator_fused(SolverSites st, PmeGeom<R> g, const R* __restrict__ pot,
                                                        NbrList L, PairAtoms<R> A, PairParams<R> P,
                                                        const R* __restrict__ mu, double selfc,
                                                        const double* __restrict__ v, double* __restrict__ Av,
                                                        double* __restrict__ partial) {
    if (skipped(P.skip)) return;
    __shared__ R sth[kOpSites][3][kOrder][2];
    __shared__ int sig[kOpSites][3];
    __shared__ double sdot[kOpSites];
    const int grp = threadIdx.x / kOpLanes, lane = threadIdx.x % kOpLanes;
    double acc = 0.0;
    for (int t0 = blockIdx.x * kOpSites; t0 < st.npol; t0 += gridDim.x * kOpSites) {
        const int t = min(t0 + grp, st.npol - 1);
        const bool tv = t0 + grp < st.npol;
        const int i = st.idx[t];
        const R4<R> pi = A.pos[i];
        R ex = 0, ey = 0, ez = 0;
        if (pot) {  // no reciprocal space without a grid
            if (lane < 3) {
                const V3<R> f = to_frac(mk(pi.x, pi.y, pi.z), g.box);
                int ig;
                R w;
                grid_coord(lane == 0 ? f.x : (lane == 1 ? f.y : f.z), g.n[lane], ig, w);
                R th[kOrder][2];
                bspline6<R, 1>(w, th);
#pragma unroll
                for (int m = 0; m < kOrder; m++) {
                    sth[grp][lane][m][0] = th[m][0];
                    sth[grp][lane][m][1] = th[m][1];
                }
                sig[grp][lane] = ig;
            }
            __syncthreads();
            const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
            const int gx = sig[grp][0], gy = sig[grp][1], gz = sig[grp][2];
            constexpr int kPoints = kOrder * kOrder * kOrder;
            constexpr int kSteps = (kPoints + kOpLanes - 1) / kOpLanes;
            R q[kSteps];
#pragma unroll
            for (int u = 0; u < kSteps; u++) {
                const int s = min(lane + u * kOpLanes, kPoints - 1);
                const int ix = s / (kOrder * kOrder), rem = s - ix * kOrder * kOrder;
                const int iy = rem / kOrder, iz = rem - iy * kOrder;
                int x = gx + ix, y = gy + iy, z = gz + iz;
                if (x >= nx) x -= nx;
                if (y >= ny) y -= ny;
                if (z >= nz) z -= nz;
                q[u] = pot[((size_t)x * ny + y) * nz + z];
            }
            R s100 = 0, s010 = 0, s001 = 0;
#pragma unroll
            for (int u = 0; u < kSteps; u++) {
                const int s0 = lane + u * kOpLanes, s = min(s0, kPoints - 1);
                const int ix = s / (kOrder * kOrder), rem = s - ix * kOrder * kOrder;
                const int iy = rem / kOrder, iz = rem - iy * kOrder;
                const R a0 = sth[grp][0][ix][0], a1 = sth[grp][0][ix][1];
                const R b0 = sth[grp][1][iy][0], b1 = sth[grp][1][iy][1];
                const R c0 = sth[grp][2][iz][0], c1 = sth[grp][2][iz][1];
                const R qv = s0 < kPoints ? q[u] : R(0);
                s100 += qv * a1 * b0 * c0;
                s010 += qv * a0 * b1 * c0;
                s001 += qv * a0 * b0 * c1;
            }
            const V3<R> e = cart_vector(mk(s100, s010, s001), g.A);
            ex = -e.x;
            ey = -e.y;
            ez = -e.z;
            __syncthreads();  // the tables are read before the next sites' replace them
        }
        R rx = 0, ry = 0, rz = 0;
        const int cnt = tv ? L.count[i] : 0;
        for (int k = lane; k < cnt; k += kOpLanes) {
            const int j = L.nbr[((size_t)(k / kNlSplit) * st.npol + t) * kNlSplit + k % kNlSplit];
            const R4<R> pj = A.pos[j];
            const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
            const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
            const V3<R> fi =
                induced_field_from<R>(uj, dr, induced_field_radial<R>(dot(dr, dr), pi.w, pj.w, P.default_thole, P));
            rx += fi.x;
            ry += fi.y;
            rz += fi.z;
        }
        const V3<R> c = partner_field<R>(i, lane, kOpLanes, A, mu, P);
        D3 e = mk((double)ex + (double)rx + (double)c.x, (double)ey + (double)ry + (double)c.y,
                  (double)ez + (double)rz + (double)c.z);
#pragma unroll
        for (int off = 1; off < kOpLanes; off <<= 1) {
            e.x += __shfl_xor(e.x, off);
            e.y += __shfl_xor(e.y, off);
            e.z += __shfl_xor(e.z, off);
        }
        if (tv && lane == 0) acc += operator_row<R>(st, t, i, e, mu, selfc, v, Av);
    }
    if (partial) {
        if (lane == 0) sdot[grp] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < kOpSites; k++) s += sdot[k];
            partial[blockIdx.x] = s;
        }
    }
}

// The same in two kernels for systems that fill the chip: the real-space field
// (k_list_field, beside the reciprocal chain on another stream), and the
// gather with the rest, 8 lanes per site (lane iz < 6: the 36 points of a z
// plane, all loads in flight).
template <class R>
__global__ __launch_bounds__(256) void k_list_field(SolverSites st, NbrList L, PairAtoms<R> A, PairParams<R> P,
                                                    const R* __restrict__ mu, double* __restrict__ field) {
    if (skipped(P.skip)) return;
    const unsigned gth = (unsigned)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int t = (int)(gth / kNlSplit), sub = (int)(gth % kNlSplit);
    const bool tv = t < st.npol;
    const int tc = tv ? t : st.npol - 1;
    const int i = st.idx[tc];
    const R4<R> pi = A.pos[i];
    const int cnt = tv ? L.count[i] : 0;
    const int* lp = L.nbr + (size_t)tc * kNlSplit + sub;
    const size_t stride = (size_t)st.npol * kNlSplit;
    int jn = sub < cnt ? lp[0] : 0;
    R ex = 0, ey = 0, ez = 0;
    for (int k = sub; k < cnt; k += kNlSplit) {
        const int j = jn;
        lp += stride;
        if (k + kNlSplit < cnt) jn = *lp;  // next index in flight during this pair
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        const V3<R> fi =
            induced_field_from<R>(uj, dr, induced_field_radial<R>(dot(dr, dr), pi.w, pj.w, P.default_thole, P));
        ex += fi.x;
        ey += fi.y;
        ez += fi.z;
    }
    const V3<R> c = partner_field<R>(i, sub, kNlSplit, A, mu, P);
    D3 e = mk((double)ex + (double)c.x, (double)ey + (double)c.y, (double)ez + (double)c.z);
#pragma unroll
    for (int off = 1; off < kNlSplit; off <<= 1) {
        e.x += __shfl_xor(e.x, off);
        e.y += __shfl_xor(e.y, off);
        e.z += __shfl_xor(e.z, off);
    }
    if (tv && sub == 0) store3(field, t, e);
}

constexpr int kGatherSites = 32;  // sites per workgroup
template <class R>
__global__ __launch_bounds__(256) void k_operator_gather(SolverSites st, PmeGeom<R> g, const R* __restrict__ pot,
                                                         const double* __restrict__ field,
                                                         const R4<R>* __restrict__ pos, const R* __restrict__ mu,
                                                         double selfc,
                                                         const double* __restrict__ v, double* __restrict__ Av,
                                                         double* __restrict__ partial) {
    if (skipped(g.skip)) return;
    __shared__ double sdot[kGatherSites];
    const int grp = threadIdx.x >> 3, iz = threadIdx.x & 7;
    double acc = 0.0;
    for (int t0 = xcd_block(blockIdx.x, gridDim.x) * kGatherSites; t0 < st.npol; t0 += gridDim.x * kGatherSites) {
        const int t = min(t0 + grp, st.npol - 1);
        const bool tv = t0 + grp < st.npol;
        const int i = st.idx[t];
        R s100 = 0, s010 = 0, s001 = 0;
        if (pot) {
            const R4<R> p = pos[i];
            int ig[3];
            R w[3];
            {
                const V3<R> f = to_frac(mk(p.x, p.y, p.z), g.box);
                grid_coord(f.x, g.n[0], ig[0], w[0]);
                grid_coord(f.y, g.n[1], ig[1], w[1]);
                grid_coord(f.z, g.n[2], ig[2], w[2]);
            }
            R tx[kOrder][2], ty[kOrder][2], tz[kOrder][2];
            bspline6<R, 1>(w[0], tx);
            bspline6<R, 1>(w[1], ty);
            bspline6<R, 1>(w[2], tz);
            const int ny = g.n[1], nz = g.n[2];
            if (iz < kOrder) {
                int z = ig[2] + iz;
                if (z >= nz) z -= nz;
                R q[kOrder][kOrder];
#pragma unroll
                for (int iy = 0; iy < kOrder; iy++) {
                    int y = ig[1] + iy;
                    if (y >= ny) y -= ny;
#pragma unroll
                    for (int ix = 0; ix < kOrder; ix++) {
                        int x = ig[0] + ix;
                        if (x >= g.n[0]) x -= g.n[0];
                        q[iy][ix] = pot[((size_t)x * ny + y) * nz + z];
                    }
                }
                R b00 = 0, b10 = 0, b01 = 0;
#pragma unroll
                for (int iy = 0; iy < kOrder; iy++) {
                    R a0 = 0, a1 = 0;
#pragma unroll
                    for (int ix = 0; ix < kOrder; ix++) {
                        a0 += q[iy][ix] * tx[ix][0];
                        a1 += q[iy][ix] * tx[ix][1];
                    }
                    b00 += a0 * ty[iy][0];
                    b10 += a1 * ty[iy][0];
                    b01 += a0 * ty[iy][1];
                }
                // this lane's z weights (a select: a runtime index would put the table in scratch memory)
                R c[2];
                spline_at<R, 1>(tz, iz, c);
                s100 = b10 * c[0];
                s010 = b01 * c[0];
                s001 = b00 * c[1];
            }
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) {
                s100 += __shfl_xor(s100, off);
                s010 += __shfl_xor(s010, off);
                s001 += __shfl_xor(s001, off);
            }
        }
        if (tv && iz == 0) {
            const V3<R> e = cart_vector(mk(s100, s010, s001), g.A);
            acc += operator_row<R>(st, t, i, load3(field, t) - mk((double)e.x, (double)e.y, (double)e.z), mu, selfc, v,
                                   Av);
        }
    }
    if (partial) {
        if (iz == 0) sdot[grp] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < kGatherSites; k++) s += sdot[k];
            partial[blockIdx.x] = s;
        }
    }
}

// ---------------------------------------------------------------------------
// Extrapolated (OPT) polarization
// (convergeInduceDipolesByExtrapolation, MPIDReferenceForce.cpp:1125-1180)
// ---------------------------------------------------------------------------
// One order at a polarisable site: E = real space + reciprocal (-A phi_1) +
// selfc mu_(m) and its gradient G = real space - A phi_2 A^T (A the
// grid-coordinate transform; :4094-4127), kept for the response forces, and
// mu_(m+1) = alpha_lab E by site in FP64 and by atom in the precision of the
// next order's kernels.  Only polarisable sites are visited: at the others
// mu is zero, and every use of E and G is multiplied by it.
// s: field and gradient (xx yy zz xy xz yz) of the lists; q: the potential's
// grid derivatives 100 010 001 200 020 002 110 101 011.
template <class R>
__device__ __forceinline__ void extrap_finish(const SolverSites& st, int t, int i, const double (&s)[9], const R (&q)[9],
                                              const FracT<double>& F, double selfc, const double* __restrict__ labpol,
                                              const ExtrapOrder& o, const double* __restrict__ mud, R* __restrict__ mu) {
    const D3 c1 = cart_vector(mk((double)q[0], (double)q[1], (double)q[2]), F);
    // A phi_2 A^T, A lower triangular
    const double xx = q[3], yy = q[4], zz = q[5], xy = q[6], xz = q[7], yz = q[8];
    double c2[6];  // xx yy zz xy xz yz
    if (!F.tri) {
        c2[0] = F.a00 * F.a00 * xx;
        c2[1] = F.a11 * F.a11 * yy;
        c2[2] = F.a22 * F.a22 * zz;
        c2[3] = F.a00 * F.a11 * xy;
        c2[4] = F.a00 * F.a22 * xz;
        c2[5] = F.a11 * F.a22 * yz;
    } else {
        const double m[3][3] = {{xx, xy, xz}, {xy, yy, yz}, {xz, yz, zz}};
        const double a[3][3] = {{F.a00, 0.0, 0.0}, {F.a10, F.a11, 0.0}, {F.a20, F.a21, F.a22}};
        double am[3][3];
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) am[r][c] = a[r][0] * m[0][c] + a[r][1] * m[1][c] + a[r][2] * m[2][c];
        auto el = [&](int r, int c) { return am[r][0] * a[c][0] + am[r][1] * a[c][1] + am[r][2] * a[c][2]; };
        c2[0] = el(0, 0);
        c2[1] = el(1, 1);
        c2[2] = el(2, 2);
        c2[3] = el(0, 1);
        c2[4] = el(0, 2);
        c2[5] = el(1, 2);
    }
    const D3 m = o.mus_in ? load3(o.mus_in, t) : load3(mud, i);
    if (!o.mus_in) store3(o.mu0, t, m);  // mu_(0) = alpha E0, so far by atom
    const D3 e = mk(s[0] - c1.x + selfc * m.x, s[1] - c1.y + selfc * m.y, s[2] - c1.z + selfc * m.z);
    store3(o.E, t, e);
#pragma unroll
    for (int c = 0; c < 6; c++) o.G[6 * (size_t)t + c] = s[3 + c] - c2[c];
    const D3 nx = sym_mul6(labpol + 6 * (size_t)i, e);
    store3(o.mus_out, t, nx);
    store_mu<R>(mu, i, nx);
}

// f = s, a lane's part of the listed neighbours' field and gradient, and in
// FP64 the lane's covalent partners'
template <class R>
__device__ __forceinline__ void add_partners(int i, int lane, int lanes, const PairAtoms<R>& A, const R* mu,
                                             const PairParams<R>& P, const R (&s)[9], double (&f)[9]) {
    R g[6] = {};
    const V3<R> c = partner_field_grad<R>(i, lane, lanes, A, mu, P, g);
    f[0] = (double)s[0] + (double)c.x;
    f[1] = (double)s[1] + (double)c.y;
    f[2] = (double)s[2] + (double)c.z;
#pragma unroll
    for (int k = 0; k < 6; k++) f[3 + k] = (double)s[3 + k] + (double)g[k];
}

// As k_operator_fused: 32 lanes per site for everything after the inverse
// transform.  mu is read of the neighbours and written in a second array.
template <class R>
__global__ __launch_bounds__(256) void k_extrap_fused(SolverSites st, PmeGeom<R> g, const R* __restrict__ pot,
                                                      NbrList L, PairAtoms<R> A, PairParams<R> P,
                                                      const R* __restrict__ mu, R* __restrict__ mu_next,
                                                      FracT<double> F, double selfc, const double* __restrict__ labpol,
                                                      ExtrapOrder o, const double* __restrict__ mud) {
    __shared__ R sth[kOpSites][3][kOrder][3];
    __shared__ int sig[kOpSites][3];
    const int grp = threadIdx.x / kOpLanes, lane = threadIdx.x % kOpLanes;
    const int t0 = blockIdx.x * kOpSites + grp;
    const int t = min(t0, st.npol - 1);
    const bool tv = t0 < st.npol;
    const int i = st.idx[t];
    const R4<R> pi = A.pos[i];
    R q[9] = {};
    if (pot) {
        if (lane < 3) {
            const V3<R> f = to_frac(mk(pi.x, pi.y, pi.z), g.box);
            int ig;
            R w;
            grid_coord(lane == 0 ? f.x : (lane == 1 ? f.y : f.z), g.n[lane], ig, w);
            R th[kOrder][3];
            bspline6<R, 2>(w, th);
#pragma unroll
            for (int m = 0; m < kOrder; m++)
#pragma unroll
                for (int d = 0; d < 3; d++) sth[grp][lane][m][d] = th[m][d];
            sig[grp][lane] = ig;
        }
        __syncthreads();
        const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
        const int gx = sig[grp][0], gy = sig[grp][1], gz = sig[grp][2];
        constexpr int kPoints = kOrder * kOrder * kOrder;
        constexpr int kSteps = (kPoints + kOpLanes - 1) / kOpLanes;
        R v[kSteps];
#pragma unroll
        for (int u = 0; u < kSteps; u++) {
            const int s = min(lane + u * kOpLanes, kPoints - 1);
            const int ix = s / (kOrder * kOrder), rem = s - ix * kOrder * kOrder;
            const int iy = rem / kOrder, iz = rem - iy * kOrder;
            int x = gx + ix, y = gy + iy, z = gz + iz;
            if (x >= nx) x -= nx;
            if (y >= ny) y -= ny;
            if (z >= nz) z -= nz;
            v[u] = pot[((size_t)x * ny + y) * nz + z];
        }
#pragma unroll
        for (int u = 0; u < kSteps; u++) {
            const int s0 = lane + u * kOpLanes, s = min(s0, kPoints - 1);
            const int ix = s / (kOrder * kOrder), rem = s - ix * kOrder * kOrder;
            const int iy = rem / kOrder, iz = rem - iy * kOrder;
            const R* a = sth[grp][0][ix];
            const R* b = sth[grp][1][iy];
            const R* c = sth[grp][2][iz];
            const R p = s0 < kPoints ? v[u] : R(0);
            q[0] += p * a[1] * b[0] * c[0];
            q[1] += p * a[0] * b[1] * c[0];
            q[2] += p * a[0] * b[0] * c[1];
            q[3] += p * a[2] * b[0] * c[0];
            q[4] += p * a[0] * b[2] * c[0];
            q[5] += p * a[0] * b[0] * c[2];
            q[6] += p * a[1] * b[1] * c[0];
            q[7] += p * a[1] * b[0] * c[1];
            q[8] += p * a[0] * b[1] * c[1];
        }
    }
    R s[9] = {};
    const int cnt = tv ? L.count[i] : 0;
    for (int k = lane; k < cnt; k += kOpLanes) {
        const int j = L.nbr[((size_t)(k / kNlSplit) * st.npol + t) * kNlSplit + k % kNlSplit];
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        const InducedRadialGrad<R> f = induced_grad_radial<R>(dot(dr, dr), pi.w, pj.w, P.default_thole, P);
        const V3<R> e = induced_field_from<R>(uj, dr, InducedRadial<R>{f.f1, f.f2});
        s[0] += e.x;
        s[1] += e.y;
        s[2] += e.z;
        induced_grad_add<R>(uj, dr, f.f2, f.f3, s + 3);
    }
    double f[9];
    add_partners<R>(i, lane, kOpLanes, A, mu, P, s, f);
#pragma unroll
    for (int off = 1; off < kOpLanes; off <<= 1)
#pragma unroll
        for (int k = 0; k < 9; k++) {
            q[k] += __shfl_xor(q[k], off);
            f[k] += __shfl_xor(f[k], off);
        }
    if (tv && lane == 0) extrap_finish<R>(st, t, i, f, q, F, selfc, labpol, o, mud, mu_next);
}

// The same in two kernels (see k_list_field and k_operator_gather)
template <class R>
__global__ __launch_bounds__(256) void k_extrap_list(SolverSites st, NbrList L, PairAtoms<R> A, PairParams<R> P,
                                                     const R* __restrict__ mu, double* __restrict__ field) {
    const unsigned gth = (unsigned)xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    const int t0 = (int)(gth / kNlSplit), sub = (int)(gth % kNlSplit);
    const bool tv = t0 < st.npol;
    const int t = tv ? t0 : st.npol - 1;
    const int i = st.idx[t];
    const R4<R> pi = A.pos[i];
    const int cnt = tv ? L.count[i] : 0;
    const int* lp = L.nbr + (size_t)t * kNlSplit + sub;
    const size_t stride = (size_t)st.npol * kNlSplit;
    int jn = sub < cnt ? lp[0] : 0;
    R s[9] = {};
    for (int k = sub; k < cnt; k += kNlSplit) {
        const int j = jn;
        lp += stride;
        if (k + kNlSplit < cnt) jn = *lp;  // next index in flight during this pair
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        const V3<R> uj = mk(mu[3 * (size_t)j], mu[3 * (size_t)j + 1], mu[3 * (size_t)j + 2]);
        const InducedRadialGrad<R> f = induced_grad_radial<R>(dot(dr, dr), pi.w, pj.w, P.default_thole, P);
        const V3<R> e = induced_field_from<R>(uj, dr, InducedRadial<R>{f.f1, f.f2});
        s[0] += e.x;
        s[1] += e.y;
        s[2] += e.z;
        induced_grad_add<R>(uj, dr, f.f2, f.f3, s + 3);
    }
    double f[9];
    add_partners<R>(i, sub, kNlSplit, A, mu, P, s, f);
#pragma unroll
    for (int off = 1; off < kNlSplit; off <<= 1)
#pragma unroll
        for (int k = 0; k < 9; k++) f[k] += __shfl_xor(f[k], off);
    if (tv && sub == 0)
#pragma unroll
        for (int k = 0; k < 9; k++) field[9 * (size_t)t + k] = f[k];
}
template <class R>
__global__ __launch_bounds__(256) void k_extrap_gather(SolverSites st, PmeGeom<R> g, const R* __restrict__ pot,
                                                       const double* __restrict__ field,
                                                       const R4<R>* __restrict__ pos, FracT<double> F, double selfc,
                                                       const double* __restrict__ labpol, ExtrapOrder o,
                                                       const double* __restrict__ mud, R* __restrict__ mu_next) {
    const int gt = xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    const int t0 = gt >> 3, iz = gt & 7;
    const bool tv = t0 < st.npol;
    const int t = tv ? t0 : st.npol - 1;
    const int i = st.idx[t];
    R q[9] = {};
    if (pot) {
        const R4<R> p = pos[i];
        int ig[3];
        R w[3];
        {
            const V3<R> f = to_frac(mk(p.x, p.y, p.z), g.box);
            grid_coord(f.x, g.n[0], ig[0], w[0]);
            grid_coord(f.y, g.n[1], ig[1], w[1]);
            grid_coord(f.z, g.n[2], ig[2], w[2]);
        }
        R tx[kOrder][3], ty[kOrder][3], tz[kOrder][3];
        bspline6<R, 2>(w[0], tx);
        bspline6<R, 2>(w[1], ty);
        bspline6<R, 2>(w[2], tz);
        const int ny = g.n[1], nz = g.n[2];
        if (iz < kOrder) {
            int z = ig[2] + iz;
            if (z >= nz) z -= nz;
            R b00 = 0, b10 = 0, b01 = 0, b20 = 0, b11 = 0, b02 = 0;
#pragma unroll
            for (int iy = 0; iy < kOrder; iy++) {
                int y = ig[1] + iy;
                if (y >= ny) y -= ny;
                R row[kOrder];
#pragma unroll
                for (int ix = 0; ix < kOrder; ix++) {
                    int x = ig[0] + ix;
                    if (x >= g.n[0]) x -= g.n[0];
                    row[ix] = pot[((size_t)x * ny + y) * nz + z];
                }
                R a0 = 0, a1 = 0, a2 = 0;
#pragma unroll
                for (int ix = 0; ix < kOrder; ix++) {
                    a0 += row[ix] * tx[ix][0];
                    a1 += row[ix] * tx[ix][1];
                    a2 += row[ix] * tx[ix][2];
                }
                b00 += a0 * ty[iy][0];
                b10 += a1 * ty[iy][0];
                b01 += a0 * ty[iy][1];
                b20 += a2 * ty[iy][0];
                b11 += a1 * ty[iy][1];
                b02 += a0 * ty[iy][2];
            }
            R c[3];
            spline_at<R, 2>(tz, iz, c);
            q[0] = b10 * c[0];
            q[1] = b01 * c[0];
            q[2] = b00 * c[1];
            q[3] = b20 * c[0];
            q[4] = b02 * c[0];
            q[5] = b00 * c[2];
            q[6] = b11 * c[0];
            q[7] = b10 * c[1];
            q[8] = b01 * c[1];
        }
#pragma unroll
        for (int off = 1; off < 8; off <<= 1)
#pragma unroll
            for (int k = 0; k < 9; k++) q[k] += __shfl_xor(q[k], off);
    }
    if (tv && iz == 0) {
        double s[9];
#pragma unroll
        for (int k = 0; k < 9; k++) s[k] = field[9 * (size_t)t + k];
        extrap_finish<R>(st, t, i, s, q, F, selfc, labpol, o, mud, mu_next);
    }
}

// ---------------------------------------------------------------------------
// conjugate gradients
// ---------------------------------------------------------------------------
// The solver's stopping test, the same expression as the host's report:
// converged when the RMS of S r, in Debye, is below stop_eps.
__device__ __forceinline__ double cg_stopped(double ss, int n, double stop_eps) {
    return kDebye * sqrt(ss / (double)n) >= stop_eps ? 0.0 : 1.0;
}
// Publishes check c of a solve (the state after c iterations): |r|^2 in
// scal[c & 1], scal[kCgCount] = c, scal[kCgStop] = the stopping test, and in
// host slot c & 1 the pair (|S r|^2, stop).  Slots alternate so that the host
// can read check c while the iteration after it is already running.
__device__ __forceinline__ void cg_publish(double* scal, double* hcheck, int c, double rr, double ss, double stop) {
    scal[c & 1] = rr;
    scal[kCgCount] = (double)c;
    scal[kCgStop] = stop;
    double* slot = hcheck + 2 * (c & 1);
    slot[0] = ss;
    slot[1] = stop;
}

// At most kOneSites sites: a whole update in one workgroup of 1024 threads
// (two sites a thread, everything loaded at once).  START: check 0 of a solve,
// r = rhs - Ax (Ax null: x = 0, r = rhs), p = r, mu = S p.  Else one iteration
// from Ap and the partials of p.Ap: a = rr / p.Ap, x += a p, r -= a Ap, the
// check, p = r + beta p and mu = S p.  More sites: the same in two kernels
// (k_cg_step, k_cg_direction) over many workgroups.  Evaluations one way and the
// other: 216 sites 0.46 and 0.50 ms, 1,000 0.52 and 0.54, 2,048 0.63 both.
constexpr int kOneThreads = 1024, kOnePer = kOneSites / kOneThreads;
template <class R, bool START>
__global__ __launch_bounds__(kOneThreads) void k_cg_one(SolverSites st, const double* __restrict__ rhs,
                                                        const double* __restrict__ Ap, double* x, double* r, double* p,
                                                        R* __restrict__ mu, const double* __restrict__ partial,
                                                        int npartial, double* scal, double* hcheck, int n,
                                                        double stop_eps) {
    if (!START && scal[kCgStop] != 0.0) return;
    __shared__ double sh[2 * kOneThreads / 64];
    const int c0 = START ? 0 : (int)scal[kCgCount];
    const double rr0 = START ? 0.0 : scal[c0 & 1];
    D3 rv[kOnePer], pv[kOnePer], av[kOnePer], xv[kOnePer];
    double S[kOnePer][6];
    int idx[kOnePer];
#pragma unroll
    for (int u = 0; u < kOnePer; u++) {
        const int t = threadIdx.x + u * kOneThreads;
        if (t >= st.npol) continue;
        idx[u] = st.idx[t];
        av[u] = Ap ? load3(Ap, t) : mk(0.0, 0.0, 0.0);
        rv[u] = load3(START ? rhs : r, t);
        if (!START) {
            pv[u] = load3(p, t);
            xv[u] = load3(x, t);
        }
    }
#pragma unroll
    for (int u = 0; u < kOnePer; u++)
        if ((int)threadIdx.x + u * kOneThreads < st.npol)
#pragma unroll
            for (int k = 0; k < 6; k++) S[u][k] = st.S[6 * (size_t)idx[u] + k];
    double a = 1.0;
    if (!START) {
        double pAp[1];
        sum_partials<kOneThreads, 1>(partial, npartial, pAp, sh);
        a = pAp[0] != 0.0 ? rr0 / pAp[0] : 0.0;
    }
    double s2[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < kOnePer; u++) {
        if ((int)threadIdx.x + u * kOneThreads >= st.npol) continue;
        if (!START) xv[u] = xv[u] + pv[u] * a;
        rv[u] = rv[u] - av[u] * a;
        const D3 sr = sym_mul6(S[u], rv[u]);
        s2[0] += dot(rv[u], rv[u]);
        s2[1] += dot(sr, sr);
    }
    group_sum<kOneThreads, 2>(s2, sh);  // every thread has read scal by its barriers
    const double beta = START || rr0 == 0.0 ? 0.0 : s2[0] / rr0;
    if (threadIdx.x == 0)
        cg_publish(scal, hcheck, START ? 0 : c0 + 1, s2[0], s2[1], cg_stopped(s2[1], n, stop_eps));
#pragma unroll
    for (int u = 0; u < kOnePer; u++) {
        const int t = threadIdx.x + u * kOneThreads;
        if (t >= st.npol) continue;
        const D3 d = START ? rv[u] : rv[u] + pv[u] * beta;
        if (!START) store3(x, t, xv[u]);
        else if (!Ap) store3(x, t, mk(0.0, 0.0, 0.0));
        store3(r, t, rv[u]);
        store3(p, t, d);
        store_mu<R>(mu, idx[u], sym_mul6(S[u], d));
    }
}

// x += a p, r -= a Ap (START: r = rhs - Ax) with partial sums of r.r and |S r|^2
template <bool START>
__global__ __launch_bounds__(256) void k_cg_step(SolverSites st, const double* __restrict__ rhs,
                                                 const double* __restrict__ Ap, double* x, double* r,
                                                 const double* __restrict__ p, const double* __restrict__ pap,
                                                 int npap, double* __restrict__ partial, double* scal) {
    if (!START && scal[kCgStop] != 0.0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) scal[kCgCur] = -1.0;
        return;
    }
    __shared__ double sh[2 * 4];
    double a = 1.0;
    if (!START) {
        const int c = (int)scal[kCgCount];
        double pAp[1];
        sum_partials<256, 1>(pap, npap, pAp, sh);
        a = pAp[0] != 0.0 ? scal[c & 1] / pAp[0] : 0.0;
        // k_cg_direction takes the count from here: it rewrites the other
        if (blockIdx.x == 0 && threadIdx.x == 0) scal[kCgCur] = (double)c;
    }
    double s2[2] = {0.0, 0.0};
    for (int t = blockIdx.x * 256 + threadIdx.x; t < st.npol; t += gridDim.x * 256) {
        D3 rv = load3(START ? rhs : r, t);
        if (Ap) rv = rv - load3(Ap, t) * a;
        if (!START) store3(x, t, load3(x, t) + load3(p, t) * a);
        else if (!Ap) store3(x, t, mk(0.0, 0.0, 0.0));
        store3(r, t, rv);
        const D3 sr = sym_mul6(st.S + 6 * (size_t)st.idx[t], rv);
        s2[0] += dot(rv, rv);
        s2[1] += dot(sr, sr);
    }
    group_sum<256, 2>(s2, sh);
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = s2[0];
        partial[kMaxPartials + blockIdx.x] = s2[1];
    }
}
// beta and the iteration's check (workgroup 0 publishes it), p = r + beta p
// and the next operator input mu = S p.  The iteration's number comes from
// k_cg_step in scal[kCgCur] (-1: the solve had stopped), which no workgroup
// of this kernel writes.
template <class R, bool START>
__global__ __launch_bounds__(256) void k_cg_direction(SolverSites st, const double* __restrict__ r, double* p,
                                                      R* __restrict__ mu, const double* __restrict__ partial,
                                                      int npartial, double* scal, double* hcheck, int n,
                                                      double stop_eps) {
    __shared__ double sh[2 * 4];
    const int c = START ? 0 : (int)scal[kCgCur];
    if (c < 0) return;
    const double rr0 = START ? 0.0 : scal[c & 1];
    double s2[2];
    sum_partials<256, 2>(partial, npartial, s2, sh);
    const double beta = rr0 != 0.0 ? s2[0] / rr0 : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0)
        cg_publish(scal, hcheck, START ? 0 : c + 1, s2[0], s2[1], cg_stopped(s2[1], n, stop_eps));
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= st.npol) return;
    D3 d = load3(r, t);
    if (!START) d = d + load3(p, t) * beta;
    store3(p, t, d);
    const int i = st.idx[t];
    store_mu<R>(mu, i, sym_mul6(st.S + 6 * (size_t)i, d));
}

// ---------------------------------------------------------------------------
// vectors
// ---------------------------------------------------------------------------
// Permanent field at a polarisable site: every kFixedLanes-th listed
// neighbour from `lane` on, in R, and of the covalent partners in FP64 (their
// screened and unscreened parts nearly cancel).  A whole wavefront per site
// where the sites do not fill the chip (216 sites: 12 us against 20 us with 16
// lanes), 16 lanes where they do.
constexpr int kListLanes = 16, kInitLanes = 64;
template <class R, int kFixedLanes>
__device__ __forceinline__ D3 fixed_field_part(const SolverSites& st, int t, int i, int lane, const NbrList& L,
                                               const PairAtoms<R>& A, const PairParams<R>& P,
                                               const PairAtoms<double>& A64, const PairParams<double>& P64) {
    const R4<R> pi = A.pos[i];
    const R2<R> tdi = A.td[i];
    const int cnt = L.count[i];
    R ex = 0, ey = 0, ez = 0;
    for (int k = lane; k < cnt; k += kFixedLanes) {
        const int j = L.nbr[((size_t)(k / kNlSplit) * st.npol + t) * kNlSplit + k % kNlSplit];
        const R4<R> pj = A.pos[j];
        const V3<R> dr = min_image(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), P.box);
        R mj[kMP];
#pragma unroll
        for (int c = 0; c < kMP; c++) mj[c] = A.lab[(size_t)j * kMP + c];
        // listed pairs are not covalent partners: scale 1, default Thole width
        const FixedRadial<R> gr = fixed_field_radial<R>(dot(dr, dr), tdi, R2<R>{R(0), pj.w}, R(1), P);
        const V3<R> f = fixed_field_from<R>(mj, dr, gr);
        ex += f.x;
        ey += f.y;
        ez += f.z;
    }
    D3 e = mk((double)ex, (double)ey, (double)ez);
    const int np = A64.npart[i];
    for (int k = lane; k < np; k += kFixedLanes) {
        const int en = A64.partners[(size_t)i * A64.pstride + k];
        const int j = en >> 2;
        const double4 qi = A64.pos[i], qj = A64.pos[j];
        const D3 dr = min_image(mk(qj.x - qi.x, qj.y - qi.y, qj.z - qi.z), P64.box);
        const double r2 = dot(dr, dr);
        if (r2 > P64.rc2) continue;
        const FixedRadial<double> gr =
            fixed_field_radial<double>(r2, A64.td[i], A64.td[j], partner_scale<double>(en, P64.scale14), P64);
        e = e + fixed_field_from<double>(A64.lab + (size_t)j * kMP, dr, gr);
    }
#pragma unroll
    for (int off = 1; off < kFixedLanes; off <<= 1) {
        e.x += __shfl_xor(e.x, off);
        e.y += __shfl_xor(e.y, off);
        e.z += __shfl_xor(e.z, off);
    }
    return e;
}
template <class R>
__global__ __launch_bounds__(256) void k_fixed_list(SolverSites st, NbrList L, PairAtoms<R> A, PairParams<R> P,
                                                    PairAtoms<double> A64, PairParams<double> P64,
                                                    double* __restrict__ field) {
    const int g = (int)(blockIdx.x * 256 + threadIdx.x) / kListLanes, lane = threadIdx.x % kListLanes;
    const int t = min(g, st.npol - 1);
    const D3 e = fixed_field_part<R, kListLanes>(st, t, st.idx[t], lane, L, A, P, A64, P64);
    if (g < st.npol && lane == 0) store3(field, t, e);
}
// E0 = real space + reciprocal (-A phi_1) + self, b = x = S E0 and the first
// operator input mu = S x.  LIST: the real-space part here, kInitLanes lanes
// per site (two dispatches less; the list walk then waits for phi); else one
// thread per site with the part of k_fixed_list.
template <class R, bool LIST>
__global__ __launch_bounds__(256) void k_solver_init(SolverSites st, NbrList L, PairAtoms<R> A, PairParams<R> P,
                                                     PairAtoms<double> A64, PairParams<double> P64,
                                                     const double* __restrict__ field, const double* __restrict__ phi,
                                                     FracT<double> F, double selfc, double* __restrict__ E0, double* b,
                                                     double* x, R* __restrict__ mu, double* __restrict__ mud,
                                                     const int* __restrict__ nl_scalars, int* hnl) {
    constexpr int kLanes = LIST ? kInitLanes : 1;
    const int g = (int)(blockIdx.x * 256 + threadIdx.x) / kLanes, lane = threadIdx.x % kLanes;
    if (blockIdx.x == 0 && threadIdx.x < 2) hnl[threadIdx.x] = nl_scalars[threadIdx.x];
    if (st.npol == 0) return;
    const int t = min(g, st.npol - 1);
    const int i = st.idx[t];
    D3 e;
    if (LIST) e = fixed_field_part<R, kInitLanes>(st, t, i, lane, L, A, P, A64, P64);
    else e = load3(field, t);
    if (g >= st.npol || lane != 0) return;
    const double* ph = phi + 35 * (size_t)i;
    const double* m = A64.lab + (size_t)i * kMP;
    const D3 c1 = cart_vector(mk(ph[1], ph[2], ph[3]), F);
    e.x += selfc * m[1] - c1.x;
    e.y += selfc * m[2] - c1.y;
    e.z += selfc * m[3] - c1.z;
    store3(E0, i, e);
    const double* S = st.S + 6 * (size_t)i;
    const D3 v = sym_mul6(S, e);
    store3(b, t, v);
    store3(x, t, v);
    const D3 u = sym_mul6(S, v);
    store_mu<R>(mu, i, u);
    store3(mud, i, u);
}

// mu = S v by atom (and mud, its FP64 copy); at: by site (DIIS's errors)
template <class R>
__global__ __launch_bounds__(256) void k_apply_S(SolverSites st, const double* __restrict__ v, R* mu, double* mud,
                                                 double* at) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= st.npol) return;
    const int i = st.idx[t];
    const D3 m = sym_mul6(st.S + 6 * (size_t)i, load3(v, t));
    if (mu) store_mu<R>(mu, i, m);
    if (mud) store3(mud, i, m);
    if (at) store3(at, t, m);
}

// v: the mutual solution (mu = S v); null: the dipoles are in place
// (Direct), or with ex.n > 0 the sum of the extrapolated orders, mu = sum_o
// c'_o mu_(o) with c'_o = sum_{j >= o} c_j (setExtrapolationCoefficients,
// MPIDReferenceForce.cpp:173-183; the sum at :1170-1177).  A single order is
// the dipoles in place, scaled.
template <class R>
__global__ __launch_bounds__(256) void k_final_start(SolverSites st, const double* __restrict__ v,
                                                     ExtrapCoefficients ex, const double* __restrict__ mus, R* mu,
                                                     double* mud, acc_t* __restrict__ acc, size_t count) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    for (size_t k = t; k < count; k += (size_t)gridDim.x * 256) acc[k] = 0;
    if (t >= st.npol || (!v && ex.n == 0)) return;
    const int i = st.idx[t];
    D3 m;
    if (v) {
        m = sym_mul6(st.S + 6 * (size_t)i, load3(v, t));
    } else if (ex.n == 1) {
        m = load3(mud, i) * ex.c[0];
    } else {
        m = mk(0.0, 0.0, 0.0);
        for (int o = 0; o < ex.n; o++) m = m + load3(mus + (size_t)o * 3 * st.npol, t) * ex.c[o];
    }
    store_mu<R>(mu, i, m);
    store3(mud, i, m);
}

// rt = b - A x (given Ax; null: rt is read), |S rt|^2 and x.rt: partial sums
// per workgroup, then one workgroup writes out[0], out[1] (mapped host memory)
__global__ __launch_bounds__(256) void k_residual(SolverSites st, const double* __restrict__ b,
                                                  const double* __restrict__ Ax, const double* __restrict__ x,
                                                  double* rt, double* __restrict__ partial) {
    __shared__ double sh[2 * 4];
    double s2[2] = {0.0, 0.0};
    for (int t = blockIdx.x * 256 + threadIdx.x; t < st.npol; t += gridDim.x * 256) {
        D3 v;
        if (Ax) {
            v = load3(b, t) - load3(Ax, t);
            store3(rt, t, v);
        } else {
            v = load3(rt, t);
        }
        const D3 sr = sym_mul6(st.S + 6 * (size_t)st.idx[t], v);
        s2[0] += dot(sr, sr);
        s2[1] += dot(load3(x, t), v);
    }
    group_sum<256, 2>(s2, sh);
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = s2[0];
        partial[kMaxPartials + blockIdx.x] = s2[1];
    }
}
__global__ __launch_bounds__(256) void k_residual_sum(const double* __restrict__ partial, int npartial, double* out,
                                                      double* passed, int n, double target) {
    __shared__ double sh[2 * 4];
    double s2[2];
    sum_partials<256, 2>(partial, npartial, s2, sh);
    if (threadIdx.x == 0) {
        out[0] = s2[0];
        out[1] = s2[1];
        if (passed) *passed = kDebye * sqrt(s2[0] / (double)n) < target ? 1.0 : 0.0;  // NaN does not pass
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static int site_blocks(int npol) { return std::max(1, std::min((npol + 255) / 256, kMaxPartials)); }

template <class R>
void launch_list_field(hipStream_t s, SolverSites st, NbrList l, PairAtoms<R> a, PairParams<R> p, const R* mu,
                       double* field) {
    if (st.npol <= 0) return;
    const unsigned blocks = ((unsigned)st.npol * kNlSplit + 255) / 256;
    hipLaunchKernelGGL(k_list_field<R>, dim3(blocks), dim3(256), 0, s, st, l, a, p, mu, field);
}
template <class R>
int launch_operator(hipStream_t s, SolverSites st, PmeGeom<R> g, const R* pot, const double* field, NbrList l,
                    PairAtoms<R> a, PairParams<R> p, const R* mu, double selfc, const double* v, double* Av,
                    double* partial) {
    if (st.npol <= 0) return 0;
    const int per = field ? kGatherSites : kOpSites;
    const int blocks = std::min((st.npol + per - 1) / per, kMaxPartials);
    if (field)
        hipLaunchKernelGGL(k_operator_gather<R>, dim3(blocks), dim3(256), 0, s, st, g, pot, field, a.pos, mu, selfc, v,
                           Av, partial);
    else
        hipLaunchKernelGGL(k_operator_fused<R>, dim3(blocks), dim3(256), 0, s, st, g, pot, l, a, p, mu, selfc, v, Av,
                           partial);
    return blocks;
}
template <class R>
void launch_cg_start(hipStream_t s, SolverSites st, const double* rhs, const double* Ax, double* x, double* r,
                     double* p, R* mu, double* partial, double* scal, double* hcheck, int n, double stop_eps) {
    if (st.npol <= kOneSites) {
        hipLaunchKernelGGL((k_cg_one<R, true>), dim3(1), dim3(kOneThreads), 0, s, st, rhs, Ax, x, r, p, mu, nullptr, 0,
                           scal, hcheck, n, stop_eps);
        return;
    }
    const int blocks = site_blocks(st.npol);
    hipLaunchKernelGGL(k_cg_step<true>, dim3(blocks), dim3(256), 0, s, st, rhs, Ax, x, r, p, nullptr, 0, partial, scal);
    hipLaunchKernelGGL((k_cg_direction<R, true>), dim3((st.npol + 255) / 256), dim3(256), 0, s, st, r, p, mu, partial,
                       blocks, scal, hcheck, n, stop_eps);
}
template <class R>
void launch_cg_iteration(hipStream_t s, SolverSites st, const double* Ap, double* x, double* r, double* p, R* mu,
                         int npap, double* partial, double* scal, double* hcheck, int n, double stop_eps) {
    if (st.npol <= kOneSites) {
        hipLaunchKernelGGL((k_cg_one<R, false>), dim3(1), dim3(kOneThreads), 0, s, st, nullptr, Ap, x, r, p, mu,
                           partial, npap, scal, hcheck, n, stop_eps);
        return;
    }
    const int blocks = site_blocks(st.npol);
    double* norms = partial + kMaxPartials;
    hipLaunchKernelGGL(k_cg_step<false>, dim3(blocks), dim3(256), 0, s, st, nullptr, Ap, x, r, p, partial, npap, norms,
                       scal);
    hipLaunchKernelGGL((k_cg_direction<R, false>), dim3((st.npol + 255) / 256), dim3(256), 0, s, st, r, p, mu, norms,
                       blocks, scal, hcheck, n, stop_eps);
}
template <class R>
void launch_fixed_list(hipStream_t s, SolverSites st, NbrList l, PairAtoms<R> a, PairParams<R> p,
                       PairAtoms<double> a64, PairParams<double> p64, double* field) {
    if (st.npol <= 0) return;
    const unsigned blocks = ((unsigned)st.npol * kListLanes + 255) / 256;
    hipLaunchKernelGGL(k_fixed_list<R>, dim3(blocks), dim3(256), 0, s, st, l, a, p, a64, p64, field);
}
template <class R>
void launch_solver_init(hipStream_t s, SolverSites st, NbrList l, PairAtoms<R> a, PairParams<R> p,
                        PairAtoms<double> a64, PairParams<double> p64, const double* field, const double* phi,
                        FracT<double> A, double selfc, double* E0, double* b, double* x, R* mu, double* mud,
                        const int* nl_scalars, int* hnl) {
    const unsigned threads = std::max(1u, (unsigned)st.npol * (field ? 1 : kInitLanes));
    const dim3 blocks((threads + 255) / 256);
    if (field)
        hipLaunchKernelGGL((k_solver_init<R, false>), blocks, dim3(256), 0, s, st, l, a, p, a64, p64, field, phi, A,
                           selfc, E0, b, x, mu, mud, nl_scalars, hnl);
    else
        hipLaunchKernelGGL((k_solver_init<R, true>), blocks, dim3(256), 0, s, st, l, a, p, a64, p64, field, phi, A,
                           selfc, E0, b, x, mu, mud, nl_scalars, hnl);
}
template <class R>
void launch_apply_S(hipStream_t s, SolverSites st, const double* v, R* mu, double* mud, double* at) {
    if (st.npol <= 0) return;
    hipLaunchKernelGGL(k_apply_S<R>, dim3((st.npol + 255) / 256), dim3(256), 0, s, st, v, mu, mud, at);
}
template <class R>
void launch_final_start(hipStream_t s, SolverSites st, const double* v, const ExtrapCoefficients& ex,
                        const double* mus, R* mu, double* mud, acc_t* acc, size_t count) {
    const size_t blocks = std::max<size_t>((st.npol + 255) / 256, std::min<size_t>((count + 255) / 256, 2048));
    hipLaunchKernelGGL(k_final_start<R>, dim3((unsigned)std::max<size_t>(blocks, 1)), dim3(256), 0, s, st, v, ex, mus,
                       mu, mud, acc, count);
}
template <class R>
void launch_extrap_list(hipStream_t s, SolverSites st, NbrList l, PairAtoms<R> a, PairParams<R> p, const R* mu,
                        double* field) {
    if (st.npol <= 0) return;
    const unsigned blocks = ((unsigned)st.npol * kNlSplit + 255) / 256;
    hipLaunchKernelGGL(k_extrap_list<R>, dim3(blocks), dim3(256), 0, s, st, l, a, p, mu, field);
}
template <class R>
void launch_extrap_order(hipStream_t s, SolverSites st, PmeGeom<R> g, const R* pot, const double* field, NbrList l,
                         PairAtoms<R> a, PairParams<R> p, const R* mu, R* mu_next, FracT<double> A, double selfc,
                         const double* labpol, const ExtrapOrder& o, const double* mud) {
    if (st.npol <= 0) return;
    if (field)
        hipLaunchKernelGGL(k_extrap_gather<R>, dim3(((unsigned)st.npol * 8 + 255) / 256), dim3(256), 0, s, st, g, pot,
                           field, a.pos, A, selfc, labpol, o, mud, mu_next);
    else
        hipLaunchKernelGGL(k_extrap_fused<R>, dim3((st.npol + kOpSites - 1) / kOpSites), dim3(256), 0, s, st, g, pot, l,
                           a, p, mu, mu_next, A, selfc, labpol, o, mud);
}
void launch_residual(hipStream_t s, SolverSites st, const double* b, const double* Ax, const double* x, double* rt,
                     double* partial, double* out, double* passed, int n, double target) {
    const int blocks = site_blocks(st.npol);
    hipLaunchKernelGGL(k_residual, dim3(blocks), dim3(256), 0, s, st, b, Ax, x, rt, partial);
    hipLaunchKernelGGL(k_residual_sum, dim3(1), dim3(256), 0, s, partial, blocks, out, passed, n,
                       target);
}

#define MPID_INSTANTIATE(R)                                                                                         \
    template void launch_list_field<R>(hipStream_t, SolverSites, NbrList, PairAtoms<R>, PairParams<R>, const R*,    \
                                       double*);                                                                   \
    template int launch_operator<R>(hipStream_t, SolverSites, PmeGeom<R>, const R*, const double*, NbrList,         \
                                    PairAtoms<R>, PairParams<R>, const R*, double, const double*, double*,          \
                                    double*);                                                                      \
    template void launch_cg_start<R>(hipStream_t, SolverSites, const double*, const double*, double*, double*,      \
                                     double*, R*, double*, double*, double*, int, double);                          \
    template void launch_cg_iteration<R>(hipStream_t, SolverSites, const double*, double*, double*, double*, R*,    \
                                         int, double*, double*, double*, int, double);                              \
    template void launch_fixed_list<R>(hipStream_t, SolverSites, NbrList, PairAtoms<R>, PairParams<R>,              \
                                       PairAtoms<double>, PairParams<double>, double*);                            \
    template void launch_solver_init<R>(hipStream_t, SolverSites, NbrList, PairAtoms<R>, PairParams<R>,             \
                                        PairAtoms<double>, PairParams<double>, const double*, const double*,        \
                                        FracT<double>, double, double*, double*, double*, R*, double*, const int*,  \
                                        int*);                                                                     \
    template void launch_final_start<R>(hipStream_t, SolverSites, const double*, const ExtrapCoefficients&,         \
                                        const double*, R*, double*, acc_t*, size_t);                               \
    template void launch_extrap_list<R>(hipStream_t, SolverSites, NbrList, PairAtoms<R>, PairParams<R>, const R*,   \
                                        double*);                                                                  \
    template void launch_extrap_order<R>(hipStream_t, SolverSites, PmeGeom<R>, const R*, const double*, NbrList,    \
                                         PairAtoms<R>, PairParams<R>, const R*, R*, FracT<double>, double,          \
                                         const double*, const ExtrapOrder&, const double*);                        \
    template void launch_apply_S<R>(hipStream_t, SolverSites, const double*, R*, double*, double*);
MPID_INSTANTIATE(float)
MPID_INSTANTIATE(double)
#undef MPID_INSTANTIATE

}  // namespace mpid
