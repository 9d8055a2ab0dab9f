// Right-hand side and facet traction of the elasticity operator on the GPU (FP64).
//
// rhs      : b = rhsVolume (one lane per element and basis function, zero without a force) + rhsFacet
//            over the Dirichlet and Fault facets, one workgroup per element that has such a face, in one
//            launch (Elasticity.cpp:521-696; elasticity.py:151-180).  Facet data are
//            the Dirichlet values on Dirichlet facets and the slip on Fault facets; a Fault on the
//            boundary takes half the slip (bc_boundary, Elasticity.cpp:559-573).  A skeleton facet
//            adds to both of its elements with c10 = eps/2 and c20 = +penalty (side 0) /
//            -penalty (side 1), both with the side-0 normal (rhs_skeleton, :575-643); a boundary
//            facet with c10 = eps, c20 = penalty (rhs_boundary, :645-696).
// traction : per facet and facet point, 1/2 (traction_0 + traction_1) - penalty (u_0 - u_1 - f) on
//            skeleton facets and traction_0 - penalty (u_0 - f) on boundary facets, with the unit
//            normal of side 0 (compute_traction / compute_traction_bnd, elasticity.py:242-250;
//            Elasticity.cpp:949-1018).
// Both use the apply kernels' facet data: the face-0 reference table with the node relabelling
// perm_f and the per-side facet geometry G' = J_f^-1 J^-1.
#include "kernels.h"

#include <climits>
#include <type_traits>

namespace tdg {

namespace {

constexpr int binom_(int n, int k) { return k == 0 ? 1 : binom_(n - 1, k - 1) * n / k; }
constexpr int vol_points_(int D, int N) {
    return D == 2 ? (N == 1 ? 4 : N == 2 ? 7 : N == 3 ? 15 : N == 4 ? 19 : N == 5 ? 28 : 37)
                  : (N == 1 ? 6 : N == 2 ? 14 : N == 3 ? 31 : 57);
}
constexpr int fct_points_(int D, int N) { return D == 2 ? N + 1 : (N == 1 ? 4 : N == 2 ? 7 : N == 3 ? 15 : 19); }

constexpr int kBC_Fault = 3, kBC_Dirichlet = 5;
constexpr int kThreads = 256;

// Facet part of one element by the lanes of a workgroup: a lane per (face, point) forms the lift weights of
// its data (value channel and the D reference gradients) in LDS, then entry `it` of the element is a
// contraction of them.  Visiting every element with a lane per basis function, each lane repeating its
// points' geometry, took 46-52 us for the 1,800 boundary faces of 20,160 P3 tetrahedra.
constexpr int kFacetThreads = 128;
template <int D, int N> struct FacetLifts {
    static constexpr int Nbf = binom_(N + D, D), nq = fct_points_(D, N), Q = D, DD = D * D, NF = D + 1, C = D + 1;
    double W[NF][nq][C][Q];
    int on[NF];

    __device__ void form(RhsArgs const& a, int64_t e, double sign, double const* fd) {
        for (int it = threadIdx.x; it < NF * nq; it += kFacetThreads) {
            const int f = it / nq, q = it % nq;
            const int4 info = a.ef[e * NF + f];
            const int64_t fct = info.x;
            const int fb = a.fbc[fct], bc = fb & 0xff;
            const bool skel = (fb >> 8) & 1, data = bc == kBC_Dirichlet || bc == kBC_Fault;
            if (q == 0) on[f] = data;
            if (!data) continue;
            const int side = (info.z >> 2) & 1;
            const int64_t fs = (fct * 2 + side) * nq + q;
            const double scale = (!skel && bc == kBC_Fault) ? 0.5 : 1.0;
            const double c10 = skel ? -0.5 : -1.0, c20 = side == 0 ? a.fpen[fct] : -a.fpen[fct];
            const double lq = a.fc0[fs], mq = a.fc1[fs], w = sign * a.w[q];
            double n[D], g[Q], nn = 0.0, fn = 0.0;
#pragma unroll
            for (int j = 0; j < D; ++j) {
                n[j] = a.fn[(fct * nq + q) * D + j];
                nn += n[j] * n[j];
            }
#pragma unroll
            for (int p = 0; p < Q; ++p) {
                g[p] = scale * fd[(fct * Q + p) * nq + q];
                fn += g[p] * n[p];
            }
            const double nl = sqrt(nn);
#pragma unroll
            for (int p = 0; p < Q; ++p) W[f][q][0][p] = c20 * w * nl * g[p];
#pragma unroll
            for (int ee = 0; ee < D; ++ee)
#pragma unroll
                for (int p = 0; p < Q; ++p) {
                    double v = 0.0;
#pragma unroll
                    for (int j = 0; j < D; ++j) {
                        double S = mq * (n[j] * g[p] + g[j] * n[p]);
                        if (j == p) S += lq * fn;
                        v += a.fG[fs * DD + ee + j * D] * S;
                    }
                    W[f][q][1 + ee][p] = c10 * w * v;
                }
        }
    }
    __device__ double sum(RhsArgs const& a, int it) const {
        const int p = it / Nbf, k = it % Nbf;
        double acc = 0.0;
#pragma unroll 1
        for (int f = 0; f < NF; ++f) {
            if (!on[f]) continue;
            double const* t = a.tabFt + a.iperm[f * Nbf + k]; // face-0 label of basis function k on face f
            for (int q = 0; q < nq; ++q)
#pragma unroll
                for (int c = 0; c < C; ++c) acc += t[(c * nq + q) * Nbf] * W[f][q][c][p];
        }
        return acc;
    }
};

// b = volume part + facet part in one launch: the first nf workgroups (the longer ones) take an element with
// facet data each, the others a lane per element and basis function of the rest (zero without a force).
// In two launches (zero or volume, then the facets in place) a call with facet data took 8.9 us on meshes of a
// few thousand elements, in one 6.4; 3D P3 7,986 elements with a force 18.8 and 15.6, P4 16,464: 78.3 and 79.3.
template <int D, int N>
__global__ __launch_bounds__(kFacetThreads) void elasticity_rhs_kernel(RhsArgs a, double const* __restrict__ force,
                                                                       double const* __restrict__ fdata,
                                                                       double* __restrict__ b, int64_t ld_force,
                                                                       int64_t ld_fdata, int64_t ld_b, unsigned nf) {
    constexpr int Nbf = binom_(N + D, D), Nq = vol_points_(D, N), Q = D, BS = Nbf * Q;
    __shared__ FacetLifts<D, N> lifts;
    double const* const fo = force ? force + blockIdx.y * ld_force : nullptr;
    double* const bc = b + blockIdx.y * ld_b;
    if (blockIdx.x >= nf) {
        const int64_t item = int64_t(blockIdx.x - nf) * kFacetThreads + threadIdx.x, e = item / Nbf;
        if (e >= a.num_elements || (fdata && a.edata[e])) return;
        const int k = int(item % Nbf);
        double acc[Q];
#pragma unroll
        for (int p = 0; p < Q; ++p) acc[p] = 0.0;
        if (fo) {
            for (int q = 0; q < Nq; ++q) {
                const double t = a.jw[e * Nq + q] * a.tabE[k * Nq + q];
#pragma unroll
                for (int p = 0; p < Q; ++p) acc[p] += t * fo[(e * Q + p) * Nq + q];
            }
        }
#pragma unroll
        for (int p = 0; p < Q; ++p) bc[e * BS + k + p * Nbf] = acc[p];
        return;
    }
    __shared__ double jw[Nq], f[Q * Nq];
    const int64_t e = a.elist[blockIdx.x];
    if (fo) {
        for (int i = threadIdx.x; i < Nq; i += kFacetThreads) jw[i] = a.jw[e * Nq + i];
        for (int i = threadIdx.x; i < Q * Nq; i += kFacetThreads) f[i] = fo[e * Q * Nq + i];
    }
    lifts.form(a, e, 1.0, fdata + blockIdx.y * ld_fdata);
    __syncthreads();
    for (int it = threadIdx.x; it < BS; it += kFacetThreads) {
        const int p = it / Nbf, k = it % Nbf;
        double acc = 0.0;
        if (fo)
            for (int q = 0; q < Nq; ++q) acc += jw[q] * a.tabE[k * Nq + q] * f[p * Nq + q];
        bc[e * BS + it] = acc + lifts.sum(a, it);
    }
}

// b += sign times the facet part on the elements that have data.
template <int D, int N>
__global__ __launch_bounds__(kFacetThreads) void elasticity_rhs_facet_kernel(RhsArgs a, double sign,
                                                                             double const* __restrict__ fdata,
                                                                             double* __restrict__ b, int64_t ld_fdata,
                                                                             int64_t ld_b) {
    constexpr int BS = binom_(N + D, D) * D;
    __shared__ FacetLifts<D, N> lifts;
    const int64_t e = a.elist[blockIdx.x];
    lifts.form(a, e, sign, fdata + blockIdx.y * ld_fdata);
    __syncthreads();
    double* const bo = b + blockIdx.y * ld_b + e * BS;
    for (int it = threadIdx.x; it < BS; it += kFacetThreads) bo[it] += lifts.sum(a, it);
}

template <int D, int N>
__global__ __launch_bounds__(kThreads) void elasticity_traction_kernel(RhsArgs a, double const* __restrict__ xs,
                                                                       double const* __restrict__ fds,
                                                                       double* __restrict__ tqs,
                                                                       int32_t const* __restrict__ sub, int64_t nsub,
                                                                       int64_t ld_x, int64_t ld_f, int64_t ld_t) {
    constexpr int Nbf = binom_(N + D, D), nq = fct_points_(D, N);
    constexpr int Q = D, BS = Nbf * Q, DD = D * D, C = D + 1;
    const int64_t item = int64_t(blockIdx.x) * kThreads + threadIdx.x;
    if (item >= nsub * nq) return;
    // facet `fct` of the list (all facets, or the subset sub), output row `row`, column blockIdx.y
    const int64_t row = item / nq;
    const int64_t fct = sub ? int64_t(sub[row]) : row;
    const int q = int(item % nq);
    double const* __restrict__ x = xs + int64_t(blockIdx.y) * ld_x;
    double const* __restrict__ fdata = fds ? fds + int64_t(blockIdx.y) * ld_f : nullptr;
    double* __restrict__ tq = tqs + int64_t(blockIdx.y) * ld_t;
    const int4 fi = a.fct[fct]; // {element 0, element 1, local face 0 | local face 1 << 4, -}
    const int fb = a.fbc[fct];
    const int bc = fb & 0xff;
    const bool skel = (fb >> 8) & 1;
    const int ns = skel ? 2 : 1;
    double n[D], nn = 0.0;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        n[j] = a.fn[(fct * nq + q) * D + j];
        nn += n[j] * n[j];
    }
    const double inl = 1.0 / sqrt(nn);
    double tr[Q], jump[Q];
#pragma unroll
    for (int p = 0; p < Q; ++p) tr[p] = jump[p] = 0.0;
    for (int s = 0; s < ns; ++s) {
        const int64_t el = s == 0 ? fi.x : fi.y;
        const int lf = s == 0 ? (fi.z & 15) : ((fi.z >> 4) & 15);
        double const* u = x + el * BS;
        int32_t const* pm = &a.perm[lf * Nbf];
        double uv[Q], gx[D][Q];
#pragma unroll
        for (int r = 0; r < Q; ++r) {
            uv[r] = 0.0;
#pragma unroll
            for (int ee = 0; ee < D; ++ee) gx[ee][r] = 0.0;
        }
        for (int l = 0; l < Nbf; ++l) {
            const int kk = pm[l];
            double const* t = &a.tabF[(l * C) * nq + q];
#pragma unroll
            for (int r = 0; r < Q; ++r) {
                const double ul = u[kk + r * Nbf];
                uv[r] += t[0] * ul;
#pragma unroll
                for (int ee = 0; ee < D; ++ee) gx[ee][r] += t[(1 + ee) * nq] * ul;
            }
        }
        double G[DD];
#pragma unroll
        for (int i = 0; i < DD; ++i) G[i] = a.fG[((fct * 2 + s) * nq + q) * DD + i];
        const double lq = a.fc0[(fct * 2 + s) * nq + q], mq = a.fc1[(fct * 2 + s) * nq + q];
        double J[Q][D]; // J[r][j] = du_r/dx_j
        double div = 0.0;
#pragma unroll
        for (int r = 0; r < Q; ++r)
#pragma unroll
            for (int j = 0; j < D; ++j) {
                double v = 0.0;
#pragma unroll
                for (int ee = 0; ee < D; ++ee) v += G[ee + j * D] * gx[ee][r];
                J[r][j] = v;
            }
#pragma unroll
        for (int r = 0; r < D; ++r) div += J[r][r];
        const double h = skel ? 0.5 : 1.0;
#pragma unroll
        for (int p = 0; p < Q; ++p) {
            double v = lq * div * n[p] * inl;
#pragma unroll
            for (int j = 0; j < D; ++j) v += mq * (J[p][j] + J[j][p]) * n[j] * inl;
            tr[p] += h * v;
            jump[p] += s == 0 ? uv[p] : -uv[p];
        }
    }
    const bool data = fdata && (bc == kBC_Dirichlet || bc == kBC_Fault);
    const double scale = (!skel && bc == kBC_Fault) ? 0.5 : 1.0;
    const double c00 = -a.fpen[fct];
#pragma unroll
    for (int p = 0; p < Q; ++p) {
        const double f = data ? scale * fdata[(fct * Q + p) * nq + q] : 0.0;
        tq[(row * Q + p) * nq + q] = tr[p] + c00 * (jump[p] - f);
    }
}

template <int D, int N>
hipError_t run_rhs_facets(RhsArgs const& a, double sign, double const* fdata, double* b, int ncols, int64_t ld_fdata,
                          int64_t ld_b, hipStream_t s) {
    if (a.num_elist == 0) return hipSuccess;
    hipLaunchKernelGGL((elasticity_rhs_facet_kernel<D, N>), dim3(unsigned(a.num_elist), unsigned(ncols)),
                       dim3(kFacetThreads), 0, s, a, sign, fdata, b, ld_fdata, ld_b);
    return hipGetLastError();
}

template <int D, int N>
hipError_t run_rhs(RhsArgs const& a, double const* force, double const* fdata, double* b, int ncols,
                   int64_t ld_force, int64_t ld_fdata, int64_t ld_b, hipStream_t s) {
    constexpr int Nbf = binom_(N + D, D);
    const int64_t nv = (a.num_elements * Nbf + kFacetThreads - 1) / kFacetThreads, nf = fdata ? a.num_elist : 0;
    if (nv + nf > int64_t(INT_MAX)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((elasticity_rhs_kernel<D, N>), dim3(unsigned(nv + nf), unsigned(ncols)), dim3(kFacetThreads), 0, s,
                       a, force, fdata, b, ld_force, ld_fdata, ld_b, unsigned(nf));
    return hipGetLastError();
}

template <int D, int N>
hipError_t run_traction(RhsArgs const& a, double const* x, double const* fdata, double* t, int32_t const* sub,
                        int64_t nsub, int ncols, int64_t ld_x, int64_t ld_f, int64_t ld_t, hipStream_t s) {
    constexpr int nq = fct_points_(D, N);
    const int64_t items = nsub * nq;
    if (items == 0) return hipSuccess;
    dim3 grid(unsigned((items + kThreads - 1) / kThreads), unsigned(ncols));
    hipLaunchKernelGGL((elasticity_traction_kernel<D, N>), grid, dim3(kThreads), 0, s, a, x, fdata, t, sub, nsub, ld_x,
                       ld_f, ld_t);
    return hipGetLastError();
}

template <class F> hipError_t by_degree(int dim, int degree, F&& f) {
    if (dim == 3) {
        switch (degree) {
        case 1: return f(std::integral_constant<int, 3>{}, std::integral_constant<int, 1>{});
        case 2: return f(std::integral_constant<int, 3>{}, std::integral_constant<int, 2>{});
        case 3: return f(std::integral_constant<int, 3>{}, std::integral_constant<int, 3>{});
        case 4: return f(std::integral_constant<int, 3>{}, std::integral_constant<int, 4>{});
        }
    } else if (dim == 2) {
        switch (degree) {
        case 1: return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
        case 2: return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
        case 3: return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{});
        case 4: return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 4>{});
        case 5: return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 5>{});
        case 6: return f(std::integral_constant<int, 2>{}, std::integral_constant<int, 6>{});
        }
    }
    return hipErrorInvalidValue;
}

} // namespace

hipError_t launch_elasticity_rhs(int dim, int degree, RhsArgs const& a, double const* force, double const* fdata,
                                 double* b, int ncols, int64_t ld_force, int64_t ld_fdata, int64_t ld_b,
                                 hipStream_t s) {
    return by_degree(dim, degree, [&](auto Dc, auto Nc) {
        return run_rhs<decltype(Dc)::value, decltype(Nc)::value>(a, force, fdata, b, ncols, ld_force, ld_fdata, ld_b,
                                                                  s);
    });
}

hipError_t launch_elasticity_rhs_facets(int dim, int degree, RhsArgs const& a, double sign, double const* fdata,
                                        double* b, int ncols, int64_t ld_fdata, int64_t ld_b, hipStream_t s) {
    return by_degree(dim, degree, [&](auto Dc, auto Nc) {
        return run_rhs_facets<decltype(Dc)::value, decltype(Nc)::value>(a, sign, fdata, b, ncols, ld_fdata, ld_b, s);
    });
}

hipError_t launch_elasticity_traction(int dim, int degree, RhsArgs const& a, double const* x, double const* fdata,
                                      double* t, hipStream_t s) {
    return by_degree(dim, degree, [&](auto Dc, auto Nc) {
        return run_traction<decltype(Dc)::value, decltype(Nc)::value>(a, x, fdata, t, nullptr, a.num_facets, 1, 0, 0,
                                                                       0, s);
    });
}

hipError_t launch_elasticity_traction_subset(int dim, int degree, RhsArgs const& a, double const* x,
                                             double const* fdata, double* t, int32_t const* sub, int64_t nsub,
                                             int ncols, int64_t ld_x, int64_t ld_f, int64_t ld_t, hipStream_t s) {
    return by_degree(dim, degree, [&](auto Dc, auto Nc) {
        return run_traction<decltype(Dc)::value, decltype(Nc)::value>(a, x, fdata, t, sub, nsub, ncols, ld_x, ld_f,
                                                                       ld_t, s);
    });
}

} // namespace tdg
