// Elastic-wave right-hand side pieces and p-multigrid transfer on the GPU (FP64):
//   inverse mass (apply_inverse_mass, elasticity.py:236-238): y_e = Mhat^-1 E diag(w_e) E^T Mhat^-1 x_e
//     with w_e(q) = -W_q / |J_e(q)| (the weight-adjusted inverse of the curvilinear element mass
//     with density 1, Elasticity.cpp:227-253); on the matrix cores in two contractions with
//     P = Mhat^-1 E, y_e = P diag(w_e) P^T x_e, where the rule sizes are compiled, else one workgroup
//     per element with four stages in LDS;
//   nodal interpolation (NodalInterpolation.cpp:8-38): y_e = I x_e per quantity (prolongation
//     from degree `from` to degree `to`) or I^T (restriction);
#include "kernels.h"
#include "mfma_layout.h"
#include "mfma_ops.h"

#include <algorithm>
#include <climits>

namespace tdg {

namespace {

constexpr int kT = 128;

__global__ __launch_bounds__(kT) void inverse_mass_kernel(WaveArgs a, double const* __restrict__ x,
                                                          double* __restrict__ y) {
    extern __shared__ double sh[];
    const int Nbf = a.nbf, Nq = a.nq, Q = a.nquant, bs = Nbf * Q;
    double* t = sh;              // bs
    double* uq = sh + bs;        // Nq * Q
    const int64_t e = blockIdx.x;
    double const* xe = x + e * bs;
    for (int i = threadIdx.x; i < bs; i += kT) {
        const int k = i % Nbf, p = i / Nbf;
        double v = 0.0;
        for (int l = 0; l < Nbf; ++l) v += a.Minv[k + l * Nbf] * xe[l + p * Nbf];
        t[i] = v;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < Nq * Q; i += kT) {
        const int q = i % Nq, p = i / Nq;
        double v = 0.0;
        for (int k = 0; k < Nbf; ++k) v += a.E[k * Nq + q] * t[k + p * Nbf];
        uq[i] = v * a.w[e * Nq + q];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < bs; i += kT) {
        const int k = i % Nbf, p = i / Nbf;
        double v = 0.0;
        for (int q = 0; q < Nq; ++q) v += a.E[k * Nq + q] * uq[q + p * Nq];
        t[i] = v; // stage 3 reads only uq
    }
    __syncthreads();
    for (int i = threadIdx.x; i < bs; i += kT) {
        const int k = i % Nbf, p = i / Nbf;
        double v = 0.0;
        for (int l = 0; l < Nbf; ++l) v += a.Minv[k + l * Nbf] * t[l + p * Nbf];
        y[e * bs + i] = v;
    }
}

__global__ __launch_bounds__(256) void interpolate_kernel(double const* __restrict__ I, int n_to, int n_from, int nquant,
                                                          int64_t nelem, int transpose, double const* __restrict__ x,
                                                          double* __restrict__ y) {
    const int n_out = transpose ? n_from : n_to, n_in = transpose ? n_to : n_from;
    const int64_t total = nelem * n_out * nquant;
    for (int64_t t = int64_t(blockIdx.x) * 256 + threadIdx.x; t < total; t += int64_t(gridDim.x) * 256) {
        const int64_t e = t / (int64_t(n_out) * nquant);
        const int r = int(t % (int64_t(n_out) * nquant)), p = r / n_out, k = r % n_out;
        double const* xe = x + e * int64_t(n_in) * nquant + p * n_in;
        double v = 0.0;
        if (transpose)
            for (int l = 0; l < n_in; ++l) v += I[l * n_from + k] * xe[l];
        else
            for (int l = 0; l < n_in; ++l) v += I[k * n_from + l] * xe[l];
        y[e * int64_t(n_out) * nquant + p * n_out + k] = v;
    }
}

// y = P diag(w) P^T x, one wave per 16 consecutive elements (the columns of every tile): per block of 16
// points the point values C = P^T U on the matrix cores, scaled by w in registers, are the B operands
// of Y += P C (register i of lane group g is point 16 b + mfma_row(g, i)).  Streams x, w and y once
// (8 (2 bs + Nq) bytes an element); the per-element kernel below, which reads its tables from L1 for
// every multiply-add, took 88 us for 20,160 P3 tetrahedra (0.27 TB/s).  With this kernel and the facet
// part added in place, the whole wave right-hand side of that mesh went from 237 to 105 us.
template <int D, int N, int W>
__global__ __launch_bounds__(64 * W) void inverse_mass_mfma_kernel(WaveArgs a, double const* x, double* y) {
    using L = MfmaLayout<D, N>;
    using acc = Mma<double>::acc;
    constexpr int Nbf = L::Nbf, Nq = L::Nq, Q = D, BS = Nbf * Q, KS = L::KS, QB = L::QB, MT = L::MT;
    constexpr int NO = (16 * BS + 63) / 64;
    __shared__ double sP[Nq * Nbf];
    __shared__ double sU[W][16 * BS];
    for (int i = threadIdx.x; i < Nq * Nbf; i += 64 * W) sP[i] = a.P[i];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const int64_t grp = int64_t(blockIdx.x) * W + wv, e0 = grp * 16;
    const int nel = e0 < a.num_elements ? int(min(int64_t(16), a.num_elements - e0)) : 0;
    const int nout = nel * BS;
    double* const U = sU[wv];
    {
        double const* xw = x + (nel ? e0 : 0) * BS;
        double v[NO];
#pragma unroll
        for (int o = 0; o < NO; ++o) v[o] = 64 * o + lane < nout ? xw[64 * o + lane] : 0.0;
#pragma unroll
        for (int o = 0; o < NO; ++o)
            if (64 * o + lane < 16 * BS) U[64 * o + lane] = v[o];
    }
    __syncthreads();
    if (nel == 0) return; // no barrier below: the staged vectors are this wave's
    double const* const Uj = U + j * BS;
    acc Y[MT][Q];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int r = 0; r < Q; ++r) Y[m][r] = acc{0, 0, 0, 0};
#pragma unroll 1
    for (int b = 0; b < QB; ++b) {
        double wq[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = 16 * b + mfma_row<double>(g, i);
            wq[i] = q < Nq ? a.w[(grp * Nq + q) * 16 + j] : 0.0;
        }
        acc C[Q];
#pragma unroll
        for (int r = 0; r < Q; ++r) C[r] = acc{0, 0, 0, 0};
        const int qa = min(16 * b + j, Nq - 1) * Nbf;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int k = 4 * s + g, kc = min(k, Nbf - 1);
            const double av = sP[qa + kc];
#pragma unroll
            for (int r = 0; r < Q; ++r) {
                const double bv = Uj[kc + r * Nbf];
                C[r] = Mma<double>::mma(av, k < Nbf ? bv : 0.0, C[r]);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (16 * b + mfma_row<double>(0, i) >= Nq) continue; // all four lane groups past the last point
            const int qr = min(16 * b + mfma_row<double>(g, i), Nq - 1) * Nbf;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const double av = sP[qr + min(16 * m + j, Nbf - 1)];
#pragma unroll
                for (int r = 0; r < Q; ++r) Y[m][r] = Mma<double>::mma(av, wq[i] * C[r][i], Y[m][r]);
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier(); // every read of the staged vectors is complete
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * m + mfma_row<double>(g, i);
            if (k < Nbf) {
#pragma unroll
                for (int r = 0; r < Q; ++r) U[j * BS + k + r * Nbf] = Y[m][r][i];
            }
        }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int i = lane; i < nout; i += 64) y[e0 * BS + i] = U[i];
}

template <int D, int N> hipError_t run_inverse_mass(WaveArgs const& a, double const* x, double* y, hipStream_t s) {
    constexpr int W = 4;
    const int64_t blocks = ((a.num_elements + 15) / 16 + W - 1) / W;
    if (blocks > int64_t(INT_MAX)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((inverse_mass_mfma_kernel<D, N, W>), dim3(unsigned(blocks)), dim3(64 * W), 0, s, a, x, y);
    return hipGetLastError();
}

unsigned grid256(int64_t n) { return unsigned(std::min<int64_t>((n + 255) / 256, 65536)); }

} // namespace

// The degrees whose rule sizes are compiled take the matrix-core kernel; the other operators (3D P5 and
// P6, for which no apply is compiled) the kernel with run-time sizes, and so do the smallest 3D P4 meshes, where
// a workgroup an element is done sooner than a wave's chain through 16 of them (us, run-time sizes and matrix
// cores: 6 elements 10.2 and 11.3, 162: 10.5 and 12.5, 480: 11.6 and 12.6, 1,296: 21.1 and 12.7; 3D P3 6: 6.7 and 5.6).
bool inverse_mass_grouped(int dim, int degree, int64_t num_elements) {
    return degree >= 1 && degree <= (dim == 2 ? 6 : 4) && !(dim == 3 && degree == 4 && num_elements <= 512);
}

hipError_t launch_inverse_mass(int dim, int degree, WaveArgs const& a, double const* x, double* y, hipStream_t s) {
    if (!inverse_mass_grouped(dim, degree, a.num_elements)) {
        const std::size_t shm = std::size_t(a.nbf * a.nquant + a.nq * a.nquant) * sizeof(double);
        if (shm > 64 * 1024) return hipErrorInvalidValue;
        hipLaunchKernelGGL(inverse_mass_kernel, dim3(unsigned(a.num_elements)), dim3(kT), shm, s, a, x, y);
        return hipGetLastError();
    }
    if (dim == 3) {
        switch (degree) {
        case 1: return run_inverse_mass<3, 1>(a, x, y, s);
        case 2: return run_inverse_mass<3, 2>(a, x, y, s);
        case 3: return run_inverse_mass<3, 3>(a, x, y, s);
        case 4: return run_inverse_mass<3, 4>(a, x, y, s);
        }
    } else if (dim == 2) {
        switch (degree) {
        case 1: return run_inverse_mass<2, 1>(a, x, y, s);
        case 2: return run_inverse_mass<2, 2>(a, x, y, s);
        case 3: return run_inverse_mass<2, 3>(a, x, y, s);
        case 4: return run_inverse_mass<2, 4>(a, x, y, s);
        case 5: return run_inverse_mass<2, 5>(a, x, y, s);
        case 6: return run_inverse_mass<2, 6>(a, x, y, s);
        }
    }
    return hipErrorInvalidValue;
}

hipError_t launch_interpolate(double const* I, int n_to, int n_from, int nquant, int64_t nelem, int transpose,
                              double const* x, double* y, hipStream_t s) {
    const int64_t total = nelem * (transpose ? n_from : n_to) * nquant;
    hipLaunchKernelGGL(interpolate_kernel, dim3(grid256(total)), dim3(256), 0, s, I, n_to, n_from, nquant, nelem,
                       transpose, x, y);
    return hipGetLastError();
}

} // namespace tdg
