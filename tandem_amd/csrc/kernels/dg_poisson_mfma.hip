// Poisson SIPG apply on the matrix cores, in two kernels over groups of 16 consecutive elements (one wave
// per group, its elements the columns of every 16x16x4 tile).
//
// The modal basis has no face-0 frame (a face's functions are not a relabelling of face 0's), so a
// neighbour's trace cannot share an operand table with the other columns.  Each element therefore
// evaluates its own traces on its own faces, where all 16 columns share the face's table, and the two
// sides meet in memory:
//   traces   : per face f and point q  C(c, q ; el) = sum_k T_f(c, q ; k) x(k ; el), then
//              u = C(0), s = K grad u . n = sum_e kn_e C(1 + e) with kn = K G n (n outward,
//              area-scaled), stored as TR[element][f][q] = {u, s}
//   elements : volume  C(e, q) = sum_k V(e, q ; k) x(k),  Y(k) += sum_(e,q) V(e, q ; k) S_ee' C(e', q)
//                      with the symmetric S = W|J| K G G^T stored per point (3 or 6 reals);
//              face f  own and neighbour's {u, s} (the points of the two sides coincide):
//                      sigma.n = (s - s_nb) / 2 - p (u - u_nb), d = (u_nb - u) / 2 (boundary:
//                      s - p u, -u) with p = penalty |n|, and
//                      Y(k) += sum_q w (-T_f(0, q ; k) sigma.n + d sum_e T_f(1 + e, q ; k) kn_e)
// Per element and volume point 3 (2D) or 6 reals are read, per face point D + 1 and two pairs; the
// thread-per-point kernel (dg_apply.hip) reads 5 (10) and about 2 (D^2 + D), and its tables from L1 for
// every multiply-add.  51,200 P4 triangles in FP64: 106 -> 26 us; 24,576 P4
// tetrahedra 691 -> 130 us.
#include "kernels.h"
#include "mfma_layout.h"
#include "mfma_ops.h"

#include <climits>

namespace tdg {

namespace {

template <class T> struct Pair;
template <> struct Pair<double> { using type = double2; };
template <> struct Pair<float> { using type = float2; };

template <int D, int N, class T> struct PoissonShape {
    using L = MfmaLayout<D, N>;
    static constexpr int NF = D + 1, C = D + 1, NS = D * (D + 1) / 2;
    // FP32 rows padded to twice an odd number of words (distinct banks for the 16 rows of a half wave)
    static constexpr int NbfP = sizeof(T) == 4 ? (L::Nbf + 1) / 4 * 4 + 2 : L::Nbf;
    static constexpr int nT = NF * C * L::nq * NbfP, nV = D * L::Nq * NbfP;
    static constexpr int waves(int table) { // as many as fit one CU's LDS, at most 8 (two a SIMD)
        const int fit = (160 * 1024 / int(sizeof(T)) - table - 64) / (16 * NbfP);
        return fit > 8 ? 8 : fit;
    }
    static constexpr int WE = waves(nT + nV) >= 4 ? 4 : waves(nT + nV), WT = 4;
    static_assert(WE >= 1 && waves(nT) >= WT, "the tables and a wave fit the CU");
};

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T, int Nbf, int NbfP>
__device__ __forceinline__ void load_table(T* s, T const* g, int rows, int tid, int threads) {
    for (int i = tid; i < rows * Nbf; i += threads) s[(i / Nbf) * NbfP + i % Nbf] = g[i];
}

// The wave's 16 element vectors in LDS (zero past the last element).
template <class T, int Nbf, int NbfP>
__device__ __forceinline__ void stage(T* X, T const* xw, int n, int lane) {
    constexpr int NX = (16 * Nbf + 63) / 64;
    T v[NX];
#pragma unroll
    for (int o = 0; o < NX; ++o) v[o] = 64 * o + lane < n ? xw[64 * o + lane] : T(0);
#pragma unroll
    for (int o = 0; o < NX; ++o) {
        const int i = 64 * o + lane;
        if (i < 16 * Nbf) X[(i / Nbf) * NbfP + i % Nbf] = v[o];
    }
}

template <int D, int N, class T>
__global__ __launch_bounds__((64 * PoissonShape<D, N, T>::WT)) void poisson_trace_kernel(
    PoissonArgs<T> a, T const* __restrict__ xs, T* __restrict__ TR, int64_t ld, int64_t ldT) {
    using S = PoissonShape<D, N, T>;
    using L = MfmaLayout<D, N>;
    using acc = typename Mma<T>::acc;
    using T2 = typename Pair<T>::type;
    constexpr int Nbf = L::Nbf, NbfP = S::NbfP, nq = L::nq, NF = S::NF, C = S::C, KS = L::KS, FT = L::FT, W = S::WT;
    __shared__ T sT[S::nT];
    __shared__ T sX[W][16 * NbfP];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int64_t grp = int64_t(blockIdx.x) * W + wv, e0 = grp * 16;
    const int nel = e0 < a.num_elements ? int(min(int64_t(16), a.num_elements - e0)) : 0;
    T const* __restrict__ x = xs + int64_t(blockIdx.y) * ld;
    load_table<T, Nbf, NbfP>(sT, a.F, NF * C * nq, tid, 64 * W);
    stage<T, Nbf, NbfP>(sX[wv], x + (nel ? e0 : 0) * Nbf, nel * Nbf, lane);
    __syncthreads();
    if (nel == 0) return; // no barrier below
    T b[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const T v = sX[wv][j * NbfP + min(4 * s + g, Nbf - 1)];
        b[s] = 4 * s + g < Nbf ? v : T(0);
    }
    // A row j of tile t: facet point 4 t + mfma_group(j), channel mfma_reg(j); lane (j, g) then holds the
    // channels of point 4 t + g of element j
    const int tq = mfma_group<T>(j), tc = min(mfma_reg<T>(j), D);
    T2* __restrict__ out = reinterpret_cast<T2*>(TR + int64_t(blockIdx.y) * ldT) + (e0 + j) * NF * nq;
#pragma unroll 1
    for (int f = 0; f < NF; ++f) {
        T const* const pk = a.PK + (grp * NF + f) * nq * C * 16 + j;
#pragma unroll
        for (int t = 0; t < FT; ++t) {
            const int q = 4 * t + g, qc = min(q, nq - 1);
            T kn[D];
#pragma unroll
            for (int e = 0; e < D; ++e) kn[e] = pk[(qc * C + e) * 16];
            acc c = acc{0, 0, 0, 0};
            T const* const row = sT + ((f * C + tc) * nq + min(4 * t + tq, nq - 1)) * NbfP;
#pragma unroll
            for (int s = 0; s < KS; ++s) c = Mma<T>::mma(row[min(4 * s + g, Nbf - 1)], b[s], c);
            T sn = T(0);
#pragma unroll
            for (int e = 0; e < D; ++e) sn += kn[e] * c[1 + e];
            if (j < nel && q < nq) {
                T2 v;
                v.x = c[0];
                v.y = sn;
                out[f * nq + q] = v;
            }
        }
    }
}

template <int D, int N, class T>
__global__ __launch_bounds__((64 * PoissonShape<D, N, T>::WE)) void poisson_element_kernel(
    PoissonArgs<T> a, T const* __restrict__ xs, T const* __restrict__ TR, T* __restrict__ ys, int64_t ld, int64_t ldT) {
    using S = PoissonShape<D, N, T>;
    using L = MfmaLayout<D, N>;
    using acc = typename Mma<T>::acc;
    using T2 = typename Pair<T>::type;
    constexpr int Nbf = L::Nbf, NbfP = S::NbfP, Nq = L::Nq, nq = L::nq, NF = S::NF, C = S::C, NS = S::NS;
    constexpr int KS = L::KS, QB = L::QB, MT = L::MT, FT = L::FT, W = S::WE;
    __shared__ T sT[S::nT];
    __shared__ T sV[S::nV];
    __shared__ T sw[nq];
    __shared__ T sX[W][16 * NbfP];
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int64_t grp = int64_t(blockIdx.x) * W + wv, e0 = grp * 16;
    const int nel = e0 < a.num_elements ? int(min(int64_t(16), a.num_elements - e0)) : 0;
    T const* __restrict__ x = xs + int64_t(blockIdx.y) * ld;
    load_table<T, Nbf, NbfP>(sT, a.F, NF * C * nq, tid, 64 * W);
    load_table<T, Nbf, NbfP>(sV, a.V, D * Nq, tid, 64 * W);
    if (tid < nq) sw[tid] = a.w[tid];
    T* const X = sX[wv];
    stage<T, Nbf, NbfP>(X, x + (nel ? e0 : 0) * Nbf, nel * Nbf, lane);
    __syncthreads();
    if (nel == 0) return; // no workgroup barrier below
    T b[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const T v = X[j * NbfP + min(4 * s + g, Nbf - 1)];
        b[s] = 4 * s + g < Nbf ? v : T(0);
    }
    acc Y[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) Y[m] = acc{0, 0, 0, 0};

    // ---- volume
#pragma unroll 1
    for (int blk = 0; blk < QB; ++blk) {
        T s2[4][NS];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int q = min(16 * blk + mfma_row<T>(g, i), Nq - 1);
#pragma unroll
            for (int c = 0; c < NS; ++c) s2[i][c] = a.PV[((grp * Nq + q) * NS + c) * 16 + j];
        }
        acc c[D];
#pragma unroll
        for (int e = 0; e < D; ++e) c[e] = acc{0, 0, 0, 0};
        const int qa = min(16 * blk + j, Nq - 1) * NbfP;
#pragma unroll
        for (int s = 0; s < KS; ++s)
#pragma unroll
            for (int e = 0; e < D; ++e) c[e] = Mma<T>::mma(sV[e * Nq * NbfP + qa + min(4 * s + g, Nbf - 1)], b[s], c[e]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (16 * blk + mfma_row<T>(0, i) >= Nq) continue; // all four lane groups past the last point
            const int q = 16 * blk + mfma_row<T>(g, i), qr = min(q, Nq - 1) * NbfP;
#pragma unroll
            for (int e = 0; e < D; ++e) {
                T v = T(0); // S is stored by rows of its upper triangle
#pragma unroll
                for (int e2 = 0; e2 < D; ++e2) {
                    const int r = e < e2 ? e : e2, cc = e < e2 ? e2 : e;
                    v += s2[i][r * D - r * (r - 1) / 2 + cc - r] * c[e2][i];
                }
                v = q < Nq ? v : T(0);
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    Y[m] = Mma<T>::mma(sV[e * Nq * NbfP + qr + min(16 * m + j, Nbf - 1)], v, Y[m]);
            }
        }
    }

    // ---- faces
    T2 const* __restrict__ tr = reinterpret_cast<T2 const*>(TR + int64_t(blockIdx.y) * ldT);
#pragma unroll 1
    for (int f = 0; f < NF; ++f) {
        const int2 info = a.PF[(grp * NF + f) * 16 + j]; // {neighbour, its face | kind << 4}; kind 0 in padding
        const int kind = info.y >> 4;
        const int64_t own = (min(e0 + j, a.num_elements - 1) * NF + f) * nq;
        const int64_t nb = kind == 1 ? (int64_t(info.x) * NF + (info.y & 15)) * nq : own;
        T const* const pk = a.PK + (grp * NF + f) * nq * C * 16 + j;
#pragma unroll
        for (int t = 0; t < FT; ++t) {
            const int q = 4 * t + g, qc = min(q, nq - 1);
            const T2 o = tr[own + qc], n = tr[nb + qc];
            T kn[D];
#pragma unroll
            for (int e = 0; e < D; ++e) kn[e] = pk[(qc * C + e) * 16];
            const T p = pk[(qc * C + D) * 16];
            const bool act = kind != 0 && q < nq;
            const T w = act ? sw[qc] : T(0);
            const T sg = kind == 1 ? T(0.5) * (o.y - n.y) - p * (o.x - n.x) : o.y - p * o.x;
            const T d = kind == 1 ? T(0.5) * (n.x - o.x) : -o.x;
            T Wt[C];
            Wt[0] = act ? -w * sg : T(0);
#pragma unroll
            for (int e = 0; e < D; ++e) Wt[1 + e] = act ? w * d * kn[e] : T(0);
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int m = 0; m < MT; ++m)
                    Y[m] = Mma<T>::mma(sT[((f * C + c) * nq + qc) * NbfP + min(16 * m + j, Nbf - 1)], Wt[c], Y[m]);
        }
    }
    wave_sync(); // every read of the staged vectors is complete
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int k = 16 * m + mfma_row<T>(g, i);
            if (k < Nbf) X[j * NbfP + k] = Y[m][i];
        }
    wave_sync();
    T* const y = ys + int64_t(blockIdx.y) * ld + e0 * Nbf;
    for (int i = lane; i < nel * Nbf; i += 64) y[i] = X[(i / Nbf) * NbfP + i % Nbf];
}

template <int D, int N, class T>
hipError_t run(PoissonArgs<T> const& a, T const* x, T* y, T* TR, int ncols, int64_t ld, int64_t ldT, hipStream_t s) {
    using S = PoissonShape<D, N, T>;
    const int64_t groups = (a.num_elements + 15) / 16;
    if (groups > int64_t(INT_MAX) || ncols > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL((poisson_trace_kernel<D, N, T>), dim3(unsigned((groups + S::WT - 1) / S::WT), unsigned(ncols)),
                       dim3(64 * S::WT), 0, s, a, x, TR, ld, ldT);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((poisson_element_kernel<D, N, T>), dim3(unsigned((groups + S::WE - 1) / S::WE), unsigned(ncols)),
                       dim3(64 * S::WE), 0, s, a, x, static_cast<T const*>(TR), y, ld, ldT);
    return hipGetLastError();
}

} // namespace

template <class T>
hipError_t launch_poisson_mfma(int dim, int degree, PoissonArgs<T> const& a, T const* x, T* y, T* TR, int ncols,
                               int64_t ld, int64_t ldT, hipStream_t s) {
    if (dim == 3) {
        switch (degree) {
        case 1: return run<3, 1, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 2: return run<3, 2, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 3: return run<3, 3, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 4: return run<3, 4, T>(a, x, y, TR, ncols, ld, ldT, s);
        }
    } else if (dim == 2) {
        switch (degree) {
        case 1: return run<2, 1, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 2: return run<2, 2, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 3: return run<2, 3, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 4: return run<2, 4, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 5: return run<2, 5, T>(a, x, y, TR, ncols, ld, ldT, s);
        case 6: return run<2, 6, T>(a, x, y, TR, ncols, ld, ldT, s);
        }
    }
    return hipErrorInvalidValue;
}

template hipError_t launch_poisson_mfma<double>(int, int, PoissonArgs<double> const&, double const*, double*, double*,
                                                int, int64_t, int64_t, hipStream_t);
template hipError_t launch_poisson_mfma<float>(int, int, PoissonArgs<float> const&, float const*, float*, float*, int,
                                               int64_t, int64_t, hipStream_t);

} // namespace tdg
