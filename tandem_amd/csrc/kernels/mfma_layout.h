// Tile geometry and device arguments of the MFMA elasticity apply (shared by host and device).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace tdg {

// Runtime tile sizes of the MFMA layout for (D, N) with Nbf basis functions, Nq volume and nq facet
// points:
//   KS = ceil(Nbf / 4)   K-steps over the basis,         MT = ceil(Nbf / 16) basis tiles,
//   QB = ceil(Nq / 16)   16-point volume blocks,          FT = ceil(nq / 4)   4-point facet tiles,
//   KF = ceil(nf / 4)     K-steps over the nf nodes of one face (the first nf labels of the face frame),
//   NCH = D*D + 2        volume channels (JInv, lamWJ, muWJ),
//   NFC = 2 D*D + 4 + D  facet channels (own G', lam, mu, neighbour G', lam, mu, oriented normal).
struct MfmaDims {
    int D, Nbf, Nq, nq, KS, QB, MT, FT, NCH, NFC;
    __host__ __device__ constexpr MfmaDims(int D_, int Nbf_, int Nq_, int nq_)
        : D(D_), Nbf(Nbf_), Nq(Nq_), nq(nq_), KS((Nbf_ + 3) / 4), QB((Nq_ + 15) / 16), MT((Nbf_ + 15) / 16),
          FT((nq_ + 3) / 4), NCH(D_ * D_ + 2), NFC(2 * D_ * D_ + 4 + D_) {}
};

namespace detail {
constexpr int binom(int n, int k) { return k == 0 ? 1 : binom(n - 1, k - 1) * n / k; }
constexpr int vol_points(int D, int N) {
    return D == 2 ? (N == 1 ? 4 : N == 2 ? 7 : N == 3 ? 15 : N == 4 ? 19 : N == 5 ? 28 : 37)
                  : (N == 1 ? 6 : N == 2 ? 14 : N == 3 ? 31 : 57);
}
constexpr int fct_points(int D, int N) { return D == 2 ? N + 1 : (N == 1 ? 4 : N == 2 ? 7 : N == 3 ? 15 : 19); }
} // namespace detail

template <int D_, int N_> struct MfmaLayout {
    static constexpr int Nbf = detail::binom(N_ + D_, D_);
    static constexpr int Nq = detail::vol_points(D_, N_);
    static constexpr int nq = detail::fct_points(D_, N_);
    static constexpr MfmaDims dims{D_, Nbf, Nq, nq};
    static constexpr int KS = dims.KS, QB = dims.QB, MT = dims.MT, FT = dims.FT, NCH = dims.NCH, NFC = dims.NFC;
    // Face frame: the basis functions of the nodes off the face vanish on it, so values and tangential
    // derivatives there involve only the face's own nf nodes (15 of 35 at 3D P4); the normal
    // derivative involves all.  The face frame numbers the face's nodes first.
    static constexpr int nf = detail::binom(N_ + D_ - 1, D_ - 1);
    static constexpr int KF = (nf + 3) / 4;
    static_assert(nf <= 16, "the face's nodes fit one 16-row tile");
};

// Output row of a 16x16x4 MFMA tile held in register i (0..3) of lane group g = lane / 16:
// consecutive rows for the f32 instruction, rows g, g+4, g+8, g+12 for the f64 instruction.
template <class T> __host__ __device__ constexpr int mfma_row(int g, int i) {
    return sizeof(T) == 8 ? g + 4 * i : 4 * g + i;
}
// Inverse: (lane group, register) of tile row rho.
template <class T> __host__ __device__ constexpr int mfma_group(int rho) { return sizeof(T) == 8 ? rho % 4 : rho / 4; }
template <class T> __host__ __device__ constexpr int mfma_reg(int rho) { return sizeof(T) == 8 ? rho / 4 : rho % 4; }

bool mfma_supported(int dim, int degree);

// Arguments of the MFMA kernel: canonical tables (copied to LDS by every block) and the
// element-grouped point data.
template <class T> struct MfmaArgs {
    T const* V;          // [e][q][k]  d phi_k / d xi_e at volume point q
    T const* T0;         // [c][q][k]  face-0 value (c = 0) and d/dxi_(c-1) at facet point q, k a face-frame
                         // label (the face's own nodes first)
    int32_t const* perm; // [2][f][k]  face-frame label -> element node of face f, then its inverse
    T const* w;          // facet weights
    T const* VD;         // [group][q][NCH][16]
    T const* FD;         // [group][f][q][NFC][16]  both sides' G', lam, mu and the oriented normal
                         // (stored per element side: every load is a contiguous 16-element row)
    T const* FP;         // [group][f][16]
    int4 const* FI;      // [group][f][16]
    int64_t num_elements, num_groups;
    int xcd_remap;       // 1: each XCD takes one contiguous range of element groups
};

template <class T>
hipError_t launch_elasticity_mfma(int dim, int degree, MfmaArgs<T> const& a, T const* x, T* y, int ncols,
                                 int64_t ld, hipStream_t stream);

// Arguments of the two-kernel (facet + element) MFMA elasticity apply.  Facets are the ones that
// carry a term (two-sided first, then one-sided), in groups of 8 with the facet innermost:
//   FR    [fgroup][q][NFR][8]   NFR = D*D + D + 4: the tangent columns t_1 .. t_(D-1) of the facet
//                               Jacobian M = J J_f of side 0 (shared by both sides), the third
//                               column c_0 of side 0 and c_1 of side 1, lam_0, mu_0, lam_1, mu_1
//   FPen  [fgroup][8]           penalty
//   FInfo [fgroup][8]           {element 0, element 1, face 0 | face 1 << 4 | kind << 8, 0}
//                               (kind 1 two-sided, 2 one-sided, 0 padding)
// The element kernel reads the volume table V and point data VD of MfmaArgs, and the lifted facet
// contributions L[element][face][Nbf * D].
template <class T> struct SplitArgs {
    T const* V;
    T const* T0;
    int32_t const* perm; // [f][k] face-frame label -> element node
    T const* w;
    T const* VD;
    T const* FR;
    T const* FPen;
    int4 const* FInfo;
    int64_t num_elements, num_groups, num_facets, num_fgroups, num_two;
    int xcd_remap; // workgroup order: 0 linear; 1 one contiguous range of groups per XCD (one column);
                   // 2 as 1, persistent (the resident workgroups loop over the blocks)
    int cpw;       // several columns: columns a workgroup takes one after another (set by the launch)
    int small;     // kSmallFacets | kSmallElements: those kernels' waves share each group
    double* dot;   // one column, optional: per element workgroup the partial sum of x . y
};

// Number of launch shapes of the two-kernel apply (waves per workgroup, occupancy targets, element
// prefetch depth, lift tail on the vector ALU or the matrix cores), per precision.
constexpr int kSplitShapes = 4;
// Small launches of the two kernels: the waves of a workgroup share each group (one block of points or
// one facet tile each) and sum in LDS, one group a workgroup up to kSmallOneGroup groups x columns, then
// two.  us per apply, launch shapes -> elements small -> both small, by groups of 16 elements (facet
// groups of 8: about 4.3 times as many in 3D, 3 in 2D):
//   3D P4 FP64  24: 70, 29, 24   81: 72, 30, 28   192: 75, 36, 44   375: 83, 48, 74   1029: 113, 110, 172
//         FP32  24: 35, 23, 18   81: 35, 23, 21   192: 37, 25, 31   375: 44, 35, 54   1029: 75, 68, 116
//   3D P3 FP64  24: 35, 21, 17   192: 38, 24, 26   648: 53, 42, 54   1029: 65, 63, 79
//   2D P6 FP64  72: 28, 15, 13   288: 28, 18, 19   512: 33, 24, 27   1152: 43, 47, 53
//         FP32  72: 15, 12, 11   288: 16, 13, 14   512: 18, 16, 17   1152: 29, 29, 31
//   16 columns  3D P4 24: FP64 86, 51, 74  FP32 46, 35, 54
// Above the limits the launch shapes win: two waves a SIMD share one table and nothing is summed across
// waves.  With one block of points (3D P2, 2D P2 and P3) the small element kernel only spreads the waves
// over more CUs: 3D P2 FP64 24: 18 -> 14, 648: 27.0 -> 26.3, 912: 28.2 -> 28.4, FP32 648: 15 -> 17.
enum { kSmallFacets = 1, kSmallElements = 2 };
constexpr int64_t kSmallOneGroup = 256, kSmallFacetGroups = 384, kSmallElementGroups = 1024;
constexpr int64_t kSmallElementGroups1 = 512; // one block of points, FP64
// facet_groups and element_groups: times columns; Nq: volume points.
constexpr int split_small(int precision_bytes, int Nq, int64_t facet_groups, int64_t element_groups) {
    return (facet_groups <= kSmallFacetGroups ? kSmallFacets : 0) |
           (element_groups <= (Nq > 16 ? kSmallElementGroups : precision_bytes == 8 ? kSmallElementGroups1 : 0)
                ? kSmallElements
                : 0);
}
// Workgroup orders (SplitArgs::xcd_remap) searched with each shape.
constexpr int kSplitOrders = 3;

// y = A x for ncols columns (stride ld) through the facet kernel (into the slot buffer L, column
// stride ldL = E (D+1) Nbf D) and the element kernel, with launch shape `shape`.  With a.dot set
// (one column), the element kernel also writes per workgroup the partial sum of x . y into
// a.dot[0 .. split_element_workgroups(shape, num_groups)).
template <class T>
hipError_t launch_elasticity_split(int dim, int degree, int shape, SplitArgs<T> const& a, T const* x, T* y, T* L,
                                   int ncols, int64_t ld, int64_t ldL, hipStream_t stream);
// Workgroups of the element kernel of launch shape `shape` for one column (a multiple of 8).
template <class T> int64_t split_element_workgroups(int shape, int small, int64_t num_groups);

// Zeroes the facet slots listed in `slots` (slot s = entries [s bs, (s + 1) bs) of L).
template <class T> hipError_t launch_zero_slots(T* L, int32_t const* slots, int64_t nslots, int bs, hipStream_t s);

// Arguments of the two-kernel matrix-core Poisson apply (element-grouped data, element innermost):
//   V  [e][q][k]                    modal basis gradients at the volume points
//   F  [f][c][q][k]                 face f's values (c = 0) and gradients at its points
//   PV [group][q][D (D + 1) / 2][16]  upper triangle of W|J| K G G^T by rows
//   PK [group][f][q][D + 1][16]     K G n (n outward, area-scaled), then penalty |n|
//   PF [group][f][16]               {neighbour, its face | kind << 4}
template <class T> struct PoissonArgs {
    T const* V;
    T const* F;
    T const* w;
    T const* PV;
    T const* PK;
    int2 const* PF;
    int64_t num_elements;
};
// y = A x for ncols columns (stride ld) through the traces TR[element][f][q] = {u, K grad u . n} (column
// stride ldT = E (D + 1) nq 2).
template <class T>
hipError_t launch_poisson_mfma(int dim, int degree, PoissonArgs<T> const& a, T const* x, T* y, T* TR, int ncols,
                               int64_t ld, int64_t ldT, hipStream_t stream);
// Unknowns x columns from which the matrix-core Poisson apply is taken.  us per apply, thread-per-point
// kernel -> this one (two launches and their tables cost 8 us in 2D, 10 to 45 in 3D whatever the size):
//   FP64  2D P2   49k 7.0 -> 8.6  120k 13.4 -> 10.6   P4  31k 6.9 -> 11.6  123k 18 -> 12   P6  57k 17 -> 17
//         3D P1   12k 7.8 -> 8.9   41k 12.9 -> 9.6    P2  31k 13.2 -> 13.3  104k 34 -> 15   P4  45k 61 -> 46
//   FP32  2D P3   82k 6.4 -> 8.5  120k (P2) 10.7 -> 9.5   3D P4  45k 33 -> 39  108k 48 -> 39
// 2D P1 stays with the thread-per-point kernel: 540k unknowns 32 -> 28 in FP64, 20 -> 23 in FP32.
constexpr int64_t poisson_mfma_unknowns(int dim, int precision_bytes) {
    return dim == 2 ? (precision_bytes == 8 ? 70000 : 120000) : (precision_bytes == 8 ? 32000 : 64000);
}

template <class T> struct GradArgs;
// Adjoint material gradient on the matrix cores (same dimensions and degrees as the apply):
// g_lam, g_mu (E x Nq) = d/d(lam_Q, mu_Q) of psi^T A u.
template <class T>
hipError_t launch_material_gradient_mfma(int dim, int degree, MfmaArgs<T> const& a, GradArgs<T> const& g,
                                         T const* u, T const* psi, T* g_lam, T* g_mu, hipStream_t stream);

} // namespace tdg
