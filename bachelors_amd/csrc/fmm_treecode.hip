// Treecode evaluation of the source tree's multipole expansions (M2P): the reference's
// single-point MultipoleSolver::calcA / calcB(current, point) (multipole_solver.cpp:686-700 ->
// QuadratureOctreeNode::calcA / calcRot, quadrature_octree.cpp:171-258), and the same recursion
// started at the nodes of a target leaf's close list, which is how the reference's calcA / calcB
// (current) evaluate the close list (fast_multipole_solver.cpp:195-231).
//
// From a start node: a non-empty node whose box passes 4 R^2 < d^2 (R = |half sizes|, d = the
// distance from its centre) adds the M2P of its multipole expansion; a node that fails opens its
// 8 children; a leaf that fails adds nothing (the reference has no particle sum there).  The walk
// is stackless: the 8 children of a node are consecutive ids, so after a node the next one is
// its next sibling, or the next sibling of the nearest ancestor that has one.
//
// M2P: A_c(x) = sum_{l <= p, m} M_c(l, m) I_l^m(x - c) with the reference's real irregular
// harmonics I(l, 0) = (-1)^l Psi_l^0, I(l, +-m) = (-1)^l sqrt2 {Re, Im} Psi_l^m, where
// Psi_l^m = (l - m)! P_l^m(cos) e^{i m phi} / r^{l+1} follows the Cartesian recurrences
//   Psi_0^0 = 1/r, Psi_m^m = (2m - 1) (x + iy) Psi_{m-1}^{m-1} / r^2,
//   Psi_l^m = ((2l - 1) z Psi_{l-1}^m - ((l-1)^2 - m^2) Psi_{l-2}^m) / r^2.
// B = curl A from the exact gradient (no finite differences):
//   dz Psi_l^m = -Psi_{l+1}^m, (dx + i dy) Psi_l^m = -Psi_{l+1}^{m+1}, (dx - i dy) Psi_l^m = Psi_{l+1}^{m-1}
// with Psi_l^{-m} = (-1)^m conj(Psi_l^m).  With A_c = Re sum_{m >= 0} alpha_c(l, m) Psi_l^m, every
// Psi_n^k of degree <= p + 1 is used once, by the alpha of the terms it serves.  The multipoles
// are stored scaled (M_true = sigma^l M), so A = M2P(u) / sigma and grad A = grad_u / sigma^2 with
// u = (x - c) / sigma.  Everything runs in FP64.
#include "fmm_treecode.hpp"
#include "fmm_prims.hpp"

namespace fmm {

constexpr double SQRT2_T = 1.41421356237309504880;

// alpha_c(l, m) = (-1)^l M_c(l, 0) (m = 0), (-1)^l sqrt2 (M_c(l, m) - i M_c(l, -m)) (m > 0)
template <class T>
__device__ __forceinline__ void alpha_at(const T* __restrict__ Mn, int Lp, int c, int l, int m, double& ar,
                                         double& ai) {
    const T* Mc = Mn + c * Lp;
    const double s = (l & 1) ? -1.0 : 1.0;
    const int k = l * l + l;
    if (m == 0) {
        ar = s * (double)Mc[k];
        ai = 0.0;
    } else {
        ar = s * SQRT2_T * (double)Mc[k + m];
        ai = -s * SQRT2_T * (double)Mc[k - m];
    }
}

struct TreeView {
    const double* center;
    const int* first_child;
    const int* parent;
    const int* npts;
    const int* level;
    ScaleTable sig;
    double radius[MAX_LEVELS];
};

// A workgroup serves 64 points: lane i of each of its 4 waves holds point i, and the waves share the
// columns k of every expansion.  The walk is the workgroup's: it opens a node if any of its points does,
// and a point that has accepted (or dropped) a node is idle until the walk leaves that node's subtree, so
// every point meets its nodes in the order of a walk of its own.  A node some point accepts has its 12
// coefficients per Psi_n^k made once in LDS (a column index is the same for all lanes, so the reads are
// broadcasts).  Bound by the FP64 chains of the columns at 4 waves per SIMD; with a thread per point, each on
// a node of its own, 24 gathered loads and 9 gradient sums per Psi, one wave per SIMD was all there was:
// 65,536 points around a coil of 38,400 (p = 10) 3.90 -> 0.27 ms (0.22 the walk, 0.05 the sort of the points).
//
//   A_c = Re(alpha_c(n, k) Psi), and B = curl A from the alphas of degree l = n - 1,
//   with p = alpha(l, k + 1), q = alpha(l, k - 1) (doubled for k = 1, which also serves m = 0's
//   Psi^{-1}), u = (p - q) / 2, w = (p + q) / 2:
//   dz A = -Re(alpha(l, k) Psi), dx A = Re(u Psi), dy A = -Im(w Psi).
constexpr int TC_WAVES = 4;

template <class T>
__device__ __forceinline__ void node_coefficients(const T* __restrict__ Mn, int p, int Lp, double (*co)[12]) {
    const int nt = (p + 2) * (p + 3) / 2;
    for (int e = threadIdx.x; e < nt; e += 64 * TC_WAVES) {
        int n = (int)((sqrtf(8.0f * e + 1.0f) - 1.0f) * 0.5f);
        while ((n + 1) * (n + 2) / 2 <= e) n++;
        while (n * (n + 1) / 2 > e) n--;
        const int k = e - n * (n + 1) / 2, l = n - 1;
        double al[3][2] = {{0, 0}, {0, 0}, {0, 0}}, z[3][2] = {{0, 0}, {0, 0}, {0, 0}}, u[3][2], w[3][2];
        for (int c = 0; c < 3; c++) {
            double pr = 0, pi = 0, qr = 0, qi = 0;
            if (n <= p) alpha_at(Mn, Lp, c, n, k, al[c][0], al[c][1]);
            if (k <= l) alpha_at(Mn, Lp, c, l, k, z[c][0], z[c][1]);
            if (k + 1 <= l) alpha_at(Mn, Lp, c, l, k + 1, pr, pi);
            if (k >= 1) alpha_at(Mn, Lp, c, l, k - 1, qr, qi);
            if (k == 1) qr *= 2.0;
            u[c][0] = 0.5 * (pr - qr); u[c][1] = 0.5 * (pi - qi);
            w[c][0] = 0.5 * (pr + qr); w[c][1] = 0.5 * (pi + qi);
        }
        double* o = co[e];
        for (int c = 0; c < 3; c++) { o[2 * c] = al[c][0]; o[2 * c + 1] = -al[c][1]; }
        o[6] = z[1][0] - w[2][1];    o[7] = -z[1][1] - w[2][0];     // B_x = dy A_z - dz A_y
        o[8] = -z[0][0] - u[2][0];   o[9] = z[0][1] + u[2][1];      // B_y = dz A_x - dx A_z
        o[10] = u[1][0] + w[0][1];   o[11] = -u[1][1] + w[0][0];    // B_z = dx A_y - dy A_x
    }
}

// this wave's columns of one node's expansion at the scaled offset u, added to acc (A 0-2, B 3-5) with
// the scales of A and of its gradient
__device__ __forceinline__ void m2p_columns(const double (*co)[12], int p, int wave, double ux, double uy, double uz,
                                            double sA, double sB, double acc[6]) {
    const double r2 = ux * ux + uy * uy + uz * uz, ir2 = 1.0 / r2;
    double dr = sqrt(ir2), di = 0.0, a[6] = {0, 0, 0, 0, 0, 0};   // (dr, di) = Psi_k^k
    int kd = 0;
    for (int i = 0; 4 * i <= p + 1; i++) {
        const int k = 4 * i + (i & 1 ? 3 - wave : wave);   // the columns' lengths p + 2 - k even out
        if (k > p + 1) continue;
        for (; kd < k;) {
            kd++;
            const double f = (2.0 * kd - 1) * ir2;
            const double nr = (dr * ux - di * uy) * f, ni = (dr * uy + di * ux) * f;
            dr = nr;
            di = ni;
        }
        double vr = dr, vi = di, p2r = 0.0, p2i = 0.0;
        for (int n = k;;) {
            const double* o = co[n * (n + 1) / 2 + k];
#pragma unroll
            for (int e = 0; e < 6; e++)
                a[e] = __builtin_fma(o[2 * e], vr, __builtin_fma(o[2 * e + 1], vi, a[e]));
            if (++n > p + 1) break;
            const double f = (2.0 * n - 1) * uz, b = (double)((n - 1) * (n - 1) - k * k);
            const double nr = __builtin_fma(f, vr, -b * p2r) * ir2, ni = __builtin_fma(f, vi, -b * p2i) * ir2;
            p2r = vr; p2i = vi; vr = nr; vi = ni;
        }
    }
    for (int e = 0; e < 6; e++) acc[e] = __builtin_fma(a[e], e < 3 ? sA : sB, acc[e]);
}

// the treecode walk from node start for the workgroup's points (valid: this lane has one)
template <class T>
__device__ __forceinline__ void walk(const TreeView& S, const T* __restrict__ M, int p, int Lp, int start, bool valid,
                                     double x, double y, double z, double (*co)[12], double acc[6]) {
    const int wave = threadIdx.x >> 6;
    int idle = valid ? -1 : -2;   // the node whose subtree this lane waits out, -1: none
    int n = start;                // uniform over the workgroup
    for (;;) {
        bool open = false;
        const int fc = S.first_child[n];
        if (fc >= 0 || S.npts[n] > 0) {
            const double cx = S.center[3 * n], cy = S.center[3 * n + 1], cz = S.center[3 * n + 2];
            // Vector3::distanceSquared and 4 radius^2 < d^2 (quadrature_octree.cpp:177-181)
            const double dx = x - cx, dy = y - cy, dz = z - cz;
            const double d2 = dx * dx + dy * dy + dz * dz;
            const int lv = S.level[n];
            const double rad = S.radius[lv];
            const bool accept = idle == -1 && 4 * rad * rad < d2;
            open = idle == -1 && !accept && fc >= 0;
            if (__any(accept)) {   // the same in all waves: they hold the same points
                __syncthreads();   // the previous node's coefficients are no longer read
                node_coefficients(M + (size_t)n * 3 * Lp, p, Lp, co);
                __syncthreads();
                if (accept) {
                    const double inv = 1.0 / S.sig.s[lv];
                    m2p_columns(co, p, wave, dx * inv, dy * inv, dz * inv, inv, inv * inv, acc);
                }
            }
            if (idle == -1 && !open) idle = n;
        }
        if (__any(open)) {
            n = fc;
            continue;
        }
        // leave n, and its ancestors whose last child it is
        for (;;) {
            if (idle == n) idle = -1;
            if (n == start) return;
            const int par = S.parent[n];
            if (n - S.first_child[par] < 7) break;
            n = par;
        }
        n++;
    }
}

// sums the waves' shares: wave 0 gets the point's A (0-2) and B (3-5)
__device__ __forceinline__ void sum_waves(double acc[6], double (*red)[6][64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (wave)
        for (int e = 0; e < 6; e++) red[wave - 1][e][lane] = acc[e];
    __syncthreads();
    if (wave == 0)
        for (int w = 0; w < TC_WAVES - 1; w++)
            for (int e = 0; e < 6; e++) acc[e] += red[w][e][lane];
}

// order[i] (may be null: i): the point served in place i; neighbouring places hold neighbouring points
template <class T>
__global__ __launch_bounds__(64 * TC_WAVES) void k_treecode_points(TreeView S, const T* __restrict__ M, int p, int Lp,
                                                                   const double* __restrict__ x,
                                                                   const int* __restrict__ order, int n,
                                                                   double scaleB, double scaleA,
                                                                   double* __restrict__ B, double* __restrict__ A) {
    extern __shared__ double sh[];
    __shared__ double red[TC_WAVES - 1][6][64];
    const int place = blockIdx.x * 64 + (threadIdx.x & 63);
    const bool valid = place < n;
    const int i = !valid ? 0 : order ? order[place] : place;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    walk(S, M, p, Lp, 0, valid, x[3 * (size_t)i], x[3 * (size_t)i + 1], x[3 * (size_t)i + 2], (double(*)[12])sh, acc);
    sum_waves(acc, red);
    if (threadIdx.x >= 64 || !valid) return;
    for (int c = 0; c < 3; c++) {
        if (B) B[3 * (size_t)i + c] = acc[3 + c] * scaleB;
        if (A) A[3 * (size_t)i + c] = acc[c] * scaleA;
    }
}

// one workgroup per useful target leaf: the walk from every node of the leaf's close list
// (slot-order targets and outputs, unscaled)
template <class T>
__global__ __launch_bounds__(64 * TC_WAVES) void k_m2p_close(TreeView S, const T* __restrict__ M, int p, int Lp,
                                                             const int* __restrict__ leaves,
                                                             const int* __restrict__ tbegin,
                                                             const int* __restrict__ tend,
                                                             const int* __restrict__ close_begin,
                                                             const int* __restrict__ close_end,
                                                             const int* __restrict__ close_s,
                                                             const double* __restrict__ txyz,
                                                             double* __restrict__ Bnear, double* __restrict__ Anear) {
    extern __shared__ double sh[];
    __shared__ double red[TC_WAVES - 1][6][64];
    const int leaf = leaves[blockIdx.x];
    for (int k0 = tbegin[leaf]; k0 < tend[leaf]; k0 += 64) {
        const int k = k0 + (threadIdx.x & 63);
        const bool valid = k < tend[leaf];
        const size_t q = valid ? k : k0;
        double acc[6] = {0, 0, 0, 0, 0, 0};
        for (int ci = close_begin[leaf]; ci < close_end[leaf]; ci++)
            walk(S, M, p, Lp, close_s[ci], valid, txyz[3 * q], txyz[3 * q + 1], txyz[3 * q + 2], (double(*)[12])sh, acc);
        sum_waves(acc, red);
        if (threadIdx.x < 64 && valid)
            for (int c = 0; c < 3; c++) {
                if (Bnear) Bnear[3 * q + c] = acc[3 + c];
                if (Anear) Anear[3 * q + c] = acc[c];
            }
    }
}

// sort key of a point: the interleaved top 10 bits of its position in a box of 8 half sizes around the
// source root's centre (clamped: points further out accept the root or its children alike)
__global__ void k_point_keys(const double* __restrict__ x, int n, double cx, double cy, double cz, double hx,
                             double hy, double hz, uint32_t* __restrict__ key, int* __restrict__ val) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double c[3] = {cx, cy, cz}, h[3] = {hx, hy, hz};
    uint32_t k = 0;
    for (int a = 0; a < 3; a++) {
        const double u = fmin(fmax((x[3 * (size_t)i + a] - c[a]) / (8.0 * h[a]) + 0.5, 0.0), 0.9995);
        const uint32_t v = (uint32_t)(u * 1024.0);
        for (int b = 0; b < 10; b++) k |= ((v >> b) & 1u) << (3 * b + a);
    }
    key[i] = k;
    val[i] = i;
}

static TreeView view_of(const TreeDev& S, const ScaleTable& sig) {
    TreeView v;
    v.center = S.center.as<double>();
    v.first_child = S.first_child.as<int>();
    v.parent = S.parent.as<int>();
    v.npts = S.npts.as<int>();
    v.level = S.level.as<int>();
    v.sig = sig;
    for (int k = 0; k < MAX_LEVELS; k++) v.radius[k] = S.radius[k];
    return v;
}

void launch_treecode_points(bool f64, const TreeDev& S, const ScaleTable& sig, const void* M, int p, int Lp,
                            const double root_c[3], const double* x, int n, double scaleB, double scaleA, double* B,
                            double* A, TreecodeScratch& W, hipStream_t st) {
    if (n <= 0 || S.num_nodes <= 0) return;
    const TreeView v = view_of(S, sig);
    // points of one workgroup should meet the same nodes; a few workgroups gain less than the sort costs
    const int* order = nullptr;
    if (n > 1024) {
        uint32_t *k0 = W.key.get<uint32_t>(n), *k1 = W.key2.get<uint32_t>(n);
        int *v0 = W.val.get<int>(n), *v1 = W.order.get<int>(n);
        k_point_keys<<<blocks(n), 256, 0, st>>>(x, n, root_c[0], root_c[1], root_c[2], S.half[0][0], S.half[0][1],
                                                S.half[0][2], k0, v0);
        sort_pairs_u32(k0, k1, v0, v1, n, 30, W.tmp, st);
        order = v1;
    }
    const size_t lds = (size_t)(p + 2) * (p + 3) / 2 * 12 * sizeof(double);
    if (f64)
        k_treecode_points<double><<<blocks(n, 64), 64 * TC_WAVES, lds, st>>>(v, (const double*)M, p, Lp, x, order, n,
                                                                             scaleB, scaleA, B, A);
    else
        k_treecode_points<float><<<blocks(n, 64), 64 * TC_WAVES, lds, st>>>(v, (const float*)M, p, Lp, x, order, n,
                                                                            scaleB, scaleA, B, A);
    FMM_HIP(hipGetLastError());
}

void launch_m2p_close(bool f64, const TreeDev& S, const ScaleTable& sig, const void* M, int p, int Lp,
                      const int* leaves, int nleaves, const TreeDev& T, const int* close_begin, const int* close_end,
                      const int* close_s, const double* txyz, double* Bnear, double* Anear, hipStream_t st) {
    if (nleaves <= 0) return;
    const TreeView v = view_of(S, sig);
    const size_t lds = (size_t)(p + 2) * (p + 3) / 2 * 12 * sizeof(double);
    if (f64)
        k_m2p_close<double><<<nleaves, 64 * TC_WAVES, lds, st>>>(v, (const double*)M, p, Lp, leaves, T.begin.as<int>(),
                                                    T.end.as<int>(), close_begin, close_end, close_s, txyz, Bnear,
                                                    Anear);
    else
        k_m2p_close<float><<<nleaves, 64 * TC_WAVES, lds, st>>>(v, (const float*)M, p, Lp, leaves, T.begin.as<int>(),
                                                   T.end.as<int>(), close_begin, close_end, close_s, txyz, Bnear,
                                                   Anear);
    FMM_HIP(hipGetLastError());
}

}  // namespace fmm
