// Particle <-> expansion kernels: source charges, P2M, L2P (curl of the local
// expansion from analytic gradients), near-field P2P, final assembly, and the FP64
// direct Biot-Savart sum (math::calcBioSavartLaplace, integration.cpp:101-120).
//
// Harmonics use the Cartesian recurrences of the complex regular solid harmonics
// Phi_l^m = r^l P_l^m(cos) e^{im phi}/(l+m)! (m >= 0); the reference's real basis is
// R(l,0) = (-1)^l Phi_l^0, R(l,m) = (-1)^l sqrt2 Re Phi_l^m, R(l,-m) = (-1)^l sqrt2 Im Phi_l^m
// (harmonics.cpp:20-56 with the sectoral term m = p included).  All recurrences run in
// FP64 on the scaled vector u = (x - c) / sigma; only P2P runs in FP32 (with FP64
// accumulation per target).
#include <algorithm>

#include "fmm_expand.hpp"
#include "fmm_gemm.hpp"
#include "fmm_recip.hpp"

namespace fmm {

__device__ __forceinline__ int lmi(int l, int m) { return l * l + l + m; }
__device__ __forceinline__ double sgnl(int l) { return (l & 1) ? -1.0 : 1.0; }
constexpr double SQRT2 = 1.41421356237309504880;

// ---------------------------------------------------------------- charges
__global__ void k_charges(const int* __restrict__ slots, int n, const double* __restrict__ xyz,
                          const double* __restrict__ w, const double* __restrict__ J, double* __restrict__ sxyz,
                          double* __restrict__ sq, double* __restrict__ sJ) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = slots[k];
    double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
    double j0, j1, j2;
    if (J) {
        j0 = J[3 * i]; j1 = J[3 * i + 1]; j2 = J[3 * i + 2];
    } else {
        // current direction perp().normalized() (vector3.cu:154-167, 201-204)
        double px = -y, py = x;
        double l = sqrt(px * px + py * py);
        j0 = l != 0 ? px / l : 0.0;
        j1 = l != 0 ? py / l : 0.0;
        j2 = 0.0;
    }
    double ww = w[i];
    sxyz[3 * k] = x; sxyz[3 * k + 1] = y; sxyz[3 * k + 2] = z;
    sq[3 * k] = ww * j0; sq[3 * k + 1] = ww * j1; sq[3 * k + 2] = ww * j2;
    if (sJ) { sJ[3 * k] = j0; sJ[3 * k + 1] = j1; sJ[3 * k + 2] = j2; }
}

__global__ void k_gather_xyz(const int* __restrict__ slots, int n, const double* __restrict__ xyz,
                             double* __restrict__ out) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = slots[k];
    out[3 * k] = xyz[3 * i]; out[3 * k + 1] = xyz[3 * i + 1]; out[3 * k + 2] = xyz[3 * i + 2];
}

// ---------------------------------------------------------------- P2M
// M_l^{+-m} = sum_j q_j R_l^{+-m}(u_j), u = (y - c) / sigma, with R(l, 0) = (-1)^l Phi_l^0 and
// R(l, +-m) = (-1)^l sqrt2 {Re, Im} Phi_l^m (harmonics.cpp:281-320).  One wave (a one-wave
// workgroup) per useful source leaf.  The leaf's tasks (point, m) -- point-major, P + 1 per point
// -- run 64 at a time; task (point, m) makes column m of the harmonics in one loop over the
// degree l = 1 .. P (P, the order, is a template parameter, so the loop unrolls with l fixed):
// for l <= m the sectoral step Phi_l^l = Phi_{l-1}^{l-1} (x + iy) / (2l), for l > m the degree
// step Phi_l^m = ((2l - 1) z Phi_{l-1}^m - r^2 Phi_{l-2}^m) / (l^2 - m^2), both as
// (A Phi_{l-1} - b Phi_{l-2}) f with a complex A = (x + iy or (2l - 1) z), b = (0 up to l = m + 1,
// then r^2) and f from an LDS table F[m][l] (1/(2l) for l <= m, 1/(l^2 - m^2) above), so every
// lane runs the same P steps whatever its m; from l = m on each value is written to the point's
// row of a small LDS ring.  After each round the points it completed are added, lane k owning
// coefficients k, k + 64, ... (ring rows padded to whole slots of 64, so the reads need no
// masks), in point order with FP64 fused multiply-adds; the degree signs and sqrt2 are applied
// once when the leaf is written.  The ring holds the points of one round and its two boundary
// points (64 / (P + 1) + 2 rows).  T is the type of the recurrences and the ring: FP64 in the
// FP64 mode, FP32 otherwise (|u| <= sqrt3 keeps every Phi_l^m in range and the recurrences
// forward-stable).
template <class T> __device__ __forceinline__ T recip_t(int n);
template <> __device__ __forceinline__ double recip_t<double>(int n) { return recip(n); }
template <> __device__ __forceinline__ float recip_t<float>(int n) { return recipf(n); }
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <int P>
constexpr int p2m_ring() { return 64 / (P + 1) + 2; }
template <int P>
constexpr int p2m_row() { return 64 * (((P + 1) * (P + 1) + 63) / 64); }

template <class T, int P>
__global__ __launch_bounds__(64) void k_p2m(const int* __restrict__ leaves, const double* __restrict__ center,
                                            const int* __restrict__ begin, const int* __restrict__ end,
                                            const int* __restrict__ level, ScaleTable sig,
                                            const double* __restrict__ sxyz, const double* __restrict__ sq, int Lp,
                                            T* __restrict__ M, const float* __restrict__ dm, int Kp,
                                            float* __restrict__ cscale, _Float16* __restrict__ hl) {
    constexpr int P1 = P + 1, L = P1 * P1, NS = (L + 63) / 64, RS = p2m_row<P>(), RING = p2m_ring<P>();
    __shared__ T ring[RING * RS];   // complex Phi of the points in flight (Re at (l, m), Im at (l, -m))
    __shared__ T F[P1 * P1];        // F[m][l]: the step factor of column m at degree l
    const int lane = threadIdx.x;
    for (int i = lane; i < P1 * P1; i += 64) {
        const int m = i / P1, l = i - m * P1;
        F[i] = l == 0 ? (T)0 : l <= m ? recip_t<T>(2 * l) : recip_t<T>(l * l - m * m);
    }
    const int leaf = leaves[blockIdx.x];
    const double cx = center[3 * leaf], cy = center[3 * leaf + 1], cz = center[3 * leaf + 2];
    const double inv = 1.0 / sig.s[level[leaf]];
    const int jb = begin[leaf], n = end[leaf] - jb, ntask = n * P1;
    double acc[NS][3];
#pragma unroll
    for (int r = 0; r < NS; r++) acc[r][0] = acc[r][1] = acc[r][2] = 0.0;
    // this lane's task: point pt, column m; a round moves it 64 tasks on
    int pt = lane / P1, m = lane - pt * P1;
    constexpr int dpt = 64 / P1, dmv = 64 - dpt * P1;
    int done = 0;
    __syncthreads();   // F is written
    for (int t0 = 0; t0 < ntask; t0 += 64) {
        if (t0 + lane < ntask) {
            const int j = jb + pt;
            const T ux = (T)((sxyz[3 * j] - cx) * inv), uy = (T)((sxyz[3 * j + 1] - cy) * inv),
                    uz = (T)((sxyz[3 * j + 2] - cz) * inv);
            const T r2 = ux * ux + uy * uy + uz * uz;
            T* row = ring + (pt % RING) * RS;
            const T* Fm = F + m * P1;
            T p1r = 1, p1i = 0, p2r = 0, p2i = 0;
            if (m == 0) row[0] = (T)1;
#pragma unroll
            for (int l = 1; l <= P; l++) {
                const bool sect = l <= m;
                const T ar = sect ? ux : (T)(2 * l - 1) * uz, ai = sect ? uy : (T)0;
                const T b = l <= m + 1 ? (T)0 : r2, f = Fm[l];
                const T vr = fma_t(ar, p1r, fma_t(-ai, p1i, -(b * p2r))) * f;
                const T vi = fma_t(ar, p1i, fma_t(ai, p1r, -(b * p2i))) * f;
                p2r = p1r; p2i = p1i; p1r = vr; p1i = vi;
                if (l >= m) {
                    row[l * l + l + m] = vr;
                    if (m > 0) row[l * l + l - m] = vi;
                }
            }
        }
        pt += dpt;
        m += dmv;
        if (m >= P1) { m -= P1; pt++; }
        __syncthreads();   // one wave: the ring rows are written before they are read
        const int complete = min(n, (t0 + 64) / P1);
        for (int q = done; q < complete; q++) {
            const T* row = ring + (q % RING) * RS + lane;
            const double q0 = sq[3 * (jb + q)], q1 = sq[3 * (jb + q) + 1], q2 = sq[3 * (jb + q) + 2];
            T v[NS];
#pragma unroll
            for (int r = 0; r < NS; r++) v[r] = row[64 * r];   // beyond L: padding, never written out
#pragma unroll
            for (int r = 0; r < NS; r++) {
                const double x = (double)v[r];
                acc[r][0] = fma_t(q0, x, acc[r][0]);
                acc[r][1] = fma_t(q1, x, acc[r][1]);
                acc[r][2] = fma_t(q2, x, acc[r][2]);
            }
        }
        done = complete;
        __syncthreads();   // the rows are read before the next round overwrites them
    }
    T* out = M + (size_t)leaf * 3 * Lp;
    T mv[NS][3];   // the leaf's multipoles as written (zero beyond L)
#pragma unroll
    for (int r = 0; r < NS; r++) {
        const int k = lane + 64 * r;
        if (k < L) {
            const int l = (int)sqrtf((float)k + 0.5f), mm = k - l * l - l;   // k = l^2 + l + mm
            const double s = ((l & 1) ? -1.0 : 1.0) * (mm == 0 ? 1.0 : SQRT2);
            for (int cc = 0; cc < 3; cc++) mv[r][cc] = (T)(acc[r][cc] * s);
        } else {
            for (int cc = 0; cc < 3; cc++) mv[r][cc] = (T)0;
        }
        if (k < Lp)
            for (int cc = 0; cc < 3; cc++) out[cc * Lp + k] = mv[r][cc];
    }
    for (int k = lane + 64 * NS; k < Lp; k += 64)   // padding beyond what the loop above covers
        for (int cc = 0; cc < 3; cc++) out[cc * Lp + k] = (T)0;
    if constexpr (sizeof(T) == 4) {
        // F16X3: the leaf's three columns of the M2L's B operand as k_split_columns makes them
        // (the same FP32 operations: dm-scaled coefficients, power-of-2 column scale, FP16 hi and
        // lo, [column][K step][hi | lo]), so that the split after the M2M covers the other nodes
        if (hl) {
            float dmv[NS];
#pragma unroll
            for (int r = 0; r < NS; r++) {
                const int k = lane + 64 * r;
                dmv[r] = k < L && k < Kp ? dm[k] : 0.0f;
            }
            for (int cc = 0; cc < 3; cc++) {
                float x[NS], mx = 0.0f;
#pragma unroll
                for (int r = 0; r < NS; r++) {
                    x[r] = mv[r][cc] * dmv[r];
                    mx = fmaxf(mx, fabsf(x[r]));
                }
                for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
                const float sc = column_scale(mx);
                const size_t col = (size_t)leaf * 3 + cc;
                if (lane == 0) cscale[col] = sc;
                _Float16* dst = hl + col * 2 * Kp;
#pragma unroll
                for (int r = 0; r < NS; r++) {
                    const int k = lane + 64 * r;
                    if (k < Kp) {
                        const float y = x[r] * sc;
                        const _Float16 h = (_Float16)y;
                        dst[(k >> 5) * 64 + (k & 31)] = h;
                        dst[(k >> 5) * 64 + (k & 31) + 32] = (_Float16)(y - (float)h);
                    }
                }
            }
        }
    }
}

// The nodes k_p2m does not write (subdivided ones and leaves without points), cleared with
// 16-byte stores, one wave per node (n4 vectors per node).
__global__ __launch_bounds__(256) void k_zero_unwritten(const int* __restrict__ first_child,
                                                        const int* __restrict__ npts, int nnodes, int n4,
                                                        float4* __restrict__ M) {
    const int v = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (v >= nnodes || (first_child[v] < 0 && npts[v] > 0)) return;
    float4* o = M + (size_t)v * n4;
    for (int i = lane; i < n4; i += 64) o[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// ---------------------------------------------------------------- L2P
// One wave per useful target leaf; lane (m, g) evaluates column m for the targets g, g+G, ...
// (G = 64 / p) and the p lanes of a target are summed through LDS.  The local expansion is turned into the complex
// coefficients beta_c (degree <= p-1) of B = sigma^-2 Re sum beta_c(l,m) Phi_l^m(u), using
// dz Phi_l^m = Phi_{l-1}^m, (dx - i dy) Phi_l^m = Phi_{l-1}^{m-1}, (dx + i dy) Phi_l^m = -Phi_{l-1}^{m+1}.
__device__ __forceinline__ void alpha_of(const double* Ls, int L, int c, int l, int m, double& ar, double& ai) {
    const double* Lc = Ls + c * L;
    double s = sgnl(l);
    if (m == 0) { ar = s * Lc[lmi(l, 0)]; ai = 0.0; }
    else { ar = s * SQRT2 * Lc[lmi(l, m)]; ai = -s * SQRT2 * Lc[lmi(l, -m)]; }
}
// derivative coefficients of component c along axis a (0 x, 1 y, 2 z) at (l', m')
__device__ __forceinline__ void deriv_coef(const double* Ls, int L, int c, int a, int lp, int mp, double& br,
                                           double& bi) {
    int l = lp + 1;
    double r, i;
    if (a == 2) { alpha_of(Ls, L, c, l, mp, br, bi); return; }
    double sr = 0, si = 0;
    alpha_of(Ls, L, c, l, mp + 1, r, i);
    double ur = 0.5 * r, ui = 0.5 * i;            // 1/2 alpha(l, m'+1)
    double vr = 0, vi = 0;                        // 1/2 alpha(l, m'-1) (+ the m' = 1 extra)
    if (mp >= 1) {
        alpha_of(Ls, L, c, l, mp - 1, r, i);
        vr = 0.5 * r; vi = 0.5 * i;
        if (mp == 1) { vr *= 2.0; vi *= 2.0; }
    }
    if (a == 0) { sr = ur - vr; si = ui - vi; }   // x: 1/2 a(m'+1) - 1/2 a(m'-1)
    else {                                        // y: (i/2) (a(m'+1) + a(m'-1))
        double wr = ur + vr, wi = ui + vi;
        sr = -wi; si = wr;
    }
    br = sr; bi = si;
}

// POT: the vector potential A = sigma^-1 Re sum alpha_c(l,m) Phi_l^m(u) over degree <= p (the
// reference's calcA, calculation_point_octree.cpp:192-212) instead of B = curl A (degree <= p-1).
//
// One wave (a one-wave workgroup) per useful target leaf.  The leaf's local expansion is mapped
// once to the coefficients beta (LDS, type T); then each lane evaluates one target: the sectoral
// chain Phi_m^m = Phi_{m-1}^{m-1} (x + iy) / (2m) and, per m, Phi_l^m = ((2l - 1) z Phi_{l-1}^m -
// r^2 Phi_{l-2}^m) / (l^2 - m^2), every (l, m) term added to the three components as it is made.
// D (the highest degree evaluated) is a template parameter, so the loops unroll with the
// recurrence factors as constants and the term index and the beta offsets fixed; the beta reads
// are the same address in every lane (LDS broadcast); explicit fused multiply-adds.  T is FP64
// in the FP64 mode, FP32 otherwise (|u| <= sqrt3 inside the leaf box keeps the recurrences in
// range); the result is scaled and written in FP64.
__device__ __forceinline__ float fma_l(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_l(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <class T, int D, bool POT>
__global__ __launch_bounds__(64) void k_l2p(const int* __restrict__ leaves, const double* __restrict__ center,
                                            const int* __restrict__ begin, const int* __restrict__ end,
                                            const int* __restrict__ level, ScaleTable sig,
                                            const double* __restrict__ txyz, const void* __restrict__ Lexp_v, int p,
                                            int Lp, bool lexp_f64, double* __restrict__ Bfar) {
    constexpr int NB = (D + 1) * (D + 2) / 2;   // (l', m') pairs with l' <= D
    extern __shared__ __attribute__((aligned(16))) double sh[];
    const int L = (p + 1) * (p + 1);
    double* Ls = sh;                             // [3][L] the local expansion (FP64)
    T* beta = (T*)(sh + 3 * L);                  // [NB][3][2]
    const int leaf = leaves[blockIdx.x];
    const int lane = threadIdx.x;
    if (lexp_f64) {
        const double* Lsrc = (const double*)Lexp_v + (size_t)leaf * 3 * Lp;
        for (int e = lane; e < 3 * L; e += 64) {
            const int c = e / L, k = e - c * L;
            Ls[e] = Lsrc[c * Lp + k];
        }
    } else {
        const float* Lsrc = (const float*)Lexp_v + (size_t)leaf * 3 * Lp;
        for (int e = lane; e < 3 * L; e += 64) {
            const int c = e / L, k = e - c * L;
            Ls[e] = (double)Lsrc[c * Lp + k];
        }
    }
    __syncthreads();
    for (int e = lane; e < NB; e += 64) {
        int lp = 0;
        while ((lp + 1) * (lp + 2) / 2 <= e) lp++;
        const int mp = e - lp * (lp + 1) / 2;
        double bv[3][2];
        if (POT) {
            for (int c = 0; c < 3; c++) alpha_of(Ls, L, c, lp, mp, bv[c][0], bv[c][1]);
        } else {
            double d[3][3][2];   // d[comp][axis]
            for (int c = 0; c < 3; c++)
                for (int a = 0; a < 3; a++) deriv_coef(Ls, L, c, a, lp, mp, d[c][a][0], d[c][a][1]);
            for (int q = 0; q < 2; q++) {   // B = curl A
                bv[0][q] = d[2][1][q] - d[1][2][q];
                bv[1][q] = d[0][2][q] - d[2][0][q];
                bv[2][q] = d[1][0][q] - d[0][1][q];
            }
        }
        for (int c = 0; c < 3; c++) {
            beta[(e * 3 + c) * 2] = (T)bv[c][0];
            beta[(e * 3 + c) * 2 + 1] = (T)bv[c][1];
        }
    }
    __syncthreads();
    const double cx = center[3 * leaf], cy = center[3 * leaf + 1], cz = center[3 * leaf + 2];
    const double inv = 1.0 / sig.s[level[leaf]];
    const double s2 = POT ? inv : inv * inv;
    const int kb = begin[leaf], n = end[leaf] - kb;
    for (int t0 = 0; t0 < n; t0 += 64) {
        const int t = t0 + lane;
        if (t >= n) break;
        const int k = kb + t;
        const T ux = (T)((txyz[3 * k] - cx) * inv), uy = (T)((txyz[3 * k + 1] - cy) * inv),
                uz = (T)((txyz[3 * k + 2] - cz) * inv);
        const T r2 = ux * ux + uy * uy + uz * uz;
        T b0 = 0, b1 = 0, b2 = 0;
        T sr = 1, si = 0;   // Phi_m^m
#pragma unroll
        for (int m = 0; m <= D; m++) {
            if (m > 0) {
                constexpr T one = 1;
                const T h = one / (T)(2 * m);
                const T nr = (sr * ux - si * uy) * h, ni = (sr * uy + si * ux) * h;
                sr = nr;
                si = ni;
            }
            T p1r = sr, p1i = si, p2r = 0, p2i = 0;
#pragma unroll
            for (int l = m; l <= D; l++) {
                T vr = p1r, vi = p1i;
                if (l > m) {
                    const T a = (T)(2 * l - 1) * uz, f = (T)1 / (T)(l * l - m * m);
                    vr = fma_l(a, p1r, -r2 * p2r) * f;
                    vi = fma_l(a, p1i, -r2 * p2i) * f;
                    p2r = p1r; p2i = p1i; p1r = vr; p1i = vi;
                }
                const T* bt = beta + (l * (l + 1) / 2 + m) * 6;
                b0 = fma_l(bt[0], vr, fma_l(-bt[1], vi, b0));
                b1 = fma_l(bt[2], vr, fma_l(-bt[3], vi, b1));
                b2 = fma_l(bt[4], vr, fma_l(-bt[5], vi, b2));
            }
        }
        Bfar[3 * k] = (double)b0 * s2;
        Bfar[3 * k + 1] = (double)b1 * s2;
        Bfar[3 * k + 2] = (double)b2 * s2;
    }
}

// ---------------------------------------------------------------- P2P
// Near field B(x) = sum_j q_j x (x - y_j) / |x - y_j|^3 over the sources of each close
// source node (the close-list loop of FastMultipoleSolver::calcB, fast_multipole_solver.cpp:214-229;
// a close node may be internal, then all its subtree's sources are summed).
//
// For R = float positions are taken relative to one origin o (the source root centre), and both
// sides are unevaluated sums hi + lo of two floats formed in FP64 (~2^-48 of the root size),
// so the pair difference d = (x_hi - y_hi) + (x_lo - y_lo) stays accurate for very close
// pairs (x_hi - y_hi is exact when the two are within a factor 2) while the pair arithmetic
// runs in FP32.  R = double takes the coordinates themselves (o = 0): the difference of two close
// ones is exact, and an offset from o that is rounded first would not leave it so.
template <class R> struct V4;
template <> struct V4<float> {
    typedef float4 t;
    static __device__ float4 make(float a, float b, float c, float d) { return make_float4(a, b, c, d); }
};
template <> struct V4<double> {
    typedef double4 t;
    static __device__ double4 make(double a, double b, double c, double d) { return make_double4(a, b, c, d); }
};
// 1 / r^3 (POT: 1 / r) from r^2 = x in FP64, 0 for x = 0.  v_rsq_f64 gives y with a relative error
// of about 2^-24; with y2 = fl(y y) and e = 1 - x y2 one step of third order,
//   1 / r = y (1 + e (1/2 + 3/8 e)),  1 / r^3 = y^3 (1 + e (3/2 + 15/8 e)),
// leaves the next term (about 2^-70) far below the roundings: at most 1.25 ulp for the cube (the
// rounding of y2 enters e as well and half cancels), against 1.5 ulp of 1 / (x sqrt(x)), in 6
// instructions and the v_rsq instead of about 25.  Arguments whose powers leave the normal range
// (x < 2^-670, x = 0, infinities, NaN) take the IEEE operations.
// inv_power_regular gives the value where inv_power_rank is below INV_POWER_ODD.
constexpr unsigned INV_POWER_ODD = (unsigned)(2 * 670) << 20;
__device__ __forceinline__ unsigned inv_power_rank(double x) {   // negative x and NaN rank high
    return (unsigned)__double2hiint(x) - ((unsigned)(1023 - 670) << 20);
}
template <bool POT>
__device__ __forceinline__ double inv_power_regular(double x) {
    double c = POT ? 0.5 : 1.5;
    asm("" : "+v"(c));   // in a register: as a literal it is moved anew before every accumulating FMA
    const double y = __builtin_amdgcn_rsq(x), y2 = y * y, e = fma_t(-x, y2, 1.0), w = POT ? y : y2 * y;
    return fma_t(w, e * fma_t(e, POT ? 0.375 : 1.875, c), w);
}
template <bool POT>
__device__ __forceinline__ double inv_power_ieee(double x) {
    return x == 0.0 ? 0.0 : POT ? 1.0 / sqrt(x) : 1.0 / (x * sqrt(x));
}
template <bool POT>
__device__ __forceinline__ double inv_power(double x) {
    double f = inv_power_regular<POT>(x);
    if (__builtin_expect(inv_power_rank(x) >= INV_POWER_ODD, 0)) f = inv_power_ieee<POT>(x);
    return f;
}
// FP32: v_rsq_f32 directly (1 ulp): pair distances squared are far above the denormal range, so the
// denormal-scaling wrapper of rsqrtf is not needed
template <bool POT>
__device__ __forceinline__ float inv_power(float x) {
    const float ri = x > 0.0f ? __builtin_amdgcn_rsqf(x) : 0.0f;
    return POT ? ri : ri * ri * ri;
}
// P0[j] = (hi(y_j - o), q_x), P1[j] = (lo(y_j - o), q_y), P2[j] = q_z for every source slot j; in FP64 o = 0 and
// the low parts are zero, P1[j].x holds sd[j] if there is one (BEM)
template <class R>
__global__ void k_pack_sources(int n, const double* __restrict__ origin, const double* __restrict__ sxyz,
                               const double* __restrict__ sq, const double* __restrict__ sd,
                               typename V4<R>::t* __restrict__ P0, typename V4<R>::t* __restrict__ P1,
                               R* __restrict__ P2) {
    constexpr bool split = sizeof(R) == 4;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    double dx = sxyz[3 * j], dy = sxyz[3 * j + 1], dz = sxyz[3 * j + 2];
    if (split) {
        dx -= origin[0];
        dy -= origin[1];
        dz -= origin[2];
    }
    R hx = (R)dx, hy = (R)dy, hz = (R)dz;
    R lx = split ? (R)(dx - (double)hx) : sd ? (R)sd[j] : (R)0, ly = split ? (R)(dy - (double)hy) : (R)0;
    R lz = split ? (R)(dz - (double)hz) : (R)0;
    P0[j] = V4<R>::make(hx, hy, hz, (R)sq[3 * j]);
    P1[j] = V4<R>::make(lx, ly, lz, (R)sq[3 * j + 1]);
    P2[j] = (R)sq[3 * j + 2];
}

// One workgroup (4 waves) per target leaf.  The sources of the close list are taken 256 at a time
// whatever nodes they come from: 64 list entries at a time give a table of slot ranges in LDS, each
// thread finds its source in it, and the batch after the current one is on its way while the current
// one is summed from LDS.  The leaf's targets go in even blocks of at most 128, n of them spread over
// the workgroup with G = floor(256 / n) lanes each: lane g n + t takes the sources g, g + G, ... for target
// t, so the lanes of a wave read one or a few sources at a time (broadcasts).  Partial sums of at most RUN
// terms in R are added up in FP64, over the G lanes in a fixed order.  A run does not end at a node's border, so
// in FP32 it is kept to 8 terms: at 64 the median error of a target among small leaves (100,000 x 400,000 clustered
// points, 32 a leaf) was 1.27e-7, with runs within nodes 1.22e-7, now 1.20e-7 (999,983 x 750,019, 48 a leaf: 1.36e-7,
// 1.39e-7, 1.22e-7).  Full runs are unrolled by 2, which pays for the additions in FP64: near field of the 4M shells
// alone 5.9 ms with runs of 64, 6.2 with runs of 8, 5.9 unrolled; of 250,000 points 0.288, 0.314, 0.298.  By 4
// and 8: 5.9 and 6.2, 0.299 and 0.304 (more than 64 registers or longer code).
// KIND: B, the vector potential sum_j q_j / |x - y_j|, or the BEM potential (FP64), whose source has a
// strength v = q and a number d (in the place of the low part of its x).
// The batches may be shared by `parts` workgroups per leaf, each writing its own sums; out: the leaf's
// first row.
// UP: the leaf takes the lists of its ancestors as well (parent[] up to the root): the transposed
// near field, where a source leaf is reached through the close pairs of any node that holds it.
//
// Bound by VALU issue (26 instructions a pair in FP32).  With a wave per 64-source chunk of a node and
// floor(64 / n) lanes a target, a leaf of 33 .. 63 targets left 2 to 48 % of the lanes idle and a node's
// last chunk was short: B and A of 250,000 shell points 0.53 + 0.41 -> 0.36 + 0.31 ms, the transposed
// near field of 262,147 x 131,101 clustered points (3.6e8 pairs) 2.14 -> 1.27 ms.
enum { NEAR_B, NEAR_A, NEAR_BEM };
template <class R> struct P2PShared {
    typename V4<R>::t s0[256], s1[256];
    R s2[256];
    int nbegin[64], nfirst[65];   // the table: first slot and first source of each entry, and their number
};
template <class R, int KIND, bool UP>
__device__ __forceinline__ void p2p_leaf(int leaf, int part, int parts, const int* __restrict__ tbegin,
                                         const int* __restrict__ tend, const int* __restrict__ close_begin,
                                         const int* __restrict__ close_end, const int* __restrict__ close_s,
                                         const double* __restrict__ origin, const int* __restrict__ sbegin,
                                         const int* __restrict__ send, const typename V4<R>::t* __restrict__ P0,
                                         const typename V4<R>::t* __restrict__ P1, const R* __restrict__ P2,
                                         const double* __restrict__ txyz, double* __restrict__ out, P2PShared<R>& sh,
                                         const int* __restrict__ parent = nullptr) {
    typedef typename V4<R>::t v4;
    constexpr bool split = sizeof(R) == 4;
    constexpr int RUN = split ? 8 : 64;   // terms of a partial sum in R
    static_assert(KIND != NEAR_BEM || !split, "the BEM potential is FP64");
    static_assert(sizeof(sh.s0) + sizeof(sh.s1) >= 256 * 3 * sizeof(double), "the sums reuse the source buffers");
    double(*red)[3] = (double(*)[3])sh.s0;
    const int tid = threadIdx.x;
    const int tb = tbegin[leaf], te = tend[leaf];
    if (!UP && close_begin[leaf] >= close_end[leaf]) {
        for (int k = tid; k < te - tb; k += 256) out[3 * k] = out[3 * k + 1] = out[3 * k + 2] = 0.0;
        return;
    }
    const int nblk = (te - tb + 127) / 128;
    for (int blk = 0; blk < nblk; blk++) {
        const int k0 = tb + (int)((long long)(te - tb) * blk / nblk);
        const int n = tb + (int)((long long)(te - tb) * (blk + 1) / nblk) - k0;
        const int G = 256 / n, g = tid / n, ti = tid - g * n;
        const bool valid = g < G;
        double ux = 0, uy = 0, uz = 0;
        if (valid) {
            ux = txyz[3 * (k0 + ti)] - (split ? origin[0] : 0.0);
            uy = txyz[3 * (k0 + ti) + 1] - (split ? origin[1] : 0.0);
            uz = txyz[3 * (k0 + ti) + 2] - (split ? origin[2] : 0.0);
        }
        const R uhx = (R)ux, uhy = (R)uy, uhz = (R)uz;
        const R ulx = split ? (R)(ux - (double)uhx) : (R)0, uly = split ? (R)(uy - (double)uhy) : (R)0;
        const R ulz = split ? (R)(uz - (double)uhz) : (R)0;
        double a0 = 0, a1 = 0, a2 = 0;
        int run = 0;   // batches of the list entries before c0
        for (int node = leaf; node >= 0; node = UP ? parent[node] : -1)
        for (int c0 = close_begin[node], ce = close_end[node]; c0 < ce; c0 += 64) {
            __syncthreads();   // the last table is no longer read
            if (tid < 64) {
                int b = 0, cnt = 0;
                if (c0 + tid < ce) {
                    const int s = close_s[c0 + tid];
                    b = sbegin[s];
                    cnt = send[s] - b;
                }
                int incl = cnt;
                for (int d = 1; d < 64; d <<= 1) {
                    const int u = __shfl_up(incl, d, 64);
                    if (tid >= d) incl += u;
                }
                sh.nbegin[tid] = b;
                sh.nfirst[tid + 1] = incl;
                if (tid == 0) sh.nfirst[0] = 0;
            }
            __syncthreads();
            const int total = sh.nfirst[64], nbatch = (total + 255) >> 8;
            // slot of source x of the table: the last entry with nfirst <= x that is not empty
            auto slot = [&](int x) {
                x = min(x, total - 1);
                int e = 0;
#pragma unroll
                for (int d = 32; d > 0; d >>= 1)
                    if (sh.nfirst[e + d] <= x) e += d;
                return sh.nbegin[e] + (x - sh.nfirst[e]);
            };
            int b = (part - run) & (parts - 1);   // parts is a power of 2
            run += nbatch;
            if (b >= nbatch) continue;
            int j = slot(256 * b + tid);
            v4 p0 = P0[j], p1 = P1[j];
            R p2 = P2[j];
            for (; b < nbatch; b += parts) {
                __syncthreads();   // the last batch is no longer read
                sh.s0[tid] = p0;
                sh.s1[tid] = p1;
                sh.s2[tid] = p2;
                const int nj = min(256, total - 256 * b);
                j = slot(256 * (b + parts) + tid);   // beyond the end: the last source again
                p0 = P0[j];
                p1 = P1[j];
                p2 = P2[j];
                __syncthreads();
                for (int q = valid ? g : nj; q < nj;) {
                    R f0 = 0, f1 = 0, f2 = 0;
                    auto pair = [&](int q) {
                        const v4 yh = sh.s0[q];
                        const v4 yl = sh.s1[q];
                        const R qx = yh.w, qy = yl.w, qz = sh.s2[q];
                        R dx = uhx - yh.x, dy = uhy - yh.y, dz = uhz - yh.z;
                        if (split) {
                            dx += ulx - yl.x;
                            dy += uly - yl.y;
                            dz += ulz - yl.z;
                        }
                        // fused multiply-adds (explicit: this library is built without contraction)
                        const R r2 = fma_t(dx, dx, fma_t(dy, dy, dz * dz));
                        const R ip = inv_power<KIND == NEAR_A>(r2);
                        if (KIND == NEAR_BEM) {   // (d (y - x) + (y - x) x v) / |y - x|^3
                            f0 = fma_t(-fma_t(dx, yl.x, fma_t(dy, qz, -dz * qy)), ip, f0);
                            f1 = fma_t(-fma_t(dy, yl.x, fma_t(dz, qx, -dx * qz)), ip, f1);
                            f2 = fma_t(-fma_t(dz, yl.x, fma_t(dx, qy, -dy * qx)), ip, f2);
                        } else if (KIND == NEAR_A) {
                            f0 = fma_t(qx, ip, f0);
                            f1 = fma_t(qy, ip, f1);
                            f2 = fma_t(qz, ip, f2);
                        } else {
                            f0 = fma_t(fma_t(qy, dz, -qz * dy), ip, f0);
                            f1 = fma_t(fma_t(qz, dx, -qx * dz), ip, f1);
                            f2 = fma_t(fma_t(qx, dy, -qy * dx), ip, f2);
                        }
                    };
                    if (split && q + (RUN - 1) * G < nj) {
#pragma unroll 2
                        for (int k = 0; k < RUN; k++) pair(q + k * G);
                        q += RUN * G;
                    } else {
                        const int qe = min(nj, q + RUN * G);
#pragma unroll 1
                        for (; q < qe; q += G) pair(q);
                    }
                    a0 += f0;
                    a1 += f1;
                    a2 += f2;
                }
            }
        }
        __syncthreads();   // the last batch is no longer read
        red[tid][0] = a0;
        red[tid][1] = a1;
        red[tid][2] = a2;
        for (int h = G; h > 1;) {
            const int half = (h + 1) >> 1;
            __syncthreads();
            if (g + half < h)
                for (int c = 0; c < 3; c++) red[tid][c] += red[tid + half * n][c];
            h = half;
        }
        if (tid < n)
            for (int c = 0; c < 3; c++) out[3 * (k0 - tb + tid) + c] = red[tid][c];
        __syncthreads();   // the next leaf or block writes the buffers again
    }
}

// What the near field's workgroups work on: part 0 of every leaf, and the further parts of the leaves with
// long lists, extra[] = (leaf, part).  desc[leaf] = (parts, first row of `partial` of the further parts).
// counters: extra items made, rows made, items taken (by the grids that share them).  The first
// extra_wgs workgroups of a grid of its own share the extra items in equal strides (they are of one size),
// the others take a leaf each: a counter for all of 32,768 leaves, most of them short, took 0.4 ms more.
// Without desc every leaf is one item.
//
// A few leaves near the sources can hold most of the pairs: with one workgroup per leaf the time is that
// of the longest list, or of the last ones to start (1M uniform targets around a coil of 1M sources: 1.0
// ms in FP32, 2.7 ms in FP64; 32,768 x 4,096 points in 276 leaves, FP64: 470 us).  A list is therefore cut
// into 2, 4, .. 32 parts of at most `batches` batches of 256 sources (near_batches; longer ones where 32 parts
// are not enough), and the register budget is that of 7 (FP64: 5) waves a
// SIMD (unrolled by 2 at most), since the short lists are a matter of latency: 1M points 1007 (items alone: 1230) ->
// 660 us in FP32, 2.7 -> 2.0 ms in FP64, beside the slab reduction; 262,147 x 131,101 clustered points 1520
// -> 330 us, transposed 1270 -> 420 us; B and A of 250,000 points 365 + 307 -> 267 + 237 us; 276 leaves 90
// -> 75 us.
//
// The order of a target's sum follows from the parts of its leaf, so these follow from the lists alone: where
// the parts of all leaves together would take more items or rows than there are, all leaves are held to 16 parts,
// or 8, and so on (sums: what they take at 2, 4, .. 32).  Where the parts lie, by atomics, enters no sum.
constexpr int NEAR_MAX_PARTS = 32, NEAR_CUTS = 5;
struct NearWork {
    const int* leaves;
    int nleaves;
    int2* desc;
    int2* extra;
    int* counters;
    unsigned long long* sums;   // [2 q]: extra items, [2 q + 1]: rows, of all leaves with parts cut to 2 << q
    double* partial;
    int extra_cap, extra_wgs;
};

// before every near field; a kernel, because a memset recorded into a graph can fail on later replays
__global__ void k_near_clear(NearWork w) {
    if (threadIdx.x < 4) w.counters[threadIdx.x] = 0;
    if (threadIdx.x < 2 * NEAR_CUTS) w.sums[threadIdx.x] = 0;
}

// the parts every leaf asks for, and the sums; 16 leaves a workgroup, 16 lanes a leaf
template <bool UP>
__global__ __launch_bounds__(256) void k_near_loads(NearWork w, int batches, const int* __restrict__ tbegin,
                                                    const int* __restrict__ tend, const int* __restrict__ parent,
                                                    const int* __restrict__ close_begin,
                                                    const int* __restrict__ close_end, const int* __restrict__ close_s,
                                                    const int* __restrict__ sbegin, const int* __restrict__ send) {
    __shared__ int parts_of[16], targets_of[16];
    const int tid = threadIdx.x, u = tid >> 4, lane = tid & 15, li = 16 * blockIdx.x + u;
    int n = 0;
    long long load = 0;
    if (li < w.nleaves) {
        const int leaf = w.leaves[li];
        n = tend[leaf] - tbegin[leaf];
        for (int node = leaf; node >= 0; node = UP ? parent[node] : -1)
            for (int ci = close_begin[node] + lane, ce = close_end[node]; ci < ce; ci += 16) {
                const int s = close_s[ci];
                load += send[s] - sbegin[s];
            }
    }
    for (int d = 1; d < 16; d <<= 1) load += __shfl_xor(load, d);
    int parts = 1;
    while (parts < NEAR_MAX_PARTS && (long long)parts * batches * 256 < load) parts *= 2;
    while (parts > 1 && (long long)(parts - 1) * n > 1 << 24) parts >>= 1;   // a wave's rows stay in 32 bits
    if (lane == 0) {
        parts_of[u] = parts;
        targets_of[u] = n;
        if (li < w.nleaves) w.desc[li] = make_int2(parts, 0);
    }
    __syncthreads();
    if (tid < 2 * NEAR_CUTS) {
        unsigned long long s = 0;
        for (int e = 0; e < 16; e++)
            s += (unsigned long long)(min(parts_of[e], 2 << (tid >> 1)) - 1) * (tid & 1 ? targets_of[e] : 1);
        if (s) atomicAdd(w.sums + tid, s);
    }
}

// the parts every leaf gets, and their places; a thread per leaf
__global__ __launch_bounds__(256) void k_near_items(NearWork w, int rows_cap, const int* __restrict__ tbegin,
                                                    const int* __restrict__ tend) {
    const int li = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
    int cut = 1;
    for (int q = 0; q < NEAR_CUTS; q++)   // the sums grow with q
        if (w.sums[2 * q] <= (unsigned)w.extra_cap && w.sums[2 * q + 1] <= (unsigned)rows_cap) cut = 2 << q;
    int items = 0, rows = 0;
    if (li < w.nleaves) {
        const int leaf = w.leaves[li];
        items = min(w.desc[li].x, cut) - 1;
        rows = items * (tend[leaf] - tbegin[leaf]);
    }
    int ii = items, ir = rows;
    for (int d = 1; d < 64; d <<= 1) {
        const int vi = __shfl_up(ii, d, 64), vr = __shfl_up(ir, d, 64);
        if (lane >= d) {
            ii += vi;
            ir += vr;
        }
    }
    int bi = 0, br = 0;
    if (lane == 63 && ii) {
        bi = atomicAdd(&w.counters[0], ii);
        br = atomicAdd(&w.counters[1], ir);
    }
    bi = __shfl(bi, 63, 64) + ii - items;
    br = __shfl(br, 63, 64) + ir - rows;
    if (li >= w.nleaves) return;
    w.desc[li] = make_int2(items + 1, br);
    for (int q = 0; q < items; q++) w.extra[bi + q] = make_int2(li, q + 1);
}

// near[leaf] += the sums of its further parts, in their order; a wave per leaf
__global__ __launch_bounds__(256) void k_add_parts(NearWork w, const int* __restrict__ tbegin,
                                                   const int* __restrict__ tend, double* __restrict__ near) {
    const int li = 4 * blockIdx.x + (threadIdx.x >> 6);
    if (li >= w.nleaves) return;
    const int2 d = w.desc[li];
    if (d.x == 1) return;
    const int leaf = w.leaves[li], tb = tbegin[leaf], n = tend[leaf] - tb;
    for (int e = threadIdx.x & 63; e < 3 * n; e += 64) {
        double v = near[3 * (size_t)tb + e];
#pragma unroll 8
        for (int q = 0; q < d.x - 1; q++) v += w.partial[3 * ((size_t)d.y + (size_t)q * n) + e];
        near[3 * (size_t)tb + e] = v;
    }
}

// QUEUE: items from the counter (leaves, then extra items); else those of this workgroup
template <class R, int KIND, bool UP, bool QUEUE>
__device__ __forceinline__ void p2p_items(const NearWork& w, const int* __restrict__ tbegin,
                                          const int* __restrict__ tend, const int* __restrict__ close_begin,
                                          const int* __restrict__ close_end, const int* __restrict__ close_s,
                                          const double* __restrict__ origin, const int* __restrict__ sbegin,
                                          const int* __restrict__ send, const typename V4<R>::t* __restrict__ P0,
                                          const typename V4<R>::t* __restrict__ P1, const R* __restrict__ P2,
                                          const double* __restrict__ txyz, double* __restrict__ near,
                                          const int* __restrict__ parent = nullptr) {
    __shared__ P2PShared<R> sh;
    __shared__ int next;
    const int nextra = w.desc ? w.counters[0] : 0;
    // i < nleaves: part 0 of leaf i, else extra item i - nleaves
    const bool own = !QUEUE && (int)blockIdx.x >= w.extra_wgs;   // one leaf
    for (int i = own ? blockIdx.x - w.extra_wgs : w.nleaves + blockIdx.x;; i += w.extra_wgs) {
        if (QUEUE) {
            if (threadIdx.x == 0) next = atomicAdd(&w.counters[2], 1);
            __syncthreads();
            i = next;
            __syncthreads();   // every thread has read next before thread 0 takes the following item
        }
        if (i >= w.nleaves + nextra) break;
        const int2 it = i < w.nleaves ? make_int2(i, 0) : w.extra[i - w.nleaves];
        const int leaf = w.leaves[it.x], tb = tbegin[leaf];
        const int2 d = w.desc ? w.desc[it.x] : make_int2(1, 0);
        double* out = it.y ? w.partial + 3 * ((size_t)d.y + (size_t)(it.y - 1) * (tend[leaf] - tb)) : near + 3 * (size_t)tb;
        p2p_leaf<R, KIND, UP>(leaf, it.y, d.x, tbegin, tend, close_begin, close_end, close_s, origin, sbegin, send, P0,
                              P1, P2, txyz, out, sh, parent);
        if (own) break;
    }
}

template <class R, int KIND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 7 : 5))) void k_p2p(NearWork w, const int* __restrict__ tbegin, const int* __restrict__ tend,
                                             const int* __restrict__ close_begin, const int* __restrict__ close_end,
                                             const int* __restrict__ close_s, const double* __restrict__ origin,
                                             const int* __restrict__ sbegin, const int* __restrict__ send,
                                             const typename V4<R>::t* __restrict__ P0,
                                             const typename V4<R>::t* __restrict__ P1, const R* __restrict__ P2,
                                             const double* __restrict__ txyz, double* __restrict__ near) {
    p2p_items<R, KIND, false, false>(w, tbegin, tend, close_begin, close_end, close_s, origin, sbegin, send, P0, P1, P2,
                                        txyz, near);
}

// The transposed near field (adjoint): per useful source leaf, sum_i g_i x (y_j - x_i) / |y_j - x_i|^3
// over the targets x_i (strengths g_i, packed as P0, P1, P2) of every target leaf that is close to the
// leaf or to one of its ancestors.  The roles of the forward near field are swapped, so the pairs run
// in the same body: no atomics, and a sum whose order is fixed.  Bound by VALU issue like the forward
// one; one wave per target leaf adding to the sources by FP64 atomics, its differences in plain FP32,
// took 14.2 ms where this takes 1.3 (262,147 x 131,101 clustered points, 3.6e8 pairs) and had put
// 1.5e-6 into the FP32 gradient, now 1.4e-7.
template <class R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 7 : 5))) void k_p2p_transposed(
    NearWork w, const int* __restrict__ sbegin, const int* __restrict__ send,
    const int* __restrict__ parent, const int* __restrict__ close_begin, const int* __restrict__ close_end,
    const int* __restrict__ close_t, const double* __restrict__ origin, const int* __restrict__ tbegin,
    const int* __restrict__ tend, const typename V4<R>::t* __restrict__ P0, const typename V4<R>::t* __restrict__ P1,
    const R* __restrict__ P2, const double* __restrict__ sxyz, double* __restrict__ out) {
    p2p_items<R, NEAR_B, true, false>(w, sbegin, send, close_begin, close_end, close_t, origin, tbegin, tend, P0, P1,
                                         P2, sxyz, out, parent);
}

// The near field by two persistent grids that take their items from the one counter: BESIDE, one workgroup
// of which fits on a CU beside the F16X3 M2L GEMM's (at most 432 registers a lane, which leaves 80: 64 here), so the
// near field runs on the VALU slots the GEMM leaves idle, and the plain one for the items left when the
// GEMM is done.  A BESIDE workgroup that starts when the GEMM's tiles are all taken (their streams share a
// hardware queue and run one after the other) leaves the items to the other form: one workgroup per CU
// alone takes 25 ms for the 7 ms of near field of the 4M shells.
// The plain form's workgroups beyond the number of items left leave at once: of 2,048 that raced for 288 items, some
// CUs got three and others none (959,985 sources, 273 targets, p = 16: 0.9 to 1.25 ms, now 0.6).
template <class R, bool POT, bool BESIDE>
__device__ __forceinline__ void p2p_queue_body(const NearWork& w, const int* __restrict__ gemm_queues, int gemm_tiles,
                                               const int* __restrict__ tbegin, const int* __restrict__ tend,
                                               const int* __restrict__ close_begin, const int* __restrict__ close_end,
                                               const int* __restrict__ close_s, const double* __restrict__ origin,
                                               const int* __restrict__ sbegin, const int* __restrict__ send,
                                               const typename V4<R>::t* __restrict__ P0,
                                               const typename V4<R>::t* __restrict__ P1, const R* __restrict__ P2,
                                               const double* __restrict__ txyz, double* __restrict__ Bnear) {
    if (BESIDE) {
        __shared__ int tiles;
        if (threadIdx.x == 0) {
            int left = 0;   // tiles of the XCDs' eighths not yet taken
            for (int x = 0; x < 8; x++)
                left += max(0, (gemm_tiles >> 3) + (x < (gemm_tiles & 7) ? 1 : 0) -
                                   __hip_atomic_load(gemm_queues + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            tiles = left;
        }
        __syncthreads();
        if (tiles == 0) return;
    } else {
        const int left = w.nleaves + (w.desc ? w.counters[0] : 0) -
                         __hip_atomic_load(w.counters + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((int)blockIdx.x >= left) return;   // the first workgroup stays until none are left
    }
    p2p_items<R, POT ? NEAR_A : NEAR_B, false, true>(w, tbegin, tend, close_begin, close_end, close_s,
                                                                     origin, sbegin, send, P0, P1, P2, txyz, Bnear);
}
template <class R, bool POT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void k_p2p_queue(
    NearWork w, const int* __restrict__ gemm_queues, int gemm_tiles, const int* __restrict__ tbegin,
    const int* __restrict__ tend, const int* __restrict__ close_begin, const int* __restrict__ close_end,
    const int* __restrict__ close_s, const double* __restrict__ origin, const int* __restrict__ sbegin,
    const int* __restrict__ send, const typename V4<R>::t* __restrict__ P0, const typename V4<R>::t* __restrict__ P1,
    const R* __restrict__ P2, const double* __restrict__ txyz, double* __restrict__ Bnear) {
    p2p_queue_body<R, POT, true>(w, gemm_queues, gemm_tiles, tbegin, tend, close_begin, close_end, close_s, origin, sbegin,
                                 send, P0, P1, P2, txyz, Bnear);
}
template <class R, bool POT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void k_p2p_queue_rest(
    NearWork w, const int* __restrict__ gemm_queues, int gemm_tiles, const int* __restrict__ tbegin,
    const int* __restrict__ tend, const int* __restrict__ close_begin, const int* __restrict__ close_end,
    const int* __restrict__ close_s, const double* __restrict__ origin, const int* __restrict__ sbegin,
    const int* __restrict__ send, const typename V4<R>::t* __restrict__ P0, const typename V4<R>::t* __restrict__ P1,
    const R* __restrict__ P2, const double* __restrict__ txyz, double* __restrict__ Bnear) {
    p2p_queue_body<R, POT, false>(w, gemm_queues, gemm_tiles, tbegin, tend, close_begin, close_end, close_s, origin, sbegin,
                                  send, P0, P1, P2, txyz, Bnear);
}

// ---------------------------------------------------------------- Problem::BEM
// BEMQuadrature sources (bem_quadrature.hpp): weight w, field B and normal n per point.  The
// source strengths in slot order are d = w (B . n) and v = w (B x n) (3); their multipoles are
// M_c(l, m) = -sum_q (dR_lm/dy_c d_q + (grad R_lm x v_q)_c) (integration.cpp:295-353, with the
// exact gradient in place of the reference's central differences), the potential they give is
// sum_q ((y - x) d + (y - x) x v) / |y - x|^3 (integration.cpp:191-202).
__global__ void k_bem_charges(const int* __restrict__ slots, int n, const double* __restrict__ xyz,
                              const double* __restrict__ w, const double* __restrict__ Bv,
                              const double* __restrict__ nrm, double* __restrict__ sxyz, double* __restrict__ sv,
                              double* __restrict__ sd) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = slots[k];
    const double b0 = Bv[3 * i], b1 = Bv[3 * i + 1], b2 = Bv[3 * i + 2];
    const double n0 = nrm[3 * i], n1 = nrm[3 * i + 1], n2 = nrm[3 * i + 2], ww = w[i];
    sxyz[3 * k] = xyz[3 * i]; sxyz[3 * k + 1] = xyz[3 * i + 1]; sxyz[3 * k + 2] = xyz[3 * i + 2];
    sd[k] = ww * (b0 * n0 + b1 * n1 + b2 * n2);
    sv[3 * k] = ww * (b1 * n2 - b2 * n1);
    sv[3 * k + 1] = ww * (b2 * n0 - b0 * n2);
    sv[3 * k + 2] = ww * (b0 * n1 - b1 * n0);
}

// One workgroup (64 threads) per useful source leaf.  Points go through LDS in chunks of
// BEM_CHUNK: thread t builds the complex table Phi_n^k (n <= p - 1, k >= 0) of point t; then each
// thread owns coefficients i = tid + 64 r and adds the gradient of R_i at every point of the chunk:
// dz Phi_l^m = Phi_{l-1}^m, dx Phi_l^m = (Phi_{l-1}^{m-1} - Phi_{l-1}^{m+1}) / 2,
// dy Phi_l^m = i (Phi_{l-1}^{m-1} + Phi_{l-1}^{m+1}) / 2, Phi_n^{-k} = (-1)^k conj Phi_n^k.
constexpr int BEM_CHUNK = 8;
template <class T>
__global__ __launch_bounds__(64) void k_p2m_bem(const int* __restrict__ leaves, const double* __restrict__ center,
                                                const int* __restrict__ begin, const int* __restrict__ end,
                                                const int* __restrict__ level, ScaleTable sig,
                                                const double* __restrict__ sxyz, const double* __restrict__ sv,
                                                const double* __restrict__ sd, int p, int Lp, T* __restrict__ M) {
    extern __shared__ double2 tab[];   // [BEM_CHUNK][p (p + 1) / 2]
    __shared__ double str[BEM_CHUNK][4];
    const int NT = p * (p + 1) / 2, L = (p + 1) * (p + 1);
    const int leaf = leaves[blockIdx.x], tid = threadIdx.x;
    const double cx = center[3 * leaf], cy = center[3 * leaf + 1], cz = center[3 * leaf + 2];
    const double inv = 1.0 / sig.s[level[leaf]];
    constexpr int RMAX = (MAX_ORDER + 1) * (MAX_ORDER + 1) / 64 + 1;
    double acc[RMAX][3];
    for (int r = 0; r < RMAX; r++) acc[r][0] = acc[r][1] = acc[r][2] = 0.0;
    const int jb = begin[leaf], je = end[leaf];
    for (int j0 = jb; j0 < je; j0 += BEM_CHUNK) {
        const int nj = min(BEM_CHUNK, je - j0);
        __syncthreads();
        if (tid < nj) {
            const int j = j0 + tid;
            const double ux = (sxyz[3 * j] - cx) * inv, uy = (sxyz[3 * j + 1] - cy) * inv,
                         uz = (sxyz[3 * j + 2] - cz) * inv, r2 = ux * ux + uy * uy + uz * uz;
            double2* t = tab + tid * NT;
            double dr = 1.0, di = 0.0;   // Phi_k^k = (x + iy)^k / (2^k k!)
            for (int k = 0; k < p; k++) {
                if (k > 0) {
                    const double s = recip(2 * k);
                    const double nr = (dr * ux - di * uy) * s, ni = (dr * uy + di * ux) * s;
                    dr = nr; di = ni;
                }
                double p1r = dr, p1i = di, p2r = 0.0, p2i = 0.0;
                t[k * (k + 1) / 2 + k] = make_double2(dr, di);
                for (int n = k + 1; n < p; n++) {
                    const double f = recip(n * n - k * k);
                    const double vr = ((2.0 * n - 1) * uz * p1r - r2 * p2r) * f;
                    const double vi = ((2.0 * n - 1) * uz * p1i - r2 * p2i) * f;
                    p2r = p1r; p2i = p1i; p1r = vr; p1i = vi;
                    t[n * (n + 1) / 2 + k] = make_double2(vr, vi);
                }
            }
            str[tid][0] = sd[j] * inv;
            str[tid][1] = sv[3 * j] * inv;
            str[tid][2] = sv[3 * j + 1] * inv;
            str[tid][3] = sv[3 * j + 2] * inv;
        }
        __syncthreads();
        for (int r = 0; r < RMAX; r++) {
            const int i = tid + 64 * r;
            if (i >= L) break;
            int l = 0;
            while ((l + 1) * (l + 1) <= i) l++;
            const int m = i - l * l - l, am = m < 0 ? -m : m;
            if (l == 0) continue;
            const int n = l - 1;
            const double sg = ((l & 1) ? -1.0 : 1.0) * (am == 0 ? 1.0 : 1.41421356237309504880);
            for (int q = 0; q < nj; q++) {
                const double2* t = tab + q * NT;
                // Phi_{l-1}^{k} for k = am - 1, am, am + 1 (signed orders through the conjugate rule)
                auto ph = [&](int k) -> double2 {
                    if (k > n || k < -n) return make_double2(0.0, 0.0);
                    if (k >= 0) return t[n * (n + 1) / 2 + k];
                    const double2 v = t[n * (n + 1) / 2 - k];
                    const double s = (k & 1) ? -1.0 : 1.0;
                    return make_double2(s * v.x, -s * v.y);
                };
                const double2 lo = ph(am - 1), mid = ph(am), hi = ph(am + 1);
                const double gxr = 0.5 * (lo.x - hi.x), gxi = 0.5 * (lo.y - hi.y);
                const double gyr = -0.5 * (lo.y + hi.y), gyi = 0.5 * (lo.x + hi.x);
                const double gzr = mid.x, gzi = mid.y;
                const bool im = m < 0;
                const double gx = sg * (im ? gxi : gxr), gy = sg * (im ? gyi : gyr), gz = sg * (im ? gzi : gzr);
                const double d = str[q][0], v0 = str[q][1], v1 = str[q][2], v2 = str[q][3];
                acc[r][0] -= gx * d + (gy * v2 - gz * v1);
                acc[r][1] -= gy * d + (gz * v0 - gx * v2);
                acc[r][2] -= gz * d + (gx * v1 - gy * v0);
            }
        }
    }
    T* out = M + (size_t)leaf * 3 * Lp;
    for (int e = tid; e < 3 * Lp; e += 64) out[e] = (T)0;
    __syncthreads();
    for (int r = 0; r < RMAX; r++) {
        const int i = tid + 64 * r;
        if (i >= L) break;
        for (int c = 0; c < 3; c++) out[c * Lp + i] = (T)acc[r][c];
    }
}

void launch_bem_charges(const int* slots, int n, const double* xyz, const double* w, const double* Bv,
                        const double* nrm, double* sxyz, double* sv, double* sd, hipStream_t st) {
    if (n) k_bem_charges<<<blocks(n), 256, 0, st>>>(slots, n, xyz, w, Bv, nrm, sxyz, sv, sd);
    FMM_HIP(hipGetLastError());
}
void launch_p2m_bem(bool f64, const int* leaves, int nleaves, const TreeDev& S, const ScaleTable& sig,
                    const double* sxyz, const double* sv, const double* sd, int p, int Lp, void* M, hipStream_t st) {
    if (!nleaves) return;
    if (p < 1 || p > MAX_ORDER) throw Error(1, "BEM P2M: order out of range");
    const size_t lds = (size_t)BEM_CHUNK * (p * (p + 1) / 2) * sizeof(double2);
    if (f64)
        k_p2m_bem<double><<<nleaves, 64, lds, st>>>(leaves, S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(),
                                                    S.level.as<int>(), sig, sxyz, sv, sd, p, Lp, (double*)M);
    else
        k_p2m_bem<float><<<nleaves, 64, lds, st>>>(leaves, S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(),
                                                   S.level.as<int>(), sig, sxyz, sv, sd, p, Lp, (float*)M);
    FMM_HIP(hipGetLastError());
}
// ---------------------------------------------------------------- assembly
__global__ void k_assemble(const int* __restrict__ slots, int n, const double* __restrict__ Bfar,
                           const double* __restrict__ Bnear, double scale, double* __restrict__ B) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = slots[k];
    for (int c = 0; c < 3; c++) B[3 * i + c] = scale * (Bfar[3 * k + c] + Bnear[3 * k + c]);
}

// ---------------------------------------------------------------- direct sum (FP64)
// B(x) = scale sum_j q_j x (x - y_j) / |x - y_j|^3 (POT: A(x) = scale sum_j q_j / |x - y_j|),
// math::calcBioSavartLaplace (integration.cpp:101-120).  The sources are cut into nsplit
// contiguous ranges: the wave (b, s) sums range s for the 64 targets of block b into
// partial[s][t][3]; k_direct_reduce adds the nsplit partials of each target in a fixed order
// (deterministic) and scales.  Splitting the sources keeps every SIMD busy when the targets are few.
//
// Bound by FP64 VALU issue.  A source is the same for all lanes, so its six doubles come through
// scalar loads straight into the arithmetic (no LDS staging, no barriers), four sources in flight;
// with inv_power and explicit fused multiply-adds a pair costs about half the instructions of an
// IEEE square root and division without contraction.  1,048,576 sources x 16,384 targets: 33.0 ->
// 17.5 ms (9.8e11 pairs/s; the start of the Newton step from v_rsq_f32 instead, with the two
// conversions, 20.8 ms).
template <bool POT>
__global__ __launch_bounds__(64) void k_direct_partial(const double* __restrict__ sxyz, const double* __restrict__ sq,
                                                       int ns, const double* __restrict__ txyz, int nt,
                                                       double* __restrict__ partial) {
    const int t = blockIdx.x * 64 + threadIdx.x, split = blockIdx.y, nsplit = gridDim.y;
    const long long per = ((long long)ns + nsplit - 1) / nsplit;
    const int j_begin = (int)min((long long)ns, per * split), j_end = (int)min((long long)ns, per * (split + 1));
    double x = 0, y = 0, z = 0;
    if (t < nt) { x = txyz[3 * t]; y = txyz[3 * t + 1]; z = txyz[3 * t + 2]; }
    double a0 = 0, a1 = 0, a2 = 0;
    auto add = [&](double dx, double dy, double dz, double f, double qx, double qy, double qz) {
        if (POT) {
            a0 = fma_t(qx, f, a0);
            a1 = fma_t(qy, f, a1);
            a2 = fma_t(qz, f, a2);
        } else {
            a0 = fma_t(fma_t(qy, dz, -qz * dy), f, a0);
            a1 = fma_t(fma_t(qz, dx, -qx * dz), f, a1);
            a2 = fma_t(fma_t(qx, dy, -qy * dx), f, a2);
        }
    };
    int j = j_begin;
    for (; j + 4 <= j_end; j += 4) {
        double v[12], q[12], r2[4], f[4];
#pragma unroll
        for (int e = 0; e < 12; e++) {
            v[e] = sxyz[3 * (size_t)j + e];
            q[e] = sq[3 * (size_t)j + e];
        }
        unsigned rank = 0;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const double dx = x - v[3 * u], dy = y - v[3 * u + 1], dz = z - v[3 * u + 2];
            r2[u] = fma_t(dx, dx, fma_t(dy, dy, dz * dz));
            f[u] = inv_power_regular<POT>(r2[u]);
            rank = max(rank, inv_power_rank(r2[u]));
        }
        if (__builtin_expect(rank >= INV_POWER_ODD, 0))   // one test for the four keeps their chains interleaved
            for (int u = 0; u < 4; u++) f[u] = inv_power<POT>(r2[u]);
#pragma unroll
        for (int u = 0; u < 4; u++)
            add(x - v[3 * u], y - v[3 * u + 1], z - v[3 * u + 2], f[u], q[3 * u], q[3 * u + 1], q[3 * u + 2]);
    }
    for (; j < j_end; j++) {
        const double* v = sxyz + 3 * (size_t)j;
        const double* q = sq + 3 * (size_t)j;
        const double dx = x - v[0], dy = y - v[1], dz = z - v[2];
        add(dx, dy, dz, inv_power<POT>(fma_t(dx, dx, fma_t(dy, dy, dz * dz))), q[0], q[1], q[2]);
    }
    if (t < nt) {
        double* o = partial + ((size_t)split * nt + t) * 3;
        o[0] = a0;
        o[1] = a1;
        o[2] = a2;
    }
}

// 2^lg lanes per output value (target * 3 + component): lane g adds the partials g, g + 2^lg, ...
// in range order, then the lanes are summed pairwise.  With hundreds of ranges and few targets one
// lane per value would be a chain of as many loads.
__global__ void k_direct_reduce(const double* __restrict__ partial, int nt, int nsplit, int lg, double scale,
                                double* __restrict__ B) {
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long i = id >> lg, n = 3ll * nt;
    const int g = (int)(id & ((1 << lg) - 1));
    double acc = 0;
    if (i < n)
        for (int s = g; s < nsplit; s += 1 << lg) acc += partial[(size_t)s * n + i];
    for (int o = 1; o < (1 << lg); o <<= 1) acc += __shfl_xor(acc, o);
    if (i < n && g == 0) B[i] = acc * scale;
}

int direct_splits(int ns, int nt) {
    // 16 waves per CU in total (4 per SIMD hide the arithmetic latency), each range at least 1,024 sources
    const int tb = std::max(1, blocks(nt, 64));
    int s = std::max(1, 16 * num_cus() / tb);
    s = std::min(s, std::max(1, ns / 1024));
    return s;
}

void launch_direct(bool pot, const double* sxyz, const double* sq, int ns, const double* txyz, int nt, double scale,
                   double* out, double* partial, int nsplit, hipStream_t st) {
    if (!nt) return;
    if (nsplit < 1) throw Error(1, "direct sum: at least one source range");
    dim3 grid(blocks(nt, 64), nsplit);
    if (pot) k_direct_partial<true><<<grid, 64, 0, st>>>(sxyz, sq, ns, txyz, nt, partial);
    else k_direct_partial<false><<<grid, 64, 0, st>>>(sxyz, sq, ns, txyz, nt, partial);
    int lg = 0;
    while (lg < 6 && (2 << lg) <= nsplit) lg++;
    k_direct_reduce<<<blocks((3ll * nt) << lg), 256, 0, st>>>(partial, nt, nsplit, lg, scale, out);
    FMM_HIP(hipGetLastError());
}

void launch_charges(const int* slots, int n, const double* xyz, const double* w, const double* J, double* sxyz,
                    double* sq, double* sJ, hipStream_t st) {
    if (n) k_charges<<<blocks(n), 256, 0, st>>>(slots, n, xyz, w, J, sxyz, sq, sJ);
}
void launch_gather_xyz(const int* slots, int n, const double* xyz, double* out, hipStream_t st) {
    if (n) k_gather_xyz<<<blocks(n), 256, 0, st>>>(slots, n, xyz, out);
}
void launch_zero_unwritten(const TreeDev& S, int Lp, size_t esize, void* M, hipStream_t st) {
    const size_t bytes = (size_t)3 * Lp * esize;
    if (!S.num_nodes) return;
    if (bytes % 16) throw Error(1, "expansion rows must be whole 16-byte vectors");
    k_zero_unwritten<<<(S.num_nodes + 3) / 4, 256, 0, st>>>(S.first_child.as<int>(), S.npts.as<int>(), S.num_nodes,
                                                            (int)(bytes / 16), (float4*)M);
    FMM_HIP(hipGetLastError());
}
template <int P>
static void p2m_go(bool f64, const int* leaves, int nleaves, const TreeDev& S, const ScaleTable& sig,
                   const double* sxyz, const double* sq, int Lp, void* M, const F16Leaves& split, hipStream_t st) {
    if (f64)
        k_p2m<double, P><<<nleaves, 64, 0, st>>>(leaves, S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(),
                                                 S.level.as<int>(), sig, sxyz, sq, Lp, (double*)M, nullptr, 0,
                                                 nullptr, nullptr);
    else
        k_p2m<float, P><<<nleaves, 64, 0, st>>>(leaves, S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(),
                                                S.level.as<int>(), sig, sxyz, sq, Lp, (float*)M, split.dm, split.Kp,
                                                split.cscale, split.hl);
}
void launch_p2m(bool f64, const int* leaves, int nleaves, const TreeDev& S, const ScaleTable& sig, const double* sxyz,
                const double* sq, int p, int Lp, void* M, hipStream_t st, const F16Leaves& split) {
    if (!nleaves) return;
    if (p < 0 || p > MAX_ORDER) throw Error(4, "expansion order above 20");
    if (split.hl && (f64 || split.Kp % 32 || split.Kp > Lp || !split.dm || !split.cscale))
        throw Error(4, "P2M: FP16 split of the leaves needs FP32 multipoles and 32 | Kp <= Lp");
    switch (p) {
#define FMM_P2M_P(PV) \
    case PV: p2m_go<PV>(f64, leaves, nleaves, S, sig, sxyz, sq, Lp, M, split, st); break;
        FMM_P2M_P(0) FMM_P2M_P(1) FMM_P2M_P(2) FMM_P2M_P(3) FMM_P2M_P(4) FMM_P2M_P(5) FMM_P2M_P(6) FMM_P2M_P(7)
        FMM_P2M_P(8) FMM_P2M_P(9) FMM_P2M_P(10) FMM_P2M_P(11) FMM_P2M_P(12) FMM_P2M_P(13) FMM_P2M_P(14)
        FMM_P2M_P(15) FMM_P2M_P(16) FMM_P2M_P(17) FMM_P2M_P(18) FMM_P2M_P(19) FMM_P2M_P(20)
#undef FMM_P2M_P
        default: throw Error(4, "expansion order above 20");
    }
    FMM_HIP(hipGetLastError());
}
template <class T, int D, bool POT>
static void l2p_go(const int* leaves, int nleaves, const TreeDev& Tr, const ScaleTable& sig, const double* txyz,
                   const void* Lexp, bool lexp_f64, int p, int Lp, double* out, hipStream_t st) {
    constexpr int NB = (D + 1) * (D + 2) / 2;
    const size_t lds = (size_t)3 * (p + 1) * (p + 1) * sizeof(double) + (size_t)NB * 6 * sizeof(T);
    k_l2p<T, D, POT><<<nleaves, 64, lds, st>>>(leaves, Tr.center.as<double>(), Tr.begin.as<int>(), Tr.end.as<int>(),
                                               Tr.level.as<int>(), sig, txyz, Lexp, p, Lp, lexp_f64, out);
}
template <int D, bool POT>
static void l2p_d(bool f64, const int* leaves, int nleaves, const TreeDev& Tr, const ScaleTable& sig,
                  const double* txyz, const void* Lexp, int p, int Lp, double* out, hipStream_t st) {
    if (f64)
        l2p_go<double, D, POT>(leaves, nleaves, Tr, sig, txyz, Lexp, true, p, Lp, out, st);
    else
        l2p_go<float, D, POT>(leaves, nleaves, Tr, sig, txyz, Lexp, false, p, Lp, out, st);
}
template <bool POT>
static void l2p_launch(bool f64, const int* leaves, int nleaves, const TreeDev& T, const ScaleTable& sig,
                       const double* txyz, const void* Lexp, int p, int Lp, double* out, hipStream_t st) {
    const int D = POT ? p : p - 1;
    if (p < 1 || p > MAX_ORDER) throw Error(1, "L2P: order out of range");
    if (!nleaves) return;
    switch (D) {
#define FMM_L2P_D(DV) \
    case DV: l2p_d<DV, POT>(f64, leaves, nleaves, T, sig, txyz, Lexp, p, Lp, out, st); break;
        FMM_L2P_D(0) FMM_L2P_D(1) FMM_L2P_D(2) FMM_L2P_D(3) FMM_L2P_D(4) FMM_L2P_D(5) FMM_L2P_D(6) FMM_L2P_D(7)
        FMM_L2P_D(8) FMM_L2P_D(9) FMM_L2P_D(10) FMM_L2P_D(11) FMM_L2P_D(12) FMM_L2P_D(13) FMM_L2P_D(14)
        FMM_L2P_D(15) FMM_L2P_D(16) FMM_L2P_D(17) FMM_L2P_D(18) FMM_L2P_D(19) FMM_L2P_D(20)
#undef FMM_L2P_D
        default: throw Error(1, "L2P: order out of range");
    }
    FMM_HIP(hipGetLastError());
}
void launch_l2p(bool f64, const int* leaves, int nleaves, const TreeDev& T, const ScaleTable& sig, const double* txyz,
                const void* Lexp, int p, int Lp, double* Bfar, hipStream_t st) {
    if (!nleaves) return;
    l2p_launch<false>(f64, leaves, nleaves, T, sig, txyz, Lexp, p, Lp, Bfar, st);
}
void launch_l2p_A(bool f64, const int* leaves, int nleaves, const TreeDev& T, const ScaleTable& sig, const double* txyz,
                  const void* Lexp, int p, int Lp, double* Afar, hipStream_t st) {
    if (!nleaves) return;
    l2p_launch<true>(f64, leaves, nleaves, T, sig, txyz, Lexp, p, Lp, Afar, st);
}
void launch_pack_sources(bool f64, int n, const double* origin, const double* sxyz, const double* sq, void* P0,
                         void* P1, void* P2, hipStream_t st, const double* sd) {
    if (!n) return;
    if (f64)
        k_pack_sources<double><<<blocks(n), 256, 0, st>>>(n, origin, sxyz, sq, sd, (double4*)P0, (double4*)P1, (double*)P2);
    else
        k_pack_sources<float><<<blocks(n), 256, 0, st>>>(n, origin, sxyz, sq, nullptr, (float4*)P0, (float4*)P1, (float*)P2);
    FMM_HIP(hipGetLastError());
}
// batches per part: 16 (4,096 sources) where there are leaves enough for 8 workgroups a CU, fewer where
// the parts have to fill the chip
static int near_batches(int nleaves) { return std::max(2, std::min(16, 2 * nleaves / num_cus())); }
constexpr int NEAR_SPLIT_SOURCES = 1024;   // below, the items cost more launches than they save

static NearWork near_work(const int* leaves, int nleaves, size_t rows, NearScratch& scratch) {
    NearWork w;
    w.leaves = leaves;
    w.nleaves = nleaves;
    w.extra_cap = 4 * nleaves + 65536;
    w.extra_wgs = 0;
    w.desc = scratch.desc.get<int2>(nleaves);
    w.extra = scratch.extra.get<int2>(w.extra_cap);
    w.sums = scratch.counters.get<unsigned long long>(2 * NEAR_CUTS + 2);
    w.counters = (int*)(w.sums + 2 * NEAR_CUTS);
    w.partial = scratch.partial.get<double>(3 * rows);
    return w;
}
// rows of partial sums: of 2 more parts per target, and what small problems take
static size_t near_rows(int nslots) { return 2 * (size_t)nslots + 262144; }

template <bool UP>
static void make_items(const NearWork& w, const TreeDev& T, const TreeDev& S, const int* close_begin,
                       const int* close_end, const int* close_s, hipStream_t st) {
    k_near_clear<<<1, 64, 0, st>>>(w);
    k_near_loads<UP><<<(w.nleaves + 15) / 16, 256, 0, st>>>(w, near_batches(w.nleaves), T.begin.as<int>(), T.end.as<int>(),
                                                            T.parent.as<int>(), close_begin, close_end, close_s,
                                                            S.begin.as<int>(), S.end.as<int>());
    k_near_items<<<blocks(w.nleaves), 256, 0, st>>>(w, (int)std::min<size_t>(near_rows(T.num_slots), INT32_MAX),
                                                    T.begin.as<int>(), T.end.as<int>());
    FMM_HIP(hipGetLastError());
}
static void add_parts(const NearWork& w, const TreeDev& T, double* near, hipStream_t st) {
    k_add_parts<<<(w.nleaves + 3) / 4, 256, 0, st>>>(w, T.begin.as<int>(), T.end.as<int>(), near);
    FMM_HIP(hipGetLastError());
}
// the items of a near field into scratch, and its grid
template <bool UP>
static NearWork start_near(const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                           const int* close_end, const int* close_s, NearScratch& scratch, int& grid, hipStream_t st,
                           bool prepared = false) {
    NearWork w{leaves, nleaves, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0};
    grid = nleaves;
    if (S.num_slots > NEAR_SPLIT_SOURCES) {
        w = near_work(leaves, nleaves, near_rows(T.num_slots), scratch);
        if (!prepared) make_items<UP>(w, T, S, close_begin, close_end, close_s, st);
        w.extra_wgs = (int)std::min<long long>(8LL * num_cus(), (long long)NEAR_MAX_PARTS * nleaves);
        grid += w.extra_wgs;
    }
    return w;
}

template <int KIND>
static void p2p_launch(bool f64, const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S,
                       const int* close_begin, const int* close_end, const int* close_s, const void* P0,
                       const void* P1, const void* P2, const double* txyz, double* out, NearScratch& scratch,
                       hipStream_t st, bool prepared = false) {
    if (!nleaves) return;
    int grid;
    const NearWork w =
        start_near<false>(leaves, nleaves, T, S, close_begin, close_end, close_s, scratch, grid, st, prepared);
    if (f64)
        k_p2p<double, KIND><<<grid, 256, 0, st>>>(w, T.begin.as<int>(), T.end.as<int>(), close_begin, close_end, close_s,
                                                  S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(),
                                                  (const double4*)P0, (const double4*)P1, (const double*)P2, txyz, out);
    else if constexpr (KIND != NEAR_BEM)
        k_p2p<float, KIND><<<grid, 256, 0, st>>>(w, T.begin.as<int>(), T.end.as<int>(), close_begin, close_end, close_s,
                                                 S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(),
                                                 (const float4*)P0, (const float4*)P1, (const float*)P2, txyz, out);
    FMM_HIP(hipGetLastError());
    if (w.desc) add_parts(w, T, out, st);
}
void launch_p2p(bool f64, const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                const int* close_end, const int* close_s, const void* P0, const void* P1, const void* P2,
                const double* txyz, double* Bnear, NearScratch& scratch, hipStream_t st, bool prepared) {
    p2p_launch<NEAR_B>(f64, leaves, nleaves, T, S, close_begin, close_end, close_s, P0, P1, P2, txyz, Bnear, scratch, st,
                       prepared);
}
void prepare_p2p(const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                 const int* close_end, const int* close_s, NearScratch& scratch, hipStream_t st) {
    int grid;
    if (nleaves) start_near<false>(leaves, nleaves, T, S, close_begin, close_end, close_s, scratch, grid, st);
}
void launch_p2p_bem(const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                    const int* close_end, const int* close_s, const void* P0, const void* P1, const void* P2,
                    const double* txyz, double* out, NearScratch& scratch, hipStream_t st) {
    p2p_launch<NEAR_BEM>(true, leaves, nleaves, T, S, close_begin, close_end, close_s, P0, P1, P2, txyz, out, scratch, st);
}
void launch_p2p_A(bool f64, const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                  const int* close_end, const int* close_s, const void* P0, const void* P1, const void* P2,
                  const double* txyz, double* Anear, NearScratch& scratch, hipStream_t st) {
    p2p_launch<NEAR_A>(f64, leaves, nleaves, T, S, close_begin, close_end, close_s, P0, P1, P2, txyz, Anear, scratch, st);
}
void prepare_p2p_queue(const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                       const int* close_end, const int* close_s, NearScratch& scratch, hipStream_t st) {
    if (!nleaves) return;
    make_items<false>(near_work(leaves, nleaves, near_rows(T.num_slots), scratch), T, S, close_begin, close_end, close_s, st);
}
void launch_p2p_queue(const int* leaves, int nleaves, const TreeDev& T, const TreeDev& S, const int* close_begin,
                      const int* close_end, const int* close_s, const void* P0, const void* P1, const void* P2,
                      const double* txyz, double* Bnear, NearScratch& scratch, const int* gemm_queues, int gemm_tiles,
                      int grid, bool beside, hipStream_t st) {
    if (!nleaves) return;
    if (grid < 1) throw Error(1, "near field: empty persistent grid");
    const NearWork w = near_work(leaves, nleaves, near_rows(T.num_slots), scratch);
    (beside ? k_p2p_queue<float, false> : k_p2p_queue_rest<float, false>)<<<grid, 256, 0, st>>>(
        w, gemm_queues, gemm_tiles, T.begin.as<int>(), T.end.as<int>(), close_begin, close_end, close_s,
        S.center.as<double>(), S.begin.as<int>(), S.end.as<int>(), (const float4*)P0, (const float4*)P1,
        (const float*)P2, txyz, Bnear);
    FMM_HIP(hipGetLastError());
}
void finish_p2p_queue(const int* leaves, int nleaves, const TreeDev& T, double* Bnear, NearScratch& scratch,
                      hipStream_t st) {
    if (nleaves) add_parts(near_work(leaves, nleaves, near_rows(T.num_slots), scratch), T, Bnear, st);
}
void launch_p2p_transposed(bool f64, const int* leaves, int nleaves, const TreeDev& S, const TreeDev& T,
                           const int* close_begin, const int* close_end, const int* close_t, const void* P0,
                           const void* P1, const void* P2, const double* sxyz, double* out, NearScratch& scratch,
                           hipStream_t st) {
    if (!nleaves) return;
    int grid;
    const NearWork w = start_near<true>(leaves, nleaves, S, T, close_begin, close_end, close_t, scratch, grid, st);
    if (f64)
        k_p2p_transposed<double><<<grid, 256, 0, st>>>(
            w, S.begin.as<int>(), S.end.as<int>(), S.parent.as<int>(), close_begin, close_end, close_t,
            S.center.as<double>(), T.begin.as<int>(), T.end.as<int>(), (const double4*)P0, (const double4*)P1,
            (const double*)P2, sxyz, out);
    else
        k_p2p_transposed<float><<<grid, 256, 0, st>>>(
            w, S.begin.as<int>(), S.end.as<int>(), S.parent.as<int>(), close_begin, close_end, close_t,
            S.center.as<double>(), T.begin.as<int>(), T.end.as<int>(), (const float4*)P0, (const float4*)P1,
            (const float*)P2, sxyz, out);
    FMM_HIP(hipGetLastError());
    if (w.desc) add_parts(w, S, out, st);
}
void launch_assemble(const int* slots, int n, const double* Bfar, const double* Bnear, double scale, double* B,
                     hipStream_t st) {
    if (n) k_assemble<<<blocks(n), 256, 0, st>>>(slots, n, Bfar, Bnear, scale, B);
}

}  // namespace fmm
