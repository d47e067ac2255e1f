// Class-batched translation GEMMs on MFMA (gfx950).
//
// A "class" is one translation operator T (Lp x Lp, row = output coefficient) shared
// by a list of (source node, destination node) pairs: an M2L offset class, or one M2M /
// L2L orientation of a level.  Column j of a class is component j % 3 of pair j / 3:
// B[:, j] = src_exp[src][comp][:], and T B[:, j] is added to dst_exp[dst][comp][:].  One
// launch covers every 64-column tile of every class (tiles never straddle classes).
// Expansions are node-major [node][3][Lp] so a column is one contiguous vector.
//
// Each workgroup (4 waves) computes the whole Lp-row panel of its 64 columns, so every
// gathered column is read from HBM once; wave w owns the row blocks w, w + 4, ... (RB of them,
// Lp = 64 RB) times the 4 column blocks, as MFMA blocks of 16 x 16.  K is staged through double-buffered LDS with the
// next step's global loads issued before the current step's MFMAs (one barrier per step).
//
// Precisions:
//   F64    : v_mfma_f64_16x16x4f64 (rows permuted so that C register r holds row 4(lane/16) + r);
//   F32    : v_mfma_f32_16x16x4f32 (C register r holds row 4(lane/16) + r), FP32 accumulate;
//   BF16X3 : v_mfma_f32_16x16x32_bf16 on A = Ah + Al (tables split offline from FP64) and
//            B = Bh + Bl (split on load): C += Al Bh + Ah Bl + Ah Bh, FP32 accumulate.
// TRANS applies T^T (the adjoint passes) by reading the operator column-wise.
#include "fmm_gemm.hpp"
#include "fmm_groups.hpp"
#include "fmm_prims.hpp"

namespace fmm {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int BN = 64;

// The operator row that lane li supplies as row li of a 16-row MFMA block.  The FP64 MFMA returns
// rows r, 4 + r, ... in register r of lane group g (row 4r + g), the FP32 one rows 4g + r; with the
// rows of an FP64 block read in the order 4 (li mod 4) + li / 4, register r of group g holds row
// 4g + r too, so a lane writes 32 consecutive bytes and its column's four lanes a 128-byte line
// instead of four 32-byte pieces.
template <class T> __device__ __forceinline__ int mfma_row(int li) {
    return sizeof(T) == 8 ? 4 * (li & 3) + (li >> 2) : li;
}

template <class T> struct Vec4;
template <> struct Vec4<float> {
    typedef float4 t;
    static __device__ __forceinline__ float4 load(const float* p) { return *(const float4*)p; }
    static __device__ __forceinline__ float get(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }
    static __device__ __forceinline__ float4 zero() { return make_float4(0.f, 0.f, 0.f, 0.f); }
};
template <> struct Vec4<double> {
    struct t { double2 a, b; };
    static __device__ __forceinline__ t load(const double* p) { return t{*(const double2*)p, *(const double2*)(p + 2)}; }
    static __device__ __forceinline__ double get(const t& v, int i) { return i == 0 ? v.a.x : i == 1 ? v.a.y : i == 2 ? v.b.x : v.b.y; }
    static __device__ __forceinline__ t zero() { return t{make_double2(0.0, 0.0), make_double2(0.0, 0.0)}; }
};

// ---------------------------------------------------------------- FP64 / FP32
template <class T, int RB, bool TRANS, bool MULTI>
__global__ __launch_bounds__(256) void k_gemm(const T* __restrict__ ops, const GemmTile* __restrict__ tiles,
                                              const int* __restrict__ pair_src, const int* __restrict__ pair_dst,
                                              const T* __restrict__ src_exp, T* __restrict__ dst_exp, int epi,
                                              int nseg, int tri) {
    // LDS row strides: four K-rows are read by the 16-lane groups of a wave at once; strides of
    // 16 (mod 64) words put the four rows on disjoint bank ranges (FP64: 8 doubles = 16 words)
    constexpr int Lp = 64 * RB, BK = 16, PAD = sizeof(T) == 8 ? 8 : 16, SA = Lp + PAD, SB = BN + PAD, NK = Lp / BK;
    const int NKT = MULTI ? nseg * NK : NK;   // single-segment launches keep a compile-time trip count
    typedef Vec4<T> V;
    typedef typename V::t v4;
    typedef typename std::conditional<sizeof(T) == 8, f64x4, f32x4>::type acc_t;
    __shared__ T As[2][BK][SA];
    __shared__ T Bs[2][BK][SB];
    const GemmTile tile = tiles[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // B loader: one column and 4 consecutive k per thread; segment g reads node pair_src + g
    const int bc = tid >> 2, bq = (tid & 3) * 4;
    const T* bptr = nullptr;
    if (bc < tile.ncol) {
        int col = tile.col0 + bc;
        int pair = col / 3, comp = col - 3 * pair;
        bptr = src_exp + ((size_t)pair_src[pair] * 3 + comp) * Lp;
    }
    // A loader: RB quads of 4 per thread.  Non-transposed: (row, 4 consecutive k);
    // transposed: (4 consecutive rows, one k) of T^T = columns of T.  Segment g applies
    // operator tile.op + g.
    v4 ra[RB], rb;
    auto gload = [&](int kt) {
        const int seg = kt / NK, k0 = (kt - seg * NK) * BK;
        const T* A = ops + (size_t)(tile.op + seg) * Lp * Lp;
#pragma unroll
        for (int j = 0; j < RB; j++) {
            int qi = tid + 256 * j;
            if (!TRANS) {
                int row = qi >> 2, kq = (qi & 3) * 4;
                ra[j] = V::load(A + (size_t)row * Lp + k0 + kq);
            } else {
                int k = qi / (Lp / 4), rq = (qi % (Lp / 4)) * 4;
                ra[j] = V::load(A + (size_t)(k0 + k) * Lp + rq);
            }
        }
        if (bptr) rb = V::load(bptr + (size_t)seg * 3 * Lp + k0 + bq);
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int j = 0; j < RB; j++) {
            int qi = tid + 256 * j;
            if (!TRANS) {
                int row = qi >> 2, kq = (qi & 3) * 4;
                for (int i = 0; i < 4; i++) As[buf][kq + i][row] = V::get(ra[j], i);
            } else {
                int k = qi / (Lp / 4), rq = (qi % (Lp / 4)) * 4;
                for (int i = 0; i < 4; i++) As[buf][k][rq + i] = V::get(ra[j], i);
            }
        }
        for (int i = 0; i < 4; i++) Bs[buf][bq + i][bc] = bptr ? V::get(rb, i) : T(0);
    };
    acc_t acc[RB][4];
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = acc_t{0, 0, 0, 0};
    gload(0);
    lstore(0);
    __syncthreads();
    // wave w owns the row blocks w, w + 4, ..., so under a degree-triangular operator every wave
    // skips about as many blocks as the others; per block its lowest and highest degree
    int dlo[RB], dhi[RB];
#pragma unroll
    for (int a = 0; a < RB; a++) {
        const int r0 = 16 * (wave + 4 * a);
        dlo[a] = (int)sqrtf((float)r0);
        dhi[a] = (int)sqrtf((float)(r0 + 15));
    }
    for (int kt = 0; kt < NKT; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < NKT) gload(kt + 1);
        const int k0 = (kt % NK) * BK, klo = (int)sqrtf((float)k0), khi = (int)sqrtf((float)(k0 + BK - 1));
        bool live[RB];
#pragma unroll
        for (int a = 0; a < RB; a++)
            live[a] = tri == TRI_NONE || (tri == TRI_LOWER ? klo <= dhi[a] : khi >= dlo[a]);
#pragma unroll
        for (int ks = 0; ks < BK; ks += 4) {
            T af[RB], bf[4];
            const int kk = ks + (lane >> 4);
#pragma unroll
            for (int b = 0; b < 4; b++) bf[b] = Bs[cur][kk][b * 16 + (lane & 15)];
#pragma unroll
            for (int a = 0; a < RB; a++) {
                if (!live[a]) continue;   // uniform over the wave
                af[a] = As[cur][kk][16 * (wave + 4 * a) + mfma_row<T>(lane & 15)];
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    if constexpr (sizeof(T) == 8)
                        acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(af[a], bf[b], acc[a][b], 0, 0, 0);
                    else
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[a], bf[b], acc[a][b], 0, 0, 0);
                }
            }
        }
        if (kt + 1 < NKT) lstore(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 4; b++) {
        int cl = b * 16 + (lane & 15);
        if (cl >= tile.ncol) continue;
        int col = tile.col0 + cl;
        if (epi == EPI_STORE) {
            T* out = dst_exp + (size_t)col * Lp;
#pragma unroll
            for (int a = 0; a < RB; a++) *(acc_t*)(out + 16 * (wave + 4 * a) + 4 * (lane >> 4)) = acc[a][b];
            continue;
        }
        int pair = col / 3, comp = col - 3 * pair;
        T* dst = dst_exp + ((size_t)pair_dst[pair] * 3 + comp) * Lp;
        if (epi == EPI_ADD) {   // a lane's four rows are consecutive: one vector read-modify-write
#pragma unroll
            for (int a = 0; a < RB; a++) *(acc_t*)(dst + 16 * (wave + 4 * a) + 4 * (lane >> 4)) += acc[a][b];
            continue;
        }
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll   // hardware float atomics on coarse-grained device memory
            for (int r = 0; r < 4; r++) unsafeAtomicAdd(dst + 16 * (wave + 4 * a) + 4 * (lane >> 4) + r, (T)acc[a][b][r]);
    }
}

// ---------------------------------------------------------------- BF16x3
template <int RB, bool TRANS, bool MULTI>
__global__ __launch_bounds__(256) void k_gemm_bf16x3(const __bf16* __restrict__ ops_hi, const __bf16* __restrict__ ops_lo,
                                                     const GemmTile* __restrict__ tiles,
                                                     const int* __restrict__ pair_src, const int* __restrict__ pair_dst,
                                                     const float* __restrict__ src_exp, float* __restrict__ dst_exp,
                                                     int epi, int nseg) {
    constexpr int Lp = 64 * RB, BK = 32, S = BK + 8, NK = Lp / BK;
    const int NKT = MULTI ? nseg * NK : NK;
    // k-contiguous rows: each lane reads its 8 consecutive k as one 16-byte vector
    __shared__ __attribute__((aligned(16))) __bf16 Ah[2][Lp][S];
    __shared__ __attribute__((aligned(16))) __bf16 Al[2][Lp][S];
    __shared__ __attribute__((aligned(16))) __bf16 Bh[2][BN][S];
    __shared__ __attribute__((aligned(16))) __bf16 Bl[2][BN][S];
    const GemmTile tile = tiles[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bc = tid >> 2, bq = (tid & 3) * 8;
    const float* bptr = nullptr;
    if (bc < tile.ncol) {
        int col = tile.col0 + bc;
        int pair = col / 3, comp = col - 3 * pair;
        bptr = src_exp + ((size_t)pair_src[pair] * 3 + comp) * Lp;
    }
    // A loader: RB units of 8 bf16 per thread and part
    bf16x8 rah[RB], ral[RB];
    float4 rb0 = {0, 0, 0, 0}, rb1 = {0, 0, 0, 0};
    auto gload = [&](int kt) {
        const int seg = kt / NK, k0 = (kt - seg * NK) * BK;
        const size_t opoff = (size_t)(tile.op + seg) * Lp * Lp;
        const __bf16* Ahg = ops_hi + opoff;
        const __bf16* Alg = ops_lo + opoff;
#pragma unroll
        for (int j = 0; j < RB; j++) {
            int qi = tid + 256 * j;
            if (!TRANS) {
                int row = qi >> 2, kq = (qi & 3) * 8;
                rah[j] = *(const bf16x8*)(Ahg + (size_t)row * Lp + k0 + kq);
                ral[j] = *(const bf16x8*)(Alg + (size_t)row * Lp + k0 + kq);
            } else {
                int k = qi / (Lp / 8), rq = (qi % (Lp / 8)) * 8;
                rah[j] = *(const bf16x8*)(Ahg + (size_t)(k0 + k) * Lp + rq);
                ral[j] = *(const bf16x8*)(Alg + (size_t)(k0 + k) * Lp + rq);
            }
        }
        if (bptr) {
            const float* bp = bptr + (size_t)seg * 3 * Lp + k0 + bq;
            rb0 = *(const float4*)bp;
            rb1 = *(const float4*)(bp + 4);
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int j = 0; j < RB; j++) {
            int qi = tid + 256 * j;
            if (!TRANS) {
                int row = qi >> 2, kq = (qi & 3) * 8;
                *(bf16x8*)&Ah[buf][row][kq] = rah[j];
                *(bf16x8*)&Al[buf][row][kq] = ral[j];
            } else {
                int k = qi / (Lp / 8), rq = (qi % (Lp / 8)) * 8;
                for (int i = 0; i < 8; i++) {
                    Ah[buf][rq + i][k] = rah[j][i];
                    Al[buf][rq + i][k] = ral[j][i];
                }
            }
        }
        float v[8] = {rb0.x, rb0.y, rb0.z, rb0.w, rb1.x, rb1.y, rb1.z, rb1.w};
        bf16x8 h, l;
        for (int i = 0; i < 8; i++) {
            float x = bptr ? v[i] : 0.0f;
            __bf16 hh = (__bf16)x;
            h[i] = hh;
            l[i] = (__bf16)(x - (float)hh);
        }
        *(bf16x8*)&Bh[buf][bc][bq] = h;
        *(bf16x8*)&Bl[buf][bc][bq] = l;
    };
    f32x4 acc[RB][4];
#pragma unroll
    for (int a = 0; a < RB; a++)
#pragma unroll
        for (int b = 0; b < 4; b++) acc[a][b] = f32x4{0, 0, 0, 0};
    gload(0);
    lstore(0);
    __syncthreads();
    const int wrow = wave * 16 * RB;
    const int kk = 8 * (lane >> 4);
    for (int kt = 0; kt < NKT; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < NKT) gload(kt + 1);
        bf16x8 bh[4], bl[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            bh[b] = *(const bf16x8*)&Bh[cur][b * 16 + (lane & 15)][kk];
            bl[b] = *(const bf16x8*)&Bl[cur][b * 16 + (lane & 15)][kk];
        }
#pragma unroll
        for (int a = 0; a < RB; a++) {
            int r = wrow + a * 16 + (lane & 15);
            bf16x8 ah = *(const bf16x8*)&Ah[cur][r][kk];
            bf16x8 al = *(const bf16x8*)&Al[cur][r][kk];
#pragma unroll
            for (int b = 0; b < 4; b++) {
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[b], acc[a][b], 0, 0, 0);
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[b], acc[a][b], 0, 0, 0);
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[b], acc[a][b], 0, 0, 0);
            }
        }
        if (kt + 1 < NKT) lstore(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 4; b++) {
        int cl = b * 16 + (lane & 15);
        if (cl >= tile.ncol) continue;
        int col = tile.col0 + cl;
        if (epi == EPI_STORE) {
            float* out = dst_exp + (size_t)col * Lp + wrow;
#pragma unroll
            for (int a = 0; a < RB; a++)
                *(float4*)(out + a * 16 + 4 * (lane >> 4)) =
                    make_float4(acc[a][b][0], acc[a][b][1], acc[a][b][2], acc[a][b][3]);
            continue;
        }
        int pair = col / 3, comp = col - 3 * pair;
        float* dst = dst_exp + ((size_t)pair_dst[pair] * 3 + comp) * Lp + wrow;
        if (epi == EPI_ADD) {   // a lane's four rows are consecutive: one 16-byte read-modify-write
#pragma unroll
            for (int a = 0; a < RB; a++) {
                float4* q = (float4*)(dst + a * 16 + 4 * (lane >> 4));
                float4 v = *q;
                v.x += acc[a][b][0];
                v.y += acc[a][b][1];
                v.z += acc[a][b][2];
                v.w += acc[a][b][3];
                *q = v;
            }
            continue;
        }
#pragma unroll
        for (int a = 0; a < RB; a++)
#pragma unroll
            for (int r = 0; r < 4; r++) unsafeAtomicAdd(dst + a * 16 + 4 * (lane >> 4) + r, acc[a][b][r]);
    }
}

// ---------------------------------------------------------------- M2L, rows padded to 16
// The M2L launch with rows and K padded only to R = 16 NB (>= L, <= Lp) instead of Lp: wave w
// owns the 16 columns [16w, 16w + 16) of the 64-column tile and all NB row blocks, so an odd
// block count leaves no wave idle.  Each column is written to the per-pair slab with row
// stride R (rows >= L are zero: the operators are zero there).
// TRANS applies T^T (the adjoint): a thread then loads one k and four consecutive rows of a
// quad, k fastest over the lanes, so that the scattered LDS stores of a wave fall on 64 banks.
// Matrix cores are busy 66-68 % of the time (counters).  Measured: 2.02 million FP64 pairs at p = 12
// 8.2 -> 7.4 ms (128-byte stores 0.55, fragments read block by block 0.25); the transposed product of
// 1.6 million FP32 pairs at p = 14 5.5 ms (7.0 with the whole-panel kernel).  Three workgroups per CU
// instead of two (K steps of 8) or columns loaded 2 to 4 K steps ahead: 7.2 - 8.5 and 5.6 - 6.2 ms.
template <class T, int NB, bool TRANS>
__global__ __launch_bounds__(256) void k_gemm_m2l(const T* __restrict__ ops, const GemmTile* __restrict__ tiles,
                                                  const int* __restrict__ pair_src, const T* __restrict__ src_exp,
                                                  T* __restrict__ slab, int Lp) {
    constexpr int R = 16 * NB, BK = 16, NK = NB;
    // k-contiguous LDS rows: the 16-lane group g of a wave takes k = 4g .. 4g+3 of a K step, one
    // per MFMA (the same order for A and B, so the sum is unchanged), read as one 4-vector
    constexpr int SK = BK + 16 / (int)sizeof(T);   // row stride in elements (pad 16 bytes)
    constexpr int NQ = (NB * 64 + 255) / 256;      // A quads (4 elements) per thread and K step
    typedef Vec4<T> V;
    typedef typename V::t v4;
    typedef typename std::conditional<sizeof(T) == 8, f64x4, f32x4>::type acc_t;
    __shared__ __attribute__((aligned(16))) T As[2][R][SK];
    __shared__ __attribute__((aligned(16))) T Bs[2][BN][SK];
    // workgroups are dealt round-robin to the 8 XCDs: give each XCD a contiguous eighth of the
    // tiles, so the tiles of one class (one operator) share an L2 (a bijection in any case)
    const int nt = gridDim.x, xcd = blockIdx.x & 7, q = nt >> 3, rem = nt & 7;
    const int t = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
    const GemmTile tile = tiles[t];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15;
    const T* A = ops + (size_t)tile.op * Lp * Lp;
    const int bc = tid >> 2, bq = (tid & 3) * 4;
    const T* bptr = nullptr;
    if (bc < tile.ncol) {
        int col = tile.col0 + bc;
        int pair = col / 3, comp = col - 3 * pair;
        bptr = src_exp + ((size_t)pair_src[pair] * 3 + comp) * Lp;
    }
    v4 ra[NQ], rb;
    auto gload = [&](int k0) {
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            int qi = tid + 256 * j;
            if (qi < NB * 64)
                ra[j] = V::load(TRANS ? A + (size_t)(k0 + (qi & 15)) * Lp + (qi >> 4) * 4
                                      : A + (size_t)(qi >> 2) * Lp + k0 + (qi & 3) * 4);
        }
        if (bptr) rb = V::load(bptr + k0 + bq);
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            int qi = tid + 256 * j;
            if (qi >= NB * 64) continue;
            if (TRANS)
#pragma unroll
                for (int i = 0; i < 4; i++) As[buf][(qi >> 4) * 4 + i][qi & 15] = V::get(ra[j], i);
            else
                *(v4*)&As[buf][qi >> 2][(qi & 3) * 4] = ra[j];
        }
        if (bptr) *(v4*)&Bs[buf][bc][bq] = rb;
        else *(v4*)&Bs[buf][bc][bq] = V::zero();
    };
    acc_t acc[NB];
#pragma unroll
    for (int a = 0; a < NB; a++) acc[a] = acc_t{0, 0, 0, 0};
    gload(0);
    lstore(0);
    __syncthreads();
    for (int kt = 0; kt < NK; kt++) {
        const int cur = kt & 1;
        if (kt + 1 < NK) gload((kt + 1) * BK);
        const v4 bf = *(const v4*)&Bs[cur][wave * 16 + li][4 * g];
        // two row blocks at a time: their fragments are read while the previous blocks' MFMAs run, and
        // consecutive MFMAs update different accumulators
#pragma unroll
        for (int a0 = 0; a0 < NB; a0 += 2) {
            v4 af[2];
#pragma unroll
            for (int a = a0; a < a0 + 2 && a < NB; a++)
                af[a - a0] = *(const v4*)&As[cur][a * 16 + mfma_row<T>(li)][4 * g];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int a = a0; a < a0 + 2 && a < NB; a++) {
                    if constexpr (sizeof(T) == 8)
                        acc[a] = __builtin_amdgcn_mfma_f64_16x16x4f64(V::get(af[a - a0], j), V::get(bf, j), acc[a], 0, 0, 0);
                    else
                        acc[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(V::get(af[a - a0], j), V::get(bf, j), acc[a], 0, 0, 0);
                }
        }
        if (kt + 1 < NK) lstore(cur ^ 1);
        __syncthreads();
    }
    // the slab is written once and read once (by the reduction): nontemporal stores keep the
    // operators and gathered multipoles resident in L2 (measured -9 % launch time on the 1M
    // points workload against plain stores)
    const int cl = wave * 16 + li;
    if (cl >= tile.ncol) return;
    T* out = slab + (size_t)(tile.col0 + cl) * R;
#pragma unroll
    for (int a = 0; a < NB; a++) {
        if constexpr (sizeof(T) == 8) {
            __builtin_nontemporal_store(f64x2{acc[a][0], acc[a][1]}, (f64x2*)(out + a * 16 + 4 * g));
            __builtin_nontemporal_store(f64x2{acc[a][2], acc[a][3]}, (f64x2*)(out + a * 16 + 4 * g + 2));
        } else {
            __builtin_nontemporal_store(acc[a], (f32x4*)(out + a * 16 + 4 * g));
        }
    }
}

// ---------------------------------------------------------------- M2L, FP16 split
// The M2L of the F16X3 precision: every product of the FP32 GEMM is replaced by three FP16
// products on v_mfma_f32_16x16x32_f16 (FP32 accumulate), A = Ah + Al and B = Bh + Bl with
// hi and lo in FP16 (22 significant bits together), C = Al Bh + Ah Bl + Ah Bh.  FP16 has a
// narrow range, so both sides are equilibrated by powers of 2 (exact):
//   A_eq = diag(rs) T diag(1/dm)   (operator tables: row scale rs per operator, dm per input
//                                   coefficient; the tables hold A_eq split, rinv = 1 / rs)
//   B_eq = diag(dm) M diag(s)      (multipoles: dm per coefficient, s per column, split once per
//                                   evaluation by k_split_columns into FP16 hi and lo parts)
// so T M = diag(rinv) (A_eq B_eq) diag(1/s).  Rows R = 16 NB >= L, K padded to Kp = 32 NKS >= L
// (zero operator columns and multipole rows beyond L).
//
// A column is a component of one group of far pairs: up to 8 children of one source node that are far
// from one target (fmm_groups.hpp).  A tile runs over the K steps of every child in the union of its
// groups' masks, one operator per child; columns whose group lacks that child take zeros.  Every child
// has scales of its own, so its product is accumulated by itself, scaled back, and added to the group's
// sum in FP32: the roundings are those of one pair, whatever its siblings.  In one accumulator through
// all children, brought to common scales in FP16, the sum took up to 8 times the roundings at its full
// size, and a child far below a sibling lost its bits even where that sibling is no far pair (a leaf of
// 2^20 times the weight: the far field beside it off by 1e-4 of itself).
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
// eight halves on their way from memory to LDS.  As a half vector the compiler takes each register apart
// and together again wherever a load is conditional (300 instructions per K step, more than all others)
typedef int i32x4 __attribute__((ext_vector_type(4)));

// LDS rows of 32 halves without padding, their four 16-byte chunks permuted by the row: chunk q of row r
// lies at q ^ f(r / 4 mod 4), f = 0, 2, 3, 1.  16-byte LDS reads are served in lane groups
// 0-3, 12-15, 20-23, 24-27 and 4-7, 8-11, 16-19, 28-31 (and those + 32): with lane = 16 g + i reading
// chunk g of row i, each group then covers all 64 banks once, and so do the stores of 8 consecutive lanes
// (two whole rows).  Rows padded to 80 bytes conflicted in half of all LDS cycles.
__device__ __forceinline__ int lds_chunk(int q, int row) {
    const int b1 = (row >> 3) & 1, b0 = (row >> 2) & 1;
    return q ^ (2 * (b1 ^ b0) + b1);
}

struct M2LGroupArgs {
    const _Float16 *ops_hi, *ops_lo;
    const float* ops_rinv;
    const GroupTile* tiles;
    const int* cls_ops;
    const int* grp_fc;
    const int* grp_mask;
    const _Float16* src_hl;
    const float* cscale;
    float* slab;
    int ntiles, zero_col;   // the column of zeros
};

// The columns (tid >> 2) + 64 c of a tile that a thread loads, and the operators of its children.
// Columns whose group lacks a child read the column of zeros behind the nodes'.
// SINGLE: every group is one pair, child 0 with the class's one operator.
template <int R, int Kp, bool SINGLE>
struct M2LTile {
    const M2LGroupArgs& A;
    GroupTile tile;
    int col[2], gm[2];   // multipole column of child 0 and child mask of the columns' groups
    __device__ __forceinline__ M2LTile(const M2LGroupArgs& A_, const GroupTile& t, int tid) : A(A_), tile(t) {
#pragma unroll
        for (int c = 0; c < 2; c++) find((tid >> 2) + 64 * c, col[c], gm[c]);
    }
    __device__ __forceinline__ void find(int cl, int& col0, int& mask) const {
        const bool valid = cl < 3 * tile.ng;
        const int g = tile.g0 + (valid ? cl / 3 : 0);
        col0 = 3 * A.grp_fc[g] + cl % 3;
        mask = !valid ? 0 : SINGLE ? 1 : A.grp_mask[g];
    }
    __device__ __forceinline__ size_t op(int o) const {
        return SINGLE ? (size_t)tile.cls : (size_t)A.cls_ops[8 * (size_t)tile.cls + o];
    }
    // the parts of column c of child o, K step by K step hi | lo
    __device__ __forceinline__ const _Float16* column(int c, int o, bool any = true) const {
        return A.src_hl + (size_t)(any && ((gm[c] >> o) & 1) ? col[c] + 3 * o : A.zero_col) * 2 * Kp;
    }
    // what undoes the scale of a column of child o (0 where the group lacks the child: that product is 0)
    __device__ __forceinline__ float column_inv(int col0, int mask, int o) const {
        return (mask >> o) & 1 ? 1.0f / A.cscale[col0 + 3 * o] : 0.0f;
    }
    __device__ __forceinline__ float* slab(int cl) const {   // the block's column of the tile's column cl
        return A.slab + (3 * (size_t)tile.g0 + cl) * R;
    }
};

// What the threads of a workgroup load of the current child of a tile into registers: the operator's rows
// (tid >> 2) + 64 j and the columns, 8 consecutive k each.  Every load is unconditional (rows beyond R
// are clamped and not stored): after a load that may have been skipped the compiler cannot count the loads
// in flight and waits for all of them.
template <int R, int Kp, int NQ, bool SINGLE>
struct M2LTileLoads : M2LTile<R, Kp, SINGLE> {
    int tid, wave, bq, sq;           // wave: uniform; bq, sq: first k of this thread's chunk, its place in LDS
    const _Float16 *ah, *al;         // operator parts (uniform)
    const _Float16* b[2];
    __device__ __forceinline__ M2LTileLoads(const M2LGroupArgs& A_, const GroupTile& t, int tid_)
        : M2LTile<R, Kp, SINGLE>(A_, t, tid_), tid(tid_), wave(__builtin_amdgcn_readfirstlane(tid_ >> 6)),
          bq((tid_ & 3) * 8), sq(8 * lds_chunk(tid_ & 3, tid_ >> 2)) {}
    __device__ __forceinline__ int row(int j) const {
        const int r = (tid >> 2) + 64 * j;
        return 64 * (j + 1) <= R ? r : min(r, R - 1);
    }
    // a wave stages 16 rows at a time: all of them exist or none
    __device__ __forceinline__ bool has_rows(int j) const { return 64 * (j + 1) <= R || 16 * wave + 64 * j < R; }
    __device__ __forceinline__ void open(int o) {
        for (int c = 0; c < 2; c++) b[c] = this->column(c, o) + bq;
        ah = this->A.ops_hi + this->op(o) * R * Kp;
        al = this->A.ops_lo + this->op(o) * R * Kp;
    }
    __device__ __forceinline__ void load(int k0, i32x4 (&ah_)[NQ], i32x4 (&al_)[NQ], i32x4 (&bh)[2],
                                         i32x4 (&bl)[2]) const {
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            const unsigned o = (unsigned)(row(j) * Kp + k0 + bq);
            ah_[j] = *(const i32x4*)(ah + o);
            al_[j] = *(const i32x4*)(al + o);
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {
            bh[c] = *(const i32x4*)(b[c] + 2 * k0);
            bl[c] = *(const i32x4*)(b[c] + 2 * k0 + 32);
        }
    }
    template <int S>
    __device__ __forceinline__ void store(const i32x4 (&ah_)[NQ], const i32x4 (&al_)[NQ], const i32x4 (&bh)[2],
                                          const i32x4 (&bl)[2], _Float16 (*Ah)[S], _Float16 (*Al)[S],
                                          _Float16 (*Bh)[S], _Float16 (*Bl)[S]) const {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            *(i32x4*)&Bh[(tid >> 2) + 64 * c][sq] = bh[c];
            *(i32x4*)&Bl[(tid >> 2) + 64 * c][sq] = bl[c];
        }
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            if (!has_rows(j)) continue;
            *(i32x4*)&Ah[(tid >> 2) + 64 * j][sq] = ah_[j];
            *(i32x4*)&Al[(tid >> 2) + 64 * j][sq] = al_[j];
        }
    }
};

// Single pairs up to p = 13 and above 18, and groups up to p = 7: wave w owns the tile's columns
// [32w, 32w + 32) and all NB row blocks; one LDS buffer refilled from registers whose loads overlap the
// MFMAs, two workgroups per CU.  Single pairs are one operator a tile, so the work before and after its few
// K steps counts: without the class tables 13,693 x 710,485 points (p = 10) 0.65 -> 0.50 ms.
template <int NB, int NKS, bool SINGLE>
__global__ __launch_bounds__(256) void k_gemm_m2l_f16x3(M2LGroupArgs A) {
    constexpr int R = 16 * NB, Kp = 32 * NKS, BK = 32, S = BK;
    constexpr int NQ = (4 * R + 255) / 256;                          // A: 8-half vectors per thread and part
    __shared__ __attribute__((aligned(16))) _Float16 Ah[R][S];
    __shared__ __attribute__((aligned(16))) _Float16 Al[R][S];
    __shared__ __attribute__((aligned(16))) _Float16 Bh[128][S];
    __shared__ __attribute__((aligned(16))) _Float16 Bl[128][S];
    // each XCD works on a contiguous eighth of the tiles (a bijection of the grid)
    const int nt = gridDim.x, xcd = blockIdx.x & 7, q = nt >> 3, rem = nt & 7;
    const int t = xcd * q + min(xcd, rem) + (blockIdx.x >> 3);
    const GroupTile tile = A.tiles[t];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15;
    M2LTileLoads<R, Kp, NQ, SINGLE> ld(A, tile, tid);
    int wcol[2], wgm[2];   // of the columns whose products this lane holds
#pragma unroll
    for (int c = 0; c < 2; c++) ld.find(wave * 32 + 16 * c + li, wcol[c], wgm[c]);
    i32x4 rah[NQ], ral[NQ], rbh[2], rbl[2];
    f32x4 acc[NB][2], sum[SINGLE ? 1 : NB][2];
#pragma unroll
    for (int a = 0; a < NB; a++)
#pragma unroll
        for (int c = 0; c < 2; c++) acc[a][c] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int a = 0; a < (SINGLE ? 1 : NB); a++)
#pragma unroll
        for (int c = 0; c < 2; c++) sum[a][c] = f32x4{0, 0, 0, 0};
    constexpr int EB = NB < 14 ? NB : 7;   // row blocks whose scales are read at a time
    int m = SINGLE ? 1 : tile.mask, o = __builtin_ctz(m);
    ld.open(o);
    ld.load(0, rah, ral, rbh, rbl);
    while (m) {
        m &= m - 1;
        const int cur = o;
        for (int kt = 0; kt < NKS; kt++) {
            ld.template store<S>(rah, ral, rbh, rbl, Ah, Al, Bh, Bl);
            __syncthreads();
            if (kt + 1 < NKS || (!SINGLE && m)) {
                if (!SINGLE && kt + 1 == NKS) {
                    o = __builtin_ctz(m);
                    ld.open(o);
                }
                ld.load(kt + 1 < NKS ? (kt + 1) * BK : 0, rah, ral, rbh, rbl);
            }
            const int kk = 8 * lds_chunk(g, li);
            half8 bh[2], bl[2];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                bh[c] = *(const half8*)&Bh[wave * 32 + 16 * c + li][kk];
                bl[c] = *(const half8*)&Bl[wave * 32 + 16 * c + li][kk];
            }
#pragma unroll
            for (int a = 0; a < NB; a++) {
                const half8 ah = *(const half8*)&Ah[a * 16 + li][kk];
                const half8 al = *(const half8*)&Al[a * 16 + li][kk];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh[c], acc[a][c], 0, 0, 0);
                    acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bl[c], acc[a][c], 0, 0, 0);
                    acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, bh[c], acc[a][c], 0, 0, 0);
                }
            }
            __syncthreads();
        }
        if (SINGLE) break;
        // the child's product, scaled back, into the group's sum
        const float* rv = A.ops_rinv + ld.op(cur) * R;
        float sinv[2];
#pragma unroll
        for (int c = 0; c < 2; c++) sinv[c] = ld.column_inv(wcol[c], wgm[c], cur);
#pragma unroll
        for (int a = 0; a < (SINGLE ? 0 : NB); a++) {
            const float4 r = *(const float4*)(rv + a * 16 + 4 * g);
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const f32x4 x = acc[a][c];
                const float rr[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
                for (int e = 0; e < 4; e++) sum[a][c][e] = __builtin_fmaf(x[e] * rr[e], sinv[c], sum[a][c][e]);
                acc[a][c] = f32x4{0, 0, 0, 0};
            }
        }
    }
    // epilogue: the slab is written once and read once (nontemporal).  A single pair's scales are undone here, all
    // of them read before the first store: a load after a store could alias it, so it stayed there and
    // its wait was one for the store as well, and the pieces of a 128-byte line reached memory one by one
    // (209,062 x 506,545 clustered points, p = 12: 6.9 instead of 5.3 GB written, 3.9 instead of 2.9 ms)
    const float* rv = A.ops_rinv + (size_t)tile.cls * R;
    float sinv[2];
#pragma unroll
    for (int c = 0; c < 2; c++) sinv[c] = SINGLE ? ld.column_inv(wcol[c], wgm[c], 0) : 0.0f;
#pragma unroll
    for (int a0 = 0; a0 < NB; a0 += EB) {
        float4 r[EB];
        if (SINGLE)
#pragma unroll
            for (int a = 0; a < EB; a++)
                if (a0 + a < NB) r[a] = *(const float4*)(rv + (a0 + a) * 16 + 4 * g);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int cl = wave * 32 + 16 * c + li;
            if (cl >= 3 * tile.ng) continue;
            float* out = ld.slab(cl);
#pragma unroll
            for (int a = 0; a < EB; a++) {
                if (a0 + a >= NB) continue;
                f32x4 v = sum[SINGLE ? 0 : a0 + a][c];
                if (SINGLE) {
                    const f32x4 x = acc[a0 + a][c];
                    v = f32x4{x[0] * r[a].x * sinv[c], x[1] * r[a].y * sinv[c], x[2] * r[a].z * sinv[c],
                              x[3] * r[a].w * sinv[c]};
                }
                __builtin_nontemporal_store(v, (f32x4*)(out + (a0 + a) * 16 + 4 * g));
            }
        }
    }
}

// 64 lanes' 16 bytes from memory into 1 KB of LDS, without registers: lane i's to lds + 16 i (lds: uniform).
// Counted by vmcnt like any load: dma_barrier waits for it and then for the workgroup.
__device__ __forceinline__ void dma16(const _Float16* p, _Float16* lds) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                     (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}
// Waits for all but the last LEFT loads of this wave and for its LDS accesses, then for the workgroup.  A
// __syncthreads would wait for all loads.
template <int LEFT> __device__ __forceinline__ void dma_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A workgroup's part of the persistent kernel below: the tile's columns and operators, and the loads into LDS.
// A buffer of rows is [hi | lo][R][32 halves], one of columns [hi | lo][W][32].  CB: 16-column blocks per wave.
template <int NB, int NKS, bool SINGLE, int CB>
struct M2LTileDma : M2LTile<16 * NB, 32 * NKS, SINGLE> {
    static constexpr int R = 16 * NB, Kp = 32 * NKS, BK = 32, S = BK, W = 32 * CB;
    static constexpr int NQ = (4 * R + 255) / 256;   // 16-byte chunks per thread and part of the rows
    static constexpr int NB0 = (NB + 1) / 2, NS = (R + 255) / 256;
    const _Float16 *ah, *al;   // operator parts (uniform)
    const _Float16* b[2];
    int tid, wave, lane, rb0, wc, kk;
    unsigned aq, bq;   // lane's place in LDS row (tid >> 2) is slot tid & 3: the chunk that belongs there
    f32x4 acc[NB0][CB], sum[SINGLE ? 1 : NB0][CB];
    __device__ __forceinline__ M2LTileDma(const M2LGroupArgs& A_, const GroupTile& t, int tid_)
        : M2LTile<R, Kp, SINGLE>(A_, t, tid_), tid(tid_), wave(__builtin_amdgcn_readfirstlane(tid_ >> 6)),
          lane(tid_ & 63), rb0((wave & 1) * NB0), wc(wave >> 1), kk(8 * lds_chunk(lane >> 4, lane & 15)),
          aq((unsigned)((tid_ >> 2) * Kp + 8 * lds_chunk(tid_ & 3, tid_ >> 2))),
          bq((unsigned)(8 * lds_chunk(tid_ & 3, tid_ >> 2))) {
#pragma unroll
        for (int a = 0; a < NB0; a++)
#pragma unroll
            for (int c = 0; c < CB; c++) {
                acc[a][c] = f32x4{0, 0, 0, 0};
                if (!SINGLE) sum[SINGLE ? 0 : a][c] = f32x4{0, 0, 0, 0};
            }
    }
    __device__ __forceinline__ f32x4 result(int a, int c) const { return SINGLE ? acc[a][c] : sum[SINGLE ? 0 : a][c]; }
    __device__ __forceinline__ void rows(int o) {
        ah = this->A.ops_hi + this->op(o) * R * Kp;
        al = this->A.ops_lo + this->op(o) * R * Kp;
    }
    __device__ __forceinline__ void columns(int o, bool any) {
#pragma unroll
        for (int c = 0; c < 2; c++) b[c] = this->column(c, o, any) + bq;
    }
    __device__ __forceinline__ void aload(int kt, _Float16* buf) const {
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            // a wave takes 16 rows at a time: all of them exist or none
            if (64 * (j + 1) > R && 16 * wave + 64 * j >= R) continue;
            dma16(ah + (size_t)64 * j * Kp + kt * BK + aq, buf + (16 * wave + 64 * j) * S);
            dma16(al + (size_t)64 * j * Kp + kt * BK + aq, buf + (R + 16 * wave + 64 * j) * S);
        }
    }
    // BLOADS loads of every wave (dma_barrier counts them): of 96 columns the last two waves load theirs twice
    __device__ __forceinline__ void bload(int kt, _Float16* buf) const {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const bool own = c == 0 || W == 128 || 16 * wave + 64 * c < W;   // uniform over the wave
            const _Float16* p = (own ? b[c] : b[0]) + 2 * kt * BK;
            const int row = 16 * wave + (own ? 64 * c : 0);
            dma16(p, buf + row * S);
            dma16(p + 32, buf + (W + row) * S);
        }
    }
    static constexpr int BLOADS = 4;
    // K step kt of child o; on: the next child (any: there is one).  ac, bc: the operands of this step; an, bn: the
    // rows of the next step and the columns of the one after it, their buffers last read before the previous
    // barrier; sc: the scales of the current child's rows and columns [R + W].  The buffers are different ones,
    // which the compiler has to know (it waits for loads into LDS before every read that could be of them).
    // LAST: the child's last step, after which its product is scaled back and added to the sum.
    template <bool LAST>
    __device__ __forceinline__ void step(int kt, int o, int on, bool any, const _Float16* __restrict__ ac,
                                         const _Float16* __restrict__ bc, _Float16* __restrict__ an,
                                         _Float16* __restrict__ bn, float* __restrict__ sc) {
        if (LAST) rows(on);
        if (kt + 2 == NKS) columns(on, any);
        float sv[NS], cv = 0;   // the child's scales on their way to LDS
        if (!LAST && kt == 0) {
            const float* rv = this->A.ops_rinv + this->op(o) * R;
#pragma unroll
            for (int i = 0; i < NS; i++) sv[i] = rv[min(tid + 256 * i, R - 1)];
            const int c = tid & 3;
            if (c < 2) cv = this->column_inv(c ? this->col[1] : this->col[0], c ? this->gm[1] : this->gm[0], o);
        }
        const int li = lane & 15, g = lane >> 4;
        half8 bh[CB], bl[CB];
#pragma unroll
        for (int c = 0; c < CB; c++) {
            bh[c] = *(const half8*)(bc + (16 * (wc * CB + c) + li) * S + kk);
            bl[c] = *(const half8*)(bc + (W + 16 * (wc * CB + c) + li) * S + kk);
        }
        // row block by row block, each block's operator fragments read during the previous block's MFMAs; the loads
        // for later steps after the first reads, the columns' after the first block's MFMAs; the three products of an
        // accumulator back to back.  The scheduling barriers keep it so: with the loads first and the order of the
        // products the compiler's, the GEMM took 13.7 instead of 12.7 ms (4M shells) and 18.1 instead of 16.7
        // (moving clusters)
        half8 fh[2], fl[2];
#pragma unroll
        for (int a = -1; a < NB0; a++) {
            if (a + 1 < NB0) {
                // the second row half's last block is past NB when NB is odd: it is the block NB - 1 again, in
                // bounds and not stored (a branch around it costs copies of the accumulators, and the other
                // half's waves would be waited for anyway)
                const int row = min(rb0 + a + 1, NB - 1) * 16 + li;
                fh[(a + 1) & 1] = *(const half8*)(ac + row * S + kk);
                fl[(a + 1) & 1] = *(const half8*)(ac + (R + row) * S + kk);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (a < 0) {
                aload(LAST ? 0 : kt + 1, an);
                __builtin_amdgcn_sched_barrier(0);   // dma_barrier counts on the columns' loads being the last
                continue;
            }
            if (a == 1) {
                bload(kt + 2 < NKS ? kt + 2 : kt + 2 - NKS, bn);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int c = 0; c < CB; c++) {
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fl[a & 1], bh[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[a & 1], bl[c], acc[a][c], 0, 0, 0);
                acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[a & 1], bh[c], acc[a][c], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (!LAST && kt == 0) {   // last read at the end of the previous child, a barrier ago
#pragma unroll
            for (int i = 0; i < NS; i++)
                if (tid + 256 * i < R) sc[tid + 256 * i] = sv[i];
            const int cl = (tid >> 2) + 64 * (tid & 3);
            if ((tid & 3) < 2 && (W == 128 || cl < W)) sc[R + cl] = cv;
        }
        if (LAST) {
            float ci[CB];
#pragma unroll
            for (int c = 0; c < CB; c++) ci[c] = sc[R + 16 * (wc * CB + c) + li];
#pragma unroll
            for (int a = 0; a < NB0; a++) {
                const f32x4 r = *(const f32x4*)(sc + min(rb0 + a, NB - 1) * 16 + 4 * g);
#pragma unroll
                for (int c = 0; c < CB; c++) {
                    f32x4 x = acc[a][c];
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        x[e] = SINGLE ? x[e] * r[e] * ci[c] : __builtin_fmaf(x[e] * r[e], ci[c], sum[SINGLE ? 0 : a][c][e]);
                    if (!SINGLE) sum[SINGLE ? 0 : a][c] = x;
                    acc[a][c] = SINGLE ? x : f32x4{0, 0, 0, 0};
                }
            }
        }
    }
};

// The waves on a 2 x 2 grid: wave (wr, wc) owns the row blocks [wr NB0, wr NB0 + NB0) below NB
// (NB0 = ceil(NB / 2)) and half the tile's columns (128, of groups above p = 16 96), so it reads half the
// operator rows and half the columns from LDS per K step (a wave tile of 16 NB0 x 64 instead of 16 NB x 32:
// about a third less LDS traffic per MFMA).  The operands go to LDS without passing registers (dma16), which hold
// two sets of accumulators instead, a child's and the group's: two buffers for the operator rows (shared by
// the tiles of one class, mostly L2 hits), loaded one K step ahead, three for the multipole columns (gathered
// from HBM), loaded two steps ahead, one barrier per K step, all across the boundary from one child to the
// next.  Measured against one set of accumulators fed through registers: GEMM of the 4M shells, p = 16, 12.9 and
// 12.7 ms, of the moving clusters, p = 14, 17.7 and 16.7; of 1M points, p = 8, 12 and 13, 1.04 -> 0.91, 1.97 -> 1.75
// and 6.9 -> 4.2 ms (then the kernel above).  Far field of 999,983 x 750,019 clustered points, p = 14, against
// FP64: 3.8e-7 -> 3.4e-7, as pair by pair; a second set in the kernel above leaves one workgroup per CU (p = 12:
// 3.3 ms).
template <int NB, int NKS, bool SINGLE, int CB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_vgpr(216))) void k_gemm_m2l_f16x3_q(M2LGroupArgs A,
                                                                                                int* __restrict__ xq) {
    typedef M2LTileDma<NB, NKS, SINGLE, CB> Tile;
    static_assert(NKS >= 3, "two steps ahead reach at most the next child; its scales have a step of their own");
    static_assert(Tile::NB0 >= 2, "the columns are loaded behind the first of several row blocks");
    constexpr int R = Tile::R, W = Tile::W, S = Tile::S, RBUF = 2 * R * S, CBUF = 2 * W * S;
    // one variable: with several the compiler labels the accesses by variable, and then a read waits for
    // every load into LDS under way to its variable, that of the other buffers too
    __shared__ struct {
        __attribute__((aligned(16))) _Float16 rows[2 * RBUF], columns[3 * CBUF];
        __attribute__((aligned(16))) float scales[R + W];   // the current child's
        int next_tile;
    } sh;
    // persistent: the grid (a multiple of 8, workgroup b on XCD b mod 8) walks the tiles, each
    // XCD a contiguous eighth of them (one class's operators shared in one L2) taken from that
    // XCD's counter xq[xcd] (zero at launch), so a workgroup that starts late (its CU busy)
    // takes fewer tiles, and then from the other XCDs' eighths; a workgroup starts its next tile
    // while its last stores drain.  The
    // register budget leaves room for one near-field workgroup (k_p2p_queue) per CU.
    const int xcd = blockIdx.x & 7, q = A.ntiles >> 3, rem = A.ntiles & 7, tid = threadIdx.x;
    int from = xcd;   // (thread 0) the eighth this workgroup draws from: its XCD's, then the others'
    for (;;) {
        if (tid == 0) {
            // once its own eighth is done a workgroup takes tiles left in the others (in turn), so
            // XCDs that finish early help the rest; each counter hands out each index once
            int t = -1;
            for (int s = 0; s < 8 && t < 0; s++) {
                const int x = (from + s) & 7, cnt = q + (x < rem ? 1 : 0);
                const int i = atomicAdd(xq + x, 1);
                if (i < cnt) {
                    t = x * q + min(x, rem) + i;
                    from = x;
                }
            }
            sh.next_tile = t;
        }
        __syncthreads();   // also: no load into LDS of the previous tile is under way in any wave
        // read before the K loop's barriers, rewritten only after them; the same in every lane, so what
        // follows from it stays in scalar registers
        const int it = __builtin_amdgcn_readfirstlane(sh.next_tile);
        if (it < 0) break;
        Tile ld(A, A.tiles[it], tid);
        int m = SINGLE ? 1 : ld.tile.mask, o = __builtin_ctz(m);   // m: the children left after the current one o
        m &= m - 1;
        ld.rows(o);
        ld.columns(o, true);
        ld.aload(0, sh.rows);
        ld.bload(0, sh.columns);
        __builtin_amdgcn_sched_barrier(0);
        ld.bload(1, sh.columns + CBUF);
        dma_barrier<Tile::BLOADS>();
        int ab = 0, bb = 0;   // the buffers of the current step
        auto next = [&] {
            dma_barrier<Tile::BLOADS>();   // all but the columns two steps ahead
            ab ^= 1;
            bb = bb == 2 ? 0 : bb + 1;
        };
        for (bool more = true; more;) {
            more = !SINGLE && m != 0;
            // the next child; after the last one the loads ahead are of its first rows and the column of zeros, unused
            const int on = more ? __builtin_ctz(m) : o;
            m &= m - 1;
            for (int kt = 0; kt + 1 < NKS; kt++) {
                ld.template step<false>(kt, o, on, more, sh.rows + ab * RBUF, sh.columns + bb * CBUF,
                                        sh.rows + (ab ^ 1) * RBUF, sh.columns + (bb == 0 ? 2 : bb - 1) * CBUF, sh.scales);
                next();
            }
            ld.template step<true>(NKS - 1, o, on, more, sh.rows + ab * RBUF, sh.columns + bb * CBUF,
                                   sh.rows + (ab ^ 1) * RBUF, sh.columns + (bb == 0 ? 2 : bb - 1) * CBUF, sh.scales);
            next();
            o = on;
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the loads ahead that nothing reads
#pragma unroll
        for (int c = 0; c < CB; c++) {
            const int cl = 16 * (ld.wc * CB + c) + (ld.lane & 15);
            if (cl >= 3 * ld.tile.ng) continue;
            float* out = ld.slab(cl) + 4 * (ld.lane >> 4);
#pragma unroll
            for (int a = 0; a < Tile::NB0; a++) {
                if (ld.rb0 + a >= NB) break;
                __builtin_nontemporal_store(ld.result(a, c), (f32x4*)(out + (ld.rb0 + a) * 16));
            }
        }
    }
}

// per multipole column c (node * 3 + component): the power of 2 s_c that brings
// max_i |M[c][i] dm[i]| into [0.5, 1) (column_scale), and the column's equilibrated values
// x_i = M[c][i] dm[i] s_c split into FP16 hi = fp16(x) and lo = fp16(x - hi) (zero beyond L): the
// B operand of the F16X3 M2L, split once per evaluation instead of once per tile.  Layout
// [column][K step][hi 32 | lo 32]: the hi and lo halves of one K step share a 128-byte line.
// A wave per column, lane j owning the 8 coefficients [8j, 8j + 8) (Kp <= 8 * 64): two 16-byte
// loads, a maximum over the wave, two 16-byte stores; the waves of a capped grid stride over the
// columns and keep their lanes' dm in registers.  Column ncols is written as zeros.
__global__ __launch_bounds__(256) void k_split_columns(const float* __restrict__ M, int ncols, int L, int Lp, int Kp,
                                                       const float* __restrict__ dm, float* __restrict__ scale,
                                                       _Float16* __restrict__ hl,
                                                       const int* __restrict__ skip_first_child,
                                                       const int* __restrict__ skip_npts) {
    const int lane = threadIdx.x & 63, i0 = 8 * lane;
    const bool act = i0 < Kp;   // Kp and Lp are multiples of 8, Kp <= Lp
    const int off = (i0 >> 5) * 64 + (i0 & 31);   // K step i0 / 32, chunk within the step
    float d[8];
#pragma unroll
    for (int e = 0; e < 8; e++) d[e] = act && i0 + e < L ? dm[i0 + e] : 0.0f;
    for (int c = blockIdx.x * 4 + (threadIdx.x >> 6); c <= ncols; c += gridDim.x * 4) {
        if (c == ncols) {   // the column of zeros
            _Float16* z = hl + (size_t)c * 2 * Kp + off;
            if (act) *(half8*)z = *(half8*)(z + 32) = half8{0, 0, 0, 0, 0, 0, 0, 0};
            break;
        }
        if (skip_first_child) {   // leaves with points: split by the P2M already
            const int node = c / 3;
            if (skip_first_child[node] < 0 && skip_npts[node] > 0) continue;
        }
        float x[8];
        float mx = 0.0f;
        if (act) {
            const float4 u = *(const float4*)(M + (size_t)c * Lp + i0);
            const float4 v = *(const float4*)(M + (size_t)c * Lp + i0 + 4);
            x[0] = u.x * d[0]; x[1] = u.y * d[1]; x[2] = u.z * d[2]; x[3] = u.w * d[3];
            x[4] = v.x * d[4]; x[5] = v.y * d[5]; x[6] = v.z * d[6]; x[7] = v.w * d[7];
#pragma unroll
            for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(x[e]));
        }
        for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        const float sc = column_scale(mx);
        if (lane == 0) scale[c] = sc;
        if (act) {
            half8 h, l;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float y = x[e] * sc;
                h[e] = (_Float16)y;
                l[e] = (_Float16)(y - (float)h[e]);
            }
            _Float16* dst = hl + (size_t)c * 2 * Kp + off;
            *(half8*)dst = h;
            *(half8*)(dst + 32) = l;
        }
    }
}

void split_columns(const float* M, int ncols, int L, int Lp, int Kp, const float* dm, float* scale, _Float16* hl,
                   hipStream_t st, const int* skip_first_child, const int* skip_npts) {
    if (ncols <= 0) return;
    if (Kp > 8 * 64 || Kp % 32 || Lp % 8 || Kp > Lp) throw Error(4, "FP16 split: column length out of range");
    if (!skip_first_child != !skip_npts) throw Error(1, "FP16 split: node flags come in pairs");
    const int grid = std::min((ncols + 4) / 4, 8 * num_cus());
    k_split_columns<<<grid, 256, 0, st>>>(M, ncols, L, Lp, Kp, dm, scale, hl, skip_first_child, skip_npts);
    FMM_HIP(hipGetLastError());
}

// groups: k_gemm_m2l_f16x3_q from p = 8 to 18, with 128 columns a tile to p = 16 (two sets of accumulators)
constexpr int M2L_GROUP_DMA_NB = 6, M2L_GROUP_WIDE_NB = 19, M2L_GROUP_MAX_NB = 23;
int m2l_f16_rows(int L) { return 16 * ((L + 15) / 16); }
bool m2l_f16x3_persistent(int L) {
    const int nb = m2l_f16_rows(L) / 16;
    return nb >= 14 && nb <= 23;   // see launch_f16x3
}
// A class of few pairs falls into group classes of fewer still, whose tiles are mostly empty and read more
// operators, and the grouping waits twice for counts.  Whole evaluations, groups / single pairs in ms, of coils
// and clusters of 30,000 to 1,000,000 points: p = 8, 261 pairs a class 2.09 / 2.01, 316 7.5 / 8.8, 441 3.36 / 3.50;
// p = 12, 112 5.3 / 5.0, 261 2.74 / 2.63, 316 12.1 / 14.4; p = 14, 112 6.7 / 6.3, 261 3.31 / 3.23, 316 16.5 / 18.3;
// p = 16, 112 9.1 / 8.5, 261 4.06 / 4.01, 316 22.7 / 24.3, 450 4.97 / 5.14.  In the kernel of the orders up to 7
// (p = 5) 261 1.88 / 1.70, 441 3.1 / 2.9, 427 (8 million pairs) 10.1 / 10.0.  Above p = 18 the LDS
// buffers and two sets of accumulators do not fit.
int m2l_group_min_pairs(int L) {
    const int nb = m2l_f16_rows(L) / 16;
    return nb > M2L_GROUP_MAX_NB ? INT32_MAX : nb >= M2L_GROUP_DMA_NB ? 300 : 1024;
}
// p = 17 and 18: two sets of accumulators of 96 columns fit beside a near-field workgroup, of 128 not at all (1M
// shell points, p = 18: single pairs 21.6 ms, groups 19.2)
int m2l_group_tile(int L) { return m2l_f16_rows(L) <= 16 * M2L_GROUP_WIDE_NB ? GROUP_TILE : 32; }
int m2l_f16_kpad(int L) { return 32 * ((L + 31) / 32); }

// The 2 x 2 kernel for groups (from three K steps on), and for single pairs where the other one's
// accumulators leave one workgroup per CU anyway (R >= 224, p >= 14) and the LDS buffers fit (R <= 368, p <= 18)
template <int NB, int NKS>
static void launch_f16x3(const M2LGroupArgs& A, bool single, int* queues, hipStream_t st) {
    constexpr bool persistent = NB >= 14 && NB <= 23, dma_groups = NB >= M2L_GROUP_DMA_NB && NB <= M2L_GROUP_MAX_NB;
    // from p = 14 one workgroup per CU, 8 per XCD round, with a near-field workgroup beside it; below, two fit
    // on a CU at p = 8 (74 KB of LDS, 224 registers; 0.58 ms, one 0.77: 1M points) and do no harm above
    const int grid = std::min(8 * ((A.ntiles + 7) / 8), (NB >= 14 ? 8 : 16) * ((num_cus() + 7) / 8));
    if constexpr (persistent)
        if (single) {
            k_gemm_m2l_f16x3_q<NB, NKS, true, 4><<<grid, 256, 0, st>>>(A, queues);
            return;
        }
    if constexpr (dma_groups)
        if (!single) {
            k_gemm_m2l_f16x3_q<NB, NKS, false, NB <= M2L_GROUP_WIDE_NB ? 4 : 3><<<grid, 256, 0, st>>>(A, queues);
            return;
        }
    if constexpr (!persistent)
        if (single) {
            k_gemm_m2l_f16x3<NB, NKS, true><<<A.ntiles, 256, 0, st>>>(A);
            return;
        }
    if constexpr (NB < M2L_GROUP_DMA_NB) k_gemm_m2l_f16x3<NB, NKS, false><<<A.ntiles, 256, 0, st>>>(A);
    else throw Error(1, "FP16 M2L: no kernel over groups for this order");
}

void m2l_gemm_f16x3(const _Float16* ops_hi, const _Float16* ops_lo, const float* ops_rinv, const FarGroups& G,
                    const _Float16* src_hl, const float* cscale, int zero_col, float* slab, int L, int* queues,
                    hipStream_t st) {
    if (!G.num_tiles) return;
    const M2LGroupArgs A{ops_hi, ops_lo, ops_rinv, G.tiles.as<GroupTile>(), G.cls_ops.as<int>(), G.fc.as<int>(),
                         G.mask.as<int>(), src_hl, cscale, slab, G.num_tiles, zero_col};
    const int nb = m2l_f16_rows(L) / 16, nks = m2l_f16_kpad(L) / 32;
    // the row and K counts of the orders 1 .. 20
#define FMM_F16(NBV, NKV)                                      \
    if (nb == NBV && nks == NKV) {                             \
        launch_f16x3<NBV, NKV>(A, G.single, queues, st);       \
        FMM_HIP(hipGetLastError());                            \
        return;                                                \
    }
    FMM_F16(1, 1) FMM_F16(2, 1) FMM_F16(3, 2) FMM_F16(4, 2) FMM_F16(6, 3) FMM_F16(7, 4) FMM_F16(8, 4) FMM_F16(9, 5)
    FMM_F16(11, 6) FMM_F16(13, 7) FMM_F16(15, 8) FMM_F16(16, 8) FMM_F16(19, 10) FMM_F16(21, 11) FMM_F16(23, 12)
    FMM_F16(25, 13) FMM_F16(28, 14)
#undef FMM_F16
    throw Error(4, "FP16 M2L: no kernel instance for this order");
}

template <int NB, bool TRANS>
static void launch_m2l_nb(Precision prec, const void* ops, const GemmTile* d_tiles, int ntiles, const int* pair_src,
                          const void* src_exp, void* slab, int Lp, hipStream_t st) {
    if (prec == Precision::F64)
        k_gemm_m2l<double, NB, TRANS><<<ntiles, 256, 0, st>>>((const double*)ops, d_tiles, pair_src, (const double*)src_exp,
                                                       (double*)slab, Lp);
    else
        k_gemm_m2l<float, NB, TRANS><<<ntiles, 256, 0, st>>>((const float*)ops, d_tiles, pair_src, (const float*)src_exp,
                                                      (float*)slab, Lp);
    FMM_HIP(hipGetLastError());
}

int m2l_slab_rows(Precision prec, int L, int Lp) {
    if (prec == Precision::BF16X3) return Lp;
    if (prec == Precision::F16X3) return m2l_f16_rows(L);
    int nb = (L + 15) / 16;
    switch (nb) {
        case 1: case 2: case 3: case 4: case 6: case 7: case 8: case 9: case 11: case 13: case 15: case 16: case 19:
        case 21: case 23: case 25: case 28:
            return 16 * nb;
        default:
            return Lp;
    }
}

template <bool TRANS>
static void m2l_gemm_go(Precision prec, const void* ops, const void* ops_lo, const GemmTile* d_tiles, int ntiles,
                        const int* pair_src, const void* src_exp, void* slab, int L, int Lp, hipStream_t st) {
    if (ntiles == 0) return;
    const int R = m2l_slab_rows(prec, L, Lp);
    if (R == Lp) {   // the whole-panel kernel (BF16x3, or an L that fills whole panels)
        class_gemm(prec, ops, ops_lo, d_tiles, ntiles, pair_src, nullptr, src_exp, slab, Lp, EPI_STORE, st, TRANS);
        return;
    }
#define FMM_NB(N) \
    case N: launch_m2l_nb<N, TRANS>(prec, ops, d_tiles, ntiles, pair_src, src_exp, slab, Lp, st); break;
    switch (R / 16) {
        FMM_NB(1) FMM_NB(2) FMM_NB(3) FMM_NB(4) FMM_NB(6) FMM_NB(7) FMM_NB(8) FMM_NB(9) FMM_NB(11) FMM_NB(13)
        FMM_NB(15) FMM_NB(16) FMM_NB(19) FMM_NB(21) FMM_NB(23) FMM_NB(25) FMM_NB(28)
        default: throw Error(4, "no padded-row M2L kernel for this order");
    }
#undef FMM_NB
}

void m2l_gemm(Precision prec, const void* ops, const void* ops_lo, const GemmTile* d_tiles, int ntiles,
              const int* pair_src, const void* src_exp, void* slab, int L, int Lp, hipStream_t st, bool transpose) {
    if (transpose) m2l_gemm_go<true>(prec, ops, ops_lo, d_tiles, ntiles, pair_src, src_exp, slab, L, Lp, st);
    else m2l_gemm_go<false>(prec, ops, ops_lo, d_tiles, ntiles, pair_src, src_exp, slab, L, Lp, st);
}

template <int RB, bool TR, bool MU>
static void launch_rb(Precision prec, const void* ops, const void* ops_lo, const GemmTile* d_tiles, int ntiles,
                      const int* pair_src, const int* pair_dst, const void* src_exp, void* dst_exp, int epi,
                      int nseg, int tri, hipStream_t st) {
    if (prec == Precision::F64)
        k_gemm<double, RB, TR, MU><<<ntiles, 256, 0, st>>>((const double*)ops, d_tiles, pair_src, pair_dst,
                                                          (const double*)src_exp, (double*)dst_exp, epi, nseg, tri);
    else if (prec == Precision::F32)
        k_gemm<float, RB, TR, MU><<<ntiles, 256, 0, st>>>((const float*)ops, d_tiles, pair_src, pair_dst,
                                                         (const float*)src_exp, (float*)dst_exp, epi, nseg, tri);
    else
        k_gemm_bf16x3<RB, TR, MU><<<ntiles, 256, 0, st>>>((const __bf16*)ops, (const __bf16*)ops_lo, d_tiles, pair_src,
                                                         pair_dst, (const float*)src_exp, (float*)dst_exp, epi, nseg);
    FMM_HIP(hipGetLastError());
}

template <bool TR>
static void launch(int RB, Precision prec, const void* ops, const void* ops_lo, const GemmTile* d_tiles, int ntiles,
                   const int* pair_src, const int* pair_dst, const void* src_exp, void* dst_exp, int epi, int nseg,
                   int tri, hipStream_t st) {
#define FMM_RB(R)                                                                                             \
    case R:                                                                                                   \
        if (nseg > 1)                                                                                         \
            launch_rb<R, TR, true>(prec, ops, ops_lo, d_tiles, ntiles, pair_src, pair_dst, src_exp, dst_exp, epi, \
                                   nseg, tri, st);                                                            \
        else                                                                                                  \
            launch_rb<R, TR, false>(prec, ops, ops_lo, d_tiles, ntiles, pair_src, pair_dst, src_exp, dst_exp, epi, \
                                    1, tri, st);                                                              \
        break;
    switch (RB) {
        FMM_RB(1) FMM_RB(2) FMM_RB(3) FMM_RB(4) FMM_RB(5) FMM_RB(6) FMM_RB(7)
        default: throw Error(4, "padded expansion length above 448 (order > 20)");
    }
#undef FMM_RB
}

void class_gemm(Precision prec, const void* ops, const void* ops_lo, const GemmTile* d_tiles, int ntiles,
                const int* pair_src, const int* pair_dst, const void* src_exp, void* dst_exp, int Lp, int epilogue,
                hipStream_t st, bool transpose, int nseg, int tri) {
    if (ntiles == 0) return;
    if (tri < TRI_NONE || tri > TRI_UPPER) throw Error(1, "unknown operator structure");
    if (Lp % 64 != 0) throw Error(1, "padded expansion length must be a multiple of 64");
    int RB = Lp / 64;
    if (epilogue < EPI_ADD || epilogue > EPI_STORE) throw Error(1, "unknown GEMM epilogue");
    if (nseg < 1) throw Error(1, "a GEMM tile needs at least one segment");
    if (transpose)
        launch<true>(RB, prec, ops, ops_lo, d_tiles, ntiles, pair_src, pair_dst, src_exp, dst_exp, epilogue, nseg, tri,
                     st);
    else
        launch<false>(RB, prec, ops, ops_lo, d_tiles, ntiles, pair_src, pair_dst, src_exp, dst_exp, epilogue, nseg, tri,
                      st);
}

// host-side tiling of class column ranges: class c owns pairs [begin[c], begin[c+1])
void plan_tiles(const std::vector<int>& class_begin, const std::vector<int>& class_op, std::vector<GemmTile>& tiles,
                int width) {
    tiles.clear();
    int nc = (int)class_begin.size() - 1;
    for (int c = 0; c < nc; c++) {
        int c0 = 3 * class_begin[c], c1 = 3 * class_begin[c + 1];
        for (int j = c0; j < c1; j += width) tiles.push_back(GemmTile{class_op[c], j, std::min(width, c1 - j)});
    }
}

// ---------------------------------------------------------------- per-node reduction of pair slabs
__global__ void k_iota(int* v, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) v[i] = i;
}
__global__ void k_zero_ranges(int* b, int* e, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = e[i] = 0;
}
__global__ void k_key_ranges(const uint32_t* __restrict__ sk, int n, int* __restrict__ b, int* __restrict__ e) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t k = sk[i];
    if (i == 0 || sk[i - 1] != k) b[k] = i;
    if (i == n - 1 || sk[i + 1] != k) e[k] = i + 1;
}

__global__ void k_segment_counts(const int* __restrict__ b, const int* __restrict__ e, int n, uint32_t* __restrict__ cnt) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) cnt[v] = (uint32_t)(e[v] - b[v] + PAIR_SEGMENT - 1) / PAIR_SEGMENT;
    else if (v == n) cnt[v] = 0;
}
__global__ void k_segment_nodes(const uint32_t* __restrict__ off, int n, int* __restrict__ seg_node) {
    int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    for (uint32_t s = off[v]; s < off[v + 1]; s++) seg_node[s] = v;
}

static int key_bits(int nnodes) {
    int b = 1;
    while (b < 32 && (1u << b) < (unsigned)nnodes) b++;
    return b;
}

void index_sorted_pairs(const int* key, int npairs, int nnodes, PairIndex& ix, hipStream_t st) {
    ix.npairs = npairs;
    ix.nnodes = nnodes;
    int* b = ix.begin.get<int>(std::max(nnodes, 1));
    int* e = ix.end.get<int>(std::max(nnodes, 1));
    if (nnodes) k_zero_ranges<<<blocks(nnodes), 256, 0, st>>>(b, e, nnodes);
    if (!npairs) return;
    k_key_ranges<<<blocks(npairs), 256, 0, st>>>((const uint32_t*)key, npairs, b, e);
    // segments of at most PAIR_SEGMENT pairs per node, numbered node by node
    uint32_t* cnt = ix.seg_count.get<uint32_t>(nnodes + 1);
    uint32_t* off = ix.seg_off.get<uint32_t>(nnodes + 1);
    k_segment_counts<<<blocks(nnodes + 1), 256, 0, st>>>(b, e, nnodes, cnt);
    exclusive_scan_u32(cnt, off, nnodes + 1, ix.tmp, st);
    ix.max_segments = npairs / PAIR_SEGMENT + std::min(npairs, nnodes);
    k_segment_nodes<<<blocks(nnodes), 256, 0, st>>>(off, nnodes, ix.seg_node.get<int>(ix.max_segments));
    FMM_HIP(hipGetLastError());
}

void build_pair_index(const int* key, int npairs, int nnodes, PairIndex& ix, hipStream_t st) {
    uint32_t* ks = nullptr;
    if (npairs) {
        int* io = ix.iota.get<int>(npairs);
        k_iota<<<blocks(npairs), 256, 0, st>>>(io, npairs);
        ks = ix.keys_sorted.get<uint32_t>(npairs);
        // stable radix sort: pairs of one node stay in ascending pair order
        sort_pairs_u32((const uint32_t*)key, ks, io, ix.order.get<int>(npairs), npairs, key_bits(nnodes), ix.tmp, st);
    }
    index_sorted_pairs((const int*)ks, npairs, nnodes, ix, st);
}

// Two passes, so that nodes with hundreds of pairs do not serialise the launch: (1) one wave
// per segment (at most PAIR_SEGMENT consecutive pairs of one node) sums its pairs' slab blocks
// in ascending pair order into a partial block; (2) one wave per node sums its segments'
// partials, in segment order, and writes the node's expansion.  The order of every sum is fixed
// by the pair numbering alone (deterministic).  A pair's slab block is nv = 3 vr 16-byte vectors (vr per
// component: the first R of each component's Lp coefficients); lane l owns the vectors
// l + 64 r, r < NR = ceil(nv / 64); pass (1) keeps the loads of U pairs in flight.
__device__ __forceinline__ float4 zero_vec(float4) { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ double2 zero_vec(double2) { return make_double2(0.0, 0.0); }
// streaming loads of the slab (read once)
__device__ __forceinline__ float4 load_stream(const float4* p) {
    f32x4 v = __builtin_nontemporal_load((const f32x4*)p);
    return make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ double2 load_stream(const double2* p) {
    f64x2 v = __builtin_nontemporal_load((const f64x2*)p);
    return make_double2(v[0], v[1]);
}

template <class V, int NR>
__global__ __launch_bounds__(256) void k_reduce_segments(const uint32_t* __restrict__ seg_off,
                                                         const int* __restrict__ seg_node, const int* __restrict__ begin,
                                                         const int* __restrict__ end, const int* __restrict__ order,
                                                         const V* __restrict__ slab, int nnodes, int nv,
                                                         V* __restrict__ partial) {
    constexpr int U = NR <= 4 ? 4 : NR <= 8 ? 2 : 1;   // 8 to 16 vectors in flight per lane
    const int sg = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (sg >= (int)seg_off[nnodes]) return;
    const int v = seg_node[sg];
    const int k0 = begin[v] + (sg - (int)seg_off[v]) * PAIR_SEGMENT, k1 = min(k0 + PAIR_SEGMENT, end[v]);
    V acc[NR];
#pragma unroll
    for (int r = 0; r < NR; r++) acc[r] = zero_vec(V());
    int k = k0;
    for (; k + U <= k1; k += U) {
        V x[U][NR];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const V* src = slab + (size_t)order[k + u] * nv + lane;
#pragma unroll
            for (int r = 0; r < NR; r++)
                if (lane + 64 * r < nv) x[u][r] = load_stream(src + 64 * r);
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int r = 0; r < NR; r++)
                if (lane + 64 * r < nv) acc[r] = acc[r] + x[u][r];
    }
    for (; k < k1; k++) {
        const V* src = slab + (size_t)order[k] * nv + lane;
#pragma unroll
        for (int r = 0; r < NR; r++)
            if (lane + 64 * r < nv) acc[r] = acc[r] + load_stream(src + 64 * r);
    }
    V* o = partial + (size_t)sg * nv + lane;
#pragma unroll
    for (int r = 0; r < NR; r++)
        if (lane + 64 * r < nv) o[64 * r] = acc[r];
}

template <class V, int NR>
__global__ __launch_bounds__(256) void k_reduce_nodes(const uint32_t* __restrict__ seg_off, const V* __restrict__ partial,
                                                      int nnodes, int vr, int vl, V* __restrict__ out) {
    const int v = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (v >= nnodes) return;
    const int s0 = (int)seg_off[v], s1 = (int)seg_off[v + 1];
    const int nv = 3 * vr;
    V* o = out + (size_t)v * 3 * vl;
    // the node's expansion is written whole (nothing clears it beforehand): the padding vectors
    // vr .. vl - 1 of each component, and all of a node without far pairs, are zero
    for (int i = lane; i < 3 * vl; i += 64) {
        const int c = i / vl;
        if (s0 == s1 || i - c * vl >= vr) o[i] = zero_vec(V());
    }
    if (s0 == s1) return;
    // the loads of four segments are issued together; the adds keep the segment order
#pragma unroll
    for (int r = 0; r < NR; r++) {
        const int i = lane + 64 * r;
        if (i >= nv) continue;
        const int c = i / vr, q = c * vl + (i - c * vr);
        V acc = zero_vec(V());
        const V* pp = partial + (size_t)s0 * nv + i;
        int sg = s0;
        for (; sg + 4 <= s1; sg += 4, pp += 4 * (size_t)nv) {
            const V x0 = pp[0], x1 = pp[nv], x2 = pp[2 * (size_t)nv], x3 = pp[3 * (size_t)nv];
            acc = acc + x0;
            acc = acc + x1;
            acc = acc + x2;
            acc = acc + x3;
        }
        for (; sg < s1; sg++, pp += nv) acc = acc + pp[0];
        o[q] = acc;
    }
}

template <class V>
static void launch_reduce(PairIndex& ix, const void* slab, int vr, int vl, void* out, hipStream_t st) {
    const int nv = 3 * vr, nr = (nv + 63) / 64;
    const uint32_t* off = ix.seg_off.as<uint32_t>();
    const int* sn = ix.seg_node.as<int>();
    V* part = (V*)ix.partial.reserve((size_t)std::max(ix.max_segments, 1) * nv * sizeof(V));
    const int g1 = (std::max(ix.max_segments, 1) + 3) / 4, g2 = (ix.nnodes + 3) / 4;
    const int *b = ix.begin.as<int>(), *e = ix.end.as<int>(), *o = ix.order.as<int>();
#define FMM_NR(N)                                                                                            \
    case N:                                                                                                 \
        k_reduce_segments<V, N><<<g1, 256, 0, st>>>(off, sn, b, e, o, (const V*)slab, ix.nnodes, nv, part); \
        k_reduce_nodes<V, N><<<g2, 256, 0, st>>>(off, part, ix.nnodes, vr, vl, (V*)out);                   \
        break;
    switch (nr) {
        FMM_NR(1) FMM_NR(2) FMM_NR(3) FMM_NR(4) FMM_NR(5) FMM_NR(6) FMM_NR(7) FMM_NR(8) FMM_NR(9) FMM_NR(10)
        FMM_NR(11) FMM_NR(12) FMM_NR(13) FMM_NR(14) FMM_NR(15) FMM_NR(16)
        default: throw Error(4, "slab rows too long for the pair reduction");
    }
#undef FMM_NR
    FMM_HIP(hipGetLastError());
}

void reduce_pairs(bool f64, PairIndex& ix, const void* slab, int R, int Lp, void* out, hipStream_t st) {
    if (!ix.npairs || !ix.nnodes) return;
    if (f64) launch_reduce<double2>(ix, slab, R / 2, Lp / 2, out, st);
    else launch_reduce<float4>(ix, slab, R / 4, Lp / 4, out, st);
}

}  // namespace fmm
