// fp_lu_nopiv.hip -- LU of a randomized matrix without pivoting: FP32 for the
// mixed-precision refinement (FP_SOLVER_LU32_IR, the batch, the coarse space), FP64
// for FP_SOLVER_LU.
//
// Neither solver rests on the factors alone: residuals of FP64 (of twice FP64 for
// the FP64 factors) decide the result, and what does not converge is factored with
// pivoting.  Partial pivoting is what makes the blocked LU latency-bound at the
// sizes of a wing (4k-12k unknowns): every 32-column sub-panel runs a tournament of
// pivot searches.  A random butterfly transformation (RBT, Parker 1995; Baboulin,
// Dongarra, Herrmann, Tomov 2013) A_r = U^T A V with two depth-2 recursive
// butterflies U, V makes pivoting unnecessary with probability close to one, and
// the LU of A_r is then a plain blocked right-looking factorisation:
//
//   per 256-column outer block:
//     k_lu_first   the first outer block's first 64 x 64 diagonal block, with the
//                  explicit inverses of L11 and U11;
//     k_lu_update  the other outer blocks: their columns' share of the previous
//                  block's rank-256 update, and their first diagonal block;
//     k_lu_step    (four times) L21 = A21 U11^-1 and the update of the outer
//                  block's columns, one workgroup per 64 rows; the first of them
//                  factors the next diagonal block; the launch also carries tiles
//                  of the previous block's update;
//     k_lu_urow    the U rows, inside the outer block and right of it (blocked
//                  substitution);
//     fp_gemm_sub  the part of the rank-256 update that no launch carries.
//
// A x = b becomes  A_r y = U^T b,  x = V y.  A depth-2 butterfly couples only
// the four indices {p, p + m, p + 2m, p + 3m} (m = n4 / 4, n4 = n rounded up
// to a multiple of 4, the pad being a diagonal), so U^T A V is one pass of
// 4 x 4 . 4 x 4 . 4 x 4 products over the (p, q) orbit blocks, and the vector
// transforms are 4 x 4 products per orbit.  A zero or non-finite pivot is
// reported through `info` and the caller falls back to the pivoted LU.
#include "fp_internal.h"
#include "fp_elements.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

namespace {

constexpr int NPB = 64;          // block of the no-pivot LU
constexpr int NIN = 4;           // blocks per outer block
constexpr int NOB = NIN * NPB;   // outer block: columns per trailing update
constexpr int UW = 32;           // columns per workgroup of the U rows
constexpr int LT = 512;          // threads: two waves a SIMD, one's LDS reads behind the other's products
constexpr int TBIG = 512;        // rows of the diagonal-block inverses the triangular solves use

__device__ __forceinline__ float bcast(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ double bcast(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Compile-time loop: f(cint<I>{}) for I = B, ..., E - 1, so that every register-array index is a constant.
template <int V> struct cint {
    static constexpr int v = V;
};
template <int B, int E, typename F> __device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (B < E) {
        f(cint<B>{});
        static_for<B + 1, E>(f);
    }
}

// Per type: LDS row strides of left (LDA) and right (LDB, LDX) operands of the products, chosen so
// that the 64 lanes of a fragment read fall on different banks (left: 16 rows x 4 columns; right:
// 4 rows x 16 columns in FP32, 4 x 4 in FP64).
template <typename T> struct Lu;
template <> struct Lu<float> {
    static constexpr int LDA = 68, LDB = 80, LDX = 48, V = 4;
    typedef float v4 __attribute__((ext_vector_type(4)));
    typedef float vec __attribute__((ext_vector_type(4)));
    // accumulator element e of a 16 x 16 tile
    static __device__ __forceinline__ int row(int lane, int e) { return 4 * (lane >> 4) + e; }
    static __device__ __forceinline__ int col(int lane, int) { return lane & 15; }
    // reciprocal refined once, quotient corrected once (the IEEE sequence switches the denormal mode and
    // is twice as long; the chain of 64 pivots waits for it)
    static __device__ __forceinline__ float div(float a, float b)
    {
        float r = __builtin_amdgcn_rcpf(b);
        r = fmaf(r, fmaf(-b, r, 1.f), r);
        const float q = a * r;
        return fmaf(fmaf(-b, q, a), r, q);
    }
    static __device__ __forceinline__ bool bad(float p) { return !(fabsf(p) > 1e-37f) || !(fabsf(p) <= 1e37f); }
};
template <> struct Lu<double> {
    static constexpr int LDA = 68, LDB = 68, LDX = 36, V = 2;
    typedef double v4 __attribute__((ext_vector_type(4)));
    typedef double vec __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ int row(int lane, int) { return 4 * ((lane >> 2) & 3) + (lane >> 4); }
    static __device__ __forceinline__ int col(int lane, int e) { return 4 * e + (lane & 3); }
    // quotient with one residual correction (rounding to within an ulp)
    static __device__ __forceinline__ double div(double a, double b)
    {
        const double r = fp_recip_nb(b), q = a * r;
        return fma(fma(-b, q, a), r, q);
    }
    static __device__ __forceinline__ bool bad(double p) { return !(fabs(p) > 1e-290) || !(fabs(p) <= 1e290); }
};

// acc += P Q for 16 rows of P (16 x K) and NT 16-column tiles of Q (K x 16 NT), both in LDS.
// FP32: v_mfma_f32_16x16x4.  FP64: v_mfma_f64_4x4x4_4b, whose four blocks take 16 rows of P and
// the same four columns of Q (the 16x16x4 form issues at half its rate).
template <typename T, int NT>
__device__ __forceinline__ void mma(const T *P, int ldp, const T *Q, int ldq, int K, int lane,
                                    typename Lu<T>::v4 (&acc)[NT])
{
    const T *pp = P + (lane & 15) * ldp + (lane >> 4);
#pragma unroll 4
    for (int ks = 0; ks < K; ks += 4) {
        const T pa = pp[ks];
        if constexpr (sizeof(T) == 4) {
            const T *q = Q + (ks + (lane >> 4)) * ldq + (lane & 15);
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(pa, q[16 * t], acc[t], 0, 0, 0);
        } else {
            const T *q = Q + (ks + (lane >> 4)) * ldq + (lane & 3);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    acc[t][b] = __builtin_amdgcn_mfma_f64_4x4x4f64(pa, q[16 * t + 4 * b], acc[t][b], 0, 0, 0);
        }
    }
}

template <typename T, int NT> __device__ __forceinline__ void zero(typename Lu<T>::v4 (&acc)[NT])
{
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = typename Lu<T>::v4{0, 0, 0, 0};
}

// A 64 x W tile through registers, 16 bytes of a row per thread at a time.
// Entries outside rows < tr, cols < tc are zero; 16-byte accesses where the row piece is inside.
template <typename T, int W> struct Tile {
    static constexpr int V = Lu<T>::V, PER_ROW = W / V, STEP = LT / PER_ROW, N = NPB / STEP;
    typedef typename Lu<T>::vec vec;
    vec v[N];
    __device__ __forceinline__ void load(const T *p, int64_t ld, int tr, int tc, int tid)
    {
        const int c = (tid % PER_ROW) * V, r0 = tid / PER_ROW;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int r = r0 + q * STEP;
            if (r < tr && c + V <= tc) {
                v[q] = *reinterpret_cast<const vec *>(p + (int64_t)r * ld + c);
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) v[q][e] = r < tr && c + e < tc ? p[(int64_t)r * ld + c + e] : T(0);
            }
        }
    }
    __device__ __forceinline__ void put(T *s, int lds, int tid) const
    {
        const int c = (tid % PER_ROW) * V, r0 = tid / PER_ROW;
#pragma unroll
        for (int q = 0; q < N; ++q) *reinterpret_cast<vec *>(s + (r0 + q * STEP) * lds + c) = v[q];
    }
    // an LDS tile to memory (rows < tr, cols < tc), times sign
    static __device__ __forceinline__ void store(const T *s, int lds, T *p, int64_t ld, int tr, int tc, T sign, int tid)
    {
        const int c = (tid % PER_ROW) * V, r0 = tid / PER_ROW;
#pragma unroll
        for (int q = 0; q < N; ++q) {
            const int r = r0 + q * STEP;
            vec w = *reinterpret_cast<const vec *>(s + r * lds + c);
            w = w * sign;
            if (r < tr && c + V <= tc) {
                *reinterpret_cast<vec *>(p + (int64_t)r * ld + c) = w;
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e)
                    if (r < tr && c + e < tc) p[(int64_t)r * ld + c + e] = w[e];
            }
        }
    }
};

// The 64 x 64 product of a step: wave w takes rows 16 (w % 4) and columns 32 (w / 4).
template <typename T> __device__ __forceinline__ void mma64(const T *P, const T *Q, int lane, int wave, typename Lu<T>::v4 (&acc)[2])
{
    zero<T, 2>(acc);
    mma<T, 2>(P + 16 * (wave & 3) * Lu<T>::LDA, Lu<T>::LDA, Q + 32 * (wave >> 2), Lu<T>::LDB, NPB, lane, acc);
}
template <typename T> __device__ __forceinline__ int arow(int lane, int wave, int e) { return 16 * (wave & 3) + Lu<T>::row(lane, e); }
template <typename T> __device__ __forceinline__ int acol(int lane, int wave, int q, int e)
{
    return 32 * (wave >> 2) + 16 * q + Lu<T>::col(lane, e);
}

// LDS of the step kernels: three 64 x 64 tiles and two 32 x 32 staging tiles
template <typename T> struct StepLds {
    T P[NPB * Lu<T>::LDA];   // left operand, then L11^-1
    T Q[NPB * Lu<T>::LDB];   // right operand, then U11^-1
    T D[NPB * Lu<T>::LDA];   // the diagonal block
    T tmp[2 * 32 * 36];
};

// Substitution of 16 values per lane with a 16 x 16 triangle in LDS (row stride LDA): forward with the unit
// lower one, or (UP) backward with the upper one and the reciprocals rd of its diagonal, one per lane.
// Column by column: the updates by one unknown are independent of each other, and the next column is read
// meanwhile (all lanes the same word; the barrier keeps the compiler from reading all 120 ahead, which
// spills in FP64).
template <typename T, bool UP> __device__ __forceinline__ void subst16(T (&x)[16], const T *t, T rd)
{
    constexpr int LDA = Lu<T>::LDA;
    T l[2][16];
#pragma unroll
    for (int i = 1; i < 16; ++i) l[0][i] = UP ? t[(15 - i) * LDA + 15] : t[i * LDA];
    static_for<0, 16>([&](auto Q) {
        constexpr int q = decltype(Q)::v, xq = UP ? 15 - q : q;
#pragma unroll
        for (int i = q + 2; i < 16; ++i)
            l[(q + 1) & 1][i] = UP ? t[(15 - i) * LDA + 14 - q] : t[i * LDA + q + 1];
        if (UP) x[xq] *= bcast(rd, xq);
#pragma unroll
        for (int i = q + 1; i < 16; ++i) {
            const int xi = UP ? 15 - i : i;
            x[xi] = fma(-l[q & 1][i], x[xq], x[xi]);
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}

// LU without pivoting of the 64 x 64 block D in LDS, in place, and the explicit inverses Li = L11^-1
// (unit lower) and Ui = U11^-1, by 512 threads.  Four sub-panels of 16 columns: wave 0 factors the
// sub-panel with one row per lane in registers (row j broadcast by v_readlane, 120 broadcast-and-FMA
// steps instead of the 2,016 of the whole block at once), a lane per column substitutes the 16 rows
// right of it, and the waves update the rest with 16 x 16 MFMA tiles.  The inverses grow the same
// way, 16 -> 32 -> 64: X21 = -X22 (L21 X11), X12 = -X11 (U12 X22).  The chain of 64 pivots with
// their divisions bounds it.  Returns (wave 0) whether a pivot was zero or not finite.
template <typename T>
__device__ __forceinline__ bool lu_diag64(StepLds<T> &s, int tid)
{
    constexpr int LDA = Lu<T>::LDA, LDB = Lu<T>::LDB, LDT = 36;
    typedef typename Lu<T>::v4 v4;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    T *D = s.D, *Li = s.P, *Ui = s.Q;
    for (int e = tid; e < NPB * NPB; e += LT) {
        Li[(e >> 6) * LDA + (e & 63)] = T(0);
        Ui[(e >> 6) * LDB + (e & 63)] = T(0);
    }
    bool bad = false;
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
        const int c0 = 16 * p;
        if (wave == 0) {
            T a[16];
            T *row = D + lane * LDA + c0;
#pragma unroll
            for (int c = 0; c < 16; ++c) a[c] = row[c];
            static_for<0, 16>([&](auto J) {
                constexpr int j = decltype(J)::v;
                const T piv = bcast(a[j], c0 + j);
                bad = bad || Lu<T>::bad(piv);
                const bool below = lane > c0 + j;
                const T l = below ? Lu<T>::div(a[j], piv) : T(0);   // zero multiplier at and above the pivot
                a[j] = below ? l : a[j];
#pragma unroll
                for (int q0 = j + 1; q0 < 16; q0 += 4) {   // broadcasts ahead of their FMAs
                    T t[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (q0 + u < 16) t[u] = bcast(a[q0 + u], c0 + j);
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (q0 + u < 16) a[q0 + u] = fma(-l, t[u], a[q0 + u]);
                }
            });
#pragma unroll
            for (int c = 0; c < 16; ++c) row[c] = a[c];
        }
        __syncthreads();
        if (p == 3) break;
        if (wave == 0 && lane < 48 - c0) {
            T x[16];
            T *col = D + c0 * LDA + c0 + 16 + lane;
#pragma unroll
            for (int i = 0; i < 16; ++i) x[i] = col[i * LDA];
            subst16<T, false>(x, D + c0 * (LDA + 1), T(1));
#pragma unroll
            for (int i = 1; i < 16; ++i) col[i * LDA] = x[i];
        }
        __syncthreads();
        const int m = 3 - p;
        for (int q = wave; q < m * m; q += LT / 64) {
            const int r0 = c0 + 16 + 16 * (q / m), k0 = c0 + 16 + 16 * (q % m);
            v4 acc[1];
            zero<T, 1>(acc);
            mma<T, 1>(D + r0 * LDA + c0, LDA, D + c0 * LDA + k0, LDA, 16, lane, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) D[(r0 + Lu<T>::row(lane, e)) * LDA + k0 + Lu<T>::col(lane, e)] -= acc[0][e];
        }
        __syncthreads();
    }
    const int isu = wave >> 2, h = wave & 1, t2 = (wave >> 1) & 1;   // waves 0-3 for L, 4-7 for U
    {
        // 16 x 16 diagonal inverses, a column per lane
        const int c0 = 16 * (wave & 3), col = lane & 15;
        const T *t = D + c0 * (LDA + 1);
        T y[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) y[i] = i == col ? T(1) : T(0);
        if (!isu) subst16<T, false>(y, t, T(1));
        else subst16<T, true>(y, t, Lu<T>::div(T(1), t[col * (LDA + 1)]));
        T *dst = isu ? Ui + c0 * (LDB + 1) + col : Li + c0 * (LDA + 1) + col;
        const int st = isu ? LDB : LDA;
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; ++i) dst[i * st] = y[i];
    }
    __syncthreads();
    T *tw = s.tmp + isu * 32 * LDT;
    {
        // 16 -> 32: pair h (two waves of the four)
        const int b0 = 32 * h, b1 = b0 + 16;
        T *th = tw + 16 * h * LDT;
        v4 acc[1];
        if (t2 == 0) {
            zero<T, 1>(acc);
            if (!isu) mma<T, 1>(D + b1 * LDA + b0, LDA, Li + b0 * (LDA + 1), LDA, 16, lane, acc);
            else mma<T, 1>(D + b0 * LDA + b1, LDA, Ui + b1 * (LDB + 1), LDB, 16, lane, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) th[Lu<T>::row(lane, e) * LDT + Lu<T>::col(lane, e)] = acc[0][e];
        }
        __syncthreads();
        if (t2 == 0) {
            zero<T, 1>(acc);
            if (!isu) mma<T, 1>(Li + b1 * (LDA + 1), LDA, th, LDT, 16, lane, acc);
            else mma<T, 1>(Ui + b0 * (LDB + 1), LDB, th, LDT, 16, lane, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = Lu<T>::row(lane, e), c = Lu<T>::col(lane, e);
                if (!isu) Li[(b1 + r) * LDA + b0 + c] = -acc[0][e];
                else Ui[(b0 + r) * LDB + b1 + c] = -acc[0][e];
            }
        }
        __syncthreads();
    }
    {
        // 32 -> 64: wave = (L or U, 16 rows, 16 columns of the 32 x 32 block)
        v4 acc[1];
        zero<T, 1>(acc);
        if (!isu) mma<T, 1>(D + (32 + 16 * h) * LDA, LDA, Li + 16 * t2, LDA, 32, lane, acc);
        else mma<T, 1>(D + 16 * h * LDA + 32, LDA, Ui + 32 * (LDB + 1) + 16 * t2, LDB, 32, lane, acc);
#pragma unroll
        for (int e = 0; e < 4; ++e) tw[(16 * h + Lu<T>::row(lane, e)) * LDT + 16 * t2 + Lu<T>::col(lane, e)] = acc[0][e];
        __syncthreads();
        zero<T, 1>(acc);
        if (!isu) mma<T, 1>(Li + (32 + 16 * h) * LDA + 32, LDA, tw + 16 * t2, LDT, 32, lane, acc);
        else mma<T, 1>(Ui + 16 * h * LDB, LDB, tw + 16 * t2, LDT, 32, lane, acc);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = 16 * h + Lu<T>::row(lane, e), c = 16 * t2 + Lu<T>::col(lane, e);
            if (!isu) Li[(32 + r) * LDA + c] = -acc[0][e];
            else Ui[r * LDB + 32 + c] = -acc[0][e];
        }
    }
    __syncthreads();
    return bad;
}

// One matrix of the factorisation (a batch holds one per body).  DL, DU: the inverses of the TBIG x TBIG
// diagonal blocks of L and U, block q row-major at q TBIG^2; the factorisation writes their 64 x 64
// diagonal blocks, which its own products read, fp_tri_inverse grows them from there.  YL, YU:
// -L11^-1, -U11^-1 into the diagonal blocks of the full inverses (may be null).
template <typename T> struct LuMat {
    T *A;
    int64_t ld, n;
    T *DL, *DU;
    int *info;
    T *YL, *YU;
};
// entry (r, c) of the block inverses, both in the same TBIG block
template <typename T> __device__ __forceinline__ T *dent(T *D, int64_t r, int64_t c)
{
    return D + (r / TBIG) * ((int64_t)TBIG * TBIG) + (r % TBIG) * TBIG + c % TBIG;
}

// The diagonal block at (c, c), held in s.D (identity outside its bs rows): factor, store the factors and
// their inverses.
template <typename T> __device__ __forceinline__ void lu_diag(const LuMat<T> &m, int64_t c, StepLds<T> &s, int tid)
{
    constexpr int LDA = Lu<T>::LDA, LDB = Lu<T>::LDB;
    typedef Tile<T, NPB> Tl;
    const int bs = (int)min((int64_t)NPB, m.n - c);
    const bool bad = lu_diag64<T>(s, tid);
    if (bad && tid == 0) atomicCAS(m.info, 0, (int)(c + 1));
    Tl::store(s.D, LDA, m.A + c * m.ld + c, m.ld, bs, bs, T(1), tid);
    Tl::store(s.P, LDA, dent(m.DL, c, c), TBIG, NPB, NPB, T(1), tid);
    Tl::store(s.Q, LDB, dent(m.DU, c, c), TBIG, NPB, NPB, T(1), tid);
    if (m.YL) Tl::store(s.P, LDA, m.YL + c * m.ld + c, m.ld, bs, bs, T(-1), tid);
    if (m.YU) Tl::store(s.Q, LDB, m.YU + c * m.ld + c, m.ld, bs, bs, T(-1), tid);
}

// First diagonal block of the outer block at k; one workgroup.
template <typename T> __device__ __forceinline__ void lu_first_dev(const LuMat<T> &m, int64_t k, StepLds<T> &s)
{
    const int tid = threadIdx.x;
    const int bs = (int)min((int64_t)NPB, m.n - k);
    Tile<T, NPB> rd;
    rd.load(m.A + k * m.ld + k, m.ld, bs, bs, tid);
    rd.put(s.D, Lu<T>::LDA, tid);
    __syncthreads();
    if (tid < NPB && tid >= bs) s.D[tid * (Lu<T>::LDA + 1)] = T(1);
    __syncthreads();
    lu_diag<T>(m, k, s, tid);
}

// Inner step t of the outer block [k, kend), c = k + 64 t, on the 64 rows below number b: the strip's
// L tile A21 := A21 U11^-1, and A22 -= W A12 for the outer block's columns right of it, W = L21 L11^-1
// and A12 the block row as it stands (W A12 = L21 U12: the chain from one diagonal block to the next does
// not wait for U12, which lu_urow_dev forms when the outer block is done).  Workgroup 0 owns the next
// diagonal block: it goes on to factor it, so that a step is one launch and the other strips run beside
// the next block's pivot chain.  All products are 64 x 64 x 64 from LDS, the next tile loaded into
// registers meanwhile.  Workgroup 0 bounds it.  Cycles of its parts at 4,800 unknowns, FP32 and FP64 (a clock
// read at each, on the average over the steps): L tile 6,200 and 9,200, W 4,200 and 11,400, the columns' update
// 11,500 and 21,000 (two tiles), then the diagonal block's pivots 16,300 and 22,600, 16-row substitutions 7,200
// and 7,100, trailing tiles 3,700 and 5,800, inverses 7,700 and 13,500, stores 900 and 1,600; a launch takes 20.4
// and 31.9 us.  With the three U12 tiles in that workgroup and four waves the first block took 26 and 39 us and
// 4,800 unknowns 3.2 and 6.3 ms; with eight waves and U12 elsewhere 16 and 23 us, 2.8 and 5.2 ms.
template <typename T>
__device__ __forceinline__ void lu_step_dev(const LuMat<T> &m, int64_t k, int t, int64_t kend, int b, StepLds<T> &s)
{
    constexpr int LDA = Lu<T>::LDA, LDB = Lu<T>::LDB;
    typedef typename Lu<T>::v4 v4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t c = k + (int64_t)NPB * t, ld = m.ld, off = c + NPB + (int64_t)NPB * b;
    const int tr = (int)min((int64_t)NPB, m.n - off);
    T *A = m.A;
    Tile<T, NPB> ra, rq;
    ra.load(A + off * ld + c, ld, tr, NPB, tid);
    rq.load(dent(m.DU, c, c), TBIG, NPB, NPB, tid);
    ra.put(s.P, LDA, tid);
    rq.put(s.Q, LDB, tid);
    __syncthreads();
    int64_t j0 = c + NPB;
    const bool more = j0 < kend;
    if (more) {
        ra.load(dent(m.DL, c, c), TBIG, NPB, NPB, tid);
        rq.load(A + c * ld + j0, ld, NPB, (int)min((int64_t)NPB, kend - j0), tid);
    }
    v4 acc[2];
    mma64<T>(s.P, s.Q, lane, wave, acc);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = arow<T>(lane, wave, e), cc = acol<T>(lane, wave, q, e);
            if (r < tr) A[(off + r) * ld + c + cc] = acc[q][e];
        }
    if (!more) return;   // the outer block's last step: no columns right of it
    // W = L21 L11^-1
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) s.P[arow<T>(lane, wave, e) * LDA + acol<T>(lane, wave, q, e)] = acc[q][e];
    ra.put(s.Q, LDB, tid);
    __syncthreads();
    mma64<T>(s.P, s.Q, lane, wave, acc);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) s.P[arow<T>(lane, wave, e) * LDA + acol<T>(lane, wave, q, e)] = acc[q][e];
    for (; j0 < kend; j0 += NPB) {
        const int tc = (int)min((int64_t)NPB, kend - j0);
        T cv[2][4];
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = arow<T>(lane, wave, e), cc = acol<T>(lane, wave, q, e);
                cv[q][e] = A[(off + min(r, tr - 1)) * ld + j0 + min(cc, tc - 1)];
            }
        rq.put(s.Q, LDB, tid);
        __syncthreads();
        if (j0 + NPB < kend) rq.load(A + c * ld + j0 + NPB, ld, NPB, (int)min((int64_t)NPB, kend - j0 - NPB), tid);
        mma64<T>(s.P, s.Q, lane, wave, acc);
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = arow<T>(lane, wave, e), cc = acol<T>(lane, wave, q, e);
                const bool in = r < tr && cc < tc;
                const T v = cv[q][e] - acc[q][e];
                if (in) A[(off + r) * ld + j0 + cc] = v;
                if (b == 0 && j0 == c + NPB) s.D[r * LDA + cc] = in ? v : (r == cc ? T(1) : T(0));
            }
        __syncthreads();
    }
    if (b == 0) lu_diag<T>(m, c + NPB, s, tid);
}

// The part of the previous outer block's trailing update that this outer block's launches carry, C -= L U in
// 64 x 64 tiles (L in columns, U in rows [k - NOB, k)): columns from j0 on, `ntc` tile columns of them, rows
// from k on; `tile0` is the launch's first tile.
struct LuRest {
    int64_t j0;
    int ntc, tile0;
};
// The tile at (i0, j0).  The launches that factor the next 256 columns are a chain of single workgroups and at
// most one workgroup per 64 rows: these tiles run on the compute units that they leave idle.  Double-buffered
// through registers, two (FP32) or one (FP64) workgroups a compute unit.  diag: the tile is the diagonal
// block at k, which stays in s.D for lu_diag.
template <typename T>
__device__ __forceinline__ void lu_rest_dev(const LuMat<T> &m, int64_t k, int64_t i0, int64_t j0, StepLds<T> &s, bool diag)
{
    constexpr int LDA = Lu<T>::LDA, LDB = Lu<T>::LDB;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t ld = m.ld;
    const int tr = (int)min((int64_t)NPB, m.n - i0), tc = (int)min((int64_t)NPB, m.n - j0);
    const T *L = m.A + i0 * ld + k - NOB, *U = m.A + (k - NOB) * ld + j0;
    T *C = m.A + i0 * ld + j0;
    Tile<T, NPB> ra, rq;
    ra.load(L, ld, tr, NPB, tid);
    rq.load(U, ld, NPB, tc, tid);
    T cv[2][4];
    typename Lu<T>::v4 acc[2];
    zero<T, 2>(acc);
    for (int q = 0; q < NIN; ++q) {
        if (q) __syncthreads();
        ra.put(s.P, LDA, tid);
        rq.put(s.Q, LDB, tid);
        __syncthreads();
        if (q + 1 < NIN) {
            ra.load(L + NPB * (q + 1), ld, tr, NPB, tid);
            rq.load(U + (int64_t)NPB * (q + 1) * ld, ld, NPB, tc, tid);
        } else {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    cv[t][e] = C[min(arow<T>(lane, wave, e), tr - 1) * ld + min(acol<T>(lane, wave, t, e), tc - 1)];
        }
        mma<T, 2>(s.P + 16 * (wave & 3) * LDA, LDA, s.Q + 32 * (wave >> 2), LDB, NPB, lane, acc);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int i = arow<T>(lane, wave, e), j = acol<T>(lane, wave, t, e);
            const bool in = i < tr && j < tc;
            const T v = cv[t][e] - acc[t][e];
            if (diag) s.D[i * LDA + j] = in ? v : (i == j ? T(1) : T(0));
            else if (in) C[i * ld + j] = v;
        }
    if (diag) __syncthreads();
}
template <typename T> __device__ __forceinline__ void lu_rest_dev(const LuMat<T> &m, int64_t k, const LuRest &r, int x, StepLds<T> &s)
{
    x += r.tile0;
    lu_rest_dev<T>(m, k, k + (int64_t)NPB * (x / r.ntc), r.j0 + (int64_t)NPB * (x % r.ntc), s, false);
}

// U rows of the outer block [k, kend).  Workgroups b < nr: the UW columns from kend + UW b on, by blocked
// forward substitution U_t = L_tt^-1 (A_t - sum_{s<t} L_ts U_s) with the solved rows kept in LDS (ten
// 64 x 64 x 32 products).  The others: a tile right of a diagonal block inside the outer block,
// U = L_tt^-1 A, where A is what lu_step_dev left (UW columns each, lu_inner of them).
__host__ __device__ inline int lu_inner(int64_t cols)   // tiles of UW columns inside an outer block of `cols` columns
{
    int n = 0;
    for (int t = 0; t + 1 < NIN; ++t) {
        const int64_t c = cols - (int64_t)NPB * (t + 1);
        if (c > 0) n += (int)((c + UW - 1) / UW);
    }
    return n;
}
template <typename T> struct UrowLds {
    T P[NPB * Lu<T>::LDA];
    T X[NIN][NPB * Lu<T>::LDX];
    T R[NPB * Lu<T>::LDX];
};
template <typename T>
__device__ __forceinline__ void lu_urow_dev(const LuMat<T> &m, int64_t k, int64_t kend, int b, int nr, UrowLds<T> &s)
{
    constexpr int LDA = Lu<T>::LDA, LDX = Lu<T>::LDX;
    typedef typename Lu<T>::v4 v4;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = 16 * (wave & 3), wc = 16 * (wave >> 2);   // 64 x 32: a 16 x 16 tile per wave
    const int64_t ld = m.ld;
    T *A = m.A;
    int t0 = 0, t1 = NIN;
    int64_t j0 = kend + (int64_t)UW * b, jend = m.n;
    if (b >= nr) {
        int x = b - nr;
        jend = kend;
        for (t0 = 0;; ++t0) {
            j0 = k + (int64_t)NPB * (t0 + 1);
            const int w = (int)((kend - j0 + UW - 1) / UW);
            if (x < w) break;
            x -= w;
        }
        j0 += (int64_t)UW * x;
        t1 = t0 + 1;
    }
    const int tc = (int)min((int64_t)UW, jend - j0), first = b < nr ? 0 : t0;   // L tiles from block `first` on
    // left operands in order: L_t,first .. L_t,t-1, then L_tt^-1
    Tile<T, NPB> rp;
    rp.load(dent(m.DL, k + (int64_t)NPB * t0, k + (int64_t)NPB * t0), TBIG, NPB, NPB, tid);
    for (int t = t0; t < t1; ++t) {
        const int64_t c = k + (int64_t)NPB * t;
        T cv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            cv[e] = A[(c + wr + Lu<T>::row(lane, e)) * ld + j0 + min(wc + Lu<T>::col(lane, e), tc - 1)];
        v4 acc[1];
        zero<T, 1>(acc);
        for (int q = first; q < t; ++q) {
            __syncthreads();
            rp.put(s.P, LDA, tid);
            __syncthreads();
            if (q + 1 < t) rp.load(A + c * ld + k + NPB * (q + 1), ld, NPB, NPB, tid);
            else rp.load(dent(m.DL, c, c), TBIG, NPB, NPB, tid);
            mma<T, 1>(s.P + wr * LDA, LDA, s.X[q] + wc, LDX, NPB, lane, acc);
        }
        __syncthreads();
        rp.put(s.P, LDA, tid);
#pragma unroll
        for (int e = 0; e < 4; ++e) s.R[(wr + Lu<T>::row(lane, e)) * LDX + wc + Lu<T>::col(lane, e)] = cv[e] - acc[0][e];
        __syncthreads();
        if (t + 1 < t1) rp.load(A + (c + NPB) * ld + k, ld, NPB, NPB, tid);
        zero<T, 1>(acc);
        mma<T, 1>(s.P + wr * LDA, LDA, s.R + wc, LDX, NPB, lane, acc);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = wr + Lu<T>::row(lane, e), cc = wc + Lu<T>::col(lane, e);
            s.X[t][r * LDX + cc] = acc[0][e];
            if (cc < tc) A[(c + r) * ld + j0 + cc] = acc[0][e];
        }
    }
}

// (the first launch of a factorisation: it also clears the info word)
template <typename T> __global__ __launch_bounds__(LT) void k_lu_first(LuMat<T> m, int64_t k)
{
    __shared__ StepLds<T> s;
    if (threadIdx.x == 0) atomicExch(m.info, 0);
    lu_first_dev<T>(m, k, s);
}
// The previous outer block's update of the columns [k, k + 64 pc), one 64 x 64 tile per workgroup (np of them),
// and tiles of the rest; the first one goes on to factor the diagonal block at k.
template <typename T> __global__ __launch_bounds__(LT) void k_lu_update(LuMat<T> m, int64_t k, int pc, int np, LuRest r)
{
    __shared__ StepLds<T> s;
    const int x = blockIdx.x;
    if (x >= np) {
        lu_rest_dev<T>(m, k, r, x - np, s);
        return;
    }
    lu_rest_dev<T>(m, k, k + (int64_t)NPB * (x / pc), k + (int64_t)NPB * (x % pc), s, x == 0);
    if (x == 0) lu_diag<T>(m, k, s, threadIdx.x);
}
template <typename T>
__global__ __launch_bounds__(LT) void k_lu_step(LuMat<T> m, int64_t k, int t, int64_t kend, int strips, LuRest r)
{
    __shared__ StepLds<T> s;
    if ((int)blockIdx.x < strips) lu_step_dev<T>(m, k, t, kend, blockIdx.x, s);
    else lu_rest_dev<T>(m, k, r, blockIdx.x - strips, s);
}

template <typename T> __global__ __launch_bounds__(LT) void k_lu_urow(LuMat<T> m, int64_t k, int64_t kend, int nr)
{
    __shared__ UrowLds<T> s;
    lu_urow_dev<T>(m, k, kend, blockIdx.x, nr, s);
}

// ---- diagonal-block inverses for the triangular solves -------------------------
// One level of the pairwise merge of the block inverses, s -> 2s (s = 64, 128, 256): the pair of
// blocks at c0 = 2 s blockIdx.y and c1 = c0 + s, blockIdx.z 0 for L, 1 for U, one 64 x 64 tile of
// the s x s block per workgroup.  Phase 0: W = L21 X11 (U: U12 X22); phase 1: X21 = -X22 W
// (U: X12 = -X11 W).  Tiles that are zero in the triangular factor are left out.
template <typename T>
__global__ __launch_bounds__(LT) void k_tri_merge(LuMat<T> m, T *__restrict__ W, int s, int phase)
{
    constexpr int LDA = Lu<T>::LDA, LDB = Lu<T>::LDB;
    __shared__ T P[NPB * LDA], Q[NPB * LDB];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nt = s / NPB, ti = blockIdx.x / nt, tj = blockIdx.x % nt, up = blockIdx.z;
    const int64_t c0 = (int64_t)2 * s * blockIdx.y, c1 = c0 + s, n = m.n;
    if (c1 >= n) return;
    const int n1 = (int)min((int64_t)nt, (n - c1 + NPB - 1) / NPB);   // tiles of the second half that exist
    if ((up ? tj : ti) >= n1) return;
    W += ((int64_t)up * gridDim.y + blockIdx.y) * s * s;
    T *D = up ? m.DU : m.DL;
    const int64_t r0 = (up ? c0 : c1) + (int64_t)NPB * ti, q0 = (up ? c1 : c0) + (int64_t)NPB * tj;
    // K tiles: phase 0 runs over the column block's triangle, phase 1 over the row block's
    int k0, k1;
    if (phase == 0) { k0 = up ? 0 : tj; k1 = up ? tj + 1 : nt; }
    else { k0 = up ? ti : 0; k1 = up ? nt : ti + 1; }
    Tile<T, NPB> rp, rq;
    auto load = [&](int kk) {
        if (phase == 0) {
            const int64_t kc = (up ? c1 : c0) + (int64_t)NPB * kk;
            rp.load(m.A + r0 * m.ld + kc, m.ld, (int)min((int64_t)NPB, n - r0), (int)min((int64_t)NPB, n - kc), tid);
            rq.load(dent(D, kc, q0), TBIG, NPB, NPB, tid);
        } else {
            const int64_t kc = (up ? c0 : c1) + (int64_t)NPB * kk;
            rp.load(dent(D, r0, kc), TBIG, NPB, NPB, tid);
            rq.load(W + (int64_t)NPB * kk * s + NPB * tj, s, NPB, NPB, tid);
        }
    };
    typename Lu<T>::v4 acc[2];
    zero<T, 2>(acc);
    load(k0);
    for (int kk = k0; kk < k1; ++kk) {
        __syncthreads();
        rp.put(P, LDA, tid);
        rq.put(Q, LDB, tid);
        __syncthreads();
        if (kk + 1 < k1) load(kk + 1);
        mma<T, 2>(P + 16 * (wave & 3) * LDA, LDA, Q + 32 * (wave >> 2), LDB, NPB, lane, acc);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = arow<T>(lane, wave, e), c = acol<T>(lane, wave, q, e);
            if (phase == 0) W[(int64_t)(NPB * ti + r) * s + NPB * tj + c] = acc[q][e];
            else *dent(D, r0 + r, q0 + c) = -acc[q][e];
        }
}

// Rows [r0, r1) of a matrix times vectors (FP64 accumulation), 512 columns at most, one wave per R rows:
//   SOLVE: out[r] = sum over the row's triangle of the block inverse M (rows and columns from r0 on)
//   else:  out[r] -= sum_c M[r][c0 + c] v[c0 + c], c < nc
// NV vectors per grid row (ld lv and lo between vectors).  Bound by latency (a 512 x 512 inverse is
// read by 64 workgroups in about 3 us), so every load of a row group is issued together.
template <typename T, int R, int NV, bool SOLVE>
__global__ __launch_bounds__(256) void k_tri_gemv(const T *__restrict__ M, int64_t ldm, int64_t r0, int64_t r1, int64_t c0,
                                                  int nc, int upper, const double *__restrict__ v, int64_t lv,
                                                  double *__restrict__ out, int64_t lo, int nv)
{
    constexpr int V = Lu<T>::V;
    typedef typename Lu<T>::vec vec;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t rb = r0 + ((int64_t)blockIdx.x * 4 + wave) * R;
    if (rb >= r1) return;
    const int vb = blockIdx.y * NV, vn = min(NV, nv - vb);
    v += (int64_t)vb * lv;
    out += (int64_t)vb * lo;
    double acc[R][NV];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[i][j] = 0.0;
    // the columns of this row group: all nc, or the tiles of its triangle (a group lies in one 64-row tile)
    int lo_c = 0, hi_c = nc;
    if (SOLVE) {
        const int tile = (int)(rb - r0) & ~(NPB - 1);
        if (upper) lo_c = tile;
        else hi_c = min(nc, tile + NPB);
    }
    for (int cb = lo_c; cb < hi_c; cb += 64 * V) {
        const int c = cb + lane * V;
        if (c < hi_c) {
            vec a[R];
            if (c + V <= hi_c) {
#pragma unroll
                for (int i = 0; i < R; ++i)
                    a[i] = *reinterpret_cast<const vec *>(M + (min(rb + i, r1 - 1) - (SOLVE ? r0 : 0)) * ldm + c);
            } else {
#pragma unroll
                for (int i = 0; i < R; ++i)
#pragma unroll
                    for (int e = 0; e < V; ++e)
                        a[i][e] = c + e < hi_c ? M[(min(rb + i, r1 - 1) - (SOLVE ? r0 : 0)) * ldm + c + e] : T(0);
            }
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                const double *x = v + (int64_t)min(j, vn - 1) * lv + c0 + c;
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    const double xe = c + e < hi_c ? x[e] : 0.0;
#pragma unroll
                    for (int i = 0; i < R; ++i) acc[i][j] = fma((double)a[i][e], xe, acc[i][j]);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            double t = acc[i][j];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
            if (lane == 0 && rb + i < r1 && j < vn) {
                double *o = out + (int64_t)j * lo + rb + i;
                *o = SOLVE ? t : *o - t;
            }
        }
}

// U^T A V over the orbit blocks: thread (p, q) reads the 4 x 4 block of A at rows
// p + i m, columns q + j m (zeros beyond n), forms U_p^T B V_q in FP64 and
// stores it rounded to T.  W holds the 4 x 4 butterfly of every orbit,
// row-major: U's at W[16 p], V's at W[16 (m + q)].  Returns the sum of squares of the entries of A it
// read.  PAD, for p = q: beyond n the matrix is continued by a diagonal of the size of its own entries (the
// largest of the same orbit block): the butterflies mix the pad's rows with rows of A, whose digits a 1 among
// entries of 1e-12 would take.
template <bool PAD, typename Tin, typename T>
__device__ __forceinline__ double rbt_orbit(const Tin *__restrict__ A, int64_t n, int64_t lda, T *__restrict__ Ar, int64_t m,
                                            int64_t ldr, const double *__restrict__ W, int64_t p, int64_t q)
{
    double sq = 0.0;
    double B[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t gr = p + i * m;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t gc = q + j * m;
            B[i][j] = (gr < n && gc < n) ? (double)A[gr * lda + gc] : 0.0;
            sq = fma(B[i][j], B[i][j], sq);
        }
    }
    if constexpr (PAD) {
        double pad = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) pad = fmax(pad, fabs(B[i][j]));
        if (!(pad > 0.0) || isinf(pad)) pad = 1.0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (p + i * m >= n) B[i][i] = pad;
    }
    const double *U = W + 16 * p, *V = W + 16 * (m + q);
    double X[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            X[i][j] = B[i][0] * V[j] + B[i][1] * V[4 + j] + B[i][2] * V[8 + j] + B[i][3] * V[12 + j];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        T *dst = Ar + (p + i * m) * ldr + q;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            dst[j * m] = (T)(U[i] * X[0][j] + U[4 + i] * X[1][j] + U[8 + i] * X[2][j] + U[12 + i] * X[3][j]);
    }
    return sq;
}

// With part set, part[workgroup] receives the sum of squares of the entries of A the workgroup read.
template <typename Tin, typename T>
__global__ __launch_bounds__(256) void k_rbt_matrix(const Tin *__restrict__ A, int64_t n, int64_t lda,
                                                   T *__restrict__ Ar, int64_t m, int64_t ldr,
                                                   const double *__restrict__ W, double *__restrict__ part)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t p = blockIdx.y;
    double sq = 0.0;
    if (q < m) sq = rbt_orbit<false>(A, n, lda, Ar, m, ldr, W, p, q);
    if (!part) return;   // uniform
    __shared__ double sw[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
    if ((threadIdx.x & 63) == 0) sw[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = sw[0] + sw[1] + sw[2] + sw[3];
}

// The blocks with a pad once more, now with it (three at most, the last ones of the diagonal).  In the kernel above the
// same lines took its registers from 76 to 102, and the batch's launches, which share the chip, from 450 to 725 us;
// with selects from the three other diagonal entries and 76 registers they took 560 (its loads of rows then wait
// for each other).
template <typename Tin, typename T>
__global__ __launch_bounds__(64) void k_rbt_pad(const Tin *__restrict__ A, int64_t n, int64_t lda, T *__restrict__ Ar,
                                                int64_t m, int64_t ldr, const double *__restrict__ W)
{
    const int64_t p = m - 1 - threadIdx.x;
    if (p >= 0 && p + 3 * m >= n) (void)rbt_orbit<true>(A, n, lda, Ar, m, ldr, W, p, p);
}

// out[0] = sum of part[0 .. np), out[1] = smallest |A(i, i)| (0 when one is NaN); one workgroup
__global__ __launch_bounds__(1024) void k_lu_check(const double *__restrict__ part, int64_t np,
                                                   const double *__restrict__ A, int64_t n, int64_t ld,
                                                   double *__restrict__ out)
{
    __shared__ double ss[16], sm[16];
    double s = 0.0, v = INFINITY;
    for (int64_t i = threadIdx.x; i < np; i += 1024) s += part[i];
    for (int64_t i = threadIdx.x; i < n; i += 1024) {
        const double d = fabs(A[i * ld + i]);
        v = d < v ? d : (d == d ? v : 0.0);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        s += __shfl_xor(s, o);
        v = fmin(v, __shfl_xor(v, o));
    }
    if ((threadIdx.x & 63) == 0) { ss[threadIdx.x >> 6] = s; sm[threadIdx.x >> 6] = v; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) { s += ss[w]; v = fmin(v, sm[w]); }
        out[0] = s;
        out[1] = v;
    }
}

// t (n4 x k) = U^T b (n x k, zero-padded), or x (n x k) = V y (y n4 x k, the pad dropped)
__global__ void k_rbt_vec(const double *__restrict__ in, int64_t ldin, double *__restrict__ out, int64_t ldout,
                          int64_t n, int64_t m, int64_t k, const double *__restrict__ W, int transpose_u)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t col = blockIdx.y;
    if (p >= m || col >= k) return;
    const double *Wp = W + 16 * (transpose_u ? p : m + p);
    const double *src = in + col * ldin;
    double *dst = out + col * ldout;
    double v[4], o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t g = p + i * m;
        v[i] = (transpose_u && g >= n) ? 0.0 : src[g];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        o[i] = transpose_u ? Wp[i] * v[0] + Wp[4 + i] * v[1] + Wp[8 + i] * v[2] + Wp[12 + i] * v[3]
                           : Wp[4 * i] * v[0] + Wp[4 * i + 1] * v[1] + Wp[4 * i + 2] * v[2] + Wp[4 * i + 3] * v[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t g = p + i * m;
        if (transpose_u || g < n) dst[g] = o[i];
    }
}

// Two depth-2 recursive butterflies of size 4m as their m orbit blocks (row-major
// 4 x 4, acting on (x_p, x_p+m, x_p+2m, x_p+3m)): the outer butterfly pairs
// p with p + 2m, the two inner ones pair p with p + m in each half; every
// butterfly is (1/sqrt 2) [R S; R -S] with random diagonals exp(r / 10),
// r uniform in [-1/2, 1/2].  The i-th draw of a splitmix64 stream is the mix of
// seed + (i + 1) * golden, so every orbit computes its own eight draws.
__device__ __forceinline__ uint64_t mix64_at(uint64_t seed, uint64_t i)
{
    uint64_t z = seed + (i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void k_rbt_weights(int64_t m, uint64_t seed, double *__restrict__ W)
{
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= 2 * m) return;
    const bool v = p >= m;   // U's orbit blocks first, then V's
    const int64_t q = v ? p - m : p;
    const uint64_t sd = v ? seed ^ 0x5DEECE66Dull : seed;
    double r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) r[j] = exp((((double)(mix64_at(sd, 8 * (uint64_t)q + j) >> 11) * 0x1.0p-53) - 0.5) / 10.0);
    const double h = sqrt(0.5);
    const double Z[4][4] = {{h * r[0], 0, h * r[1], 0}, {0, h * r[2], 0, h * r[3]},
                            {h * r[0], 0, -h * r[1], 0}, {0, h * r[2], 0, -h * r[3]}};
    const double Y[4][4] = {{h * r[4], h * r[5], 0, 0}, {h * r[4], -h * r[5], 0, 0},
                            {0, 0, h * r[6], h * r[7]}, {0, 0, h * r[6], -h * r[7]}};
    double *o = W + 16 * p;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[4 * i + j] = Y[i][0] * Z[0][j] + Y[i][1] * Z[1][j] + Y[i][2] * Z[2][j] + Y[i][3] * Z[3][j];
}

// E (n x n, FP64, lde) = -(V C U^T) restricted to n x n, C (4m x 4m, FP32, ldc):
// thread (p, q) forms -V_p B U_q^T of the orbit block B of C at rows p + i m,
// columns q + j m (the undoing of U^T A V for an inverse: A^-1 = V A_r^-1 U^T).
__global__ __launch_bounds__(256) void k_rbt_unmatrix(const float *__restrict__ C, int64_t ldc, int64_t m,
                                                     double *__restrict__ E, int64_t n, int64_t lde,
                                                     const double *__restrict__ W)
{
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t p = blockIdx.y;
    if (q >= m) return;
    double B[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) B[i][j] = (double)C[(p + i * m) * ldc + q + j * m];
    const double *Vp = W + 16 * (m + p), *Uq = W + 16 * q;
    double T[4][4];   // B U_q^T
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            T[i][j] = B[i][0] * Uq[4 * j] + B[i][1] * Uq[4 * j + 1] + B[i][2] * Uq[4 * j + 2] + B[i][3] * Uq[4 * j + 3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t gr = p + i * m;
        if (gr >= n) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t gc = q + j * m;
            if (gc < n)
                E[gr * lde + gc] =
                    -(Vp[4 * i] * T[0][j] + Vp[4 * i + 1] * T[1][j] + Vp[4 * i + 2] * T[2][j] + Vp[4 * i + 3] * T[3][j]);
        }
    }
}

}  // namespace

int64_t fp_rbt_size(int64_t n) { return (n + 3) / 4 * 4; }

size_t fp_rbt_weights_bytes(int64_t n) { return (size_t)32 * (fp_rbt_size(n) / 4) * sizeof(double); }

// U's orbit blocks then V's, for a matrix of order n (padded to n4)
int fp_rbt_weights(fp_ctx *ctx, int64_t n, uint64_t seed, double *d_W)
{
    const int64_t m = fp_rbt_size(n) / 4;
    if (m == 0) return FP_OK;
    hipLaunchKernelGGL(k_rbt_weights, dim3((unsigned)((2 * m + 127) / 128)), dim3(128), 0, ctx->stream, m, seed, d_W);
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}

int64_t fp_rbt_norm_parts(int64_t n)
{
    const int64_t m = fp_rbt_size(n) / 4;
    return (m + 255) / 256 * m;
}

template <typename Tin, typename T>
int fp_rbt_matrix(fp_ctx *ctx, const Tin *A, int64_t n, int64_t lda, T *Ar, int64_t ldr, const double *d_W, double *part)
{
    const int64_t m = fp_rbt_size(n) / 4;
    if (m == 0) return FP_OK;
    ProfScope ps(ctx, "rbt");
    hipLaunchKernelGGL((k_rbt_matrix<Tin, T>), dim3((unsigned)((m + 255) / 256), (unsigned)m), dim3(256), 0, ctx->stream,
                       A, n, lda, Ar, m, ldr, d_W, part);
    if (n % 4) hipLaunchKernelGGL((k_rbt_pad<Tin, T>), dim3(1), dim3(64), 0, ctx->stream, A, n, lda, Ar, m, ldr, d_W);
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}
template int fp_rbt_matrix<double, float>(fp_ctx *, const double *, int64_t, int64_t, float *, int64_t, const double *,
                                          double *);
template int fp_rbt_matrix<float, float>(fp_ctx *, const float *, int64_t, int64_t, float *, int64_t, const double *,
                                         double *);
template int fp_rbt_matrix<double, double>(fp_ctx *, const double *, int64_t, int64_t, double *, int64_t,
                                           const double *, double *);

// out[0] = |A|_F^2 from fp_rbt_matrix's partial sums, out[1] = the smallest |pivot| of the factors LU (n4 x n4)
int fp_lu_check(fp_ctx *ctx, const double *part, int64_t n, const double *LU, int64_t ld, double *out)
{
    hipLaunchKernelGGL(k_lu_check, dim3(1), dim3(1024), 0, ctx->stream, part, fp_rbt_norm_parts(n), LU, fp_rbt_size(n),
                       ld, out);
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}

// transpose_u: out (n4 x k, ldout) = U^T in (n x k, ldin); else out (n x k) = V in (n4 x k)
int fp_rbt_vec(fp_ctx *ctx, const double *in, int64_t ldin, double *out, int64_t ldout, int64_t n, int64_t k,
               const double *d_W, int transpose_u)
{
    const int64_t m = fp_rbt_size(n) / 4;
    if (m == 0 || k == 0) return FP_OK;
    if (k > 65535) return fp_fail(ctx, FP_ERR_UNSUPPORTED, "getrs: too many right-hand sides in one call");   // as fp_getrs
    hipLaunchKernelGGL(k_rbt_vec, dim3((unsigned)((m + 255) / 256), (unsigned)k), dim3(256), 0, ctx->stream, in, ldin,
                       out, ldout, n, m, k, d_W, transpose_u);
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}

// the diagonal-block inverses of L, then of U, then fp_tri_inverse's products
static int64_t lu_dsize(int64_t n) { return (n + TBIG - 1) / TBIG * ((int64_t)TBIG * TBIG); }
size_t fp_getrf_nopiv_work_bytes(int64_t n, int elem_bytes)
{
    return ((size_t)2 * lu_dsize(n) + (size_t)lu_dsize(n) / 2) * elem_bytes;
}

static int64_t lu_tiles(int64_t x, int64_t w) { return x > 0 ? (x + w - 1) / w : (int64_t)0; }

// LU without pivoting of the n x n matrix A (row-major, 16-byte aligned, ld a multiple of 4), outer
// blocks of 256 columns: per inner block of 64 one launch (lu_step_dev), then the U rows right of the
// outer block and one rank-256 trailing update (a rank-64 update per inner block would read and write
// the whole trailing matrix four times as often).  info_dev receives 1 + the first row of the diagonal
// block whose pivot was zero or not finite (0 if none).
//
// That update's columns of the next outer block are brought up to date in the launch that also factors the
// next diagonal block (k_lu_update); as much of the rest as the chain of launches has room for goes into
// these launches as further workgroups (lu_rest_dev), which need nothing of the chain and are not needed by
// it before the U rows; only what is left is a launch of its own (fp_gemm_sub).  PER_CU: workgroups that a
// compute unit holds, a slot each; FIRST, STEP: tiles per slot that the launch of a diagonal
// block and a step take before the chain waits for them, by measurement.  4,800 (8,000) unknowns, ms, FP32:
// nothing carried 2.80 (6.66), 1/1 2.54 (6.18), 1/2 2.37 (5.85), 2/2 2.35 (5.79), 2/3 2.36 (5.80); FP64: nothing
// 5.23 (13.1), 1/1 4.86 (12.5), 1/2 4.50 (11.95), 2/2 4.52 (12.06), 2/4 4.77 (12.5).
template <typename T> struct LuRoom;
template <> struct LuRoom<float> { static constexpr int PER_CU = 2, FIRST = 2, STEP = 2; };
template <> struct LuRoom<double> { static constexpr int PER_CU = 1, FIRST = 1, STEP = 2; };

template <typename T>
int fp_getrf_nopiv(fp_ctx *ctx, T *A, int64_t n, int64_t ld, int *info_dev, void *work, T *YL, T *YU)
{
    if (n <= 0) return FP_OK;
    if (ld % 4) return fp_fail(ctx, FP_ERR_ARG, "internal: no-pivot LU needs a leading dimension divisible by 4");
    const LuMat<T> m{A, ld, n, (T *)work, (T *)work + lu_dsize(n), info_dev, YL, YU};
    int st;
    const int64_t slots = (int64_t)LuRoom<T>::PER_CU * ctx->num_cu;
    int64_t rest_j = n;   // columns from here on still miss the previous outer block's update
    for (int64_t k = 0; k < n; k += NOB) {
        const int64_t kend = std::min<int64_t>(k + NOB, n), rows = lu_tiles(n - k, NPB);
        LuRest r{rest_j, (int)std::max<int64_t>(lu_tiles(n - rest_j, NPB), 1), 0};
        int64_t left = rest_j < n ? r.ntc * rows : 0;
        auto take = [&](int64_t room, bool last) {   // tiles of the next launch
            const int64_t x = last ? left : std::min(left, std::max<int64_t>(room, 0));
            left -= x;
            return x;
        };
        if (k == 0) {
            ProfScope ps(ctx, "lu_nopiv_diag");
            hipLaunchKernelGGL(k_lu_first<T>, dim3(1), dim3(LT), 0, ctx->stream, m, k);
        } else {
            const int64_t pc = lu_tiles(kend - k, NPB), x = take(slots * LuRoom<T>::FIRST - pc * rows, rows == 1);
            ProfScope ps(ctx, "lu_nopiv_update");
            hipLaunchKernelGGL(k_lu_update<T>, dim3((unsigned)(pc * rows + x)), dim3(LT), 0, ctx->stream, m, k, (int)pc,
                               (int)(pc * rows), r);
            r.tile0 += (int)x;
        }
        for (int t = 0; t < NIN; ++t) {
            const int64_t strips = rows - 1 - t;
            if (strips <= 0) break;
            const int64_t x = take((slots - strips) * LuRoom<T>::STEP, t + 2 >= NIN || strips == 1);
            ProfScope ps(ctx, "lu_nopiv_step");
            hipLaunchKernelGGL(k_lu_step<T>, dim3((unsigned)(strips + x)), dim3(LT), 0, ctx->stream, m, k, t, kend, (int)strips,
                               r);
            r.tile0 += (int)x;
        }
        const int64_t right = n - kend;
        const int nr = (int)lu_tiles(right, UW), ni = lu_inner(kend - k);
        if (nr + ni > 0) {
            ProfScope ps(ctx, "lu_nopiv_urow");
            hipLaunchKernelGGL(k_lu_urow<T>, dim3((unsigned)(nr + ni)), dim3(LT), 0, ctx->stream, m, k, kend, nr);
        }
        FP_HIP(ctx, hipGetLastError());
        if (right <= 0) break;
        // tile columns of the update right of the next outer block, as many as its launches have room for
        const int64_t rt = lu_tiles(right, NPB), pt = std::min<int64_t>(NIN, rt);
        int64_t room = std::max<int64_t>(slots * LuRoom<T>::FIRST - pt * rt, 0);
        for (int t = 0; t < std::min<int64_t>(NIN - 1, rt - 1); ++t)
            room += std::max<int64_t>(slots - (rt - 1 - t), 0) * LuRoom<T>::STEP;
        const int64_t now = rt - pt - std::min(room / rt, rt - pt);   // the others, at once
        const int64_t j0 = kend + pt * NPB;
        rest_j = std::min(j0 + now * NPB, n);
        if (now > 0 && (st = fp_gemm_sub<T>(ctx, right, rest_j - j0, NOB, A + kend * ld + k, ld, A + k * ld + j0, ld,
                                            A + kend * ld + j0, ld)))
            return st;
    }
    return FP_OK;
}
template int fp_getrf_nopiv<float>(fp_ctx *, float *, int64_t, int64_t, int *, void *, float *, float *);
template int fp_getrf_nopiv<double>(fp_ctx *, double *, int64_t, int64_t, int *, void *, double *, double *);

// The inverses of the TBIG-row diagonal blocks of fp_getrf_nopiv's factors (same work), from their
// 64-row blocks: three levels of two launches.  About (2/3) n TBIG^2 flop.
template <typename T>
int fp_tri_inverse(fp_ctx *ctx, const T *A, int64_t n, int64_t ld, void *work)
{
    ProfScope ps(ctx, "lu_nopiv_blockinv");
    const LuMat<T> m{const_cast<T *>(A), ld, n, (T *)work, (T *)work + lu_dsize(n), nullptr, nullptr, nullptr};
    T *W = (T *)work + 2 * lu_dsize(n);
    for (int s = NPB; s < TBIG && s < n; s *= 2) {
        const dim3 g((unsigned)((s / NPB) * (s / NPB)), (unsigned)lu_tiles(n, 2 * s), 2);
        hipLaunchKernelGGL(k_tri_merge<T>, g, dim3(LT), 0, ctx->stream, m, W, s, 0);
        hipLaunchKernelGGL(k_tri_merge<T>, g, dim3(LT), 0, ctx->stream, m, W, s, 1);
    }
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}
template int fp_tri_inverse<float>(fp_ctx *, const float *, int64_t, int64_t, void *);
template int fp_tri_inverse<double>(fp_ctx *, const double *, int64_t, int64_t, void *);

template <typename T, int NV>
static void tri_gemvs(fp_ctx *ctx, const T *LU, int64_t n, int64_t ld, const T *D, bool upper, double *b, int64_t ldb,
                      double *y, int64_t ldy, int64_t k)
{
    const unsigned gy = (unsigned)((k + NV - 1) / NV);
    const int64_t nb = (n + TBIG - 1) / TBIG;
    for (int64_t q = 0; q < nb; ++q) {
        const int64_t j = upper ? nb - 1 - q : q, c0 = j * TBIG, c1 = std::min<int64_t>(c0 + TBIG, n);
        hipLaunchKernelGGL((k_tri_gemv<T, 2, NV, true>), dim3((unsigned)lu_tiles(c1 - c0, 8), gy), dim3(256), 0, ctx->stream,
                           D + j * ((int64_t)TBIG * TBIG), (int64_t)TBIG, c0, c1, c0, (int)(c1 - c0), upper ? 1 : 0,
                           (const double *)b, ldb, y, ldy, (int)k);
        // the rows still to be solved
        const int64_t r0 = upper ? 0 : c1, r1 = upper ? c0 : n;
        if (r1 > r0)
            hipLaunchKernelGGL((k_tri_gemv<T, 4, NV, false>), dim3((unsigned)lu_tiles(r1 - r0, 16), gy), dim3(256), 0,
                               ctx->stream, LU + c0, ld, r0, r1, c0, (int)(c1 - c0), 0, (const double *)y, ldy, b, ldb,
                               (int)k);
    }
}

// The block inverses of A^T's factors (L' = U^T, U' = L^T) from those of A's: DL' = DU^T and DU' = DL^T, block by
// block.  64 x 64 tiles through LDS.
template <typename T>
__global__ __launch_bounds__(256) void k_tri_transpose(const T *__restrict__ D, T *__restrict__ E, int64_t half)
{
    __shared__ T s[64][65];
    constexpr int NT = TBIG / 64;
    const int ti = blockIdx.x / NT, tj = blockIdx.x % NT, x = threadIdx.x & 63, y = threadIdx.x >> 6;
    const int64_t blk = (int64_t)blockIdx.y * TBIG * TBIG;
    const T *src = D + (blockIdx.z ? 0 : half) + blk;   // z = 0: DL' from DU
    T *dst = E + (blockIdx.z ? half : 0) + blk;
    for (int r = y; r < 64; r += 4) s[r][x] = src[(64 * ti + r) * TBIG + 64 * tj + x];
    __syncthreads();
    for (int r = y; r < 64; r += 4) dst[(64 * tj + r) * TBIG + 64 * ti + x] = s[x][r];
}
template <typename T> int fp_tri_inverse_transposed(fp_ctx *ctx, int64_t n, const void *work, void *work_t)
{
    if (n <= 0) return FP_OK;
    const int64_t half = lu_dsize(n), nb = (n + TBIG - 1) / TBIG;
    hipLaunchKernelGGL(k_tri_transpose<T>, dim3((TBIG / 64) * (TBIG / 64), (unsigned)nb, 2), dim3(256), 0, ctx->stream,
                       (const T *)work, (T *)work_t, half);
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}
template int fp_tri_inverse_transposed<double>(fp_ctx *, int64_t, const void *, void *);

// x (n x k, ldx, FP64) := U^-1 L^-1 x by fp_getrf_nopiv's factors and the block inverses in `work`
// (fp_tri_inverse); tmp: n k doubles.  Two launches per 512-row block and sweep: the block's solution
// y = D b, then its contribution to the rows still to be solved.  The chain of launches bounds it
// (4,800 unknowns: 20 a sweep); a sweep that polls per 128-row block walked 38 hand-overs of 8-10 us.
template <typename T>
int fp_lu_solve_nopiv(fp_ctx *ctx, const T *LU, int64_t n, int64_t ld, const void *work, double *x, int64_t k, int64_t ldx,
                      double *tmp)
{
    if (n <= 0 || k <= 0) return FP_OK;
    ProfScope ps(ctx, "getrs");
    const T *DL = (const T *)work, *DU = DL + lu_dsize(n);
    if (k == 1) {
        tri_gemvs<T, 1>(ctx, LU, n, ld, DL, false, x, ldx, tmp, n, k);
        tri_gemvs<T, 1>(ctx, LU, n, ld, DU, true, tmp, n, x, ldx, k);
    } else {
        tri_gemvs<T, 4>(ctx, LU, n, ld, DL, false, x, ldx, tmp, n, k);
        tri_gemvs<T, 4>(ctx, LU, n, ld, DU, true, tmp, n, x, ldx, k);
    }
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}
template int fp_lu_solve_nopiv<float>(fp_ctx *, const float *, int64_t, int64_t, const void *, double *, int64_t, int64_t,
                                      double *);
template int fp_lu_solve_nopiv<double>(fp_ctx *, const double *, int64_t, int64_t, const void *, double *, int64_t,
                                       int64_t, double *);

// ---- the same factorisation for many bodies at once --------------------------
// One launch per step covers every body (blockIdx.y = body): the bodies' serial chains of
// diagonal blocks run side by side, and the small products of different bodies fill the chip
// together.  Global outer blocks [kk, kk + NOB); a body takes part in the steps inside its order.

__global__ void k_fill_info_lub(const fp_lu_desc *__restrict__ desc, int nb)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < nb) *desc[b].info = 0;
}

static __device__ __forceinline__ LuMat<float> lub_mat(const fp_lu_desc &d)
{
    return LuMat<float>{d.A, d.ld, d.n, d.work, d.work + (d.n + TBIG - 1) / TBIG * ((int64_t)TBIG * TBIG), d.info,
                        nullptr, nullptr};
}

__global__ __launch_bounds__(LT) void k_lu_first_lub(const fp_lu_desc *__restrict__ desc, int64_t kk)
{
    __shared__ StepLds<float> s;
    const LuMat<float> m = lub_mat(desc[blockIdx.y]);
    if (kk >= m.n) return;   // uniform per workgroup
    lu_first_dev<float>(m, kk, s);
}

__global__ __launch_bounds__(LT) void k_lu_step_lub(const fp_lu_desc *__restrict__ desc, int64_t kk, int t)
{
    __shared__ StepLds<float> s;
    const LuMat<float> m = lub_mat(desc[blockIdx.y]);
    const int64_t below = m.n - kk - (int64_t)NPB * (t + 1);
    if ((int64_t)blockIdx.x * NPB >= below) return;
    lu_step_dev<float>(m, kk, t, min(kk + (int64_t)NOB, m.n), blockIdx.x, s);
}

__global__ __launch_bounds__(LT) void k_lu_urow_lub(const fp_lu_desc *__restrict__ desc, int64_t kk)
{
    __shared__ UrowLds<float> s;
    const LuMat<float> m = lub_mat(desc[blockIdx.y]);
    if (kk >= m.n) return;
    const int64_t kend = min(kk + (int64_t)NOB, m.n);
    const int nr = (int)((m.n - kend + UW - 1) / UW);
    if ((int)blockIdx.x >= nr + lu_inner(kend - kk)) return;
    lu_urow_dev<float>(m, kk, kend, blockIdx.x, nr, s);
}

int fp_getrf_nopiv_f32_batched(fp_ctx *ctx, const fp_lu_desc *d_desc, const int64_t *n_host, int nb)
{
    if (nb <= 0) return FP_OK;
    if (nb > 65535) return fp_fail(ctx, FP_ERR_UNSUPPORTED, "batched LU: too many bodies");
    int64_t nmax = 0;
    for (int b = 0; b < nb; ++b) nmax = std::max(nmax, n_host[b]);
    hipLaunchKernelGGL(k_fill_info_lub, dim3((unsigned)((nb + 63) / 64)), dim3(64), 0, ctx->stream, d_desc, nb);
    int st;
    for (int64_t kk = 0; kk < nmax; kk += NOB) {
        {
            ProfScope ps(ctx, "lu_nopiv_diag");
            hipLaunchKernelGGL(k_lu_first_lub, dim3(1, (unsigned)nb), dim3(LT), 0, ctx->stream, d_desc, kk);
        }
        for (int t = 0; t < NIN; ++t) {
            const int64_t strips = lu_tiles(nmax - kk - (int64_t)NPB * (t + 1), NPB);
            if (strips <= 0) break;
            ProfScope ps(ctx, "lu_nopiv_step");
            hipLaunchKernelGGL(k_lu_step_lub, dim3((unsigned)strips, (unsigned)nb), dim3(LT), 0, ctx->stream, d_desc,
                               kk, t);
        }
        const int64_t right = nmax - kk - NOB;
        int64_t gu = 0;
        for (int b = 0; b < nb; ++b) {
            const int64_t kend = std::min(kk + (int64_t)NOB, n_host[b]);
            if (kk < n_host[b]) gu = std::max(gu, lu_tiles(n_host[b] - kend, UW) + lu_inner(kend - kk));
        }
        if (gu > 0) {
            ProfScope ps(ctx, "lu_nopiv_urow");
            hipLaunchKernelGGL(k_lu_urow_lub, dim3((unsigned)gu, (unsigned)nb), dim3(LT), 0, ctx->stream, d_desc, kk);
        }
        FP_HIP(ctx, hipGetLastError());
        if (right > 0 && (st = fp_gemm_sub_lub(ctx, d_desc, nb, kk, NOB, right))) return st;
    }
    return FP_OK;
}

// Explicit inverses of the no-pivot factors, for refinement sweeps that then cost
// two GEMVs instead of two blocked triangular solves.  YL = -L^-1 and YU = -U^-1
// (row-major, ld as A; zero outside their triangles on entry, the diagonal 64 x 64
// blocks written by fp_getrf_nopiv).  With Y = -X the block recurrences
//   lower:  Y_JI = Y_JJ L_JI Y_II,   upper:  Y_IJ = Y_II U_IJ Y_JJ   (I before J)
// are two "C -= A B" products each through T = -L_JI Y_II (resp. -U_IJ Y_JJ);
// blocks merge pairwise, 64 -> 128 -> ..., one batched launch per product and
// level.  U^-1 L^-1 = YU YL: the signs cancel in the solve.  T: n x ld scratch.
int fp_trtri_nopiv_f32(fp_ctx *ctx, const float *A, int64_t n, int64_t ld, float *YL, float *YU, float *T)
{
    ProfScope ps(ctx, "lu_nopiv_trtri");
    int st;
    for (int64_t s = NPB; s < n; s *= 2) {
        const int64_t P = n / (2 * s), rem = n - 2 * s * P;
        const int64_t step = 2 * s * ld + 2 * s;   // between consecutive pairs
        if (P > 0) {
            if ((st = fp_fill_f32(ctx, T, P * s * ld, 0.f))) return st;
            // lower: T_p = -L_JI Y_II, Y_JI -= Y_JJ T_p
            if ((st = fp_gemm_sub_batched_f32(ctx, s, s, s, A + s * ld, ld, step, YL, ld, step, T, ld, s * ld, (int)P)))
                return st;
            if ((st = fp_gemm_sub_batched_f32(ctx, s, s, s, YL + s * ld + s, ld, step, T, ld, s * ld, YL + s * ld, ld,
                                              step, (int)P)))
                return st;
            if ((st = fp_fill_f32(ctx, T, P * s * ld, 0.f))) return st;
            // upper: T_p = -U_IJ Y_JJ, Y_IJ -= Y_II T_p
            if ((st = fp_gemm_sub_batched_f32(ctx, s, s, s, A + s, ld, step, YU + s * ld + s, ld, step, T, ld, s * ld,
                                              (int)P)))
                return st;
            if ((st = fp_gemm_sub_batched_f32(ctx, s, s, s, YU, ld, step, T, ld, s * ld, YU + s, ld, step, (int)P)))
                return st;
        }
        if (rem > s) {   // the last pair: I = [r, r + s), J = [r + s, n)
            const int64_t r = 2 * s * P, sj = rem - s, rj = r + s;
            if ((st = fp_fill_f32(ctx, T, s * ld, 0.f))) return st;
            if ((st = fp_gemm_sub_batched_f32(ctx, sj, s, s, A + rj * ld + r, ld, 0, YL + r * ld + r, ld, 0, T, ld, 0,
                                              1)))
                return st;
            if ((st = fp_gemm_sub_batched_f32(ctx, sj, s, sj, YL + rj * ld + rj, ld, 0, T, ld, 0, YL + rj * ld + r, ld,
                                              0, 1)))
                return st;
            if ((st = fp_fill_f32(ctx, T, s * ld, 0.f))) return st;
            if ((st = fp_gemm_sub_batched_f32(ctx, s, sj, sj, A + r * ld + rj, ld, 0, YU + rj * ld + rj, ld, 0, T, ld,
                                              0, 1)))
                return st;
            if ((st = fp_gemm_sub_batched_f32(ctx, s, sj, s, YU + r * ld + r, ld, 0, T, ld, 0, YU + r * ld + rj, ld, 0,
                                              1)))
                return st;
        }
    }
    return FP_OK;
}

// Workspace of fp_inverse_rbt_f32 for order n: the randomized copy (then the
// product), -L^-1, -U^-1, the triangular-inverse scratch (FP32, n4 x ld4 each),
// the butterflies and the LU's own work.
static int64_t inv_ld(int64_t n4) { return std::max<int64_t>(64, (n4 + 63) / 64 * 64); }
size_t fp_inverse_rbt_work_bytes(int64_t n)
{
    const int64_t n4 = fp_rbt_size(n), ld4 = inv_ld(n4);
    return (size_t)4 * n4 * ld4 * sizeof(float) + fp_rbt_weights_bytes(n) + fp_getrf_nopiv_work_bytes(n4, sizeof(float)) + 1024;
}

// E^-1 in place (n x n, FP64, lde) by the LU without pivoting of the randomized
// FP32 matrix U^T E V, the explicit inverses of its factors and one product:
// E^-1 = V (U_r^-1 L_r^-1) U^T.  No chain of n / 64 Gauss-Jordan passes with
// their products: the factorisation's own chain is a few launches per 64
// columns and the rest are large MFMA products.  info_dev as fp_getrf_nopiv.
// Nothing is allocated and the host is not synchronised (a side stream may run it).
int fp_inverse_rbt_f32(fp_ctx *ctx, double *E, int64_t n, int64_t lde, void *work, size_t work_bytes, int *info_dev,
                       uint64_t seed)
{
    if (n <= 0) return FP_OK;
    if (work_bytes < fp_inverse_rbt_work_bytes(n)) return fp_fail(ctx, FP_ERR_ARG, "internal: inverse workspace too small");
    ProfScope ps(ctx, "inverse_rbt");
    const int64_t n4 = fp_rbt_size(n), m = n4 / 4, ld4 = inv_ld(n4), sz = n4 * ld4;
    float *Ar = (float *)work, *YL = Ar + sz, *YU = YL + sz, *T = YU + sz;
    double *W = (double *)(T + sz);
    void *nwork = (char *)W + fp_rbt_weights_bytes(n);
    hipLaunchKernelGGL(k_rbt_weights, dim3((unsigned)((2 * m + 127) / 128)), dim3(128), 0, ctx->stream, m, seed, W);
    int st;
    if ((st = fp_rbt_matrix<double, float>(ctx, E, n, lde, Ar, ld4, W))) return st;
    if ((st = fp_fill_f32(ctx, YL, sz, 0.f)) || (st = fp_fill_f32(ctx, YU, sz, 0.f))) return st;
    if ((st = fp_getrf_nopiv<float>(ctx, Ar, n4, ld4, info_dev, nwork, YL, YU))) return st;
    if ((st = fp_trtri_nopiv_f32(ctx, Ar, n4, ld4, YL, YU, T))) return st;
    // Ar <- -(YU YL) = -U^-1 L^-1 (the factors are no longer needed)
    if ((st = fp_fill_f32(ctx, Ar, sz, 0.f))) return st;
    if ((st = fp_gemm_sub<float>(ctx, n4, n4, n4, YU, ld4, YL, ld4, Ar, ld4))) return st;
    hipLaunchKernelGGL(k_rbt_unmatrix, dim3((unsigned)((m + 255) / 256), (unsigned)m), dim3(256), 0, ctx->stream,
                       (const float *)Ar, ld4, m, E, n, lde, (const double *)W);
    FP_HIP(ctx, hipGetLastError());
    return FP_OK;
}
