// The local analysis without an eigensolve: the update needs C^(-1/2) on the nine
// member-perturbation vectors of a gridpoint and C^(-1) on one more vector, and both
// functions of C = a I + A (a = (M-1)/beta, A = G^T G >= 0) are Chebyshev series of
// moderate degree when the spectrum [a, a + lambda_max(A)] is not too wide.
//
//   X_a = xbar 1^T + dX (sqrt(M-1) C^(-1/2) + C^(-1) b 1^T)     (letkf_solver.h:288-316)
//
// with x = 2 (C - a) / lambda - 1 in [-1, 1], lambda >= lambda_max(A):
//   f(C) r = sum_n c_n T_n(x) r = sum_k T_4k(x) sum_{j<4} d_kj T_j(x) r,
// the inner sums from V_j = T_j(x) r (three products of A with a block of ten vectors),
// the outer one by Clenshaw's recurrence in Y = T_4(x) = 2 T_2(x)^2 - 1, one product of Y
// with the block per step.  Two full products (A^2 and T_2^2) and about 2.2 sqrt(kappa)
// block products replace the Jacobi sweeps; nothing but matrix products is left.
//
// Products: v_mfma_f32_16x16x32_bf16 (x16 for one tile) with every operand split into
// three bf16 parts (24 mantissa bits) and the six products of weight above 2^-24, FP32
// accumulation: the FP32 matrix instructions take 2.7 times as long for the same bits.
// Against 64 bits the products and the series leave an error of 1e-7 to 1e-6 of the
// result (kappa up to 400), a tenth or less of what the split Gram matrix leaves.
// An accumulator tile is an operand as it stands: lane (c, g) holds rows 16 T + 4 g + r,
// r = 0..3, of column c, so summing over k in the order (T, g, r), the tile (K, J) of a
// matrix is the B operand of K-block K and, the matrix being symmetric, the tile (K, I)
// its A operand.  No value moves between lanes from the Gram matrix to the analysed state.
#pragma once
#include <algorithm>
#include <cmath>
#include <vector>

#include "context.hpp"

namespace lbmletkf {

// ---- the series, on the host ------------------------------------------------------
// Classes of condition number kappa = 2^(k/4), k = 1, 2, ..; per class the degree that
// leaves the series of x^(-1/2) and 1/x on [1, kappa] off by about eps of their value at
// 1, and the coefficients d_kj of both.
constexpr int SERIES_CLASS0 = 80;     // quadruples of the header (first quadruple of each class)
// The widest class lies where the eigensolve of the same kernel family costs as much: in
// the mixed analysis at N = 64 a block product costs 1/110 of the warm-started sweeps
// (kappa 2000), in FP64 1/4000 of them; there the table ends it (0.7 MB).
constexpr int SERIES_CLASSES32 = 40, SERIES_CLASSES64 = 64;  // kappa up to 1024 and 65536
constexpr double SERIES_EPS32 = 3e-8, SERIES_EPS64 = 1e-13;

// Quadruples of T: entry k of the header is (first quadruple, blocks K, 0, 0) of class k,
// as values; then per block the two quadruples d_k0..d_k3 of x^(-1/2) and of 1/x.
template <class T>
std::vector<T> series_table(int classes, double eps) {
    std::vector<T> t(4 * SERIES_CLASS0, T(0));
    for (int cl = 1; cl <= classes; ++cl) {
        const double kappa = std::exp2(cl / 4.0), q = (std::sqrt(kappa) - 1.0) / (std::sqrt(kappa) + 1.0);
        const int degree = int(std::ceil(std::log(1.0 / eps) / -std::log(q))) + 1;
        const int K = std::max(2, (degree + 3) / 4), n = 4 * K;
        std::vector<double> c[2];
        // 1/y, y = ((kappa-1) x + kappa + 1)/2: c_k = (2 - [k = 0]) (-q)^k / sqrt(kappa)
        c[1].resize(n);
        for (int k = 0; k < n; ++k) c[1][k] = (k ? 2.0 : 1.0) * std::pow(-q, k) / std::sqrt(kappa);
        // y^(-1/2) = f: 2 (x + al) f' + f = 0, al = (kappa+1)/(kappa-1), gives for the
        // coefficients d_k of f'
        //   (1 + 1/2k) d_{k-1} + 2 al d_k + (1 - 1/2k) d_{k+1} = 0,  c_k = (d_{k-1} - d_{k+1})/2k,
        // of which they are the decaying solution: taken downwards from far above the
        // degree, and scaled to f = 1 at y = 1 (x = -1) and f = kappa^(-1/2) at x = 1
        const double al = (kappa + 1.0) / (kappa - 1.0);
        const int top = 2 * n + 40;
        std::vector<double> d(top + 2, 0.0);
        d[top] = 1e-280;
        for (int k = top; k >= 1; --k)
            d[k - 1] = -(2.0 * al * d[k] + (1.0 - 0.5 / k) * d[k + 1]) / (1.0 + 0.5 / k);
        c[0].resize(n);
        double lo = 0.0, hi = 0.0;  // sum_{k>0} of the unscaled series at x = -1 and x = 1
        for (int k = top; k >= 1; --k) {
            const double ck = (d[k - 1] - d[k + 1]) / (2.0 * k);
            lo += k % 2 ? -ck : ck;
            hi += ck;
            if (k < n) c[0][k] = ck;
        }
        const double scale = (1.0 - 1.0 / std::sqrt(kappa)) / (lo - hi);
        for (int k = 1; k < n; ++k) c[0][k] *= scale;
        c[0][0] = 1.0 - scale * lo;
        t[4 * cl] = T(t.size() / 4);
        t[4 * cl + 1] = T(K);
        std::vector<double> e(size_t(K) * 8);
        for (int f = 0; f < 2; ++f)
            // T_{4k+j} = 2 T_4k T_j - T_{4(k-1) + (4-j)}
            for (int k = K - 1; k >= 0; --k)
                for (int j = 0; j < 4; ++j) {
                    const double ck = c[f][4 * k + j];
                    e[size_t(k) * 8 + 4 * f + j] = k > 0 && j > 0 ? 2.0 * ck : ck;
                    if (k > 0 && j > 0) c[f][4 * (k - 1) + 4 - j] -= ck;
                }
        for (double x : e) t.push_back(T(x));
    }
    return t;
}

// ---- on the device ------------------------------------------------------------------
namespace {
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float quiet_nan() { return __int_as_float(0x7fc00000); }

// Operands of one K-block: two accumulator tiles (32 values of k), or the only one of a
// 16 x 16 problem.
template <int N>
struct SeriesOp {
    static constexpr int TILES = N >= 32 ? 2 : 1;
    typedef bf16x8 vec;
};
template <>
struct SeriesOp<16> {
    static constexpr int TILES = 1;
    typedef bf16x4 vec;
};

__device__ __forceinline__ f32x4 series_mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 series_mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0,
                                                     0, 0);
}

// x = p0 + p1 + p2, each bf16 (rounded to nearest), for a pair of values
__device__ __forceinline__ void split_pair(float a, float b, bf16x2 (&p)[3]) {
#pragma unroll
    for (int s = 0; s < 3; ++s) {
        p[s] = __builtin_convertvector(f32x2{a, b}, bf16x2);
        if (s < 2) {
            const unsigned bits = __builtin_bit_cast(unsigned, p[s]);
            a -= __builtin_bit_cast(float, bits << 16);
            b -= __builtin_bit_cast(float, bits & 0xffff0000u);
        }
    }
}
__device__ __forceinline__ void split_tiles(const f32x4* t, bf16x8 (&p)[3]) {
    bf16x2 q[4][3];
#pragma unroll
    for (int k = 0; k < 4; ++k) split_pair(t[k / 2][2 * (k % 2)], t[k / 2][2 * (k % 2) + 1], q[k]);
#pragma unroll
    for (int s = 0; s < 3; ++s)
        p[s] = __builtin_shufflevector(__builtin_shufflevector(q[0][s], q[1][s], 0, 1, 2, 3),
                                       __builtin_shufflevector(q[2][s], q[3][s], 0, 1, 2, 3), 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ void split_tiles(const f32x4* t, bf16x4 (&p)[3]) {
    bf16x2 q[2][3];
#pragma unroll
    for (int k = 0; k < 2; ++k) split_pair(t[0][2 * k], t[0][2 * k + 1], q[k]);
#pragma unroll
    for (int s = 0; s < 3; ++s) p[s] = __builtin_shufflevector(q[0][s], q[1][s], 0, 1, 2, 3);
}

// c + a b over one K-block, the small products first
template <class V>
__device__ __forceinline__ f32x4 series_fma(const V (&a)[3], const V (&b)[3], f32x4 c) {
    c = series_mfma(a[0], b[2], c);
    c = series_mfma(a[2], b[0], c);
    c = series_mfma(a[1], b[1], c);
    c = series_mfma(a[0], b[1], c);
    c = series_mfma(a[1], b[0], c);
    return series_mfma(a[0], b[0], c);
}

// a symmetric matrix as operands: K-block kb, tile column j
template <int N>
struct SeriesMat {
    static constexpr int NT = N / 16, KB = NT / SeriesOp<N>::TILES;
    typename SeriesOp<N>::vec p[KB][NT][3];
    // from its tiles (K NT + J) scaled by s
    __device__ __forceinline__ void set(const f32x4* t, float scale) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                f32x4 x[SeriesOp<N>::TILES];
#pragma unroll
                for (int h = 0; h < SeriesOp<N>::TILES; ++h) x[h] = t[(kb * SeriesOp<N>::TILES + h) * NT + j] * scale;
                split_tiles(x, p[kb][j]);
                // opaque: under register pressure the compiler would sink the split into
                // the loop that uses it
#pragma unroll
                for (int s = 0; s < 3; ++s) asm volatile("" : "+v"(p[kb][j][s]));
                __builtin_amdgcn_sched_barrier(0);
            }
    }
    // its tile (K, J), exactly the sum of the parts
    __device__ __forceinline__ f32x4 tile(int K, int J) const {
        f32x4 x;
        const int kb = K / SeriesOp<N>::TILES, h = 4 * (K % SeriesOp<N>::TILES);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            x[r] = float(p[kb][J][0][h + r]) + (float(p[kb][J][1][h + r]) + float(p[kb][J][2][h + r]));
        return x;
    }
    // d = this * this
    __device__ __forceinline__ void square(f32x4* d) const {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                f32x4 c{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) c = series_fma(p[kb][i], p[kb][j], c);
                d[i * NT + j] = c;
                __builtin_amdgcn_sched_barrier(0);
            }
    }
    // c += this * (s v) for a block of sixteen columns v
    __device__ __forceinline__ void times(const f32x4 (&v)[NT], float s, f32x4 (&c)[NT]) const {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            f32x4 x[SeriesOp<N>::TILES];
#pragma unroll
            for (int h = 0; h < SeriesOp<N>::TILES; ++h) x[h] = v[kb * SeriesOp<N>::TILES + h] * s;
            typename SeriesOp<N>::vec b[3];
            split_tiles(x, b);
#pragma unroll
            for (int i = 0; i < NT; ++i) c[i] = series_fma(p[kb][i], b, c[i]);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// The four vectors V_j, in registers, or where a matrix fills those (N = 64), in LDS as
// [j][T][lane].
template <int N>
struct SeriesBasis {
    static constexpr int NT = N / 16;
    f32x4 v[4][NT];
    __device__ __forceinline__ SeriesBasis(float*, int) {}
    __device__ __forceinline__ void put(int j, const f32x4 (&x)[NT]) {
#pragma unroll
        for (int T = 0; T < NT; ++T) v[j][T] = x[T];
    }
    __device__ __forceinline__ f32x4 get(int j, int T) const { return v[j][T]; }
};
template <>
struct SeriesBasis<64> {
    static constexpr int NT = 4;
    f32x4* at;
    __device__ __forceinline__ SeriesBasis(float* lds, int lane) : at(reinterpret_cast<f32x4*>(lds) + lane) {}
    __device__ __forceinline__ void put(int j, const f32x4 (&x)[NT]) {
#pragma unroll
        for (int T = 0; T < NT; ++T) at[(j * NT + T) * 64] = x[T];
    }
    __device__ __forceinline__ f32x4 get(int j, int T) const { return at[(j * NT + T) * 64]; }
};

// r := f(C) r for C = a I + A, A in the tiles `acc` (K NT + J; rows and columns past the
// members zero): columns 0..8 of the block by x^(-1/2), column 9 by 1/x.  Returns the
// number of block products taken, or 0, r untouched, where the spectrum is wider than the
// widest class (or not finite).  A is taken times a power of two that brings a to [1, 2).
// basis.get(0, .) holds the incoming r after a true return.  The scheduling barriers
// keep the tiles in order: at N = 64 two matrices leave no registers to work ahead in.
template <int N>
__device__ __forceinline__ int series_apply(const f32x4* acc, f32x4 (&r)[N / 16], float a_in, float scale_a,
                                            const float4* __restrict__ table, SeriesBasis<N>& basis, int lane) {
    constexpr int NT = N / 16;
    const float a = a_in * scale_a;
    SeriesMat<N> m;
    m.set(acc, scale_a);
    f32x4 sq[NT * NT];
    m.square(sq);
    // lambda_max(A) <= ||A^2||_F^(1/2) (at most rank^(1/4) too wide)
    float ss = 0.f;
#pragma unroll
    for (int t = 0; t < NT * NT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) ss = fmaf(sq[t][k], sq[t][k], ss);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    const float kappa = 1.f + 1.0001f * __builtin_amdgcn_sqrtf(__builtin_amdgcn_sqrtf(ss)) / a;
    if (!(kappa <= 1023.f)) return 0;  // SERIES_CLASSES32
    const int cl = __builtin_amdgcn_readfirstlane(max(1, int(ceilf(4.f * log2f(kappa)))));
    const float lam = a * (exp2f(0.25f * float(cl)) - 1.f);
    const float al = 2.f / lam;  // x = al A - 1
    const float4 hd = table[cl];
    const int first = __builtin_amdgcn_readfirstlane(int(hd.x));
    const int K = __builtin_amdgcn_readfirstlane(int(hd.y));

    // V_0 = r, V_1 = x V_0, V_j = 2 x V_{j-1} - V_{j-2}
    {
        f32x4 v[NT];
        basis.put(0, r);
#pragma unroll
        for (int T = 0; T < NT; ++T) v[T] = -r[T];
        m.times(r, al, v);
        basis.put(1, v);
#pragma unroll
        for (int j = 2; j < 4; ++j) {
            f32x4 w[NT];
#pragma unroll
            for (int T = 0; T < NT; ++T) w[T] = -2.f * v[T] - basis.get(j - 2, T);
            m.times(v, 2.f * al, w);
            basis.put(j, w);
#pragma unroll
            for (int T = 0; T < NT; ++T) v[T] = w[T];
        }
    }
    // T_2(x) = 2 al^2 A^2 - 4 al A + I, then Y = T_4 = 2 T_2^2 - I; the recurrence takes 2 Y
    __builtin_amdgcn_sched_barrier(0);
    const int c = lane & 15, g = lane >> 4;
    const float k2 = 2.f * al * al, k1 = -4.f * al;
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int J = 0; J < NT; ++J) {
            const f32x4 x = m.tile(I, J);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                sq[I * NT + J][k] = fmaf(k2, sq[I * NT + J][k], fmaf(k1, x[k], I == J && 4 * g + k == c ? 1.f : 0.f));
            __builtin_amdgcn_sched_barrier(0);
        }
    m.set(sq, 1.f);
    m.square(sq);
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int J = 0; J < NT; ++J)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                sq[I * NT + J][k] = fmaf(4.f, sq[I * NT + J][k], I == J && 4 * g + k == c ? -2.f : 0.f);
    m.set(sq, 1.f);

    // Clenshaw: B_k = Q_k + 2 Y B_{k+1} - B_{k+2}, Q_k = sum_j d_kj V_j; result Q_0 + Y B_1 - B_2
    const float4* coef = table + first + (c == 9 ? 1 : 0);
    f32x4 b1[NT], b2[NT];
    {
        const float4 d = coef[2 * (K - 1)];
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            b1[T] = d.x * basis.get(0, T) + d.y * basis.get(1, T) + d.z * basis.get(2, T) + d.w * basis.get(3, T);
            b2[T] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    float4 d = coef[2 * (K - 2)];
#pragma unroll 1
    for (int k = K - 2; k >= 0; --k) {
        const float4 dn = coef[2 * max(k - 1, 0)];
        f32x4 q[NT];
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            const f32x4 x0 = basis.get(0, T), x1 = basis.get(1, T), x2 = basis.get(2, T), x3 = basis.get(3, T);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                q[T][e] = fmaf(d.x, x0[e], fmaf(d.y, x1[e], fmaf(d.z, x2[e], fmaf(d.w, x3[e], -b2[T][e]))));
        }
        m.times(b1, k > 0 ? 1.f : 0.5f, q);
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            b2[T] = b1[T];
            b1[T] = q[T];
        }
        d = dn;
    }
    // f(C) = a^(-1/2) f(C / a), 1 / C = (1/a) 1 / (C / a)
    const float scale = c == 9 ? 1.f / a_in : 1.f / sqrtf(a_in);
#pragma unroll
    for (int T = 0; T < NT; ++T) r[T] = b1[T] * scale;
    return K + 2;
}

// ---- the same in FP64 (the PLAIN variant), on v_mfma_f64_16x16x4f64 ------------------
// A[m][k] from lane (m = lane % 16, k = lane / 16), B[k][n] from lane (n = lane % 16,
// k = lane / 16), D[lane / 16 + 4 r][lane % 16]: summed over k in the order (T, r), the
// accumulator tiles are operands as they stand here too.
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <int N>
struct SeriesMat64 {
    static constexpr int NT = N / 16;
    f64x4 t[NT * NT];  // tile (K, J)
    __device__ __forceinline__ void square(f64x4 (&d)[NT * NT]) const {
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) d[i * NT + j] = f64x4{0, 0, 0, 0};
#pragma unroll
        for (int K = 0; K < NT; ++K)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < NT; ++i)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        d[i * NT + j] = __builtin_amdgcn_mfma_f64_16x16x4f64(t[K * NT + i][r], t[K * NT + j][r],
                                                                             d[i * NT + j], 0, 0, 0);
    }
    // c += this * (s v)
    __device__ __forceinline__ void times(const f64x4 (&v)[NT], double s, f64x4 (&c)[NT]) const {
#pragma unroll
        for (int K = 0; K < NT; ++K)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double x = s * v[K][r];
#pragma unroll
                for (int i = 0; i < NT; ++i)
                    c[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(t[K * NT + i][r], x, c[i], 0, 0, 0);
            }
    }
};

// r := f(C) r, as series_apply; m holds A and is overwritten; basis: 4 N 16 doubles of
// LDS, basis[(j NT + T) 64 + lane] the incoming r (j = 0) afterwards.
template <int N>
__device__ __forceinline__ int series_apply64(SeriesMat64<N>& m, f64x4 (&r)[N / 16], double a,
                                              const double4* __restrict__ table, f64x4* basis, int lane) {
    constexpr int NT = N / 16;
    auto put = [&](int j, const f64x4 (&x)[NT]) {
#pragma unroll
        for (int T = 0; T < NT; ++T) basis[(j * NT + T) * 64 + lane] = x[T];
    };
    auto get = [&](int j, int T) { return basis[(j * NT + T) * 64 + lane]; };
    const double ia = 1.0 / a;
    f64x4 sq[NT * NT];
#pragma unroll
    for (int t = 0; t < NT * NT; ++t) m.t[t] *= ia;  // spectrum [0, kappa - 1]
    m.square(sq);
    double ss = 0;
#pragma unroll
    for (int t = 0; t < NT * NT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) ss = fma(sq[t][k], sq[t][k], ss);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    const float kappa = 1.f + 1.0001f * float(sqrt(sqrt(ss)));
    if (!(kappa <= 65500.f)) return 0;  // SERIES_CLASSES64
    const int cl = __builtin_amdgcn_readfirstlane(max(1, int(ceilf(4.f * log2f(kappa)))));
    const double lam = exp2(0.25 * double(cl)) - 1.0;
    const double al = 2.0 / lam;
    const double4 hd = table[cl];
    const int first = __builtin_amdgcn_readfirstlane(int(hd.x));
    const int K = __builtin_amdgcn_readfirstlane(int(hd.y));
    {
        f64x4 v[NT];
        put(0, r);
#pragma unroll
        for (int T = 0; T < NT; ++T) v[T] = -r[T];
        m.times(r, al, v);
        put(1, v);
#pragma unroll
        for (int j = 2; j < 4; ++j) {
            f64x4 w[NT];
#pragma unroll
            for (int T = 0; T < NT; ++T) w[T] = -2.0 * v[T] - get(j - 2, T);
            m.times(v, 2.0 * al, w);
            put(j, w);
#pragma unroll
            for (int T = 0; T < NT; ++T) v[T] = w[T];
        }
    }
    // T_2 = 2 al^2 A^2 - 4 al A + I; 2 T_4 = 4 T_2^2 - 2 I
    const int c = lane & 15, g = lane >> 4;
    const double k2 = 2.0 * al * al, k1 = -4.0 * al;
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int J = 0; J < NT; ++J)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                m.t[I * NT + J][k] = fma(k2, sq[I * NT + J][k],
                                         fma(k1, m.t[I * NT + J][k], I == J && g + 4 * k == c ? 1.0 : 0.0));
    m.square(sq);
#pragma unroll
    for (int I = 0; I < NT; ++I)
#pragma unroll
        for (int J = 0; J < NT; ++J)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                m.t[I * NT + J][k] = fma(4.0, sq[I * NT + J][k], I == J && g + 4 * k == c ? -2.0 : 0.0);
    const double4* coef = table + first + (c == 9 ? 1 : 0);
    f64x4 b1[NT], b2[NT];
    {
        const double4 d = coef[2 * (K - 1)];
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            b1[T] = d.x * get(0, T) + d.y * get(1, T) + d.z * get(2, T) + d.w * get(3, T);
            b2[T] = f64x4{0, 0, 0, 0};
        }
    }
#pragma unroll 1
    for (int k = K - 2; k >= 0; --k) {
        const double4 d = coef[2 * k];
        f64x4 q[NT];
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            const f64x4 x0 = get(0, T), x1 = get(1, T), x2 = get(2, T), x3 = get(3, T);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                q[T][e] = fma(d.x, x0[e], fma(d.y, x1[e], fma(d.z, x2[e], fma(d.w, x3[e], -b2[T][e]))));
        }
        m.times(b1, k > 0 ? 1.0 : 0.5, q);
#pragma unroll
        for (int T = 0; T < NT; ++T) {
            b2[T] = b1[T];
            b1[T] = q[T];
        }
    }
    const double scale = c == 9 ? ia : sqrt(ia);
#pragma unroll
    for (int T = 0; T < NT; ++T) r[T] = b1[T] * scale;
    return K + 2;
}

}  // namespace
}  // namespace lbmletkf
