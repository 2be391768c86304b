/* Device BLAS for the hip engine: GEMM on the gfx950 matrix cores, exposed as
 * the reference's blas_* extension methods (include/bh_blas_hip.h).
 *
 * Real types: one workgroup of 4 waves computes a BM x BN tile of C; wave w owns
 * the (w / 2, w % 2) quarter as TM x TN MFMA tiles of 16 x 16.  Per K step (16)
 * the workgroup stages op(A) (BM x BK) and op(B) (BK x BN) in LDS with padded
 * rows so that the 16-lane groups of one MFMA operand read fall in disjoint
 * banks; the LDS tiles are double-buffered and the next K step is fetched into
 * registers while the current one runs on the matrix cores.  Products with too
 * few such tiles for the chip split K over the waves of a workgroup instead
 * (gemm_slice).  MFMA operand layout (16 x 16 x 4, measured on gfx950): lane l
 * supplies A[l % 16][l / 16] and B[l / 16][l % 16]; its 4 results are
 * D[4 (l / 16) + r][l % 16] for f32 and D[4 r + l / 16][l % 16] for f64, r = 0..3.
 *
 * Complex types run on the same MFMA tiles, four real products per complex one (gemm_complex).
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <stdexcept>
#include <string>

#include <bohrium/bh_extmethod.hpp>
#include <bohrium/bh_instruction.hpp>

#include "../../../include/bh_blas_hip.h"
#include "../../../include/bh_ve_hip.h"

namespace {

typedef double bh_d4 __attribute__((ext_vector_type(4)));
typedef float bh_f4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;
template <> struct Mfma<double> {
    typedef bh_d4 Acc;
    static __device__ __forceinline__ Acc step(double a, double b, Acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // row of the 16 x 16 tile that result r of `lane` belongs to
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + (lane >> 4); }
};
template <> struct Mfma<float> {
    typedef bh_f4 Acc;
    static __device__ __forceinline__ Acc step(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

constexpr int kThreads = 256;

// Between the loads of the next K step and the products of this one.  In the 32-bit kernels the scheduler moved the loads
// down to where their registers are stored, behind the products that they were to run beside; in the 64-bit ones it
// leaves them (and lost a few per cent when told to).  Float32, 64 x 64 tiles: 1024^3 51.3 -> 32.2 us, 960 x 1100 x 1000 57.4 -> 44.0,
// 2000 x 1500 x 2500 157 -> 146; complex64 1024^3 93.0 -> 89.3.
template <typename R> __device__ __forceinline__ void loads_before_products() {
    if constexpr (sizeof(R) == 4) __builtin_amdgcn_sched_barrier(0);
}
constexpr int kPad = 16;

// 16 bytes of elements; `loose`: at any element (a global load needs no more than 4-byte alignment).
template <typename T> struct Vec;
template <> struct Vec<double> {
    typedef double type __attribute__((ext_vector_type(2)));
    typedef double loose __attribute__((ext_vector_type(2), aligned(8)));
    static constexpr int n = 2;
};
template <> struct Vec<float> {
    typedef float type __attribute__((ext_vector_type(4)));
    typedef float loose __attribute__((ext_vector_type(4), aligned(4)));
    static constexpr int n = 4;
};

// One operand tile: ROWS rows (m of op(A) or n of op(B)) by kBK steps of k.  KCONT: k is the contiguous
// dimension in memory (element (r, k) at P[r * ld + k]); otherwise r is (element at P[k * ld + r]).  A thread
// moves CH chunks of V elements along the contiguous dimension, one 16-byte load each at any alignment.
// LDS layout: [ROWS][kBK + KPAD] when KCONT, else [kBK][ROWS + kPad]; with these pads the 16-lane groups of
// an MFMA operand read (16 rows at one k, the next group at k + 1) and the chunk stores fall in disjoint
// banks.
//
// The loads of the main loop have no bounds checks (a check is a branch, and the compiler waits for the
// loads at its join: the prefetch of the next K step was not overlapped at all).  Rows past R are taken
// from inside the matrix instead, their results are not stored: KCONT chunks repeat row R - 1; the others
// move down to end at row R - 1, in LDS too (`edge`: stored element by element).  Needs R >= V.  The K % kBK
// leading columns are a step of their own (`first`), zero-filled.
template <typename T, bool KCONT, int ROWS, int kBK>
struct Tile {
    static constexpr int V = Vec<T>::n;
    static constexpr int PER = ROWS * kBK / kThreads;
    static constexpr int CH = PER / V;
    static constexpr int KPAD = sizeof(T) == 8 ? 2 : 4;
    static constexpr int LDS = KCONT ? ROWS * (kBK + KPAD) : kBK * (ROWS + kPad);
    static_assert(CH * V == PER && CH * kThreads * V == ROWS * kBK, "tile / thread count");
    typedef typename Vec<T>::loose Loose;

    const T *p[CH];  // the chunks of the next step
    int64_t advance;
    T reg[PER];

    static __device__ __forceinline__ void chunk(int e, int &r, int &k) {
        const int c = static_cast<int>(threadIdx.x) + e * kThreads;
        if (KCONT) {
            r = c / (kBK / V);
            k = (c % (kBK / V)) * V;
        } else {
            k = c / (ROWS / V);
            r = (c % (ROWS / V)) * V;
        }
    }
    // The row that chunk (r) of a tile at r0 is loaded from.
    static __device__ __forceinline__ int64_t source(int64_t r0, int r, int64_t R) {
        const int64_t last = KCONT ? R - 1 : R - V;
        return r0 + r < last ? r0 + r : last;
    }
    // Loads columns [0, kn) of the tile (kn <= kBK, zeros past it) and points at column kn.
    __device__ __forceinline__ void first(const T *__restrict__ P, int64_t ld, int64_t r0, int64_t R, int kn) {
        advance = KCONT ? kBK : kBK * ld;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            int r, k;
            chunk(e, r, k);
            const int64_t gr = source(r0, r, R);
            p[e] = KCONT ? P + gr * ld + k : P + k * ld + gr;
        }
        // A whole step by 16-byte loads, like the others (element by element 2048 x 2048 x 64 float32 took 11.1 us, 9.8 so).
        if (kn == kBK) {
            next();
            return;
        }
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            int r, k;
            chunk(e, r, k);
#pragma unroll
            for (int j = 0; j < V; ++j) reg[e * V + j] = (KCONT ? k + j : k) < kn ? p[e][j] : T(0);
            p[e] += KCONT ? kn : kn * ld;
        }
    }
    __device__ __forceinline__ void next() {
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const Loose v = *reinterpret_cast<const Loose *>(p[e]);
            p[e] += advance;
#pragma unroll
            for (int j = 0; j < V; ++j) reg[e * V + j] = v[j];
        }
    }
    __device__ __forceinline__ void store(T *lds, bool edge, int64_t r0, int64_t R) const {
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            int r, k;
            chunk(e, r, k);
            if (!KCONT && edge) {
                const int at = static_cast<int>(source(r0, r, R) - r0);
#pragma unroll
                for (int j = 0; j < V; ++j)
                    if (at + j >= 0) lds[k * (ROWS + kPad) + at + j] = reg[e * V + j];
                continue;
            }
            typename Vec<T>::type v;
#pragma unroll
            for (int j = 0; j < V; ++j) v[j] = reg[e * V + j];
            *reinterpret_cast<typename Vec<T>::type *>(KCONT ? lds + r * (kBK + KPAD) + k : lds + k * (ROWS + kPad) + r) = v;
        }
    }
    static __device__ __forceinline__ T read(const T *lds, int r, int k) {
        return KCONT ? lds[r * (kBK + KPAD) + k] : lds[k * (ROWS + kPad) + r];
    }
};

// C = op(A) op(B), or alpha op(A) op(B) + beta C when SCALED (C is not read when beta is 0); op(A)(m, k)
// = TA ? A[k * lda + m] : A[m * lda + k], op(B)(k, n) = TB ? B[n * ldb + k] : B[k * ldb + n].  UPPER:
// only C(m, n) with m <= n is stored.  The scaled epilogue is a separate instantiation: in the plain
// product it costs the f64 128 x 128 kernel ~120 VGPRs and half its throughput.
// The LDS tiles are double-buffered: while the matrix cores work on one K step, the next one is
// loaded into registers and then stored into the other buffer; one barrier per K step.  Two waves a SIMD: the
// epilogue alone would take the f64 128 x 128 kernel to 278 registers and one wave.
// Bound by the MFMA rate (counters: the matrix cores are busy 83 % of the cycles of the f64 128 x 128 kernel).
// Measured against loads that wait at bounds checks in the loop: 4096^3 f64 2363 -> 2072 us (66.3 TFLOP/s; the library
// 67-69), f32 1120 -> 1017 us; 2000 x 1500 x 2500 f64 344 -> 269 us, f32 189 -> 144 us.
template <typename T, bool TA, bool TB, bool UPPER, int TM, int TN, int BK, bool SCALED>
__global__ void __launch_bounds__(kThreads, 2)
gemm_mfma(const T *__restrict__ A, const T *__restrict__ B, T *__restrict__ C, int64_t M, int64_t N, int64_t K,
          int64_t lda, int64_t ldb, int64_t ldc, T alpha, T beta) {
    constexpr int BM = 32 * TM, BN = 32 * TN;
    typedef Tile<T, !TA, BM, BK> ATile;
    typedef Tile<T, TB, BN, BK> BTile;
    __shared__ __attribute__((aligned(16))) T As[2][ATile::LDS];
    __shared__ __attribute__((aligned(16))) T Bs[2][BTile::LDS];

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t bm = static_cast<int64_t>(blockIdx.y) * BM, bn = static_cast<int64_t>(blockIdx.x) * BN;
    if (UPPER && bm > bn + BN - 1) return;  // the whole tile lies below the diagonal
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    const bool a_edge = bm + BM > M, b_edge = bn + BN > N;

    typename Mfma<T>::Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = T(0);

    auto multiply = [&](int buf) {
        const T *as = As[buf], *bs = Bs[buf];
#pragma unroll
        for (int ks = 0; ks < BK; ks += 4) {
            const int kr = ks + (lane >> 4);
            T a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = ATile::read(as, wm + i * 16 + (lane & 15), kr);
#pragma unroll
            for (int j = 0; j < TN; ++j) b[j] = BTile::read(bs, wn + j * 16 + (lane & 15), kr);
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = Mfma<T>::step(a[i], b[j], acc[i][j]);
        }
    };
    ATile ta;
    BTile tb;
    if (K > 0) {
        const int kn = K % BK != 0 ? static_cast<int>(K % BK) : BK;
        ta.first(A, lda, bm, M, kn);
        tb.first(B, ldb, bn, N, kn);
        ta.store(As[0], a_edge, bm, M);
        tb.store(Bs[0], b_edge, bn, N);
        __syncthreads();
        int buf = 0;
        for (int64_t k = kn; k < K; k += BK) {
            ta.next();
            tb.next();
            loads_before_products<T>();
            multiply(buf);
            buf ^= 1;
            ta.store(As[buf], a_edge, bm, M);
            tb.store(Bs[buf], b_edge, bn, N);
            // the buffer is complete, and every wave is done reading the other before it is refilled
            __syncthreads();
        }
        multiply(buf);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = bm + wm + i * 16 + Mfma<T>::row(lane, r);
                const int64_t col = bn + wn + j * 16 + (lane & 15);
                if (row < M && col < N && (!UPPER || row <= col)) {
                    if (SCALED) {
                        T v = alpha * acc[i][j][r];
                        if (beta != T(0)) v += beta * C[row * ldc + col];
                        C[row * ldc + col] = v;
                    } else {
                        C[row * ldc + col] = acc[i][j][r];
                    }
                }
            }
}

template <typename R> struct alignas(2 * sizeof(R)) Cplx {
    R re, im;
};

template <typename T> __device__ __forceinline__ T conj_of(T x) { return x; }
template <typename R> __device__ __forceinline__ Cplx<R> conj_of(Cplx<R> z) { return {z.re, -z.im}; }
template <typename T> __device__ __forceinline__ T real_of(T x) { return x; }
template <typename R> __device__ __forceinline__ Cplx<R> real_of(Cplx<R> z) { return {z.re, R(0)}; }
template <typename T> struct One {
    static __device__ __forceinline__ T get() { return T(1); }
};
template <typename R> struct One<Cplx<R>> {
    static __device__ __forceinline__ Cplx<R> get() { return {R(1), R(0)}; }
};
// s - a x
template <typename T> __device__ __forceinline__ T msub(T s, T a, T x) { return fma(-a, x, s); }
template <typename R> __device__ __forceinline__ Cplx<R> msub(Cplx<R> s, Cplx<R> a, Cplx<R> x) {
    return {fma(a.im, x.im, fma(-a.re, x.re, s.re)), fma(-a.im, x.re, fma(-a.re, x.im, s.im))};
}

// Complex on the matrix cores: C = alpha op(A) op(B) + beta C with op(B)(k, n) = conj(B[n * ldb + k]) when
// CONJB; REALDIAG stores the diagonal with a zero imaginary part (Hermitian results).  Each complex MFMA
// tile is four real ones (re += ar br, re += (-ai) bi, im += ar bi, im += ai br), so one LDS read of a complex
// element feeds two operands and the kernel is bound by the MFMA rate: per K step of BK a wave issues
// TM TN BK MFMAs of 64 (f64) or 32 (f32) cycles for (TM + TN) BK / 4 LDS reads.  Tiles, staging and double
// buffering as in gemm_mfma; the LDS rows are padded to an odd number of 16-byte elements (c128) or to two
// 8-byte elements more than a multiple of 16 (c64), so the 16-lane groups of a read fall in disjoint banks.
// Measured against one FMA thread per element of C: 4096^3 c128 24.4 -> 7.74 ms (22.5 -> 71.0 TFLOP/s), c64
// 34.5 -> 131.8 TFLOP/s; 2000 x 1500 x 2500 c128 2771 -> 920 us.  The matrix cores are busy 86 % of the cycles (c128).
template <typename R, bool KCONT, int ROWS, int kBK>
struct CTile {
    static constexpr int CH = ROWS * kBK / kThreads;
    static constexpr int KPAD = sizeof(R) == 8 ? 1 : 2;
    static constexpr int RPAD = sizeof(R) == 8 ? 0 : 16;
    static constexpr int LDS = KCONT ? ROWS * (kBK + KPAD) : kBK * (ROWS + RPAD);
    static_assert(CH * kThreads == ROWS * kBK, "tile / thread count");

    const Cplx<R> *p[CH];  // the elements of the next step
    int64_t advance;
    Cplx<R> reg[CH];

    static __device__ __forceinline__ void place(int e, int &r, int &k) {
        const int c = static_cast<int>(threadIdx.x) + e * kThreads;
        r = KCONT ? c / kBK : c % ROWS;
        k = KCONT ? c % kBK : c / ROWS;
    }
    // As Tile::first and next; rows past Rn repeat row Rn - 1.
    __device__ __forceinline__ void first(const Cplx<R> *__restrict__ P, int64_t ld, int64_t r0, int64_t Rn, int kn) {
        advance = KCONT ? kBK : kBK * ld;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            int r, k;
            place(e, r, k);
            const int64_t gr = r0 + r < Rn ? r0 + r : Rn - 1;
            const Cplx<R> *q = KCONT ? P + gr * ld + k : P + k * ld + gr;
            reg[e] = k < kn ? *q : Cplx<R>{R(0), R(0)};
            p[e] = q + (KCONT ? kn : kn * ld);
        }
    }
    __device__ __forceinline__ void next() {
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            reg[e] = *p[e];
            p[e] += advance;
        }
    }
    __device__ __forceinline__ void store(Cplx<R> *lds) const {
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            int r, k;
            place(e, r, k);
            lds[KCONT ? r * (kBK + KPAD) + k : k * (ROWS + RPAD) + r] = reg[e];
        }
    }
    static __device__ __forceinline__ Cplx<R> read(const Cplx<R> *lds, int r, int k) {
        return lds[KCONT ? r * (kBK + KPAD) + k : k * (ROWS + RPAD) + r];
    }
};

template <typename R, bool TA, bool TB, bool CONJB, bool UPPER, bool REALDIAG, bool SCALED, int TM, int TN, int BK>
__global__ void __launch_bounds__(kThreads, 2)
gemm_complex(const Cplx<R> *__restrict__ A, const Cplx<R> *__restrict__ B, Cplx<R> *__restrict__ C, int64_t M,
             int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, R alpha, R beta) {
    constexpr int BM = 32 * TM, BN = 32 * TN;
    typedef CTile<R, !TA, BM, BK> ATile;
    typedef CTile<R, TB, BN, BK> BTile;
    __shared__ __attribute__((aligned(16))) Cplx<R> As[2][ATile::LDS];
    __shared__ __attribute__((aligned(16))) Cplx<R> Bs[2][BTile::LDS];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t bm = static_cast<int64_t>(blockIdx.y) * BM, bn = static_cast<int64_t>(blockIdx.x) * BN;
    if (UPPER && bm > bn + BN - 1) return;  // the whole tile lies below the diagonal
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    typename Mfma<R>::Acc re[TM][TN], im[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) re[i][j][r] = im[i][j][r] = R(0);
    auto multiply = [&](int buf) {
        const Cplx<R> *as = As[buf], *bs = Bs[buf];
#pragma unroll
        for (int ks = 0; ks < BK; ks += 4) {
            const int kr = ks + (lane >> 4);
            Cplx<R> a[TM], b[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) a[i] = ATile::read(as, wm + i * 16 + (lane & 15), kr);
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                b[j] = BTile::read(bs, wn + j * 16 + (lane & 15), kr);
                if (CONJB) b[j].im = -b[j].im;
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const R nai = -a[i].im;
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    re[i][j] = Mfma<R>::step(a[i].re, b[j].re, re[i][j]);
                    im[i][j] = Mfma<R>::step(a[i].re, b[j].im, im[i][j]);
                    re[i][j] = Mfma<R>::step(nai, b[j].im, re[i][j]);
                    im[i][j] = Mfma<R>::step(a[i].im, b[j].re, im[i][j]);
                }
            }
        }
    };
    ATile ta;
    BTile tb;
    if (K > 0) {
        const int kn = K % BK != 0 ? static_cast<int>(K % BK) : BK;
        ta.first(A, lda, bm, M, kn);
        tb.first(B, ldb, bn, N, kn);
        ta.store(As[0]);
        tb.store(Bs[0]);
        __syncthreads();
        int buf = 0;
        for (int64_t k = kn; k < K; k += BK) {
            ta.next();
            tb.next();
            loads_before_products<R>();
            multiply(buf);
            buf ^= 1;
            ta.store(As[buf]);
            tb.store(Bs[buf]);
            // the buffer is complete, and every wave is done reading the other before it is refilled
            __syncthreads();
        }
        multiply(buf);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t row = bm + wm + i * 16 + Mfma<R>::row(lane, r);
                const int64_t col = bn + wn + j * 16 + (lane & 15);
                if (row < M && col < N && (!UPPER || row <= col)) {
                    Cplx<R> v = {re[i][j][r], im[i][j][r]};
                    if (SCALED) {
                        v.re *= alpha;
                        v.im *= alpha;
                        if (beta != R(0)) {
                            const Cplx<R> c = C[row * ldc + col];
                            v.re = fma(beta, c.re, v.re);
                            v.im = fma(beta, c.im, v.im);
                        }
                    }
                    if (REALDIAG && row == col) v.im = 0;
                    C[row * ldc + col] = v;
                }
            }
}

// ---- small products: K split over the waves of a workgroup.  A product with few tiles leaves most CUs idle
// in the kernels above (100 x 100 x 4000: 4 workgroups), and each of its tiles is one serial chain over
// K.  Here a workgroup computes a 16 TM x 16 TN tile with WAVES waves, wave w the K steps w, w + WAVES, ...
// of 16, straight from global memory (no sharing to stage for; a lane loads 4 neighbouring k where K is
// contiguous), and the partial tiles are folded through LDS in a fixed order.  Measured: 100 x 100 x 4000 f64
// 323 -> 24 us, f32 204 -> 11, c128 292 -> 43; 512^3 f64 30 -> 9.4; 256^3 f64 16 -> 4.1, c128 14.6 -> 5.6;
// 2048 x 64 x 2048 f32 67 -> 11.4 us.
template <typename E> struct Prod {
    typedef typename Mfma<E>::Acc Acc;
    typedef E Real;
    static __device__ __forceinline__ E zero() { return E(0); }
    static __device__ __forceinline__ void clear(Acc &c) { c = Acc{}; }
    static __device__ __forceinline__ void step(E a, E b, Acc &c) { c = Mfma<E>::step(a, b, c); }
    static __device__ __forceinline__ void add(Acc &c, const Acc &d) { c += d; }
    static __device__ __forceinline__ E get(const Acc &c, int r) { return c[r]; }
    static __device__ __forceinline__ int row(int lane, int r) { return Mfma<E>::row(lane, r); }
    static __device__ __forceinline__ E scaled(E v, E alpha, E beta, const E *old) {
        v *= alpha;
        return beta != E(0) ? v + beta * *old : v;
    }
    static __device__ __forceinline__ E real_diagonal(E v) { return v; }
};
template <typename R> struct Prod<Cplx<R> > {
    typedef Cplx<R> E;
    typedef R Real;
    struct Acc {
        typename Mfma<R>::Acc re, im;
    };
    static __device__ __forceinline__ E zero() { return E{R(0), R(0)}; }
    static __device__ __forceinline__ void clear(Acc &c) { c.re = c.im = typename Mfma<R>::Acc{}; }
    static __device__ __forceinline__ void step(E a, E b, Acc &c) {
        c.re = Mfma<R>::step(a.re, b.re, c.re);
        c.im = Mfma<R>::step(a.re, b.im, c.im);
        c.re = Mfma<R>::step(-a.im, b.im, c.re);
        c.im = Mfma<R>::step(a.im, b.re, c.im);
    }
    static __device__ __forceinline__ void add(Acc &c, const Acc &d) {
        c.re += d.re;
        c.im += d.im;
    }
    static __device__ __forceinline__ E get(const Acc &c, int r) { return E{c.re[r], c.im[r]}; }
    static __device__ __forceinline__ int row(int lane, int r) { return Mfma<R>::row(lane, r); }
    static __device__ __forceinline__ E scaled(E v, R alpha, R beta, const E *old) {
        v.re *= alpha;
        v.im *= alpha;
        if (beta != R(0)) {
            v.re = fma(beta, old->re, v.re);
            v.im = fma(beta, old->im, v.im);
        }
        return v;
    }
    static __device__ __forceinline__ E real_diagonal(E v) { return E{v.re, R(0)}; }
};

template <typename E, bool TA, bool TB, bool CONJB, bool UPPER, bool REALDIAG, bool SCALED, int TM, int TN, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
gemm_slice(const E *__restrict__ A, const E *__restrict__ B, E *__restrict__ C, int64_t M, int64_t N, int64_t K,
           int64_t lda, int64_t ldb, int64_t ldc, typename Prod<E>::Real alpha, typename Prod<E>::Real beta) {
    typedef Prod<E> P;
    constexpr int BM = 16 * TM, BN = 16 * TN, KC = 16;
    __shared__ __attribute__((aligned(16))) typename P::Acc part[WAVES > 1 ? WAVES / 2 : 1][TM * TN][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t bm = static_cast<int64_t>(blockIdx.y) * BM, bn = static_cast<int64_t>(blockIdx.x) * BN;
    if (UPPER && bm > bn + BN - 1) return;  // the whole tile lies below the diagonal
    typename P::Acc acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) P::clear(acc[i][j]);
    // rows and columns past the edges repeat the last one: their results are not stored
    int64_t row[TM], col[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) row[i] = bm + i * 16 + (lane & 15) < M ? bm + i * 16 + (lane & 15) : M - 1;
#pragma unroll
    for (int j = 0; j < TN; ++j) col[j] = bn + j * 16 + (lane & 15) < N ? bn + j * 16 + (lane & 15) : N - 1;
    const int q = (lane >> 4) * 4;
    E a[2][TM][4], b[2][TN][4];
    auto load = [&](int64_t k0, int w) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int64_t k = k0 + q + s;
            const bool in = k < K;
#pragma unroll
            for (int i = 0; i < TM; ++i) a[w][i][s] = in ? (TA ? A[k * lda + row[i]] : A[row[i] * lda + k]) : P::zero();
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                E v = in ? (TB ? B[col[j] * ldb + k] : B[k * ldb + col[j]]) : P::zero();
                b[w][j][s] = CONJB ? conj_of(v) : v;
            }
        }
    };
    auto load_in = [&](int64_t k0, int w) {  // a whole step: no bounds checks
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int64_t k = k0 + q + s;
#pragma unroll
            for (int i = 0; i < TM; ++i) a[w][i][s] = TA ? A[k * lda + row[i]] : A[row[i] * lda + k];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const E v = TB ? B[col[j] * ldb + k] : B[k * ldb + col[j]];
                b[w][j][s] = CONJB ? conj_of(v) : v;
            }
        }
    };
    auto multiply = [&](int w) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) P::step(a[w][i][s], b[w][j][s], acc[i][j]);
    };
    const int64_t whole = K / KC;  // steps of 16 without a remainder
    int64_t c = wave;
    if (c < whole) load_in(c * KC, 0);
    for (; c + WAVES < whole; c += 2 * WAVES) {  // two steps a round, the next one loaded while one is multiplied
        load_in((c + WAVES) * KC, 1);
        multiply(0);
        if (c + 2 * WAVES < whole) load_in((c + 2 * WAVES) * KC, 0);
        multiply(1);
    }
    if (c < whole) multiply(0);
    if (whole * KC < K && wave == static_cast<int>(whole % WAVES)) {
        load(whole * KC, 0);
        multiply(0);
    }
#pragma unroll
    for (int h = WAVES / 2; h >= 1; h /= 2) {
        if (wave >= h && wave < 2 * h)
#pragma unroll
            for (int t = 0; t < TM * TN; ++t) part[wave - h][t][lane] = acc[t / TN][t % TN];
        __syncthreads();
        if (wave < h)
#pragma unroll
            for (int t = 0; t < TM * TN; ++t) P::add(acc[t / TN][t % TN], part[wave][t][lane]);
        __syncthreads();
    }
    if (wave != 0) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t m = bm + i * 16 + P::row(lane, r), n = bn + j * 16 + (lane & 15);
                if (m >= M || n >= N || (UPPER && m > n)) continue;
                E v = P::get(acc[i][j], r);
                if (SCALED) v = P::scaled(v, alpha, beta, C + m * ldc + n);
                if (REALDIAG && m == n) v = P::real_diagonal(v);
                C[m * ldc + n] = v;
            }
}

// out (m x m, leading dimension m) from the upper triangle of A (i <= j read, the rest not
// referenced): SYM mirrors it, HERM mirrors it conjugated with a real diagonal, UNIT is the unit
// upper triangular matrix (ones on the diagonal, zeros below).
enum class Fill { SYM, HERM, UNIT };

template <typename T, Fill F>
__global__ void __launch_bounds__(256) fill_from_upper(const T *__restrict__ A, int64_t lda, T *__restrict__ out,
                                                       int64_t m) {
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 16 + (threadIdx.x & 15);
    const int64_t i = static_cast<int64_t>(blockIdx.y) * 16 + (threadIdx.x >> 4);
    if (i >= m || j >= m) return;
    T v;
    if (i < j)
        v = A[i * lda + j];
    else if (i > j)
        v = F == Fill::UNIT ? T{} : F == Fill::HERM ? conj_of(A[j * lda + i]) : A[j * lda + i];
    else
        v = F == Fill::UNIT ? One<T>::get() : F == Fill::HERM ? real_of(A[i * lda + i]) : A[i * lda + i];
    out[i * m + j] = v;
}

// Solves U X = B in place for one diagonal block of a unit upper triangular system: U is the nb x nb
// block at A (leading dimension lda; its diagonal and lower part are not referenced), B the nb rows
// at B (leading dimension ldb, n columns).  One thread per column keeps the column in registers
// (rows past nb are zero and not stored) and substitutes backwards with U's block from LDS.
template <typename T, int NB>
__global__ void __launch_bounds__(256) trsm_unit_upper_block(const T *__restrict__ A, int64_t lda,
                                                             T *__restrict__ B, int64_t ldb, int nb, int64_t n) {
    __shared__ T U[NB][NB + 1];
    for (int e = threadIdx.x; e < NB * NB; e += 256) {
        const int i = e / NB, k = e % NB;
        U[i][k] = (k > i && k < nb) ? A[static_cast<int64_t>(i) * lda + k] : T{};
    }
    __syncthreads();
    const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (j >= n) return;
    T x[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) x[i] = i < nb ? B[i * ldb + j] : T{};
#pragma unroll
    for (int i = NB - 2; i >= 0; --i) {
        T s = x[i];
#pragma unroll
        for (int k = i + 1; k < NB; ++k) s = msub(s, U[i][k], x[k]);
        x[i] = s;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
        if (i < nb) B[i * ldb + j] = x[i];
}

thread_local std::string g_err;

// One GEMM call: C = alpha op(A) op(B) + beta C.
struct Gemm {
    int dtype;
    int64_t m, n, k;
    const void *A;
    int64_t lda;
    const void *B;
    int64_t ldb;
    void *C;
    int64_t ldc;
    double alpha, beta;
    hipStream_t s;
};

int64_t tiles(const Gemm &g, int64_t bm, int64_t bn) { return ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn); }

// The 256 CUs need a workgroup each: fewer 64 x 64 tiles than that, and K is split over waves instead
// (gemm_slice), with the largest tile that still gives 256 workgroups.  Measured, tile / slice: 1001 x 777 x
// 1303 (208 tiles) f64 66 / 60 us, f32 40 / 38, c128 186 / 201, c64 113 / 99; 512^3 (64 tiles) f64 25 / 9.4,
// f32 15 / 6.1, c128 73 / 24, c64 46 / 13; 1024^3 (256 tiles) f64 49 / 51, f32 30 / 29, c128 148 / 157, c64 90 / 78; 2000 x
// 1500 x 2500 (768 tiles) f64 269 / 349, f32 144 / 210, c128 919 / 1101, c64 510 / 540.
// (The tiles' chunks need as many rows and columns as a vector has elements.)
constexpr int64_t kFill = 256;
bool use_tiles(const Gemm &g) { return tiles(g, 64, 64) >= kFill && g.m >= 16 && g.n >= 16; }

template <typename E, bool TA, bool TB, bool CONJB, bool UPPER, bool REALDIAG, bool SCALED, int TM, int TN, int WAVES>
void launch_slice_tile(const Gemm &g) {
    typedef typename Prod<E>::Real R;
    const dim3 grid(static_cast<unsigned>((g.n + 16 * TN - 1) / (16 * TN)),
                    static_cast<unsigned>((g.m + 16 * TM - 1) / (16 * TM)));
    gemm_slice<E, TA, TB, CONJB, UPPER, REALDIAG, SCALED, TM, TN, WAVES><<<grid, 64 * WAVES, 0, g.s>>>(
        static_cast<const E *>(g.A), static_cast<const E *>(g.B), static_cast<E *>(g.C), g.m, g.n, g.k, g.lda, g.ldb,
        g.ldc, static_cast<R>(g.alpha), static_cast<R>(g.beta));
}

template <typename E, bool TA, bool TB, bool CONJB, bool UPPER, bool REALDIAG, bool SCALED>
void launch_slice(const Gemm &g) {
    // One or two steps of K: further waves would only wait for the fold (8 x 30000 x 16 c128 17.9 us with a 32 x 32 tile of
    // 4 waves, 4.4 so; 900 x 900 x 16 f64 6.6 -> 4.6).  16 rows or columns at most: a tile of 32 is at least half padding, and
    // complex products are bound by its MFMAs (15 x 20000 x 200 c128 37.5 us, 20.4 with the small tile).
    constexpr bool complex = sizeof(E) != sizeof(typename Prod<E>::Real);
    if (g.k <= 32)
        launch_slice_tile<E, TA, TB, CONJB, UPPER, REALDIAG, SCALED, 1, 1, 2>(g);
    else if (tiles(g, 32, 32) >= kFill && !(complex && std::min(g.m, g.n) <= 16))
        launch_slice_tile<E, TA, TB, CONJB, UPPER, REALDIAG, SCALED, 2, 2, 4>(g);
    else if (!complex && tiles(g, 16, 32) >= kFill)
        launch_slice_tile<E, TA, TB, CONJB, UPPER, REALDIAG, SCALED, 1, 2, 8>(g);
    else
        launch_slice_tile<E, TA, TB, CONJB, UPPER, REALDIAG, SCALED, 1, 1, 8>(g);
}

template <typename T, bool TA, bool TB, bool UPPER, bool SCALED, int TM>
void launch_real_tile(const Gemm &g) {
    const dim3 grid(static_cast<unsigned>((g.n + 32 * TM - 1) / (32 * TM)),
                    static_cast<unsigned>((g.m + 32 * TM - 1) / (32 * TM)));
    gemm_mfma<T, TA, TB, UPPER, TM, TM, 16, SCALED><<<grid, kThreads, 0, g.s>>>(
        static_cast<const T *>(g.A), static_cast<const T *>(g.B), static_cast<T *>(g.C), g.m, g.n, g.k, g.lda, g.ldb,
        g.ldc, static_cast<T>(g.alpha), static_cast<T>(g.beta));
}

template <typename T, bool TA, bool TB, bool UPPER, bool SCALED>
void launch_real_scaled(const Gemm &g) {
    // 128 x 128 tiles when the matrix gives every CU two workgroups of them, else 64 x 64
    if (!use_tiles(g))
        launch_slice<T, TA, TB, false, UPPER, false, SCALED>(g);
    else if (tiles(g, 128, 128) >= 2 * kFill)
        launch_real_tile<T, TA, TB, UPPER, SCALED, 4>(g);
    else
        launch_real_tile<T, TA, TB, UPPER, SCALED, 2>(g);
}

template <typename T, bool TA, bool TB, bool UPPER>
bool launch_real(const Gemm &g) {
    if (g.alpha == 1.0 && g.beta == 0.0) {
        launch_real_scaled<T, TA, TB, UPPER, false>(g);
    } else if constexpr (!TA) {  // trsm's updates and syr2k's second pass
        launch_real_scaled<T, TA, TB, UPPER, true>(g);
    } else {
        g_err = "bhblas: scaled product with a transposed A is not provided";
        return false;
    }
    return true;
}

template <typename R, bool TA, bool TB, bool CONJB, bool UPPER, bool REALDIAG, bool SCALED>
void launch_complex_scaled(const Gemm &g) {
    if (!use_tiles(g)) {
        launch_slice<Cplx<R>, TA, TB, CONJB, UPPER, REALDIAG, SCALED>(g);
        return;
    }
    constexpr int BK = sizeof(R) == 8 ? 8 : 16;
    const dim3 grid(static_cast<unsigned>((g.n + 63) / 64), static_cast<unsigned>((g.m + 63) / 64));
    gemm_complex<R, TA, TB, CONJB, UPPER, REALDIAG, SCALED, 2, 2, BK><<<grid, kThreads, 0, g.s>>>(
        static_cast<const Cplx<R> *>(g.A), static_cast<const Cplx<R> *>(g.B), static_cast<Cplx<R> *>(g.C), g.m, g.n,
        g.k, g.lda, g.ldb, g.ldc, static_cast<R>(g.alpha), static_cast<R>(g.beta));
}

template <typename R, bool TA, bool TB, bool CONJB, bool UPPER, bool REALDIAG>
void launch_complex(const Gemm &g) {
    if (g.alpha == 1.0 && g.beta == 0.0)
        launch_complex_scaled<R, TA, TB, CONJB, UPPER, REALDIAG, false>(g);
    else
        launch_complex_scaled<R, TA, TB, CONJB, UPPER, REALDIAG, true>(g);
}

int launch_status() {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_err = std::string("bhblas: launch failed: ") + hipGetErrorString(e);
        return 1;
    }
    return 0;
}

bool is_complex(int dtype) { return dtype == BHBLAS_C64 || dtype == BHBLAS_C128; }

int64_t elem_size(int dtype) {
    switch (dtype) {
        case BHBLAS_F32: return 4;
        case BHBLAS_F64: return 8;
        case BHBLAS_C64: return 8;
        case BHBLAS_C128: return 16;
        default: return 0;
    }
}

// Checks the sizes and the type of a call over m x n (and k); false with g_err set when they are
// unusable.  Grid y carries 16-row tiles, at most 65535 of them.
bool check_call(int dtype, int64_t m, int64_t n, int64_t k) {
    if (elem_size(dtype) == 0) {
        g_err = "bhblas: unsupported type";
        return false;
    }
    if (m < 0 || n < 0 || k < 0) {
        g_err = "bhblas: negative matrix size";
        return false;
    }
    if ((m + 15) / 16 > 65535 || (n + 15) / 16 > 0x7fffffffLL) {
        g_err = "bhblas: matrix too large for one launch";
        return false;
    }
    return true;
}

template <bool TA, bool TB, bool UPPER, bool CONJB = false, bool REALDIAG = false>
int dispatch(const Gemm &g) {
    if (!check_call(g.dtype, g.m, g.n, g.k)) return 1;
    if (g.m == 0 || g.n == 0) return 0;
    switch (g.dtype) {
        case BHBLAS_F32:
            if (!launch_real<float, TA, TB, UPPER>(g)) return 1;
            break;
        case BHBLAS_F64:
            if (!launch_real<double, TA, TB, UPPER>(g)) return 1;
            break;
        case BHBLAS_C64: launch_complex<float, TA, TB, CONJB, UPPER, REALDIAG>(g); break;
        case BHBLAS_C128: launch_complex<double, TA, TB, CONJB, UPPER, REALDIAG>(g); break;
    }
    return launch_status();
}

Gemm make_gemm(int dtype, int64_t m, int64_t n, int64_t k, const void *A, int64_t lda, const void *B, int64_t ldb,
               void *C, int64_t ldc, void *stream, double alpha = 1.0, double beta = 0.0) {
    return Gemm{dtype, m, n, k, A, lda, B, ldb, C, ldc, alpha, beta, static_cast<hipStream_t>(stream)};
}

// Stream-ordered device temporary, released on the same stream.
struct DeviceTemp {
    void *p = nullptr;
    hipStream_t s;
    explicit DeviceTemp(hipStream_t st) : s(st) {}
    bool alloc(size_t bytes) {
        if (bytes == 0) return true;
        if (hipMallocAsync(&p, bytes, s) != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();
            g_err = "bhblas: out of device memory for a temporary of " + std::to_string(bytes) + " bytes";
            return false;
        }
        return true;
    }
    ~DeviceTemp() {
        if (p != nullptr) (void)hipFreeAsync(p, s);
    }
};

template <Fill F> int fill(int dtype, const void *A, int64_t lda, void *out, int64_t m, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>((m + 15) / 16), static_cast<unsigned>((m + 15) / 16));
    switch (dtype) {
        case BHBLAS_F32: fill_from_upper<float, F><<<grid, 256, 0, s>>>(static_cast<const float *>(A), lda,
                                                                         static_cast<float *>(out), m); break;
        case BHBLAS_F64: fill_from_upper<double, F><<<grid, 256, 0, s>>>(static_cast<const double *>(A), lda,
                                                                          static_cast<double *>(out), m); break;
        case BHBLAS_C64: fill_from_upper<Cplx<float>, F><<<grid, 256, 0, s>>>(
            static_cast<const Cplx<float> *>(A), lda, static_cast<Cplx<float> *>(out), m); break;
        case BHBLAS_C128: fill_from_upper<Cplx<double>, F><<<grid, 256, 0, s>>>(
            static_cast<const Cplx<double> *>(A), lda, static_cast<Cplx<double> *>(out), m); break;
    }
    return launch_status();
}

// C = F(A) B with F(A) expanded from A's upper triangle into an m x m buffer: a stream-ordered
// temporary, or `staging` when the caller supplies one of at least m * m elements.
template <Fill F>
int expanded_product(int dtype, int64_t m, int64_t n, const void *A, int64_t lda, const void *B, int64_t ldb,
                     void *C, int64_t ldc, void *stream, void *staging = nullptr) {
    if (!check_call(dtype, m, n, m)) return 1;
    if (m == 0 || n == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    DeviceTemp full(s);
    void *expanded = staging;
    if (expanded == nullptr) {
        if (!full.alloc(static_cast<size_t>(m * m * elem_size(dtype)))) return 1;
        expanded = full.p;
    }
    if (fill<F>(dtype, A, lda, expanded, m, s) != 0) return 1;
    return dispatch<false, false, false>(make_gemm(dtype, m, n, m, expanded, m, B, ldb, C, ldc, stream));
}

template <typename T, int NB>
void trsm_block(const void *A, int64_t lda, void *B, int64_t ldb, int nb, int64_t n, hipStream_t s) {
    trsm_unit_upper_block<T, NB><<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(
        static_cast<const T *>(A), lda, static_cast<T *>(B), ldb, nb, n);
}

// ------------------------------------------------------------ extension methods

using bohrium::extmethod::ExtmethodImpl;

int blas_type(const bh_view &v) {
    switch (v.base->dtype()) {
        case bh_type::FLOAT32: return BHBLAS_F32;
        case bh_type::FLOAT64: return BHBLAS_F64;
        case bh_type::COMPLEX64: return BHBLAS_C64;
        case bh_type::COMPLEX128: return BHBLAS_C128;
        default: return -1;
    }
}

// A 2-D C-contiguous view: row-major with unit inner stride and outer stride = columns.
void require_matrix(const bh_view &v, const char *what, const std::string &method) {
    if (v.isConstant() || v.ndim != 2 || v.stride[1] != 1 || v.stride[0] != v.shape[1])
        throw std::runtime_error(method + ": " + what + " must be a C-contiguous 2-d array");
}

enum class Kind { GEMM, GEMMT, SYMM, HEMM, SYRK, HERK, SYR2K, HER2K, TRMM, TRSM };

// The reference's methods table (extmethods/blas/templates/methods.json): operands (C, A[, B]),
// row-major, CblasUpper / CblasLeft / CblasNoTrans / CblasUnit, alpha 1 and beta 0.
class BlasMethod : public ExtmethodImpl {
    Kind kind;
    std::string name;

public:
    BlasMethod(Kind k, const char *n) : kind(k), name(n) {}
    void execute(bh_instruction *instr, void *arg) override {
        const bh_hip_ext_context *ctx = static_cast<const bh_hip_ext_context *>(arg);
        if (ctx == nullptr || ctx->version != 1) throw std::runtime_error(name + ": needs the hip engine's context");
        const bool only_a = kind == Kind::SYRK || kind == Kind::HERK;
        if (instr->operand.size() != (only_a ? 2u : 3u)) throw std::runtime_error(name + ": wrong number of operands");
        const bool triangular = kind == Kind::TRMM || kind == Kind::TRSM;  // C is not used
        const bh_view &C = instr->operand[0], &A = instr->operand[1];
        if (!triangular) require_matrix(C, "C", name);
        require_matrix(A, "A", name);
        const int dt = blas_type(A);
        const bool complex_only = kind == Kind::HEMM || kind == Kind::HERK || kind == Kind::HER2K;
        if (dt < 0 || (complex_only && !is_complex(dt)))
            throw std::runtime_error(std::string(bh_type_text(A.base->dtype())) + " not supported by BLAS for '" +
                                     name + "'.");
        if (!triangular && C.base->dtype() != A.base->dtype())
            throw std::runtime_error(name + ": operands differ in type");
        const int64_t am = A.shape[0], ak = A.shape[1];
        const int esize = bh_type_size(A.base->dtype());
        auto ptr = [&](const bh_view &v) {
            return static_cast<char *>(ctx->device_pointer(ctx->engine, v.base)) + v.start * esize;
        };
        auto shape_error = [&](const char *what) { throw std::runtime_error(name + ": " + what); };
        if (only_a) {
            if (C.shape[0] != am || C.shape[1] != am) shape_error("C must be n x n for A n x k");
            if (ctx->dry_run) return;
            const int rc = kind == Kind::SYRK ? bhblas_syrk(dt, am, ak, ptr(A), ak, ptr(C), am, ctx->stream)
                                              : bhblas_herk(dt, am, ak, ptr(A), ak, ptr(C), am, ctx->stream);
            if (rc != 0) throw std::runtime_error(name + ": " + g_err);
            return;
        }
        const bh_view &B = instr->operand[2];
        require_matrix(B, "B", name);
        if (B.base->dtype() != A.base->dtype()) throw std::runtime_error(name + ": operands differ in type");
        const int64_t bm = B.shape[0], bn = B.shape[1];
        int rc = 0;
        switch (kind) {
            case Kind::GEMM:
                if (bm != ak || C.shape[0] != am || C.shape[1] != bn)
                    shape_error("shapes do not chain (A m x k, B k x n, C m x n)");
                if (ctx->dry_run) return;
                rc = bhblas_gemm(dt, 0, am, bn, ak, ptr(A), ak, ptr(B), bn, ptr(C), bn, ctx->stream);
                break;
            case Kind::GEMMT:
                if (bm != am || C.shape[0] != ak || C.shape[1] != bn)
                    shape_error("shapes do not chain (A m x k, B m x n, C k x n)");
                if (ctx->dry_run) return;
                rc = bhblas_gemm(dt, 1, ak, bn, am, ptr(A), ak, ptr(B), bn, ptr(C), bn, ctx->stream);
                break;
            case Kind::SYMM:
            case Kind::HEMM:
                if (ak != am || bm != am || C.shape[0] != am || C.shape[1] != bn)
                    shape_error("shapes do not chain (A m x m, B m x n, C m x n)");
                if (ctx->dry_run) return;
                rc = (kind == Kind::SYMM ? bhblas_symm : bhblas_hemm)(dt, am, bn, ptr(A), ak, ptr(B), bn, ptr(C), bn,
                                                                      ctx->stream);
                break;
            case Kind::SYR2K:
            case Kind::HER2K:
                if (bm != am || bn != ak || C.shape[0] != am || C.shape[1] != am)
                    shape_error("shapes do not chain (A n x k, B n x k, C n x n)");
                if (ctx->dry_run) return;
                rc = (kind == Kind::SYR2K ? bhblas_syr2k : bhblas_her2k)(dt, am, ak, ptr(A), ak, ptr(B), bn, ptr(C),
                                                                         am, ctx->stream);
                break;
            case Kind::TRMM:
            case Kind::TRSM:
                if (ak != am || bm != am) shape_error("shapes do not chain (A m x m, B m x n)");
                if (ctx->dry_run) return;
                rc = (kind == Kind::TRMM ? bhblas_trmm : bhblas_trsm)(dt, am, bn, ptr(A), ak, ptr(B), bn, ctx->stream);
                break;
            default: break;
        }
        if (rc != 0) throw std::runtime_error(name + ": " + g_err);
    }
};

} // namespace

// Staging area of bhblas_symm_noalloc: the expanded m x m matrix lives here instead of in a
// temporary.  Every device that runs the library holds its own copy (at its own address) until
// the process ends.  In host code `scratch` names a host-side stand-in, never the device memory:
// host code uses only the address that hipGetSymbolAddress returned for the current device.
static constexpr size_t kScratchBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_addr[kMaxDevices] = {};

// The device address of `scratch` on the current device, looked up once per device.
int scratch_address(void **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        (void)hipGetLastError();
        g_err = "bhblas: no usable current device for the staging area";
        return 1;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_addr[dev] == nullptr) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            (void)hipGetLastError();
            g_err = std::string("bhblas: hipGetSymbolAddress of the staging area failed: ") + hipGetErrorString(e);
            return 1;
        }
        g_scratch_addr[dev] = p;
    }
    *out = g_scratch_addr[dev];
    return 0;
}

} // namespace

extern "C" {

int bhblas_gemm(int dtype, int trans_a, int64_t m, int64_t n, int64_t k, const void *A, int64_t lda, const void *B,
                int64_t ldb, void *C, int64_t ldc, void *stream) {
    const Gemm g = make_gemm(dtype, m, n, k, A, lda, B, ldb, C, ldc, stream);
    return trans_a ? dispatch<true, false, false>(g) : dispatch<false, false, false>(g);
}

int bhblas_syrk(int dtype, int64_t m, int64_t k, const void *A, int64_t lda, void *C, int64_t ldc, void *stream) {
    // C = A A^T: op(B)(kk, n) = A[n][kk], i.e. B = A read transposed.
    return dispatch<false, true, true>(make_gemm(dtype, m, m, k, A, lda, A, lda, C, ldc, stream));
}

int bhblas_herk(int dtype, int64_t n, int64_t k, const void *A, int64_t lda, void *C, int64_t ldc, void *stream) {
    if (!is_complex(dtype)) {
        g_err = "bhblas: herk needs a complex type";
        return 1;
    }
    return dispatch<false, true, true, true, true>(make_gemm(dtype, n, n, k, A, lda, A, lda, C, ldc, stream));
}

int bhblas_syr2k(int dtype, int64_t n, int64_t k, const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                 int64_t ldc, void *stream) {
    if (dispatch<false, true, true>(make_gemm(dtype, n, n, k, A, lda, B, ldb, C, ldc, stream)) != 0) return 1;
    return dispatch<false, true, true>(make_gemm(dtype, n, n, k, B, ldb, A, lda, C, ldc, stream, 1.0, 1.0));
}

int bhblas_her2k(int dtype, int64_t n, int64_t k, const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                 int64_t ldc, void *stream) {
    if (!is_complex(dtype)) {
        g_err = "bhblas: her2k needs a complex type";
        return 1;
    }
    if (dispatch<false, true, true, true, false>(make_gemm(dtype, n, n, k, A, lda, B, ldb, C, ldc, stream)) != 0)
        return 1;
    return dispatch<false, true, true, true, true>(make_gemm(dtype, n, n, k, B, ldb, A, lda, C, ldc, stream, 1.0, 1.0));
}

int bhblas_symm(int dtype, int64_t m, int64_t n, const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                int64_t ldc, void *stream) {
    return expanded_product<Fill::SYM>(dtype, m, n, A, lda, B, ldb, C, ldc, stream);
}

int bhblas_symm_noalloc(int dtype, int64_t m, int64_t n, const void *A, int64_t lda, const void *B, int64_t ldb,
                        void *C, int64_t ldc, void *stream) {
    if (!check_call(dtype, m, n, m)) return 1;
    if (m == 0 || n == 0) return 0;
    const uint64_t need = static_cast<uint64_t>(m) * static_cast<uint64_t>(m) * static_cast<uint64_t>(elem_size(dtype));
    if (need > kScratchBytes) {
        g_err = "bhblas: symm_noalloc needs m * m * element size <= " + std::to_string(kScratchBytes) +
                " bytes of staging, got " + std::to_string(need) + " (m = " + std::to_string(m) + ")";
        return 1;
    }
    void *staging = nullptr;
    if (scratch_address(&staging) != 0) return 1;
    return expanded_product<Fill::SYM>(dtype, m, n, A, lda, B, ldb, C, ldc, stream, staging);
}

int bhblas_hemm(int dtype, int64_t m, int64_t n, const void *A, int64_t lda, const void *B, int64_t ldb, void *C,
                int64_t ldc, void *stream) {
    if (!is_complex(dtype)) {
        g_err = "bhblas: hemm needs a complex type";
        return 1;
    }
    return expanded_product<Fill::HERM>(dtype, m, n, A, lda, B, ldb, C, ldc, stream);
}

int bhblas_trmm(int dtype, int64_t m, int64_t n, const void *A, int64_t lda, void *B, int64_t ldb, void *stream) {
    if (!check_call(dtype, m, n, m)) return 1;
    if (m == 0 || n == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t es = elem_size(dtype);
    DeviceTemp prod(s);
    if (!prod.alloc(static_cast<size_t>(m * n * es))) return 1;
    if (expanded_product<Fill::UNIT>(dtype, m, n, A, lda, B, ldb, prod.p, n, stream) != 0) return 1;
    if (hipMemcpy2DAsync(B, static_cast<size_t>(ldb * es), prod.p, static_cast<size_t>(n * es),
                         static_cast<size_t>(n * es), static_cast<size_t>(m), hipMemcpyDeviceToDevice, s) != hipSuccess) {
        (void)hipGetLastError();
        g_err = "bhblas: copy of the trmm product failed";
        return 1;
    }
    return 0;
}

int bhblas_trsm(int dtype, int64_t m, int64_t n, const void *A, int64_t lda, void *B, int64_t ldb, void *stream) {
    if (!check_call(dtype, m, n, m)) return 1;
    if (m == 0 || n == 0) return 0;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t es = elem_size(dtype);
    // Diagonal blocks of NB rows from the bottom up: solve the block in place, then take its
    // contribution out of every row above it with one GEMM (C = B above, alpha -1, beta 1).
    const int64_t NB = dtype == BHBLAS_C128 ? 32 : 64;
    const char *a = static_cast<const char *>(A);
    char *b = static_cast<char *>(B);
    for (int64_t r0 = ((m - 1) / NB) * NB; r0 >= 0; r0 -= NB) {
        const int nb = static_cast<int>(std::min(NB, m - r0));
        const void *ad = a + (r0 * lda + r0) * es;
        void *bd = b + r0 * ldb * es;
        switch (dtype) {
            case BHBLAS_F32: trsm_block<float, 64>(ad, lda, bd, ldb, nb, n, s); break;
            case BHBLAS_F64: trsm_block<double, 64>(ad, lda, bd, ldb, nb, n, s); break;
            case BHBLAS_C64: trsm_block<Cplx<float>, 64>(ad, lda, bd, ldb, nb, n, s); break;
            case BHBLAS_C128: trsm_block<Cplx<double>, 32>(ad, lda, bd, ldb, nb, n, s); break;
        }
        if (launch_status() != 0) return 1;
        if (r0 > 0 &&
            dispatch<false, false, false>(make_gemm(dtype, r0, n, nb, a + r0 * es, lda, bd, ldb, B, ldb, stream, -1.0,
                                                    1.0)) != 0)
            return 1;
    }
    return 0;
}

const char *bhblas_last_error(void) { return g_err.c_str(); }

#define BH_BLAS_METHOD(NAME, KIND)                                                                          \
    bh_extmethod_impl *blas_##NAME##_create(void) { return new BlasMethod(Kind::KIND, "blas_" #NAME); }    \
    void blas_##NAME##_destroy(bh_extmethod_impl *self) { delete self; }

BH_BLAS_METHOD(gemm, GEMM)
BH_BLAS_METHOD(gemmt, GEMMT)
BH_BLAS_METHOD(symm, SYMM)
BH_BLAS_METHOD(hemm, HEMM)
BH_BLAS_METHOD(syrk, SYRK)
BH_BLAS_METHOD(herk, HERK)
BH_BLAS_METHOD(syr2k, SYR2K)
BH_BLAS_METHOD(her2k, HER2K)
BH_BLAS_METHOD(trmm, TRMM)
BH_BLAS_METHOD(trsm, TRSM)

} // extern "C"
