// utr_fft.hpp -- LDS-resident Stockham FFT for gfx950 (device side).
//
// A workgroup transforms `nb` sequences of length N that sit contiguously in
// LDS (sequence-major).  Each radix-R pass with p = product of the previous
// radices reads x[i + r*N/R], twiddles it by w^(r*(i mod p)) with
// w = exp(sign*2*pi*i/(p*R)), applies a length-R DFT and writes
// y[(i/p)*p*R + (i mod p) + q*p]; after the last pass the data are in natural
// order (Stockham autosort, no bit reversal).  Two LDS buffers are used in
// ping-pong.  Twiddles come from a table computed in FP64 on the host.
//
// The forward transform replaces the FFTW plans of Fftwd2fc / Fftwd3frc used
// at UTR.cpp:851,994,1223-1232 (exponent sign -1 forward, +1 inverse,
// unnormalised).
#pragma once

#include <hip/hip_runtime.h>

namespace utr {

template <typename T>
struct cplx {
    T x, y;
};

// fused multiply-adds written out where a sum of two products leaves the
// compiler a choice, so that a transform rounds the same in every kernel
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
    return {fma_t(a.x, b.x, -(a.y * b.y)), fma_t(a.x, b.y, a.y * b.x)};
}
template <typename T>
__device__ __forceinline__ cplx<T> cadd(cplx<T> a, cplx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cplx<T> csub(cplx<T> a, cplx<T> b) { return {a.x - b.x, a.y - b.y}; }
// multiply by sign*i
template <typename T>
__device__ __forceinline__ cplx<T> mul_si(cplx<T> a, int sign) {
    return sign > 0 ? cplx<T>{-a.y, a.x} : cplx<T>{a.y, -a.x};
}

// ------------------------------------------------------------- LDS layout
// One pad entry after every 8: the strided writes of the first Stockham
// passes (stride R, then R*p for p < 64) then fall on distinct LDS banks
// instead of 4 to 16 lanes sharing one.  (The transposed column loads of
// 8 sequences of 256 still share banks; two layouts that spread them, an
// extra pad per 128 entries and an XOR swizzle, measured slower overall.)
// A buffer of n logical entries holds lds_len(n); entry i sits at lx(i).
__host__ __device__ constexpr int lds_len(int n) { return n + (n >> 3); }
__device__ __forceinline__ int lx(int i) { return i + (i >> 3); }

// ---------------------------------------------------------------- factors
struct FacList {
    int nf;
    int f[24];
    int p[24];    // product of earlier radices
    int off[24];  // twiddle-table offset of each pass
    int ntw;      // table length
};

// Radix order: an 8 first where 8 divides n, then the odd radices, then the
// other powers of two (8s, a 4, a 2): the first and the last radix divide 8,
// as fft_reg needs.
constexpr FacList factorize(int n) {
    FacList L{};
    L.nf = 0;
    int m = n;
    if (m % 8 == 0) { L.f[L.nf++] = 8; m /= 8; }
    while (m % 3 == 0) { L.f[L.nf++] = 3; m /= 3; }
    while (m % 5 == 0) { L.f[L.nf++] = 5; m /= 5; }
    int odd = m;
    while (odd % 2 == 0) odd /= 2;
    for (int q = 7; odd > 1; q += 2)
        while (odd % q == 0) { L.f[L.nf++] = q; m /= q; odd /= q; }
    while (m % 8 == 0) { L.f[L.nf++] = 8; m /= 8; }
    while (m % 4 == 0) { L.f[L.nf++] = 4; m /= 4; }
    while (m % 2 == 0) { L.f[L.nf++] = 2; m /= 2; }
    int p = 1, off = 0;
    for (int s = 0; s < L.nf; s++) {
        L.p[s] = p;
        L.off[s] = off;
        off += p * (L.f[s] - 1);
        p *= L.f[s];
    }
    L.ntw = off;
    return L;
}

// ---------------------------------------------------------- small DFTs
// In-place length-R DFT of u[0..R-1] with exponent sign*2*pi*i*r*q/R.
template <typename T, int R>
__device__ __forceinline__ void dft_small(cplx<T>* u, int sign) {
    if constexpr (R == 2) {
        cplx<T> a = u[0], b = u[1];
        u[0] = cadd(a, b);
        u[1] = csub(a, b);
    } else if constexpr (R == 4) {
        cplx<T> a0 = cadd(u[0], u[2]), a1 = csub(u[0], u[2]);
        cplx<T> b0 = cadd(u[1], u[3]), b1 = mul_si(csub(u[1], u[3]), sign);
        u[0] = cadd(a0, b0);
        u[2] = csub(a0, b0);
        u[1] = cadd(a1, b1);
        u[3] = csub(a1, b1);
    } else if constexpr (R == 8) {
        const T h = T(0.70710678118654752440);
        // radix-2 split: even/odd 4-point DFTs
        cplx<T> e[4] = {u[0], u[2], u[4], u[6]};
        cplx<T> o[4] = {u[1], u[3], u[5], u[7]};
        dft_small<T, 4>(e, sign);
        dft_small<T, 4>(o, sign);
        // o[q] times exp(sign*2*pi*i*q/8): o1, o3 are h t1, h t3
        const cplx<T> t1 = {o[1].x - sign * o[1].y, o[1].y + sign * o[1].x};
        const cplx<T> o2 = mul_si(o[2], sign);
        const cplx<T> t3 = {-o[3].x - sign * o[3].y, -o[3].y + sign * o[3].x};
        u[0] = cadd(e[0], o[0]);
        u[4] = csub(e[0], o[0]);
        u[1] = {fma_t(h, t1.x, e[1].x), fma_t(h, t1.y, e[1].y)};
        u[5] = {fma_t(-h, t1.x, e[1].x), fma_t(-h, t1.y, e[1].y)};
        u[2] = cadd(e[2], o2);
        u[6] = csub(e[2], o2);
        u[3] = {fma_t(h, t3.x, e[3].x), fma_t(h, t3.y, e[3].y)};
        u[7] = {fma_t(-h, t3.x, e[3].x), fma_t(-h, t3.y, e[3].y)};
    } else if constexpr (R == 3) {
        const T c1 = T(-0.5), s1 = T(0.86602540378443864676) * T(sign);
        cplx<T> a = u[0], b = u[1], c = u[2];
        cplx<T> t = cadd(b, c), d = csub(b, c);
        u[0] = cadd(a, t);
        cplx<T> m = {fma_t(c1, t.x, a.x), fma_t(c1, t.y, a.y)};
        u[1] = {fma_t(-s1, d.y, m.x), fma_t(s1, d.x, m.y)};
        u[2] = {fma_t(s1, d.y, m.x), fma_t(-s1, d.x, m.y)};
    } else if constexpr (R == 5) {
        const T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);
        const T s1 = T(0.95105651629515357212) * T(sign), s2 = T(0.58778525229247312917) * T(sign);
        cplx<T> a = u[0];
        cplx<T> t1 = cadd(u[1], u[4]), d1 = csub(u[1], u[4]);
        cplx<T> t2 = cadd(u[2], u[3]), d2 = csub(u[2], u[3]);
        u[0] = {a.x + t1.x + t2.x, a.y + t1.y + t2.y};
        cplx<T> m1 = {fma_t(c2, t2.x, fma_t(c1, t1.x, a.x)), fma_t(c2, t2.y, fma_t(c1, t1.y, a.y))};
        cplx<T> m2 = {fma_t(c1, t2.x, fma_t(c2, t1.x, a.x)), fma_t(c1, t2.y, fma_t(c2, t1.y, a.y))};
        cplx<T> r1 = {-fma_t(s1, d1.y, s2 * d2.y), fma_t(s1, d1.x, s2 * d2.x)};
        cplx<T> r2 = {-fma_t(s2, d1.y, -(s1 * d2.y)), fma_t(s2, d1.x, -(s1 * d2.x))};
        u[1] = cadd(m1, r1);
        u[4] = csub(m1, r1);
        u[2] = cadd(m2, r2);
        u[3] = csub(m2, r2);
    } else {
        // generic odd prime: direct O(R^2) DFT with sincos (rare sizes only)
        cplx<T> v[R];
        for (int q = 0; q < R; q++) {
            T sr = 0, si = 0;
            for (int r = 0; r < R; r++) {
                double ang = 6.283185307179586476925 * (double)((r * q) % R) / R * sign;
                T c = T(cos(ang)), s = T(sin(ang));
                sr += u[r].x * c - u[r].y * s;
                si += u[r].x * s + u[r].y * c;
            }
            v[q] = {sr, si};
        }
        for (int q = 0; q < R; q++) u[q] = v[q];
    }
}

// One Stockham pass for all nb sequences.
template <typename T, int N, int R>
__device__ __forceinline__ void fft_pass(const cplx<T>* __restrict__ src, cplx<T>* __restrict__ dst,
                                         int nb, int p, const cplx<T>* __restrict__ tw, int sign,
                                         int tid, int nthr) {
    constexpr int M = N / R;
    const int total = nb * M;
    for (int t = tid; t < total; t += nthr) {
        const int seq = t / M;
        const int i = t - seq * M;
        const int k = i % p;
        const int s0 = seq * N + i;
        cplx<T> u[R];
#pragma unroll
        for (int r = 0; r < R; r++) u[r] = src[lx(s0 + r * M)];
        if (p > 1) {
            const cplx<T>* w = tw + k * (R - 1);
#pragma unroll
            for (int r = 1; r < R; r++) {
                cplx<T> c = w[r - 1];
                if (sign > 0) c.y = -c.y;
                u[r] = cmul(u[r], c);
            }
        }
        dft_small<T, R>(u, sign);
        const int d0 = seq * N + (i / p) * p * R + k;
#pragma unroll
        for (int q = 0; q < R; q++) dst[lx(d0 + q * p)] = u[q];
    }
}

template <typename T, int N, int S>
__device__ __forceinline__ void fft_passes(cplx<T>*& a, cplx<T>*& b, int nb,
                                           const cplx<T>* __restrict__ tw, int sign, int tid,
                                           int nthr) {
    constexpr FacList F = factorize(N);
    if constexpr (S < F.nf) {
        constexpr int R = F.f[S];
        fft_pass<T, N, R>(a, b, nb, F.p[S], tw + F.off[S], sign, tid, nthr);
        __syncthreads();
        cplx<T>* t = a;
        a = b;
        b = t;
        fft_passes<T, N, S + 1>(a, b, nb, tw, sign, tid, nthr);
    }
}

// Transforms nb sequences of length N held in `a` (LDS, entry i of the
// concatenated sequences at lx(i)).  `b` is scratch of the same size.  On return `a` points at the buffer holding the result.
// The caller must __syncthreads() before the call (data loaded) and reads
// the result after it (this function ends with a barrier).
// tw: forward-sign twiddle table for length N (FacList layout).
template <typename T, int N>
__device__ __forceinline__ void fft_lds(cplx<T>*& a, cplx<T>*& b, int nb,
                                        const cplx<T>* __restrict__ tw, int sign, int tid,
                                        int nthr) {
    fft_passes<T, N, 0>(a, b, nb, tw, sign, tid, nthr);
}

// ------------------------------------------------- FFT through registers
//
// A workgroup of NT threads transforms FftReg<N, NT>::NB sequences of length N
// (a multiple of 8).  Thread (i, c), i < M = N / 8, holds the eight elements
// i + M r (r = 0 .. 7) of sequence c in registers, before and after the
// transform: the first radix-8 pass works on the registers as loaded, each
// later pass but the last takes one LDS exchange, and the last pass leaves its
// results in registers at the same eight places, so a transform, a pointwise
// product and the inverse transform follow one another without touching LDS
// in between.  Against fft_lds (load to LDS, every pass from LDS to LDS, read
// back) an element of a 256-point transform makes 4 LDS accesses instead of 8,
// and one buffer instead of two leaves room for twice the workgroups.
//
// Sequences sit SEQ entries apart in LDS, SEQ = 4 mod 32, with the pad of lx:
// for 8 sequences of 256 the accesses with neighbouring lanes on neighbouring
// sequences (columns) and on neighbouring elements (rows) are both free of
// avoidable bank conflicts.
// Threads of a workgroup: 8 k sequences, k = 1 from N = 129 on, so that a row of
// columns is whole 64-byte pieces and no thread is left without a place.
__host__ __device__ constexpr int fft_threads(int n) { return n >= 256 ? n : 256 / n * n; }

template <int N, int NT>
struct FftReg {
    static_assert(N % 8 == 0, "first radix is 8");
    static constexpr int M = N / 8;
    static constexpr int NB = NT / M;  // sequences of a workgroup
    static_assert(NB >= 1 && NB * M == NT, "one thread per eight elements");
    static constexpr int SEQ = (lds_len(N) + 31 - 4) / 32 * 32 + 4;
    static constexpr int LDS = NB * SEQ;  // entries
    // this thread's sequence and first element; columns: neighbouring lanes on
    // neighbouring sequences, rows: on neighbouring elements
    __device__ static __forceinline__ int col_c(int tid) { return tid % NB; }
    __device__ static __forceinline__ int col_i(int tid) { return tid / NB; }
    __device__ static __forceinline__ int row_c(int tid) { return tid / M; }
    __device__ static __forceinline__ int row_i(int tid) { return tid % M; }
};

// Middle passes S .. nf - 2, LDS to LDS.
template <typename T, int N, int NT, int S>
__device__ __forceinline__ void fft_reg_mid(cplx<T>* __restrict__ sm, const cplx<T>* __restrict__ tw, int sign, int tid,
                                            bool cols) {
    constexpr FacList F = factorize(N);
    if constexpr (S < F.nf - 1) {
        using Q = FftReg<N, NT>;
        constexpr int R = F.f[S], p = F.p[S], M = N / R, G = (Q::NB * M + NT - 1) / NT;
        cplx<T> u[G][R];
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int t = tid + NT * g;
            const int c = cols ? t % Q::NB : t / M, i = cols ? t / Q::NB : t % M;
            if (c < Q::NB && i < M) {
#pragma unroll
                for (int r = 0; r < R; r++) u[g][r] = sm[c * Q::SEQ + lx(i + r * M)];
            }
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < G; g++) {
            const int t = tid + NT * g;
            const int c = cols ? t % Q::NB : t / M, i = cols ? t / Q::NB : t % M;
            if (c < Q::NB && i < M) {
                const int k = i % p;
                const cplx<T>* w = tw + F.off[S] + k * (R - 1);
#pragma unroll
                for (int r = 1; r < R; r++) {
                    cplx<T> f = w[r - 1];
                    if (sign > 0) f.y = -f.y;
                    u[g][r] = cmul(u[g][r], f);
                }
                dft_small<T, R>(u[g], sign);
                const int d0 = (i / p) * p * R + k;
#pragma unroll
                for (int q = 0; q < R; q++) sm[c * Q::SEQ + lx(d0 + q * p)] = u[g][q];
            }
        }
        __syncthreads();
        fft_reg_mid<T, N, NT, S + 1>(sm, tw, sign, tid, cols);
    }
}

// u: elements i + M r of sequence c, in and out.  The thread's place is (ci, ii)
// before and (co, io) after (the same, or columns in and rows out); threads
// with no place (c >= NB or i >= M) take part in the barriers only.  sm: LDS
// entries of FftReg, free when called with fresh = true; otherwise the previous
// transform's reads are waited for first.
template <typename T, int N, int NT>
__device__ __forceinline__ void fft_reg(cplx<T>* u, cplx<T>* __restrict__ sm, const cplx<T>* __restrict__ tw, int sign,
                                        int tid, int ci, int ii, int co, int io, bool cols, bool fresh) {
    using Q = FftReg<N, NT>;
    constexpr FacList F = factorize(N);
    static_assert(F.f[0] == 8, "first radix is 8");
    constexpr int RL = F.f[F.nf - 1], GL = 8 / RL, ML = N / RL;
    static_assert(F.nf >= 2 && 8 % RL == 0, "last radix divides 8");
    if (!fresh) __syncthreads();
    dft_small<T, 8>(u, sign);
#pragma unroll
    for (int q = 0; q < 8; q++) sm[ci * Q::SEQ + lx(ii * 8 + q)] = u[q];
    __syncthreads();
    fft_reg_mid<T, N, NT, 1>(sm, tw, sign, tid, cols);
#pragma unroll
    for (int g = 0; g < GL; g++) {
        const int k = io + g * Q::M;
        cplx<T> v[RL];
#pragma unroll
        for (int r = 0; r < RL; r++) v[r] = sm[co * Q::SEQ + lx(k + r * ML)];
        const cplx<T>* w = tw + F.off[F.nf - 1] + k * (RL - 1);
#pragma unroll
        for (int r = 1; r < RL; r++) {
            cplx<T> f = w[r - 1];
            if (sign > 0) f.y = -f.y;
            v[r] = cmul(v[r], f);
        }
        dft_small<T, RL>(v, sign);
#pragma unroll
        for (int q = 0; q < RL; q++) u[g + q * GL] = v[q];
    }
}

// The transform of columns (neighbouring lanes on neighbouring sequences) or of
// rows (on neighbouring elements), in place.
template <int N, typename T = float, int NT_ = fft_threads(N)>
struct Fft {
    static constexpr int NT = NT_;
    using Q = FftReg<N, NT>;
    static constexpr int NB = Q::NB, M = Q::M, LDS = Q::LDS;
    // workgroups a CU holds at most, by threads and by LDS (registers may allow fewer)
    static constexpr int WPC = 2048 / NT < 163840 / (LDS * (int)sizeof(cplx<T>)) ? 2048 / NT
                                                                               : 163840 / (LDS * (int)sizeof(cplx<T>));
    __device__ static __forceinline__ void cols(cplx<T>* u, cplx<T>* sm, const cplx<T>* tw, int sign, int tid,
                                                bool fresh) {
        const int c = Q::col_c(tid), i = Q::col_i(tid);
        fft_reg<T, N, NT>(u, sm, tw, sign, tid, c, i, c, i, true, fresh);
    }
    __device__ static __forceinline__ void rows(cplx<T>* u, cplx<T>* sm, const cplx<T>* tw, int sign, int tid,
                                                bool fresh) {
        const int c = Q::row_c(tid), i = Q::row_i(tid);
        fft_reg<T, N, NT>(u, sm, tw, sign, tid, c, i, c, i, false, fresh);
    }
    // columns in, rows out
    __device__ static __forceinline__ void cols_to_rows(cplx<T>* u, cplx<T>* sm, const cplx<T>* tw, int sign,
                                                        int tid, bool fresh) {
        fft_reg<T, N, NT>(u, sm, tw, sign, tid, Q::col_c(tid), Q::col_i(tid), Q::row_c(tid), Q::row_i(tid), true,
                          fresh);
    }
};

}  // namespace utr
