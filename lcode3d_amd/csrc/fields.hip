// Field solves of the xi step (lcode.py:122-364) on gfx950.
//
// Every solve inverts a five-point operator whose boundary conditions make
// it diagonal under a type-1 sine or cosine transform along each axis.  Along
// j the solve transforms; along i it does not: after the transform along j
// every line k is a tridiagonal system, which two first-order recurrences
// solve directly (the same matrix, without a forward and an inverse transform
// along i).  Three passes, batched over all fields:
//
//   pass A  RHS rows i: assemble the RHS on the fly, transform along j, store
//           the spectra row by row, T[i][k]
//   pass B  the tridiagonal systems along i, in place, a group of lines k per
//           block
//   pass C  output rows i: transform T[i][.] along j, then the epilogue (Bz
//           mean, Variant A, averaging)
//
// A type-1 transform of length n is one complex FFT of length L = 2 (n + 1)
// (sine) or 2 (n - 1) (cosine) of the odd or even extension; two real lines
// ride in one complex FFT (real and imaginary parts).  All six fields of a
// step share L = 2 (N - 1).  The FFT keeps half of the extension (below).
//
// The transforms and the spectra T are in S = double (plain path) or S =
// float (mixed-precision path); the RHS assembly, the recurrences of pass B
// and their tables, the Bz mean and the epilogue are FP64 in both.

#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace lcode {

namespace {

template <typename S> struct Vec;
template <> struct Vec<double> { using T = double2; };
template <> struct Vec<float> { using T = float2; };

template <typename V>
__device__ __forceinline__ V mk(decltype(V::x) x, decltype(V::x) y) {
    V v;
    v.x = x;
    v.y = y;
    return v;
}
template <typename V>
__device__ __forceinline__ V cmul(V a, V b) {
    return mk<V>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <typename V>
__device__ __forceinline__ V cadd(V a, V b) { return mk<V>(a.x + b.x, a.y + b.y); }
template <typename V>
__device__ __forceinline__ V csub(V a, V b) { return mk<V>(a.x - b.x, a.y - b.y); }
template <typename V>
__device__ __forceinline__ V conj(V a) { return mk<V>(a.x, -a.y); }
template <typename V>
__device__ __forceinline__ V neg(V a) { return mk<V>(-a.x, -a.y); }
// multiply by -i
template <typename V>
__device__ __forceinline__ V mul_mi(V a) { return mk<V>(a.y, -a.x); }

// Forward DFT of R points held in registers: y_p = sum_q x_q e^{-2 pi i pq/R}.
template <int R, typename V> struct Dft;

template <typename V> struct Dft<2, V> {
    static __device__ __forceinline__ void run(V* v) {
        const V a = v[0], b = v[1];
        v[0] = cadd(a, b);
        v[1] = csub(a, b);
    }
};

template <typename V> struct Dft<4, V> {
    static __device__ __forceinline__ void run(V* v) {
        const V s02 = cadd(v[0], v[2]), d02 = csub(v[0], v[2]);
        const V s13 = cadd(v[1], v[3]), d13 = mul_mi(csub(v[1], v[3]));
        v[0] = cadd(s02, s13);
        v[2] = csub(s02, s13);
        v[1] = cadd(d02, d13);
        v[3] = csub(d02, d13);
    }
};

// Radix 8 as two radix-4 DFTs of the even and odd points combined with
// the eighth roots of unity: y_p = e_p + w8^p o_p, y_(p+4) = e_p - w8^p o_p.
template <typename V> struct Dft<8, V> {
    static __device__ __forceinline__ void run(V* v) {
        using S = decltype(V::x);
        constexpr S r = (S)0.70710678118654752440;   // 1 / sqrt(2)
        V e[4] = {v[0], v[2], v[4], v[6]};
        V o[4] = {v[1], v[3], v[5], v[7]};
        Dft<4, V>::run(e);
        Dft<4, V>::run(o);
        const V o1 = mk<V>(r * (o[1].x + o[1].y), r * (o[1].y - o[1].x));    // (1 - i) / sqrt 2
        const V o2 = mul_mi(o[2]);                                           // -i
        const V o3 = mk<V>(r * (o[3].y - o[3].x), -r * (o[3].x + o[3].y));   // -(1 + i) / sqrt 2
        v[0] = cadd(e[0], o[0]);
        v[4] = csub(e[0], o[0]);
        v[1] = cadd(e[1], o1);
        v[5] = csub(e[1], o1);
        v[2] = cadd(e[2], o2);
        v[6] = csub(e[2], o2);
        v[3] = cadd(e[3], o3);
        v[7] = csub(e[3], o3);
    }
};

template <typename V> struct Dft<3, V> {
    static __device__ __forceinline__ void run(V* v) {
        using S = decltype(V::x);
        constexpr S s = (S)0.86602540378443864676;  // sin(2 pi / 3)
        const V t = cadd(v[1], v[2]), d = csub(v[1], v[2]);
        const V base = mk<V>(v[0].x - (S).5 * t.x, v[0].y - (S).5 * t.y);
        const V rot = mk<V>(s * d.y, -s * d.x);     // -i s d
        v[0] = cadd(v[0], t);
        v[1] = cadd(base, rot);
        v[2] = csub(base, rot);
    }
};

template <typename V> struct Dft<5, V> {
    static __device__ __forceinline__ void run(V* v) {
        using S = decltype(V::x);
        constexpr S c1 = (S)0.30901699437494742410;   // cos(2 pi / 5)
        constexpr S c2 = (S)-0.80901699437494742410;  // cos(4 pi / 5)
        constexpr S s1 = (S)0.95105651629515357212;   // sin(2 pi / 5)
        constexpr S s2 = (S)0.58778525229247312917;   // sin(4 pi / 5)
        const V x0 = v[0];
        const V t1 = cadd(v[1], v[4]), d1 = csub(v[1], v[4]);
        const V t2 = cadd(v[2], v[3]), d2 = csub(v[2], v[3]);
        const V a1 = mk<V>(x0.x + c1 * t1.x + c2 * t2.x, x0.y + c1 * t1.y + c2 * t2.y);
        const V a2 = mk<V>(x0.x + c2 * t1.x + c1 * t2.x, x0.y + c2 * t1.y + c1 * t2.y);
        const V b1 = mk<V>(s1 * d1.x + s2 * d2.x, s1 * d1.y + s2 * d2.y);
        const V b2 = mk<V>(s2 * d1.x - s1 * d2.x, s2 * d1.y - s1 * d2.y);
        v[0] = cadd(x0, cadd(t1, t2));
        v[1] = cadd(a1, mul_mi(b1));
        v[4] = csub(a1, mul_mi(b1));
        v[2] = cadd(a2, mul_mi(b2));
        v[3] = csub(a2, mul_mi(b2));
    }
};

// N1 N2 points (gcd 1) by Good-Thomas: n = (N2 n1 + N1 n2) mod R, k = (E1 k1 +
// E2 k2) mod R with E1 = N2 (N2^-1 mod N1), E2 = N1 (N1^-1 mod N2), so that
// W_R^(nk) = W_N1^(n1 k1) W_N2^(n2 k2): no twiddles between the two.
constexpr int inverse_mod(int a, int n) {
    for (int k = 1; k < n; ++k)
        if (a * k % n == 1) return k;
    return 0;
}

template <int N1, int N2, typename V>
__device__ __forceinline__ void dft_coprime(V* x) {
    constexpr int R = N1 * N2, E1 = N2 * inverse_mod(N2 % N1, N1),
                  E2 = N1 * inverse_mod(N1 % N2, N2);
    V a[N2][N1];
#pragma unroll
    for (int n2 = 0; n2 < N2; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < N1; ++n1) a[n2][n1] = x[(N2 * n1 + N1 * n2) % R];
        Dft<N1, V>::run(a[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) {
        V b[N2];
#pragma unroll
        for (int n2 = 0; n2 < N2; ++n2) b[n2] = a[n2][k1];
        Dft<N2, V>::run(b);
#pragma unroll
        for (int k2 = 0; k2 < N2; ++k2) x[(E1 * k1 + E2 * k2) % R] = b[k2];
    }
}

template <typename V> struct Dft<6, V> {
    static __device__ __forceinline__ void run(V* v) { dft_coprime<2, 3>(v); }
};
template <typename V> struct Dft<10, V> {
    static __device__ __forceinline__ void run(V* v) { dft_coprime<2, 5>(v); }
};
template <typename V> struct Dft<12, V> {
    static __device__ __forceinline__ void run(V* v) { dft_coprime<4, 3>(v); }
};
template <typename V> struct Dft<15, V> {
    static __device__ __forceinline__ void run(V* v) { dft_coprime<3, 5>(v); }
};
template <typename V> struct Dft<20, V> {
    static __device__ __forceinline__ void run(V* v) { dft_coprime<4, 5>(v); }
};

// M^2 points as M DFTs of stride M, the twiddles W^(n2 k1) and M DFTs across.
template <int M, typename V, typename W>
__device__ __forceinline__ void dft_square(V* x, W&& w) {
    V a[M][M];
#pragma unroll
    for (int n2 = 0; n2 < M; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < M; ++n1) a[n2][n1] = x[M * n1 + n2];
        Dft<M, V>::run(a[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < M; ++k1) {
        V b[M];
#pragma unroll
        for (int n2 = 0; n2 < M; ++n2) b[n2] = n2 * k1 ? w(a[n2][k1], n2 * k1) : a[n2][k1];
        Dft<M, V>::run(b);
#pragma unroll
        for (int k2 = 0; k2 < M; ++k2) x[k1 + M * k2] = b[k2];
    }
}

template <typename V> struct Dft<9, V> {
    static __device__ __forceinline__ void run(V* v) {
        using S = decltype(V::x);
        dft_square<3>(v, [](V a, int e) {   // W_9^e, e = 1, 2, 4
            const S c = e == 1 ? (S)0.76604444311897803520 : e == 2 ? (S)0.17364817766693034885
                                                                    : (S)-0.93969262078590838405;
            const S s = e == 1 ? (S)0.64278760968653932632 : e == 2 ? (S)0.98480775301220805937
                                                                    : (S)0.34202014332566873304;
            return cmul(a, mk<V>(c, -s));
        });
    }
};

template <typename V> struct Dft<16, V> {
    static __device__ __forceinline__ void run(V* v) {
        using S = decltype(V::x);
        constexpr S r = (S)0.70710678118654752440;
        constexpr S c1 = (S)0.92387953251128675613, s1 = (S)0.38268343236508977173;
        dft_square<4>(v, [](V a, int e) {   // W_16^e, e = 1, 2, 3, 4, 6, 9
            switch (e) {
                case 1: return cmul(a, mk<V>(c1, -s1));
                case 2: return mk<V>(r * (a.x + a.y), r * (a.y - a.x));
                case 3: return cmul(a, mk<V>(s1, -c1));
                case 4: return mul_mi(a);
                case 6: return mk<V>(r * (a.y - a.x), -r * (a.x + a.y));
                default: return cmul(a, mk<V>(-c1, s1));   // 9
            }
        });
    }
};

// ---------------------------------------------------------------------------
// The FFT of an extension: x[L - p] = +x[p] (cosine) or -x[p] (sine), and so
// X[L - k] = +-X[k].  With L = R1 T, n = l + T m and k = kappa + R1 k2,
//   X[kappa + R1 k2] = sum_l W_T^(l k2) C_l[kappa],
//   C_l[kappa] = W_L^(l kappa) A_l[kappa],  A_l = DFT_R1 of x[l + T m] over m,
// and the symmetry halves the work twice: lane T - l's points are lane l's
// mirrored, so lane l <= T / 2 writes both rows of C,
//   C_(T-l)[kappa] = +-conj(W_L^(l kappa)) A_l[(R1 - kappa) mod R1],
// and only the columns kappa <= R1 / 2 are transformed: the residues above hold
// the mirror images of those below.  The first stage takes its points straight
// from global memory (every point once: the lanes 0 .. T / 2 of
// a row pair hold columns l + T m or L - l - T m), the K = R1 / 2 + 1 transforms of
// length T run as Stockham stages in LDS, z[row KP + kappa] with kappa fastest
// (KP = K made odd: the first stage's stores of consecutive rows then spread over all
// banks), one butterfly per thread, and the last stage unfolds its outputs into
// X[0 .. L / 2] in order, so that the passes store whole lines.  The host picks R1
// and the radices (solver_fft_plan).
//
// Bound: the chain of a block (loads, three or four LDS exchanges, stores) with a few
// wavefronts per SIMD on small grids, memory on large ones (1281^2: pass C 320 MB in
// 67 us).  Six fields, passes A / C, us per launch, transforms of the whole extension
// (radix 4 in LDS; 20 points per lane at 641^2 and 1281^2) -> of half of it:
// 129^2 6.4 / 6.4 -> 6.3 / 6.2, 257^2 9.7 / 9.2 -> 8.6 / 8.2, 361^2 19.2 / 19.0 ->
// 12.3 / 11.3, 641^2 23.8 / 21.2 -> 21.2 / 17.0, with FP32 transforms and grids 18.4 / 20.2
// -> 14.0 / 15.0, 1281^2 96.8 / 80.3 -> 80.5 / 66.3.
// ---------------------------------------------------------------------------

// Roots held per butterfly of radix R: w^q, q = 1, 2, 3, 4, 8, 12 (below R).
__host__ __device__ constexpr int root_count(int R) { return (R < 4 ? R : 4) - 1 + (R + 3) / 4 - 1; }

// The plan of radices R1; r[0 .. nst).  A constant for the lengths with kernels of their
// own (static_fft: the powers of two from 64 to 2048 and 640, 1280 and 2560, the grids
// that a run is refined through by halving its step), whose index arithmetic then
// folds away.  The same plan from kernel arguments and as a constant, us: A + C of
// six fields 129^2 14.8 and 12.4, 257^2 19.9 and 17.1, 641^2 41.5 and 38.9.  The rest of
// the two families, 80, 160, 320 and 4096, has none: a step at 81^2 81.9 and 81.8, at
// 161^2 93.0 and 90.4, six FP32 solves at 2049^2 442 and 433, but with their 18 kernels in
// the library the steps of other sizes took longer (641^2 with FP32 grids 198.0 -> 200.9,
// FP64 217.4 -> 218.4, 361^2 143.2 -> 143.8).
__host__ __device__ constexpr FftPlan make_plan(int L, int R1, int nst, const int* r) {
    FftPlan p{};
    p.L = L;
    p.R1 = R1;
    p.T = L / R1;
    p.K = R1 / 2 + 1;
    p.KP = p.K | 1;
    p.lanes = p.T / 2 + 1;
    p.nfirst = p.lanes * root_count(p.K);
    p.nst = nst;
    p.k_inv = (unsigned)((0x100000000ull + p.K - 1) / p.K);
    int threads = p.lanes, span = 1;
    for (int s = 0; s < nst; ++s) {
        const int stride = p.T / r[s], tasks = p.K * stride;
        p.word[s] = fft_word(r[s], span, stride);
        if (span > 1) {
            p.span_inv[s] = (unsigned)((0x100000000ull + span - 1) / span);
            p.nroots += span * root_count(r[s]);
        }
        if (tasks > threads) threads = tasks;
        span *= r[s];
    }
    p.threads = (threads + 63) / 64 * 64;
    return p;
}

struct StaticFft {
    int L, R1, nst, r[3];
};
constexpr StaticFft kStaticFft[] = {
    {64, 4, 2, {4, 4}},    {128, 4, 2, {4, 8}},     {256, 4, 3, {4, 4, 4}},
    {512, 4, 3, {4, 4, 8}}, {640, 4, 3, {4, 4, 10}}, {1024, 8, 2, {8, 16}},
    {1280, 10, 2, {16, 8}}, {2048, 8, 2, {16, 16}},  {2560, 10, 2, {16, 16}},
};
constexpr int static_fft(int L) {   // index, or -1
    for (int k = 0; k < (int)(sizeof(kStaticFft) / sizeof(kStaticFft[0])); ++k)
        if (kStaticFft[k].L == L) return k;
    return -1;
}

// n / d for n < 2^16 and 1 < d < 2^16, inv = ceil(2^32 / d).
__device__ __forceinline__ int div_by(int n, unsigned inv) {
    return (int)__umulhi((unsigned)n, inv);
}

// The roots w^q, q < R, of one butterfly, from the q = 1, 2, 3, 4, 8, 12 of a table
// [root][stride] (the plan's order): the others, q = 4 a + c, are one product,
// formed in FP64, and all are rounded once to the transform's precision.
template <int R>
struct Roots {
    static constexpr int NL = R < 4 ? R : 4, NA = (R + 3) / 4;
    double2 lo[4], hi[NA];
    __device__ __forceinline__ void load(const double2* __restrict__ tw, int stride, int k) {
#pragma unroll
        for (int c = 1; c < NL; ++c) lo[c] = tw[(c - 1) * stride + k];
#pragma unroll
        for (int a = 1; a < NA; ++a) hi[a] = tw[(a + 2) * stride + k];
    }
    template <typename V>
    __device__ __forceinline__ V at(int q) const {
        const int a = q / 4, c = q % 4;
        const double2 w = a == 0 ? lo[c] : c == 0 ? hi[a] : cmul(hi[a], lo[c]);
        return mk<V>(w.x, w.y);
    }
};

// The stages' roots, copied to LDS at the start of a block: loaded before the block's
// inputs, stored after they are on their way.
struct StageRoots {
    static constexpr int kHeld = 2;
    double2 v[kHeld];
    __device__ __forceinline__ void load(const FftPlan& p, const double2* __restrict__ tw) {
#pragma unroll
        for (int u = 0; u < kHeld; ++u)
            v[u] = tw[p.nfirst + min((int)(threadIdx.x + u * blockDim.x), p.nroots - 1)];
    }
    __device__ __forceinline__ void store(const FftPlan& p, const double2* __restrict__ tw,
                                          double2* lds) const {
#pragma unroll
        for (int u = 0; u < kHeld; ++u) {
            const int k = threadIdx.x + u * blockDim.x;
            if (k < p.nroots) lds[k] = v[u];
        }
        for (int k = threadIdx.x + kHeld * blockDim.x; k < p.nroots; k += blockDim.x)
            lds[k] = tw[p.nfirst + k];
    }
};

// First stage, lane l: rows l and T - l of C from the points x.
template <int R1, typename V>
__device__ __forceinline__ void fft_first(V (&x)[R1], V* z, const FftPlan& p, bool sine, int l,
                                          const Roots<R1 / 2 + 1>& w) {
    constexpr int K = R1 / 2 + 1;
    Dft<R1, V>::run(x);
    V* const up = z + l * p.KP;
    V* const down = z + (p.T - l) * p.KP;
    const bool both = l > 0 && 2 * l < p.T;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const V a = x[k], m = x[(R1 - k) % R1];
        if (k == 0) {
            up[k] = a;
            if (both) down[k] = sine ? neg(m) : m;
        } else {
            const V r = w.template at<V>(k);
            up[k] = cmul(a, r);
            const V d = cmul(m, conj(r));
            if (both) down[k] = sine ? neg(d) : d;
        }
    }
}

// One Stockham stage over the K columns: thread beta takes butterfly b = beta / K of
// column beta mod K.  Every read of the stage precedes its first write (block-wide
// barriers: all threads call it).  The last stage writes X[k], k <= L / 2, to z[k].
template <int R, bool FIXED, typename V>
__device__ __forceinline__ void fft_stage(V* z, const FftPlan& p, unsigned word, unsigned span_inv,
                                          bool last, bool sine, const double2* tw) {
    const int span = fft_word_span(word), stride = fft_word_stride(word);
    const int beta = threadIdx.x;
    const bool act = beta < p.K * stride;
    const int b = FIXED ? (int)((unsigned)beta / (unsigned)p.K) : div_by(beta, p.k_inv);
    const int kap = beta - b * p.K;
    const int k = span == 1 ? 0
                  : FIXED   ? (int)((unsigned)b % (unsigned)span)
                            : b - div_by(b, span_inv) * span;
    V v[R];
    if (act) {
        if (span == 1) {
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = z[(b + q * stride) * p.KP + kap];
        } else {
            Roots<R> w;
            w.load(tw, span, k);
#pragma unroll
            for (int q = 0; q < R; ++q) v[q] = z[(b + q * stride) * p.KP + kap];
#pragma unroll
            for (int q = 1; q < R; ++q) v[q] = cmul(v[q], w.template at<V>(q));
        }
        Dft<R, V>::run(v);
    }
    __syncthreads();
    if (act) {
        if (last) {
            const bool edge = kap == 0 || 2 * kap == p.R1;   // mirrored into itself
#pragma unroll
            for (int q = 0; q < R; ++q) {
                const int i = kap + p.R1 * (b + q * span);
                if (2 * i <= p.L) z[i] = v[q];
                else if (!edge) z[p.L - i] = sine ? neg(v[q]) : v[q];
            }
        } else {
            const int j = (b - k) * R + k;
#pragma unroll
            for (int q = 0; q < R; ++q) z[(j + q * span) * p.KP + kap] = v[q];
        }
    }
    __syncthreads();
}

template <typename V>
__device__ __forceinline__ void run_stages(V* z, const FftPlan& p, bool sine, const double2* tw) {
    // the stages' descriptors, all read at once: a stage shifts them down
    unsigned word[kMaxStages], inv[kMaxStages];
#pragma unroll
    for (int s = 0; s < kMaxStages; ++s) {
        word[s] = p.word[s];
        inv[s] = p.span_inv[s];
    }
    __syncthreads();   // the first stage's rows
    for (int s = 0; s < p.nst; ++s) {
        const unsigned w = word[0], v = inv[0];
        const bool last = s == p.nst - 1;
        const int R = fft_word_radix(w);
        switch (R) {
            case 2: fft_stage<2, false>(z, p, w, v, last, sine, tw); break;
            case 3: fft_stage<3, false>(z, p, w, v, last, sine, tw); break;
            case 4: fft_stage<4, false>(z, p, w, v, last, sine, tw); break;
            case 5: fft_stage<5, false>(z, p, w, v, last, sine, tw); break;
            case 6: fft_stage<6, false>(z, p, w, v, last, sine, tw); break;
            case 8: fft_stage<8, false>(z, p, w, v, last, sine, tw); break;
            case 9: fft_stage<9, false>(z, p, w, v, last, sine, tw); break;
            case 10: fft_stage<10, false>(z, p, w, v, last, sine, tw); break;
            case 12: fft_stage<12, false>(z, p, w, v, last, sine, tw); break;
            case 15: fft_stage<15, false>(z, p, w, v, last, sine, tw); break;
            default: fft_stage<16, false>(z, p, w, v, last, sine, tw); break;
        }
        if (s > 0) tw += fft_word_span(w) * root_count(R);
#pragma unroll
        for (int u = 0; u + 1 < kMaxStages; ++u) {
            word[u] = word[u + 1];
            inv[u] = inv[u + 1];
        }
    }
}

template <int L, int STAGE, typename V>
__device__ __forceinline__ void static_stages(V* z, bool sine, const double2* tw) {
    constexpr StaticFft f = kStaticFft[static_fft(L)];
    constexpr FftPlan p = make_plan(L, f.R1, f.nst, f.r);
    if constexpr (STAGE < f.nst) {
        constexpr int R = f.r[STAGE], span = fft_word_span(p.word[STAGE]);
        fft_stage<R, true>(z, p, p.word[STAGE], 0, STAGE == f.nst - 1, sine, tw);
        static_stages<L, STAGE + 1>(z, sine, tw + (STAGE > 0 ? span * root_count(R) : 0));
    }
}

template <int L, typename V>
__device__ __forceinline__ void fft_stages(V* z, const FftPlan& p, bool sine, const double2* tw) {
    if constexpr (L != 0) {
        __syncthreads();   // the first stage's rows
        static_stages<L, 0>(z, sine, tw);
    } else {
        run_stages(z, p, sine, tw);
    }
}

// The block's plan: the constant of L, or (0) the geometry's.
template <int L>
__device__ __forceinline__ FftPlan plan_of(const SolverGeom& g) {
    if constexpr (L != 0) {
        constexpr StaticFft f = kStaticFft[static_fft(L)];
        return make_plan(L, f.R1, f.nst, f.r);
    } else {
        return g.fft;
    }
}

// Outputs of the pair's two lines at column j of the grid, 0 <= j <= L / 2:
// cosine Re and Im of X[j], sine -Im and Re.
template <typename V>
__device__ __forceinline__ void get_pair(const V* z, bool sine, int j, double& a, double& c) {
    const V v = z[j];
    a = sine ? -(double)v.y : (double)v.x;
    c = sine ? (double)v.x : (double)v.y;
}

// Grid column of point l + T m: itself up to L / 2, its mirror image above.
template <int R1>
__device__ __forceinline__ int point_column(const FftPlan& p, int l, int m) {
    const int n = l + p.T * m;
    return 2 * m < R1 ? n : p.L - n;
}

// The extension's points l + T m of a lane from the values v(m, column) of the two
// lines (sine: odd, 0 at both ends).
template <int R1, typename V, typename F>
__device__ __forceinline__ void extend(V (&x)[R1], const FftPlan& p, bool sine, int l, F&& v) {
#pragma unroll
    for (int m = 0; m < R1; ++m) {
        x[m] = v(m, point_column<R1>(p, l, m));
        if (sine && 2 * m >= R1) x[m] = neg(x[m]);
        if ((m == 0 || 2 * m == R1) && sine && l == 0) x[m] = mk<V>(0, 0);
    }
}

// Right-hand sides of rows i and i + 1 (clamped to the grid: a row outside it, or
// without data, is dropped by the caller) at column j; the values of rhs_value_k.  The
// grids' bases are uniform and the lane holds one 32-bit offset per row, for all grids (a base
// per row and grid took more scalar registers than there are: 641^2 22.4 us against 21.2,
// 1281^2 86.7 against 80.5); a derivative along i takes the
// sources of its four rows once.
template <typename G>
__device__ __forceinline__ double at(const G* base, unsigned e) {
    return (double)*reinterpret_cast<const G*>(reinterpret_cast<const char*>(base) +
                                               e * (unsigned)sizeof(G));
}

template <int KIND, typename G>
__device__ __forceinline__ void rhs_pair_k(int i, int j, int N, const RhsInputs& in, double& a,
                                           double& c) {
    const int i1 = min(i + 1, N - 1);
    const int rows[4] = {max(i - 1, 0), i, i1, min(i1 + 1, N - 1)};
    const bool in0 = i >= 1 && i <= N - 2, in1 = i1 >= 1 && i1 <= N - 2;
    auto over_h2 = [&](double x) { return quotient(x, in.h * 2, in.inv_h2); };
    auto over_dxi = [&](double x) { return quotient(x, in.dxi, in.inv_dxi); };
    const G *jx = gp<G>(in.jx), *jy = gp<G>(in.jy);
    const bool jin = j >= 1 && j <= N - 2;
    const unsigned oj = jin ? 1 : 0;
    unsigned o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (unsigned)(rows[r] * N + j);
    if constexpr (KIND == F_EZ) {
        // the interior only carries this right-hand side (zero elsewhere)
        const double x0 = at(jx, o[0]), x1 = at(jx, o[1]),
                     x2 = at(jx, o[2]), x3 = at(jx, o[3]);
        const double ya = at(jy, o[1] + oj) - at(jy, o[1] - oj);
        const double yc = at(jy, o[2] + oj) - at(jy, o[2] - oj);
        a = over_h2(-((x2 - x0) + ya));
        c = over_h2(-((x3 - x1) + yc));
    } else if constexpr (KIND == F_BZ) {
        const double x0 = at(jy, o[0]), x1 = at(jy, o[1]),
                     x2 = at(jy, o[2]), x3 = at(jy, o[3]);
        const double ya = at(jx, o[1] + oj) - at(jx, o[1] - oj);
        const double yc = at(jx, o[2] + oj) - at(jx, o[2] - oj);
        const bool n0 = in0 && jin, n1 = in1 && jin;
        a = over_h2(-((n0 ? ya : 0.) - (n0 ? x2 - x0 : 0.)));
        c = over_h2(-((n1 ? yc : 0.) - (n1 ? x3 - x1 : 0.)));
    } else {
        constexpr bool rho = KIND == F_EX || KIND == F_EY;
        constexpr bool along_i = KIND == F_EX || KIND == F_BY;
        constexpr bool xcur = along_i;
        constexpr int ft = KIND == F_EX ? 0 : KIND == F_EY ? 1 : KIND == F_BX ? 2 : 3;
        const G* src = gp<G>(rho ? in.ro : in.jz);
        const double* sp0 = rho ? in.ro_prev : in.jz_prev;
        const G* prev = sp0 ? gp<G>(sp0) : src;
        const double* dummy = std::is_same<G, double>::value ? in.ro : in.zero64;
        const double* beam = in.beam ? in.beam : dummy;
        const double on = in.beam ? 1. : 0., off = in.beam ? 0. : in.beam_scalar;
        // (a beam is added to the source of every derivative: lcode.py:862-863)
        auto source = [&](unsigned e) {
            const double s = (at(src, e) + at(prev, e)) / 2;
            return s + (at(beam, e) * on + off);
        };
        double da, dc;
        if constexpr (along_i) {
            const double s0 = source(o[0]), s1 = source(o[1]);
            const double s2 = source(o[2]), s3 = source(o[3]);
            da = s2 - s0;
            dc = s3 - s1;
        } else {
            da = source(o[1] + oj) - source(o[1] - oj);
            dc = source(o[2] + oj) - source(o[2] - oj);
        }
        const G* jp = gp<G>(xcur ? in.jx_prev : in.jy_prev);
        const G* jc = xcur ? jx : jy;
        const G* tr = gp<G>(in.Ftrick[ft]);
        const double ja = over_dxi(at(jp, o[1]) - at(jc, o[1]));
        const double jc1 = over_dxi(at(jp, o[2]) - at(jc, o[2]));
        const double ta = at(tr, o[1]) * in.trick;
        const double tc = at(tr, o[2]) * in.trick;
        const double fa = (in0 && jin ? over_h2(da) : 0.) - ja;
        const double fc = (in1 && jin ? over_h2(dc) : 0.) - jc1;
        if constexpr (KIND == F_BX) {
            a = fa + ta;
            c = fc + tc;
        } else {
            a = -(fa - ta);
            c = -(fc - tc);
        }
    }
}

template <typename G>
__device__ __forceinline__ void rhs_pair(int kind, int i, int j, int N, const RhsInputs& in,
                                         double& a, double& c) {
    switch (kind) {
        case F_EX: rhs_pair_k<F_EX, G>(i, j, N, in, a, c); break;
        case F_EY: rhs_pair_k<F_EY, G>(i, j, N, in, a, c); break;
        case F_BX: rhs_pair_k<F_BX, G>(i, j, N, in, a, c); break;
        case F_BY: rhs_pair_k<F_BY, G>(i, j, N, in, a, c); break;
        case F_EZ: rhs_pair_k<F_EZ, G>(i, j, N, in, a, c); break;
        default: rhs_pair_k<F_BZ, G>(i, j, N, in, a, c); break;
    }
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Sum over the block, to every thread (scratch: one double per wave).
__device__ __forceinline__ double block_sum(double v, double* scratch) {
    v = wave_sum(v);
    if (blockDim.x == 64) return v;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += scratch[w];
    return t;
}

// XCD-aware block order.  Workgroups go to the 8 XCDs round-robin by
// linear id and each XCD has its own L2; neighbouring row pairs share the
// 128-B lines of their sources, so give every XCD a
// contiguous range of (field, row pair)s.  A bijection on the grid.
struct BlockPos {
    int field, block;
};

__device__ __forceinline__ BlockPos xcd_block() {
    const int gx = gridDim.x, total = gx * gridDim.y;
    const int logical = xcd_logical(blockIdx.y * gx + blockIdx.x, total);
    return BlockPos{logical / gx, logical % gx};
}

// Pass A's order: the fields of one row pair get consecutive logical
// ids, so one XCD assembles all six right-hand sides of its rows and reads
// their shared sources (densities, currents, beam) into its L2 once.
__device__ __forceinline__ BlockPos xcd_block_rows() {
    const int gx = gridDim.x, nf = gridDim.y, total = gx * nf;
    const int logical = xcd_logical(blockIdx.y * gx + blockIdx.x, total);
    return BlockPos{logical % nf, logical / nf};
}

// ---------------------------------------------------------------------------
// Passes
// ---------------------------------------------------------------------------

// Pass A: a block takes one field's grid rows ga (even) and ga + 1.  All its threads
// assemble right-hand sides, a column of both rows at a time (at 641^2 21.2 us; two
// columns in flight 22.6: more registers; the first stage's lanes alone, at their own
// points, 30.3), and the first stage reads them back from LDS.
// G: storage type of the source grids (FP64 arithmetic in both).
template <int R1, int L_, typename S, typename G>
__global__ void __launch_bounds__(512)
pass_a_kernel(SolverGeom g, SolveBatch b) {
    using V = typename Vec<S>::T;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if (!gate_open(b.gate)) return;
    const BlockPos bp = xcd_block_rows();
    const FieldPlan& fp = b.f[bp.field];
    const FftPlan p = plan_of<L_>(g);
    double2* const tw = reinterpret_cast<double2*>(lds_raw);
    V* const z = reinterpret_cast<V*>(tw + p.nroots);
    const int N = g.N, ga = bp.block * 2, gb = ga + 1;
    auto has = [&](int r) { return r >= fp.rowsA0 && r < fp.rowsA0 + fp.rowsA; };
    fetch_lines(g);
    fetch_lines(fp);
    fetch_lines(b.in);
    const bool va = has(ga), vb = has(gb);
    if (!va && !vb) return;
    const bool sine = fp.xfA == XF_DST;
    StageRoots sr;
    sr.load(p, g.tw);
    const int l = threadIdx.x, nt = L_ ? p.threads : (int)blockDim.x;
    Roots<R1 / 2 + 1> w;
    w.load(g.tw, p.lanes, min(l, p.lanes - 1));
    for (int j = l; j < N; j += nt) {
        double a, c;
        rhs_pair<G>(fp.kind, ga, j, N, b.in, a, c);
        z[j] = mk<V>(va ? (S)a : (S)0, vb ? (S)c : (S)0);
    }
    sr.store(p, g.tw, tw);
    __syncthreads();
    V x[R1];
    if (l < p.lanes) extend<R1>(x, p, sine, l, [&](int, int j) { return z[j]; });
    __syncthreads();
    if (l < p.lanes) fft_first<R1>(x, z, p, sine, l, w);
    fft_stages<L_>(z, p, sine, tw);
    S* const Ta = static_cast<S*>(fp.T) + (size_t)ga * g.ld;
    S* const Tb = Ta + g.ld;
#pragma unroll 4
    for (int k = threadIdx.x; k < fp.lenA; k += blockDim.x) {
        double a, c;
        get_pair(z, sine, fp.colA0 + k, a, c);
        if (va) Ta[k] = (S)a;
        if (vb) Tb[k] = (S)c;
    }
}

// Pass B: the tridiagonal systems along i.  With g = h^2 f / (2 (N - 1)) (the
// normalisation of the transform along j and its inverse) and sigma = h^2
// (lambda_k + trick), line k reads
//   -u(i-1) + (2 + sigma) u(i) - u(i+1) = g(i)
// with u = 0 beyond both ends (sine along i) or with (1 + sigma / 2) u - u' =
// g / 2 at them (cosine along i).  Elimination from the top leaves the
// multipliers l(i) = 1 / (2 + sigma - l(i-1)), all in (0, 1], and
//   y(i) = g(i) + l(i-1) y(i-1),    u(i) = l(i) (y(i) + u(i+1)).
// The table holds s = 1 - l, rounded once from long double: where l is near
// 1 (the smooth lines) 1 - l carries the decay, and y - s y keeps its
// relative accuracy where l y would not.  No step subtracts like-sized
// numbers, so the error is that of the transforms it replaces: relative 2-norm
// 1.5e-16 .. 2.5e-16 against 1.6e-16 .. 2.7e-16 (FFT) for smooth lines at
// N = 361 .. 1281.
//
// A block takes CB lines; lane = (chunk, line) with 64 / CB chunks of R
// consecutive rows per wave, so a load reads 64 / CB runs of CB values.  Every chunk solves its rows from a zero carry in registers,
// carries are combined within the wave by shuffles and across the waves
// through LDS (a carry enters as v + c - S c, S = 1 - prod l of the rows
// between), and each row then takes its carry.  Bound: HBM and Infinity
// Cache traffic (8 N^2 values in, and 6 N^2 out per six fields: the
// multipliers of Ey, Bx and of Ex, By are shared) against a round trip of
// latency each way; the arithmetic is about 20 FP64 operations per value.
// Six fields, us per launch, against the transform along i, multiplier and
// transform back that this replaced: 361^2 28.6 -> 9.4, 641^2 23.4 -> 13.7,
// 1281^2 122 -> 62, 641^2 with FP32 spectra 17.5 -> 12.9.
//
// All but the smoothest lines' multipliers are constant after a few rows (the
// elimination has converged to the last bit): on large grids the rows behind that
// one read it again (tri_last), which keeps most of the tables out of the traffic:
// 1281^2 62.4 -> 54.1 us, 641^2 14.0 -> 13.8, with FP32 spectra 13.4 -> 12.6.
template <int R, int CB, typename S>
__global__ void __launch_bounds__(1024)
pass_b_kernel(SolverGeom g, SolveBatch b) {
    constexpr int kChunks = 64 / CB;      // chunks per wave
    __shared__ double2 agg[2][16][CB];    // (S, v) of each wave, both sweeps
    __shared__ double red[16][CB];
    if (!gate_open(b.gate)) return;
    // the fields of one line group adjacent: Ey and Bx (Ex and By) read the
    // same multipliers
    const BlockPos bp = xcd_block_rows();
    const FieldPlan& fp = b.f[bp.field];
    fetch_lines(g);
    fetch_lines(fp);
    const int n = fp.rowsA, k0 = bp.block * CB;
    if (k0 >= fp.lenA) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int col = lane % CB, chunk = wave * kChunks + lane / CB, r0 = chunk * R;
    const int k = k0 + col, kc = min(k, fp.lenA - 1);
    const bool neumann = fp.xfB == XF_DCT;
    S* const T = static_cast<S*>(fp.T) + (size_t)fp.rowsA0 * g.ld;
    const double* const tab = fp.tri;
    // (32-bit offsets from uniform bases: a field has at most 2^24 values)
    auto at = [&](int row) { return (unsigned)(min(max(row, 0), n - 1) * g.ld + kc); };

    // all loads first, rows clamped in bounds; the rows from n on become
    // zero rows (s = 1) whose solution is 0
    double y[R], s[R];
    const int last = fp.tri_last ? fp.tri_last[kc] : n - 1;
#pragma unroll
    for (int i = 0; i < R; ++i) y[i] = (double)T[at(r0 + i)];
    // the multipliers are constant from row `last` on (but for the cosine's last row)
    auto tri_at = [&](int row) {
        return tab[at(neumann && row >= n - 1 ? n - 1 : min(row, last))];
    };
#pragma unroll
    for (int i = 0; i < R; ++i) s[i] = tri_at(r0 + i);
    const double s_before = tri_at(r0 - 1);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int row = r0 + i;
        y[i] = row < n ? y[i] * fp.tri_scale : 0.;
        if (neumann && (row == 0 || row == n - 1)) y[i] *= .5;
        if (row >= n) s[i] = 1.;
    }
    // sum over the rows of column `col` (every thread of the block calls it)
    auto column_sum = [&](double v) {
#pragma unroll
        for (int d = CB; d < 64; d *= 2) v += __shfl_xor(v, d, 64);
        __syncthreads();
        if (lane < CB) red[wave][col] = v;
        __syncthreads();
        double t = 0.;
        for (int w = 0; w < waves; ++w) t += red[w][col];
        return t;
    };
    // Bz, k = 0: the operator has the constants as its null space; the zero
    // mode of the right-hand side and of the solution is dropped (weights
    // 1/2 at the ends, as the cosine transform sums)
    const bool zero = fp.zero_mode && k0 == 0;   // (block-uniform)
    if (zero) {
        double t = 0.;
#pragma unroll
        for (int i = 0; i < R; ++i) t += y[i];
        t = column_sum(t) / (n - 1);
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int row = r0 + i;
            if (k == 0 && row < n) y[i] -= (row == 0 || row == n - 1) ? .5 * t : t;
        }
    }

    // forward sweep
    double v = 0., P = 0., sp = s_before;
#pragma unroll
    for (int i = 0; i < R; ++i) {
        v = fma(-sp, v, y[i] + v);
        P = fma(sp, 1. - P, P);
        y[i] = v;
        sp = s[i];
    }
#pragma unroll
    for (int d = CB; d < 64; d *= 2) {
        const double Po = __shfl_up(P, d, 64), vo = __shfl_up(v, d, 64);
        if (lane >= d) {
            v = fma(-P, vo, v + vo);
            P = fma(P, 1. - Po, Po);
        }
    }
    if (lane >= 64 - CB) agg[0][wave][col] = make_double2(P, v);
    P = __shfl_up(P, CB, 64);
    v = __shfl_up(v, CB, 64);
    if (lane < CB) P = v = 0.;
    __syncthreads();
    double carry = 0.;
    for (int w = 0; w < wave; ++w) {
        const double2 a = agg[0][w][col];
        carry = fma(-a.x, carry, a.y + carry);
    }
    carry = fma(-P, carry, v + carry);
    P = 0.;
    sp = s_before;
#pragma unroll
    for (int i = 0; i < R; ++i) {
        P = fma(sp, 1. - P, P);
        y[i] = fma(-P, carry, y[i] + carry);
        sp = s[i];
    }

    // backward sweep
    v = P = 0.;
#pragma unroll
    for (int i = R - 1; i >= 0; --i) {
        const double t = y[i] + v;
        v = fma(-s[i], t, t);
        P = fma(s[i], 1. - P, P);
        y[i] = v;
    }
#pragma unroll
    for (int d = CB; d < 64; d *= 2) {
        const double Po = __shfl_down(P, d, 64), vo = __shfl_down(v, d, 64);
        if (lane < 64 - d) {
            v = fma(-P, vo, v + vo);
            P = fma(P, 1. - Po, Po);
        }
    }
    if (lane < CB) agg[1][wave][col] = make_double2(P, v);
    P = __shfl_down(P, CB, 64);
    v = __shfl_down(v, CB, 64);
    if (lane >= 64 - CB) P = v = 0.;
    __syncthreads();
    carry = 0.;
    for (int w = waves - 1; w > wave; --w) {
        const double2 a = agg[1][w][col];
        carry = fma(-a.x, carry, a.y + carry);
    }
    carry = fma(-P, carry, v + carry);
    P = 0.;
#pragma unroll
    for (int i = R - 1; i >= 0; --i) {
        P = fma(s[i], 1. - P, P);
        y[i] = fma(-P, carry, y[i] + carry);
    }
    if (zero) {
        double t = 0.;
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int row = r0 + i;
            if (row < n) t += (row == 0 || row == n - 1) ? .5 * y[i] : y[i];
        }
        t = column_sum(t) / (n - 1);
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (k == 0) y[i] -= t;
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
        if (r0 + i < n && k < fp.lenA) T[at(r0 + i)] = (S)y[i];
    if (fp.partial) {
        // Bz mean: the sum of all Bz equals sum_k colsum[k] sum_i T[i][k]
        double t = 0.;
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (r0 + i < n) t += y[i];
        t = column_sum(t);
        if (wave == 0 && lane < CB && k < fp.lenA) fp.partial[k] = fp.colsum[k] * t;
    }
}

// Pass C: a block takes one field's rows ra (even) and ra + 1.  The first stage's lanes
// load their points directly.  (Prev and guess values loaded ahead of the FFT
// cost a wave per SIMD: 641^2 18.8 -> 24.7 us.)
// G: storage type of the fields, averages and guess (FP64 epilogue
// arithmetic in both).
template <int R1, int L_, typename S, typename G>
__global__ void __launch_bounds__(512)
pass_c_kernel(SolverGeom g, SolveBatch b) {
    using V = typename Vec<S>::T;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ double red[8];
    if (!gate_open(b.gate)) return;
    const BlockPos bp = xcd_block();
    const FieldPlan& fp = b.f[bp.field];
    const FftPlan p = plan_of<L_>(g);
    double2* const tw = reinterpret_cast<double2*>(lds_raw);
    V* const z = reinterpret_cast<V*>(tw + p.nroots);
    const int N = g.N, ra = bp.block * 2, rb = ra + 1;
    auto has = [&](int r) { return r >= fp.rowsA0 && r < fp.rowsA0 + fp.rowsA; };
    fetch_lines(g);
    fetch_lines(fp);
    const bool ha = has(ra), hb = has(rb);
    const bool sine = fp.xfA == XF_DST;
    const int l = threadIdx.x;
    StageRoots sr;
    sr.load(p, g.tw);
    if (l < p.lanes) {
        // (rows without data read a valid row, and are dropped; so is what the
        // ends of a sine line read)
        const S* Ta = static_cast<const S*>(fp.T) + (size_t)(ha ? ra : fp.rowsA0) * g.ld;
        const S* Tb = static_cast<const S*>(fp.T) + (size_t)(hb ? rb : fp.rowsA0) * g.ld;
        S a[R1], c[R1];
#pragma unroll
        for (int m = 0; m < R1; ++m) {
            const int k = min(max(point_column<R1>(p, l, m) - fp.colA0, 0), fp.lenA - 1);
            a[m] = Ta[k];
            c[m] = Tb[k];
        }
        Roots<R1 / 2 + 1> w;
        w.load(g.tw, p.lanes, l);
        V x[R1];
        extend<R1>(x, p, sine, l, [&](int m, int) {
            return mk<V>(ha ? a[m] : (S)0, hb ? c[m] : (S)0);
        });
        fft_first<R1>(x, z, p, sine, l, w);
    }
    sr.store(p, g.tw, tw);
    double mean = 0.;
    if (fp.partial) {
        double s = 0.;
        for (int k = threadIdx.x; k < fp.lenA; k += blockDim.x) s += fp.partial[k];
        mean = block_sum(s, red) / ((double)N * N);
    }

    const int nt = L_ ? p.threads : (int)blockDim.x;
    const G* guess = b.resid ? gp<G>(b.guess[fp.kind]) : nullptr;
    const G* prevF = gp<G>(fp.prevF);
    const size_t oa = (size_t)ra * N, ob = (size_t)min(rb, N - 1) * N;
    // prev and guess values of kCols columns of both rows (columns clamped in
    // bounds), all on their way before the first is used
    constexpr int kCols = 4;
    G qa[kCols], qb[kCols], ga[kCols], gb[kCols];
    auto fetch = [&](int j0) {
#pragma unroll
        for (int u = 0; u < kCols; ++u) {
            const int j = min(j0 + u * nt, N - 1);
            qa[u] = qb[u] = ga[u] = gb[u] = (G)0;
            if (prevF) {
                qa[u] = prevF[oa + j];
                qb[u] = prevF[ob + j];
            }
            if (guess) {
                ga[u] = guess[oa + j];
                gb[u] = guess[ob + j];
            }
        }
    };
    fft_stages<L_>(z, p, sine, tw);

    const bool transverse = fp.kind == F_EX || fp.kind == F_EY ||
                            fp.kind == F_BX || fp.kind == F_BY;
    const bool varA = b.variantA && transverse;
    G* const outF = gp<G>(fp.outF);
    G* const outAvg = gp<G>(fp.outAvg);
    double r_num = 0., r_den = 0.;
    // one output point: F from the spectrum value v, prev and guess values q, r
    auto emit = [&](size_t idx, double v, double q, double r) {
        double F = v;
        if (fp.partial) F -= mean;                         // lcode.py:362
        if (varA) F = 2 * F - q;                           // lcode.py:869-871
        if (outF) outF[idx] = (G)F;
        if (outAvg) outAvg[idx] = (G)((F + q) / 2);        // lcode.py:876-881
        if (guess) {
            const double d = F - r;
            r_num += d * d;
            r_den += F * F;
        }
    };
    for (int j0 = threadIdx.x; j0 < N; j0 += kCols * nt) {
        fetch(j0);
#pragma unroll
        for (int u = 0; u < kCols; ++u) {
            const int j = j0 + u * nt;
            if (j >= N) break;
            // columns outside the transform are exact zeros, and so is a row without
            // data (not the noise of the row that shares its transform)
            double a, c;
            get_pair(z, sine, j, a, c);
            const bool inside = j >= fp.colA0 && j < fp.colA0 + fp.lenA;
            emit(oa + j, inside && ha ? a : 0., qa[u], ga[u]);
            if (rb < N) emit(ob + j, inside && hb ? c : 0., qb[u], gb[u]);
        }
    }
    if (b.resid) {
        // guided step: this block's share of the corrector's residual against
        // the guess, summed over its waves; one reduction kernel adds the
        // blocks' partials afterwards (no same-address atomics)
        r_num = block_sum(r_num, red);
        r_den = block_sum(r_den, red);
        if (threadIdx.x == 0) {
            const int lin = blockIdx.y * gridDim.x + blockIdx.x;
            b.resid_part[2 * lin] = r_num;
            b.resid_part[2 * lin + 1] = r_den;
        }
    }
}

// resid[0..1] = sums of the blocks' partials (fixed order)
__global__ void __launch_bounds__(256)
resid_reduce_kernel(const double* part, int nblocks, double* resid) {
    __shared__ double red[2][256];
    double a = 0., d = 0.;
    for (int k = threadIdx.x; k < nblocks; k += 256) {
        a += part[2 * k];
        d += part[2 * k + 1];
    }
    red[0][threadIdx.x] = a;
    red[1][threadIdx.x] = d;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            red[0][threadIdx.x] += red[0][threadIdx.x + off];
            red[1][threadIdx.x] += red[1][threadIdx.x + off];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        resid[0] = red[0][0];
        resid[1] = red[1][0];
    }
}

// Guided step set-up: guess = sum_t c[t] hist[t] for the six fields, the
// predictor-pass averages (guess + prev) / 2 (lcode.py:876-881 with the
// guess in place of the predicted fields), and zeroed residual sums.
// Bound: memory, (6 NT + 6) grids in and 12 out; the number of terms is a template
// parameter so that the loads of all fields are in flight at once (a loop over them:
// 641^2 FP32 grids, three terms, 13.1 us; now 11.6).
template <int NT, typename G>
__global__ void __launch_bounds__(256)
guess_kernel(GuessArgs p) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (p.acc_zero && k < 2) p.acc_zero[k] = 0.;
    if (k >= p.n) return;
    G h[NT][6], prev[6];
#pragma unroll
    for (int f = 0; f < 6; ++f) {
#pragma unroll
        for (int t = 0; t < NT; ++t) h[t][f] = gp<G>(p.h[t][f])[k];
        prev[f] = gp<G>(p.prev[f])[k];
    }
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        double gsum = 0.;
#pragma unroll
        for (int t = 0; t < NT; ++t) gsum += p.c[t] * (double)h[t][f];
        const G gs = (G)gsum;
        gp<G>(p.guess[f])[k] = gs;
        gp<G>(p.avg[f])[k] = (G)(((double)gs + (double)prev[f]) / 2);
    }
}

}  // namespace

// Pass B's shape: 8 lines per block (a wave reads runs of 64 bytes) and 12
// rows per thread, while 16 waves of 8 chunks hold a line (1536 rows); 6 rows
// on short lines, where the chain of one thread is the whole time; beyond
// 1536 rows 4 lines and 16 rows, for 4096 rows (more than any transform length
// that fits LDS).  Six fields at 129^2 / 361^2 / 641^2 / 1281^2, us per launch
// (rows x lines): 6 x 8 5.9 / 9.3 / 18.5 / -, 12 x 8 6.6 / 9.5 / 13.7 / 61.6,
// 16 x 8 7.4 / 10.0 / 19.6 / -, 24 x 8 8.3 / 11.3 / 14.8 / 63.1 (fewer rows:
// more carries to combine; more: too few waves); 12 x 16 6.8 / 9.8 / 16.4 / -,
// 12 x 4 6.3 / 9.6 / 15.8 / 79.6 (longer and shorter runs).
template <typename S>
static int launch_pass_b(const SolverGeom& g, const SolveBatch& b, hipStream_t s,
                         Profiler* prof) {
    int rows = 0, lines = 0;
    for (int f = 0; f < b.nfields; ++f) {
        rows = rows > b.f[f].rowsA ? rows : b.f[f].rowsA;
        lines = lines > b.f[f].lenA ? lines : b.f[f].lenA;
    }
    ProfScope ps(prof, "solve_pass_b", s, true);
    auto go = [&](auto kernel, int R, int CB) {
        const int per_wave = R * (64 / CB);
        launch_timed(ps, kernel, dim3((lines + CB - 1) / CB, b.nfields),
                     dim3(64 * ((rows + per_wave - 1) / per_wave)), 0, s, g, b);
    };
    if (rows <= 192) go(pass_b_kernel<6, 8, S>, 6, 8);
    else if (rows <= 1536) go(pass_b_kernel<12, 8, S>, 12, 8);
    else if (rows <= 4096) go(pass_b_kernel<16, 4, S>, 16, 4);
    else {
        set_error("internal: line too long for the tridiagonal pass");
        return LCODE_E_UNSUPPORTED;
    }
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

template <int R1, int L_, typename S, typename G>
static int launch_passes(const SolverGeom& g, const SolveBatch& b, hipStream_t s,
                         Profiler* prof) {
    // one block per field and pair of grid rows
    const dim3 grid((g.N + 1) / 2, b.nfields), block(g.fft.threads);
    const size_t lds = (size_t)solver_lds_bytes(g);
    {
        ProfScope ps(prof, "solve_pass_a", s, true);
        launch_timed(ps, pass_a_kernel<R1, L_, S, G>, grid, block, lds, s, g, b);
    }
    LCODE_HIP(hipGetLastError());
    {
        const int rc = launch_pass_b<S>(g, b, s, prof);
        if (rc) return rc;
    }
    {
        ProfScope ps(prof, "solve_pass_c", s, true);
        launch_timed(ps, pass_c_kernel<R1, L_, S, G>, grid, block, lds, s, g, b);
    }
    LCODE_HIP(hipGetLastError());
    if (b.resid) {
        ProfScope ps(prof, "resid_reduce", s);
        resid_reduce_kernel<<<1, 256, 0, s>>>(b.resid_part, (int)(grid.x * grid.y), b.resid);
        LCODE_HIP(hipGetLastError());
    }
    return LCODE_OK;
}

int solver_lds_bytes(const SolverGeom& g) {
    return g.fft.nroots * (int)sizeof(double2) +
           g.fft.T * g.fft.KP * (int)(g.fp32 ? sizeof(float2) : sizeof(double2));
}

std::vector<double2> solver_fft_roots(const FftPlan& p) {
    std::vector<double2> t;
    auto add = [&](int R, int n, int step) {   // W_L^(step k q), [root][k < n]
        for (int q = 1; q < R; q += q < 4 ? 1 : 4)
            for (int k = 0; k < n; ++k) {
                const long double a = 2.0L * 3.14159265358979323846264338327950288L *
                                      ((long)step * k * q % p.L) / p.L;
                t.push_back(make_double2((double)std::cos(a), (double)-std::sin(a)));
            }
    };
    add(p.K, p.lanes, 1);
    for (int s = 1; s < p.nst; ++s) {
        const int R = fft_word_radix(p.word[s]), span = fft_word_span(p.word[s]);
        add(R, span, p.L / (span * R));
    }
    return t;
}

// The plan of a length without one of its own: the cheapest of all factorisations
// under
//   (sum of the radices + 8 per stage + 4 per 64 w columns) x rounds,
// a block's chain (DFTs in registers, an LDS exchange per stage, columns per thread in the
// assembly and the stores; a unit is about 0.1 us a pass) times how often the CU's
// wave slots are filled: w waves per block, 16 resident per CU (128 registers), rounds =
// the mean of the exact and the rounded-up number, at least 1.  Passes A + C,
// six fields, us, with the plan's cost in brackets:
//   301^2  4;5,5,6 21.5 (64)     4;15,10 22.0 (65)    10;6,10 23.7 (70)
//   361^2  4;4,5,9 24.3 (62)     12;6,10 24.7 (64)    8;9,10 27.2 (75)
//   451^2  20;5,9 30.0 (74)      12;5,15 31.0 (72)    4;5,5,9 37.0 (103)
//   801^2  10;10,16 64.8 (140)   8;5,5,8 68.7 (198)
//   901^2  8;15,15 82.1 (156)    20;9,10 84.7 (158)   4;5,9,10 128.7 (286)
//   1081^2 12;12,15 116 (178)    16;9,15 129 (244)    8;5,6,9 168 (350)
bool solver_fft_plan(int L, FftPlan* out) {
    if (const int k = static_fft(L); k >= 0) {
        const StaticFft& f = kStaticFft[k];
        *out = make_plan(L, f.R1, f.nst, f.r);
        return true;
    }
    constexpr int kCUs = 256, kSlots = 16, kMaxThreads = 512;
    const int N = L / 2 + 1;
    const double blocks = 6. * ((N + 1) / 2) / kCUs;
    double best = 0;
    bool found = false;
    int r[kMaxStages];
    for (int R1 : {4, 8, 10, 12, 16, 20}) {
        if (L % R1) continue;
        auto search = [&](auto&& self, int depth, int rest, int sum) -> void {
            if (rest == 1) {
                const FftPlan p = make_plan(L, R1, depth, r);
                if (p.threads > kMaxThreads) return;
                const int w = p.threads / 64;
                const double x = blocks / (kSlots / w);
                const double rounds = std::max(1., (x + std::ceil(x)) / 2);
                const double cost =
                    (sum + 8 * (depth + 1) + 4 * ((N + p.threads - 1) / p.threads)) * rounds;
                if (found && cost >= best) return;
                found = true;
                best = cost;
                *out = p;
                return;
            }
            if (depth == kMaxStages) return;
            for (int R : {2, 3, 4, 5, 6, 8, 9, 10, 12, 15, 16}) {
                if (rest % R) continue;
                r[depth] = R;
                self(self, depth + 1, rest / R, sum + R);
            }
        };
        search(search, 0, L / R1, R1);
    }
    return found;
}

template <typename S, typename G>
static int launch_solve_t(const SolverGeom& g, const SolveBatch& b,
                          hipStream_t s, Profiler* prof) {
    // a cosine line has the N points from column 0, a sine line the N - 2 from 1
    for (int f = 0; f < b.nfields; ++f) {
        const FieldPlan& p = b.f[f];
        const bool ok = p.xfA == XF_DCT ? p.lenA == g.N && p.colA0 == 0
                                        : p.lenA == g.N - 2 && p.colA0 == 1;
        if (!ok) {
            set_error("internal: field plan outside the transform's layout");
            return LCODE_E_INVALID;
        }
    }
    switch (g.fft.L) {
#define LCODE_CASE(LL) \
    case LL: return launch_passes<kStaticFft[static_fft(LL)].R1, LL, S, G>(g, b, s, prof);
        LCODE_CASE(64) LCODE_CASE(128) LCODE_CASE(256) LCODE_CASE(512) LCODE_CASE(640)
        LCODE_CASE(1024) LCODE_CASE(1280) LCODE_CASE(2048) LCODE_CASE(2560)
#undef LCODE_CASE
    }
    switch (g.fft.R1) {
        case 4: return launch_passes<4, 0, S, G>(g, b, s, prof);
        case 8: return launch_passes<8, 0, S, G>(g, b, s, prof);
        case 10: return launch_passes<10, 0, S, G>(g, b, s, prof);
        case 12: return launch_passes<12, 0, S, G>(g, b, s, prof);
        case 16: return launch_passes<16, 0, S, G>(g, b, s, prof);
        default: return launch_passes<20, 0, S, G>(g, b, s, prof);
    }
}

int launch_guess(const GuessArgs& p, hipStream_t s, Profiler* prof) {
    {
        ProfScope ps(prof, "guess", s);
        auto go = [&](auto k32, auto k64) {
            if (p.grid32) k32<<<(p.n + 255) / 256, 256, 0, s>>>(p);
            else k64<<<(p.n + 255) / 256, 256, 0, s>>>(p);
        };
        switch (p.nt) {
            case 1: go(guess_kernel<1, float>, guess_kernel<1, double>); break;
            case 2: go(guess_kernel<2, float>, guess_kernel<2, double>); break;
            case 3: go(guess_kernel<3, float>, guess_kernel<3, double>); break;
            default: go(guess_kernel<4, float>, guess_kernel<4, double>); break;
        }
    }
    LCODE_HIP(hipGetLastError());
    return LCODE_OK;
}

int launch_solve(const SolverGeom& g, const SolveBatch& b, hipStream_t s,
                 Profiler* prof) {
    if (b.nfields == 0) return LCODE_OK;
    // FP32 grids come only with FP32 transforms (the mixed form)
    if (b.grid32 && !g.fp32) {
        set_error("FP32 grids need the FP32 transforms");
        return LCODE_E_INVALID;
    }
    if (b.grid32) return launch_solve_t<float, float>(g, b, s, prof);
    return g.fp32 ? launch_solve_t<float, double>(g, b, s, prof)
                  : launch_solve_t<double, double>(g, b, s, prof);
}

}  // namespace lcode
