// One-dimensional FFTs of length N = R1 R2 (2 <= R1 <= R2 <= 16) in two
// register stages with one exchange through LDS, for the meshes that are not
// powers of two (those have p2_fft).
//
// With n = j + R2 r and k = k1 + R1 k2 (j, k2 < R2; r, k1 < R1):
//   X[k1 + R1 k2] = sum_j W_R2^(j k2) [ W_N^(j k1) sum_r x[j + R2 r] W_R1^(r k1) ].
// Stage 1: thread (line, j) loads its R1 points from global memory, takes
// their DFT in registers, multiplies by W_N^(j k1) and writes LDS; stage 2:
// thread (line, k1) reads its R2 points, takes their DFT and stores to global
// memory.  The backward transform is the forward one between swaps of real
// and imaginary parts.  Every radix is a compile-time DFT with constant
// twiddles (odd primes by the symmetric form, composites by two factors); a
// switch that is uniform over the workgroup picks it, so one kernel serves
// every mesh of a batch.
//
// The FP32 form stores FP32 (mesh and LDS) and computes in FP64 registers:
// FP64 runs at the FP32 rate here (no packed FP32), and FP32 constants leave
// systematic errors (every point of a radix multiplied by the same rounded
// cosine): FP32 forward transforms of 120^3 random points are 6.2e-8 off
// their FP64 values, against 1.5e-7 with FP32 arithmetic.
//
// What bounds it: HBM (a pass reads and writes the mesh once).  The passes it
// replaces went through LDS once per radix, three or four times, with integer
// divisions by run-time lengths and twiddle loads per radix point.  Measured,
// one pass over 120^3 FP32 26 -> 12 us (27.6 MB, 2.3 TB/s), its fused x pass
// with three outputs 102 -> 31 us; 256 batched FP32 meshes of 16-48 points a
// side 139 -> 56 us a pass, fused x pass 257 -> 146 us.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "device_common.hpp"
#include "fft_tiles.hpp"

namespace p3m {
namespace fft {

constexpr int kMaxTwoRadix = 16;

// N = r1 r2; div1 / div2: u / r = (u div) >> 16 for u < 1024
struct TwoPlan {
    int r1, r2, div1, div2; // r1 = 0: no such split
};

inline TwoPlan make_two(int n) {
    TwoPlan p = {0, 0, 0, 0};
    for (int a = 2; a * a <= n && a <= kMaxTwoRadix; a++)
        if (n % a == 0 && n / a <= kMaxTwoRadix)
            p.r1 = a; // the largest such a: the most balanced split
    if (p.r1 > 0) {
        p.r2 = n / p.r1;
        p.div1 = 65536 / p.r1 + 1;
        p.div2 = 65536 / p.r2 + 1;
    }
    return p;
}

// ---- constant twiddles -------------------------------------------------------

constexpr double kPiConst = 3.14159265358979323846;

// Taylor series on [0, pi / 4]
constexpr double sin_small(double x) {
    double t = x, s = 0.0;
    for (int k = 1; k < 25; k += 2) {
        s += t;
        t *= -x * x / ((k + 1) * (k + 2));
    }
    return s;
}
constexpr double cos_small(double x) {
    double t = 1.0, s = 0.0;
    for (int k = 0; k < 24; k += 2) {
        s += t;
        t *= -x * x / ((k + 1) * (k + 2));
    }
    return s;
}

struct CosSin {
    double c, s;
};
// cos and sin of 2 pi k / n, 0 <= k < n
constexpr CosSin unit_root(int k, int n) {
    const int quarter = 4 * k / n, rem = 4 * k - quarter * n;
    double c = 0.0, s = 0.0;
    if (2 * rem <= n) {
        const double x = 0.5 * kPiConst * rem / n;
        c = cos_small(x);
        s = sin_small(x);
    } else {
        const double x = 0.5 * kPiConst * (n - rem) / n;
        c = sin_small(x);
        s = cos_small(x);
    }
    switch (quarter) {
    case 0: return {c, s};
    case 1: return {-s, c};
    case 2: return {-c, -s};
    default: return {s, -c};
    }
}

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// v exp(-2 pi i K / N)
template <int K, int N, typename V> __device__ __forceinline__ V rotate(V v) {
    using T = decltype(V::x);
    constexpr int k = K % N;
    V r;
    if constexpr (k == 0) {
        r = v;
    } else if constexpr (4 * k == N) {
        r.x = v.y;
        r.y = -v.x;
    } else if constexpr (2 * k == N) {
        r.x = -v.x;
        r.y = -v.y;
    } else if constexpr (4 * k == 3 * N) {
        r.x = -v.y;
        r.y = v.x;
    } else {
        constexpr CosSin w = unit_root(k, N);
        r.x = v.x * T(w.c) + v.y * T(w.s);
        r.y = v.y * T(w.c) - v.x * T(w.s);
    }
    return r;
}

// ---- DFTs in registers (forward, natural order) -------------------------------

constexpr int first_factor(int r) {
    return r == 4 || r == 16 ? r / (r == 4 ? 2 : 4)
                             : (r == 12 ? 4 : (r % 2 == 0 ? 2 : (r % 3 == 0 && r > 3 ? 3 : r)));
}

constexpr bool coprime(int a, int b) {
    while (b) {
        const int r = a % b;
        a = b;
        b = r;
    }
    return a == 1;
}
// a^-1 mod m (m = 1: 0)
constexpr int inverse_mod(int a, int m) {
    for (int k = 1; k < m; k++)
        if (a * k % m == 1)
            return k;
    return 0;
}

template <int R, typename V> struct RegDft {
    __device__ static __forceinline__ void run(V *v) {
        using T = decltype(V::x);
        constexpr int A = first_factor(R), B = R / A;
        if constexpr (R == 2) {
            const V a = v[0], b = v[1];
            v[0] = cadd(a, b);
            v[1] = csub(a, b);
        } else if constexpr (B == 1) {
            // odd prime: pairs v_r, v_(R-r) share their cosines and sines
            constexpr int H = (R - 1) / 2;
            V s[H], d[H];
            V sum = v[0];
            static_for<H>([&](auto r) {
                s[r] = cadd(v[r + 1], v[R - 1 - r]);
                d[r] = csub(v[r + 1], v[R - 1 - r]);
                sum = cadd(sum, s[r]);
            });
            V out[R];
            out[0] = sum;
            static_for<H>([&](auto mi) {
                constexpr int m = decltype(mi)::value + 1;
                V a = v[0], b;
                b.x = T(0);
                b.y = T(0);
                static_for<H>([&](auto r) {
                    constexpr CosSin w = unit_root((decltype(r)::value + 1) * m % R, R);
                    a.x += s[r].x * T(w.c);
                    a.y += s[r].y * T(w.c);
                    b.x += d[r].x * T(w.s);
                    b.y += d[r].y * T(w.s);
                });
                out[m].x = a.x + b.y;
                out[m].y = a.y - b.x;
                out[R - m].x = a.x - b.y;
                out[R - m].y = a.y + b.x;
            });
            static_for<R>([&](auto k) { v[k] = out[k]; });
        } else if constexpr (coprime(A, B)) {
            // coprime factors: index n = B n1 + A n2, k the matching residue,
            // no twiddles between the factors (Good's prime-factor mapping):
            // fewer roundings than the two-factor step below
            constexpr int eA = B * inverse_mod(B, A), eB = A * inverse_mod(A, B);
            V t[R];
            static_for<B>([&](auto n2) {
                V a[A];
                static_for<A>([&](auto n1) { a[n1] = v[(B * decltype(n1)::value + A * decltype(n2)::value) % R]; });
                RegDft<A, V>::run(a);
                static_for<A>([&](auto k1) { t[n2 + B * k1] = a[k1]; });
            });
            static_for<A>([&](auto k1) {
                RegDft<B, V>::run(t + B * k1);
                static_for<B>([&](auto k2) {
                    v[(eA * decltype(k1)::value + eB * decltype(k2)::value) % R] = t[B * k1 + k2];
                });
            });
        } else {
            V t[R];
            static_for<B>([&](auto n2) {
                V a[A];
                static_for<A>([&](auto n1) { a[n1] = v[B * n1 + n2]; });
                RegDft<A, V>::run(a);
                static_for<A>([&](auto k1) {
                    t[n2 + B * k1] = rotate<decltype(n2)::value * decltype(k1)::value, R>(a[k1]);
                });
            });
            static_for<A>([&](auto k1) {
                RegDft<B, V>::run(t + B * k1);
                static_for<B>([&](auto k2) { v[k1 + A * k2] = t[B * k1 + k2]; });
            });
        }
    }
};

// f(integral_constant<int, r>) for the run-time radix r (uniform over the workgroup)
template <typename F> __device__ __forceinline__ void with_radix(int r, F &&f) {
    switch (r) {
#define CASE(R) case R: f(std::integral_constant<int, R>{}); break;
        CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
        CASE(13) CASE(14) CASE(15) CASE(16)
#undef CASE
    default: break;
    }
}

template <typename V> __device__ __forceinline__ V swap_if(V v, int inv) {
    V r;
    r.x = inv ? v.y : v.x;
    r.y = inv ? v.x : v.y;
    return r;
}

// A copy of v the compiler cannot see through: inside the loops over field
// components it keeps the address arithmetic and twiddle loads of all
// radices from being moved in front of the loop (256 registers, one
// wavefront per SIMD).
__device__ __forceinline__ int opaque(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// ---- the two stages over a tile of lines ----------------------------------------

// Thread u of a tile of lt = 2^lg lines: its line and its index among `r`
// per line.  CONTIG (z axis): the indexes of one line are neighbours, so a
// stage's loads and stores run along the line; otherwise the lines are.
template <bool CONTIG>
__device__ __forceinline__ void two_index(int u, int lg, int r, int div, int &l, int &j) {
    if (CONTIG) {
        l = (u * div) >> 16;
        j = u - l * r;
    } else {
        l = u & ((1 << lg) - 1);
        j = u >> lg;
    }
}

// LDS slot of (line l, k1, j): along the line with an odd row pitch (rows of
// r2 | 1 points keep stage 2's stride odd), or lines fastest
template <bool CONTIG>
__device__ __forceinline__ int two_slot(int l, int k1, int j, int r1, int r2, int lg) {
    if (CONTIG)
        return l * (r1 * (r2 | 1)) + k1 * (r2 | 1) + j;
    return ((k1 * r2 + j) << lg) + l;
}

// complex points of LDS a tile takes
__host__ __device__ inline int two_lds_points(const TwoPlan &p, int lt) {
    const int a = p.r1 * (p.r2 | 1), b = p.r2 * (p.r1 | 1);
    return lt * (a > b ? a : b);
}

// stage 1 of a tile: load(l, e) -> point e of line l
template <bool CONTIG, typename V, typename Load>
__device__ __forceinline__ void two_stage1(int r1, int r2, int div2, int lg, const double2 *__restrict__ tw,
                                           V *buf, int inv, Load &&load) {
    int l, j;
    two_index<CONTIG>(opaque(threadIdx.x), lg, r2, div2, l, j);
    if (l >= (1 << lg) || j >= r2)
        return;
    with_radix(r1, [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        V in[R];
        static_for<R>([&](auto r) { in[r] = load(l, j + r2 * r); });
        double2 v[R];
        static_for<R>([&](auto r) { v[r] = widen(swap_if(in[r], inv)); });
        RegDft<R, double2>::run(v);
        static_for<R>([&](auto k) {
            buf[two_slot<CONTIG>(l, k, j, r1, r2, lg)] = narrow<V>(k == 0 ? v[k] : cmul(v[k], tw[j * k]));
        });
    });
}

// stage 2 of a tile: store(l, e, v)
template <bool CONTIG, typename V, typename Store>
__device__ __forceinline__ void two_stage2(int r1, int r2, int div1, int lg, const V *buf, int inv,
                                           Store &&store) {
    int l, k1;
    two_index<CONTIG>(opaque(threadIdx.x), lg, r1, div1, l, k1);
    if (l >= (1 << lg) || k1 >= r1)
        return;
    with_radix(r2, [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        double2 v[R];
        static_for<R>([&](auto j) { v[j] = widen(buf[two_slot<CONTIG>(l, k1, j, r1, r2, lg)]); });
        RegDft<R, double2>::run(v);
        static_for<R>([&](auto k2) { store(l, k1 + r1 * k2, swap_if(narrow<V>(v[k2]), inv)); });
    });
}

// in-place pass over lines of a mesh
template <typename T, bool CONTIG>
__device__ __forceinline__ void two_pass_tile(c2_t<T> *data, const LineMap &m, const TwoPlan &p,
                                              const double2 *__restrict__ tw, int inv, int lg, long L0,
                                              unsigned char *smem) {
    using V = c2_t<T>;
    V *buf = reinterpret_cast<V *>(smem);
    auto start = [&](int l, bool &ok) {
        const unsigned L = (unsigned)L0 + (unsigned)l;
        ok = (long)L < m.nlines;
        const unsigned a = L / (unsigned)m.C;
        return (long)a * m.sa + (long)(L - a * (unsigned)m.C);
    };
    int l1, l2, unused;
    two_index<CONTIG>(threadIdx.x, lg, p.r2, p.div2, l1, unused);
    two_index<CONTIG>(threadIdx.x, lg, p.r1, p.div1, l2, unused);
    bool ok1, ok2;
    const long s1 = start(l1, ok1), s2 = start(l2, ok2);
    two_stage1<CONTIG>(p.r1, p.r2, p.div2, lg, tw, buf, inv, [&](int, int e) {
        V v;
        v.x = v.y = T(0);
        if (ok1)
            v = data[s1 + e * m.es];
        return v;
    });
    __syncthreads();
    two_stage2<CONTIG>(p.r1, p.r2, p.div1, lg, buf, inv, [&](int, int e, const V &v) {
        if (ok2)
            data[s2 + e * m.es] = v;
    });
}

// r2c along z: real lines of n points -> the first n / 2 + 1 coefficients
template <typename T>
__device__ __forceinline__ void two_r2c_tile(const T *__restrict__ in, c2_t<T> *__restrict__ out, long nlines,
                                             const TwoPlan &p, const double2 *__restrict__ tw, int lg,
                                             long L0, unsigned char *smem) {
    using V = c2_t<T>;
    V *buf = reinterpret_cast<V *>(smem);
    const int n = p.r1 * p.r2, H = n / 2 + 1;
    two_stage1<true>(p.r1, p.r2, p.div2, lg, tw, buf, 0, [&](int l, int e) {
        V v;
        v.x = L0 + l < nlines ? in[(L0 + l) * n + e] : T(0);
        v.y = T(0);
        return v;
    });
    __syncthreads();
    two_stage2<true>(p.r1, p.r2, p.div1, lg, buf, 0, [&](int l, int e, const V &v) {
        if (e < H && L0 + l < nlines)
            out[(L0 + l) * H + e] = v;
    });
}

// c2r along z: Hermitian lines of n / 2 + 1 coefficients -> n real values
// (X[n - k] = conj X[k]; the real part of the backward transform)
template <typename T>
__device__ __forceinline__ void two_c2r_tile(const c2_t<T> *__restrict__ in, T *__restrict__ out, long nlines,
                                             const TwoPlan &p, const double2 *__restrict__ tw, int lg,
                                             long L0, unsigned char *smem) {
    using V = c2_t<T>;
    V *buf = reinterpret_cast<V *>(smem);
    const int n = p.r1 * p.r2, H = n / 2 + 1;
    two_stage1<true>(p.r1, p.r2, p.div2, lg, tw, buf, 1, [&](int l, int e) {
        V v;
        v.x = v.y = T(0);
        if (L0 + l < nlines) {
            v = in[(L0 + l) * H + (e < H ? e : n - e)];
            v.y = e < H ? v.y : -v.y;
        }
        return v;
    });
    __syncthreads();
    two_stage2<true>(p.r1, p.r2, p.div1, lg, buf, 1, [&](int l, int e, const V &v) {
        if (L0 + l < nlines)
            out[(L0 + l) * n + e] = v.x;
    });
}

// The fused x pass.  The forward transform's stage 2 leaves thread (line, k1)
// with the points k1 + R1 k2, which are stage 1's inputs of the backward
// transform with the factors' roles exchanged, so the multiplied spectrum
// goes from one to the other in registers.

// this thread's points X[k1 + R1 k2] from LDS, handed to use(k2, value);
// the results of use are kept in x
template <typename V, typename X, typename Use>
__device__ __forceinline__ void two_forward_points(const TwoPlan &p, X (&x)[kMaxTwoRadix], int l, int k1, int lg,
                                                   const V *buf, Use &&use) {
    with_radix(p.r2, [&](auto rc) {
        constexpr int R = decltype(rc)::value;
        double2 v[R];
        static_for<R>([&](auto j) { v[j] = widen(buf[two_slot<false>(l, k1, j, p.r1, p.r2, lg)]); });
        RegDft<R, double2>::run(v);
        static_for<R>([&](auto k) { x[k] = narrow<X>(use(k, v[k])); });
    });
}

// backward transform of the points make(k2) of this thread's (line, k1),
// which arrive with real and imaginary parts swapped; barriers before (other
// threads may still read buf) and between the stages
template <typename V, typename Make, typename Store>
__device__ __forceinline__ void two_backward(const TwoPlan &p, bool active, int l, int k1, int lg,
                                             const double2 *__restrict__ tw, V *buf, Make &&make, Store &&store) {
    __syncthreads();
    if (active)
        with_radix(p.r2, [&](auto rc) {
            constexpr int R = decltype(rc)::value;
            double2 w[R];
            static_for<R>([&](auto k) { w[k] = make(k); });
            RegDft<R, double2>::run(w);
            static_for<R>([&](auto k) {
                buf[two_slot<false>(l, k, k1, p.r2, p.r1, lg)] = narrow<V>(k == 0 ? w[k] : cmul(w[k], tw[k1 * k]));
            });
        });
    __syncthreads();
    two_stage2<false>(p.r2, p.r1, p.div2, lg, buf, 1, store);
}

// The fused x pass (convolve_x_tile): forward along x, X <- G X (FP64
// product rounded to T), backward into out0 (NOUT == 1) or backward of
// i (2 pi / L) Dn[n_d] X into out_d (NOUT == 3).  Lines c = j W + k of
// stride nl.
template <int NOUT, typename T>
__device__ __forceinline__ void
two_convolve_tile(const c2_t<T> *in, c2_t<T> *out0, c2_t<T> *out1, c2_t<T> *out2, long nl, int W,
                  const TwoPlan &p, const double2 *__restrict__ tw, const double *__restrict__ G,
                  const double *__restrict__ Dn, double twopi_L, int lg, long L0, unsigned char *smem) {
    using V = c2_t<T>;
    V *buf = reinterpret_cast<V *>(smem);
    const int M = p.r1 * p.r2;
    const int l = threadIdx.x & ((1 << lg) - 1), k1 = threadIdx.x >> lg;
    const long L = L0 + l;
    const bool ok = L < nl, active = k1 < p.r1;
    two_stage1<false>(p.r1, p.r2, p.div2, lg, tw, buf, 0, [&](int, int e) {
        V v;
        v.x = v.y = T(0);
        if (ok)
            v = in[L + (long)e * nl];
        return v;
    });
    const int jy = ok ? (int)((unsigned)L / (unsigned)W) : 0, kz = ok ? (int)L - jy * W : 0;
    const double *Gl = G + ((long)k1 * M + jy) * M + kz;
    const long gstep = (long)p.r1 * M * M;
    V x[kMaxTwoRadix];
    __syncthreads();
    if (active)
        two_forward_points(p, x, l, k1, lg, buf, [&](auto k, double2 v) {
            const double g = ok ? Gl[gstep * k] : 0.0;
            return make_double2(v.x * g, v.y * g);
        });
#pragma unroll 1
    for (int d = 0; d < NOUT; d++) {
        V *out = d == 0 ? out0 : (d == 1 ? out1 : out2);
        const int kd = opaque(k1), ld = opaque(l);
        const double fl = NOUT == 1 || d == 0 ? 0.0 : twopi_L * Dn[d == 1 ? jy : kz];
        two_backward(
            p, active, ld, kd, lg, tw, buf,
            [&](auto k) {
                if constexpr (NOUT == 1)
                    return make_double2(x[k].y, x[k].x);
                // i f X = (-f y, f x), swapped
                const double f = d == 0 ? twopi_L * Dn[kd + p.r1 * k] : fl;
                return make_double2(f * x[k].x, -f * x[k].y);
            },
            [&](int, int e, const V &v) {
                if (ok)
                    out[L + (long)e * nl] = v;
            });
    }
}

// Adjoint of the ik gradient step (divergence_x_tile): forward of three
// spectra, out = sum_d (-i (2 pi / L) Dn[n_d] G) X_d, backward.
template <typename T>
__device__ __forceinline__ void
two_divergence_tile(const c2_t<T> *in0, const c2_t<T> *in1, const c2_t<T> *in2, c2_t<T> *out, long nl, int W,
                    const TwoPlan &p, const double2 *__restrict__ tw, const double *__restrict__ G,
                    const double *__restrict__ Dn, double twopi_L, int lg, long L0, unsigned char *smem) {
    using V = c2_t<T>;
    V *buf = reinterpret_cast<V *>(smem);
    const int M = p.r1 * p.r2;
    const int l = threadIdx.x & ((1 << lg) - 1), k1 = threadIdx.x >> lg;
    const long L = L0 + l;
    const bool ok = L < nl, active = k1 < p.r1;
    const int jy = ok ? (int)((unsigned)L / (unsigned)W) : 0, kz = ok ? (int)L - jy * W : 0;
    const double *Gl = G + ((long)k1 * M + jy) * M + kz;
    const long gstep = (long)p.r1 * M * M;
    double2 acc[kMaxTwoRadix];
#pragma unroll 1
    for (int d = 0; d < 3; d++) {
        const int kd = opaque(k1), ld = opaque(l);
        const V *in = d == 0 ? in0 : (d == 1 ? in1 : in2);
        two_stage1<false>(p.r1, p.r2, p.div2, lg, tw, buf, 0, [&](int, int e) {
            V v;
            v.x = v.y = T(0);
            if (ok)
                v = in[L + (long)e * nl];
            return v;
        });
        __syncthreads();
        const double fl = d == 0 ? 0.0 : twopi_L * Dn[d == 1 ? jy : kz];
        if (active)
            two_forward_points(p, acc, ld, kd, lg, buf, [&](auto k, const double2 &v) {
                const double f = (d == 0 ? twopi_L * Dn[kd + p.r1 * k] : fl) * (ok ? Gl[gstep * k] : 0.0);
                // -i f X = (f y, -f x), swapped
                double2 w = make_double2(-f * v.x, f * v.y);
                if (d > 0)
                    w = cadd(w, acc[k]);
                return w;
            });
        __syncthreads();
    }
    two_backward(
        p, active, l, k1, lg, tw, buf, [&](auto k) { return acc[k]; },
        [&](int, int e, const V &v) {
            if (ok)
                out[L + (long)e * nl] = v;
        });
}

}  // namespace fft
}  // namespace p3m
