// Mixed-radix Stockham FFT for the P3M meshes (radices 2,3,4,5,7,8,11,13).
//
// A 3D transform is three passes of batched 1D transforms, one per axis.
// Lengths 16 ... 256 of powers of two hold their lines in registers (p2_fft,
// below), lengths with two factors up to 16 take two register stages
// (fft_two.hpp); the rest (162, 200, 220, above 256, ...) one pass per radix
// through two LDS buffers (fft_tiles.hpp).  The x pass of the forward
// transform is fused with the multiplication by the influence function (and,
// for ik, the gradient i 2pi/L Dn) and with the x pass of the backward
// transform, so the spectrum never makes an extra round trip through HBM.
//
// Conventions are FFTW's (the reference's transforms, p3m-ik.c:84-88 etc.):
// forward X[k] = sum x[n] exp(-2 pi i nk/N), backward with +, unnormalised.
#include <hip/hip_runtime.h>

#include <cmath>
#include <new>

#include "batch_desc.hpp"
#include "device_common.hpp"
#include "fft_tiles.hpp"
#include "fft_two_launch.hpp"
#include "k_internal.hpp"

using namespace p3m;
using namespace p3m::fft;

namespace {

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_fft_pass(c2_t<T> *data, LineMap m, Radices rp, const c2_t<T> *__restrict__ tw, int inv, int lt,
           int contig) {
    extern __shared__ unsigned char smem[];
    fft_pass_tile<T>(data, m, rp, tw, inv, lt, contig, (long)blockIdx.x * lt, smem);
}

// Power-of-two lines: register-resident passes (p2_fft), 256 / (N / 8)
// lines per workgroup, one LDS row per line.  Contiguous lines (z axis):
// a line's threads are consecutive, so each load of the eight covers N / 8
// neighbouring elements; strided lines (y, x): consecutive threads take
// neighbouring lines.
template <int N, typename T, bool CONTIG>
__global__ void __launch_bounds__(kThreads)
k_fft_p2(Three<c2_t<T> *> set, LineMap m, const double2 *__restrict__ tw, int inv) {
    using V = c2_t<T>;
    V *data = set.p[blockIdx.y];
    constexpr int TPL = N / 8, LPW = kThreads / TPL, PITCH = N + 1;
    __shared__ V buf[LPW * PITCH];
    const int tid = threadIdx.x;
    const int l = CONTIG ? tid / TPL : tid % LPW;
    const int t = CONTIG ? tid % TPL : tid / LPW;
    const long L = (long)blockIdx.x * LPW + l;
    const bool ok = L < m.nlines;
    const long base = ok ? line_start(m, L) : 0;
    V in[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        in[s].x = in[s].y = T(0);
        if (ok)
            in[s] = data[base + (long)(t + TPL * s) * m.es];
    }
    double2 v[8];
#pragma unroll
    for (int s = 0; s < 8; s++)
        v[s] = widen(in[s]);
    p2_fft<N>(v, buf + l * PITCH, t, tw, inv);
    if (ok) {
#pragma unroll
        for (int s = 0; s < 8; s++)
            data[base + (long)(t + TPL * s) * m.es] = narrow<V>(v[s]);
    }
}

// The fused x pass (convolve_x_tile) for power-of-two meshes on registers:
// forward along x, X <- G X, then for nout == 1
// backward into out0, for nout == 3 backward of i (2 pi / L) Dn[n_d] X into
// out_d.  Lines c = j W + k (strided by nl = M W), element e = n_x.
template <int N, typename T>
__global__ void __launch_bounds__(kThreads)
k_convolve_p2(const c2_t<T> *in, c2_t<T> *out0, c2_t<T> *out1, c2_t<T> *out2, long nl, int W,
              const double2 *__restrict__ tw, const double *__restrict__ G,
              const double *__restrict__ Dn, double twopi_L, int nout) {
    using V = c2_t<T>;
    constexpr int TPL = N / 8, LPW = kThreads / TPL, PITCH = N + 1;
    __shared__ V buf[LPW * PITCH];
    const int tid = threadIdx.x;
    const int l = tid % LPW, t = tid / LPW;
    const long L = (long)blockIdx.x * LPW + l;
    const bool ok = L < nl;
    const int j = ok ? (int)(L / W) : 0, k = ok ? (int)(L - (long)j * W) : 0;
    V x[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        x[s].x = x[s].y = T(0);
        if (ok)
            x[s] = in[L + (long)(t + TPL * s) * nl];
    }
    double2 v[8];
#pragma unroll
    for (int s = 0; s < 8; s++)
        v[s] = widen(x[s]);
    V *line = buf + l * PITCH;
    p2_fft<N>(v, line, t, tw, 0);
#pragma unroll
    for (int s = 0; s < 8; s++) {
        const int e = t + TPL * s;
        const double g = ok ? G[((long)e * N + j) * N + k] : 0.0;
        v[s].x *= g;
        v[s].y *= g;
    }
    if (nout == 1) {
        p2_fft<N>(v, line, t, tw, 1);
        if (ok) {
#pragma unroll
            for (int s = 0; s < 8; s++)
                out0[L + (long)(t + TPL * s) * nl] = narrow<V>(v[s]);
        }
        return;
    }
    V *outs[3] = {out0, out1, out2};
    for (int d = 0; d < 3; d++) {
        double2 w[8];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int e = t + TPL * s;
            const int nd = (d == 0) ? e : ((d == 1) ? j : k);
            const double f = twopi_L * Dn[nd];
            w[s].x = -f * v[s].y;
            w[s].y = f * v[s].x;
        }
        p2_fft<N>(w, line, t, tw, 1);
        if (ok) {
#pragma unroll
            for (int s = 0; s < 8; s++)
                outs[d][L + (long)(t + TPL * s) * nl] = narrow<V>(w[s]);
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_fft_r2c_z(const T *__restrict__ in, c2_t<T> *__restrict__ out, long nlines, int n, Radices rp,
            const c2_t<T> *__restrict__ tw, int lt) {
    extern __shared__ unsigned char smem[];
    fft_r2c_z_tile<T>(in, out, nlines, n, rp, tw, lt, (long)blockIdx.x * lt, smem);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_fft_c2r_z(const c2_t<T> *__restrict__ in, T *__restrict__ out, long nlines, int n, Radices rp,
            const c2_t<T> *__restrict__ tw, int lt) {
    extern __shared__ unsigned char smem[];
    fft_c2r_z_tile<T>(in, out, nlines, n, rp, tw, lt, (long)blockIdx.x * lt, smem);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_convolve_x(const c2_t<T> *in, c2_t<T> *out0, c2_t<T> *out1, c2_t<T> *out2, LineMap m, int W,
             Radices rp, const c2_t<T> *__restrict__ tw, const double *__restrict__ G,
             const double *__restrict__ Dn, double twopi_L, int nout, int lt) {
    extern __shared__ unsigned char smem[];
    convolve_x_tile<T>(in, out0, out1, out2, m, W, rp, tw, G, Dn, twopi_L, nout, lt,
                       (long)blockIdx.x * lt, smem);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_divergence_x(const c2_t<T> *in0, const c2_t<T> *in1, const c2_t<T> *in2, c2_t<T> *out, LineMap m,
               int W, Radices rp, const c2_t<T> *__restrict__ tw, const double *__restrict__ G,
               const double *__restrict__ Dn, double twopi_L, int lt) {
    extern __shared__ unsigned char smem[];
    divergence_x_tile<T>(in0, in1, in2, out, m, W, rp, tw, G, Dn, twopi_L, lt,
                         (long)blockIdx.x * lt, smem);
}

}  // namespace

struct p3mk_fft {
    p3mk_geom g;
    int M, H;
    Radices rp;
    TwoPlan two;
    double2 *tw64;
    float2 *tw32;
};

extern "C" size_t p3mk_mesh_bytes(const p3mk_geom *g) {
    const size_t M3 = (size_t)g->M * g->M * g->M;
    const size_t s = g->fp32 ? sizeof(float) : sizeof(double);
    return g->r2c ? M3 * s : 2 * M3 * s;
}

extern "C" size_t p3mk_spec_bytes(const p3mk_geom *g) {
    const size_t s = g->fp32 ? sizeof(float) : sizeof(double);
    const size_t H = g->r2c ? (size_t)(g->M / 2 + 1) : (size_t)g->M;
    return 2 * (size_t)g->M * g->M * H * s;
}

extern "C" int p3mk_fft_create(p3mk_fft **out, const p3mk_geom *g) {
    *out = nullptr;
    Radices rp;
    if (g->M < 2 || !make_radices(g->M, rp))
        return p3mk_fail(P3MK_EINVAL, "mesh size is not a product of 2,3,5,7,11,13", 0);
    p3mk_fft *f = new (std::nothrow) p3mk_fft;
    if (!f)
        return p3mk_fail(P3MK_ENOMEM, "fft plan allocation", 0);
    f->g = *g;
    f->M = g->M;
    f->H = g->M / 2 + 1;
    f->rp = rp;
    f->two = make_two(g->M);
    f->tw64 = nullptr;
    f->tw32 = nullptr;
    const int n = g->M;
    double2 *h64 = new (std::nothrow) double2[n];
    float2 *h32 = new (std::nothrow) float2[n];
    if (!h64 || !h32) {
        delete[] h64;
        delete[] h32;
        delete f;
        return p3mk_fail(P3MK_ENOMEM, "twiddle table", 0);
    }
    for (int k = 0; k < n; k++) {
        // exp(-2 pi i k/n), from long double for correctly rounded doubles
        const long double a = -2.0L * 3.141592653589793238462643383279502884L * k / n;
        h64[k] = make_double2((double)cosl(a), (double)sinl(a));
        h32[k] = make_float2((float)cosl(a), (float)sinl(a));
    }
    int rc = p3mk_alloc((void **)&f->tw64, sizeof(double2) * n);
    if (rc == P3MK_OK)
        rc = p3mk_alloc((void **)&f->tw32, sizeof(float2) * n);
    if (rc == P3MK_OK) {
        hipError_t e = hipMemcpy(f->tw64, h64, sizeof(double2) * n, hipMemcpyHostToDevice);
        if (e == hipSuccess)
            e = hipMemcpy(f->tw32, h32, sizeof(float2) * n, hipMemcpyHostToDevice);
        if (e != hipSuccess)
            rc = p3mk_fail(P3MK_EDEVICE, "twiddle upload", (int)e);
    }
    delete[] h64;
    delete[] h32;
    if (rc != P3MK_OK) {
        p3mk_fft_destroy(f);
        return rc;
    }
    *out = f;
    return P3MK_OK;
}

extern "C" void p3mk_fft_destroy(p3mk_fft *f) {
    if (!f)
        return;
    p3mk_release(f->tw64);
    p3mk_release(f->tw32);
    delete f;
}

namespace {

// Lines per workgroup of a launch over one mesh: pow2_tile_lines, halved
// (down to 8) while the launch would have fewer workgroups than the GPU has
// CUs (256).
template <typename T> int launch_lines(int n, int nbuf, long nlines) {
    int lt = pow2_tile_lines<T>(n, nbuf);
    while (lt > 8 && (nlines + lt - 1) / lt < 256)
        lt /= 2;
    return lt;
}

template <int N, typename T>
int pass_p2(p3mk_fft *f, Three<c2_t<T> *> data, int k, const LineMap &m, int inv, bool contig, p3mk_queue *q) {
    constexpr int LPW = kThreads / (N / 8);
    const long blocks = (m.nlines + LPW - 1) / LPW;
    const double2 *tw = f->tw64;
    if (contig)
        hipLaunchKernelGGL((k_fft_p2<N, T, true>), dim3((unsigned)blocks, (unsigned)k), dim3(kThreads), 0,
                           p3mk_stream(q), data, m, tw, inv);
    else
        hipLaunchKernelGGL((k_fft_p2<N, T, false>), dim3((unsigned)blocks, (unsigned)k), dim3(kThreads), 0,
                           p3mk_stream(q), data, m, tw, inv);
    return p3mk_launch_check("fft pass");
}

// one pass over k <= 3 meshes
template <typename T>
int pass(p3mk_fft *f, Three<c2_t<T> *> data, int k, const LineMap &m, int inv, bool contig, p3mk_queue *q) {
    switch (m.n) {
    case 16: return pass_p2<16, T>(f, data, k, m, inv, contig, q);
    case 32: return pass_p2<32, T>(f, data, k, m, inv, contig, q);
    case 64: return pass_p2<64, T>(f, data, k, m, inv, contig, q);
    case 128: return pass_p2<128, T>(f, data, k, m, inv, contig, q);
    case 256: return pass_p2<256, T>(f, data, k, m, inv, contig, q);
    default: break;
    }
    const c2_t<T> *tw = sizeof(T) == 8 ? (const c2_t<T> *)f->tw64 : (const c2_t<T> *)f->tw32;
    if (f->two.r1 > 0)
        return two_pass<T>(f->two, data, k, m, f->tw64, inv, contig, p3mk_stream(q));
    const int lt = launch_lines<T>(m.n, 2, m.nlines);
    const size_t lds = 2 * (size_t)lt * (m.n + 1) * sizeof(c2_t<T>);
    const long blocks = (m.nlines + lt - 1) / lt;
    for (int j = 0; j < k; j++)
        hipLaunchKernelGGL(k_fft_pass<T>, dim3((unsigned)blocks), dim3(kThreads), lds, p3mk_stream(q),
                           data.p[j], m, f->rp, tw, inv, lt, contig ? 1 : 0);
    return p3mk_launch_check("fft pass");
}

template <typename P> Three<P> three(int k, void *const p[3]) {
    Three<P> r = {};
    for (int j = 0; j < k; j++)
        r.p[j] = (P)p[j];
    return r;
}

template <typename T>
int forward_zy(p3mk_fft *f, int k, void *const mesh[3], void *const spec[3], p3mk_queue *q) {
    using V = c2_t<T>;
    const int M = f->M, H = f->H;
    if (!f->g.r2c) {
        const Three<V *> d = three<V *>(k, mesh);
        LineMap z = {M, 1, 1, M, (long)M * M};
        P3MK_TRY(pass<T>(f, d, k, z, 0, true, q));
        LineMap y = {M, M, M, (long)M * M, (long)M * M};
        return pass<T>(f, d, k, y, 0, false, q);
    }
    const long nl = (long)M * M;
    const Three<V *> s = three<V *>(k, spec);
    if (f->two.r1 > 0) {
        P3MK_TRY(two_r2c<T>(f->two, three<const T *>(k, mesh), s, k, nl, f->tw64, p3mk_stream(q)));
    } else {
        const c2_t<T> *tw = sizeof(T) == 8 ? (const V *)f->tw64 : (const V *)f->tw32;
        const int lt = launch_lines<T>(M, 2, nl);
        const size_t lds = 2 * (size_t)lt * (M + 1) * sizeof(V);
        for (int j = 0; j < k; j++)
            hipLaunchKernelGGL(k_fft_r2c_z<T>, dim3((unsigned)((nl + lt - 1) / lt)), dim3(kThreads), lds,
                               p3mk_stream(q), (const T *)mesh[j], s.p[j], nl, M, f->rp, tw, lt);
        P3MK_TRY(p3mk_launch_check("fft r2c"));
    }
    LineMap y = {M, H, H, (long)M * H, (long)M * H};
    return pass<T>(f, s, k, y, 0, false, q);
}

template <typename T>
int backward_yz(p3mk_fft *f, int k, void *const spec[3], void *const mesh[3], p3mk_queue *q) {
    using V = c2_t<T>;
    const int M = f->M, H = f->H;
    const Three<V *> s = three<V *>(k, spec);
    if (!f->g.r2c) {
        LineMap y = {M, M, M, (long)M * M, (long)M * M};
        P3MK_TRY(pass<T>(f, s, k, y, 1, false, q));
        LineMap z = {M, 1, 1, M, (long)M * M};
        return pass<T>(f, s, k, z, 1, true, q);
    }
    LineMap y = {M, H, H, (long)M * H, (long)M * H};
    P3MK_TRY(pass<T>(f, s, k, y, 1, false, q));
    const long nl = (long)M * M;
    if (f->two.r1 > 0)
        return two_c2r<T>(f->two, three<const V *>(k, spec), three<T *>(k, mesh), k, nl, f->tw64, p3mk_stream(q));
    const c2_t<T> *tw = sizeof(T) == 8 ? (const V *)f->tw64 : (const V *)f->tw32;
    const int lt = launch_lines<T>(M, 2, nl);
    const size_t lds = 2 * (size_t)lt * (M + 1) * sizeof(V);
    for (int j = 0; j < k; j++)
        hipLaunchKernelGGL(k_fft_c2r_z<T>, dim3((unsigned)((nl + lt - 1) / lt)), dim3(kThreads), lds,
                           p3mk_stream(q), (const V *)spec[j], (T *)mesh[j], nl, M, f->rp, tw, lt);
    return p3mk_launch_check("fft c2r");
}

template <int N, typename T>
int convolve_p2(p3mk_fft *f, int nout, const double *G, const double *Dn, void *spec,
                void *const out[3], long nl, int W, p3mk_queue *q) {
    using V = c2_t<T>;
    constexpr int LPW = kThreads / (N / 8);
    const double2 *tw = f->tw64;
    V *o0 = (V *)out[0];
    V *o1 = nout == 3 ? (V *)out[1] : nullptr;
    V *o2 = nout == 3 ? (V *)out[2] : nullptr;
    hipLaunchKernelGGL((k_convolve_p2<N, T>), dim3((unsigned)((nl + LPW - 1) / LPW)), dim3(kThreads), 0,
                       p3mk_stream(q), (const V *)spec, o0, o1, o2, nl, W, tw, G, Dn,
                       2.0 * 3.14159265358979323846 / f->g.L, nout);
    return p3mk_launch_check("convolve");
}

template <typename T>
int convolve(p3mk_fft *f, int nout, const double *G, const double *Dn, void *spec,
             void *const out[3], p3mk_queue *q) {
    using V = c2_t<T>;
    const int M = f->M;
    const int W = f->g.r2c ? f->H : M;
    const long nl = (long)M * W;
    switch (M) {
    case 16: return convolve_p2<16, T>(f, nout, G, Dn, spec, out, nl, W, q);
    case 32: return convolve_p2<32, T>(f, nout, G, Dn, spec, out, nl, W, q);
    case 64: return convolve_p2<64, T>(f, nout, G, Dn, spec, out, nl, W, q);
    case 128: return convolve_p2<128, T>(f, nout, G, Dn, spec, out, nl, W, q);
    case 256: return convolve_p2<256, T>(f, nout, G, Dn, spec, out, nl, W, q);
    default: break;
    }
    const c2_t<T> *tw = sizeof(T) == 8 ? (const V *)f->tw64 : (const V *)f->tw32;
    const double twopi_L = 2.0 * 3.14159265358979323846 / f->g.L;
    if (f->two.r1 > 0)
        return two_convolve<T>(f->two, (const V *)spec, (V *const *)out, nout, nl, W, f->tw64, G, Dn, twopi_L,
                               p3mk_stream(q));
    LineMap x = {M, nl, nl, 0, nl};
    const int nbuf = (nout == 3) ? 3 : 2;
    const int lt = launch_lines<T>(M, nbuf, nl);
    const size_t lds = (size_t)nbuf * lt * (M + 1) * sizeof(V);
    V *o0 = (V *)out[0];
    V *o1 = nout == 3 ? (V *)out[1] : nullptr;
    V *o2 = nout == 3 ? (V *)out[2] : nullptr;
    hipLaunchKernelGGL(k_convolve_x<T>, dim3((unsigned)((nl + lt - 1) / lt)), dim3(kThreads), lds,
                       p3mk_stream(q), (const V *)spec, o0, o1, o2, x, W, f->rp, tw, G, Dn, twopi_L,
                       nout, lt);
    return p3mk_launch_check("convolve");
}

template <typename T>
int divergence(p3mk_fft *f, const double *G, const double *Dn, void *const in[3], void *out,
               p3mk_queue *q) {
    using V = c2_t<T>;
    const int M = f->M;
    const int W = f->g.r2c ? f->H : M;
    const long nl = (long)M * W;
    const c2_t<T> *tw = sizeof(T) == 8 ? (const V *)f->tw64 : (const V *)f->tw32;
    const double twopi_L = 2.0 * 3.14159265358979323846 / f->g.L;
    if (f->two.r1 > 0)
        return two_divergence<T>(f->two, (const V *const *)in, (V *)out, nl, W, f->tw64, G, Dn, twopi_L,
                                 p3mk_stream(q));
    LineMap x = {M, nl, nl, 0, nl};
    const int lt = launch_lines<T>(M, 3, nl);
    const size_t lds = (size_t)3 * lt * (M + 1) * sizeof(V);
    hipLaunchKernelGGL(k_divergence_x<T>, dim3((unsigned)((nl + lt - 1) / lt)), dim3(kThreads), lds,
                       p3mk_stream(q), (const V *)in[0], (const V *)in[1], (const V *)in[2],
                       (V *)out, x, W, f->rp, tw, G, Dn, twopi_L, lt);
    return p3mk_launch_check("divergence");
}

}  // namespace

// ---- batched passes over many systems ------------------------------------

namespace p3m {

int bfft_lines_per_tile(const BForm &f, int M, int kind) {
    const int lg = btwo_lg(make_two(M));
    if (lg >= 0)
        return 1 << lg;
    const int nbuf = (kind == kPassX && !f.ad) ? 3 : 2;
    return f.fp32 ? batch_tile_lines<float>(M, nbuf) : batch_tile_lines<double>(M, nbuf);
}

size_t bfft_lds_bytes(const BForm &f, int M, int kind) {
    const size_t v = f.fp32 ? sizeof(float2) : sizeof(double2);
    const TwoPlan two = make_two(M);
    if (two.r1 > 0)
        return (size_t)two_lds_points(two, 1 << btwo_lg(two)) * v;
    const int nbuf = (kind == kPassX && !f.ad) ? 3 : 2;
    return (size_t)nbuf * bfft_lines_per_tile(f, M, kind) * (M + 1) * v;
}

int bfft_pass(const BForm &f, const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int axis,
              int slot, int inv, p3mk_queue *q) {
    if (nblocks <= 0)
        return P3MK_OK;
    hipStream_t st = p3mk_stream(q);
    return f.fp32 ? btwo_pass<float>(sys, blk, nsys, nblocks, lds, axis, slot, inv, f.r2c, st)
                  : btwo_pass<double>(sys, blk, nsys, nblocks, lds, axis, slot, inv, f.r2c, st);
}

int bfft_r2c_z(const BForm &f, const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int in_slot,
               int out_slot, p3mk_queue *q) {
    if (nblocks <= 0)
        return P3MK_OK;
    hipStream_t st = p3mk_stream(q);
    return f.fp32 ? btwo_r2c<float>(sys, blk, nsys, nblocks, lds, in_slot, out_slot, st)
                  : btwo_r2c<double>(sys, blk, nsys, nblocks, lds, in_slot, out_slot, st);
}

int bfft_c2r_z(const BForm &f, const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int in_slot,
               int out_slot, p3mk_queue *q) {
    if (nblocks <= 0)
        return P3MK_OK;
    hipStream_t st = p3mk_stream(q);
    return f.fp32 ? btwo_c2r<float>(sys, blk, nsys, nblocks, lds, in_slot, out_slot, st)
                  : btwo_c2r<double>(sys, blk, nsys, nblocks, lds, in_slot, out_slot, st);
}

int bfft_convolve_x(const BForm &f, const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds,
                    int nout, int in_slot, int out_slot, p3mk_queue *q) {
    if (nblocks <= 0)
        return P3MK_OK;
    hipStream_t st = p3mk_stream(q);
    return f.fp32 ? btwo_convolve<float>(sys, blk, nsys, nblocks, lds, nout, in_slot, out_slot, f.r2c, st)
                  : btwo_convolve<double>(sys, blk, nsys, nblocks, lds, nout, in_slot, out_slot, f.r2c, st);
}

}  // namespace p3m

extern "C" int p3mk_fft_forward_zy_many(p3mk_fft *f, int k, void *const mesh[3], void *const spec[3],
                                        p3mk_queue *q) {
    return f->g.fp32 ? forward_zy<float>(f, k, mesh, spec, q) : forward_zy<double>(f, k, mesh, spec, q);
}

extern "C" int p3mk_fft_backward_yz_many(p3mk_fft *f, int k, void *const spec[3], void *const mesh[3],
                                         p3mk_queue *q) {
    return f->g.fp32 ? backward_yz<float>(f, k, spec, mesh, q) : backward_yz<double>(f, k, spec, mesh, q);
}

extern "C" int p3mk_fft_forward_zy(p3mk_fft *f, void *mesh, void *spec, p3mk_queue *q) {
    void *const m[3] = {mesh, nullptr, nullptr}, *const s[3] = {spec, nullptr, nullptr};
    return p3mk_fft_forward_zy_many(f, 1, m, s, q);
}

extern "C" int p3mk_fft_backward_yz(p3mk_fft *f, void *spec, void *mesh, p3mk_queue *q) {
    void *const m[3] = {mesh, nullptr, nullptr}, *const s[3] = {spec, nullptr, nullptr};
    return p3mk_fft_backward_yz_many(f, 1, s, m, q);
}

extern "C" int p3mk_convolve(p3mk_fft *f, int nout, const double *G, const double *Dn, void *spec,
                             void *const out[3], p3mk_queue *q) {
    if (nout != 1 && nout != 3)
        return p3mk_fail(P3MK_EINVAL, "convolve: nout must be 1 or 3", 0);
    return f->g.fp32 ? convolve<float>(f, nout, G, Dn, spec, out, q)
                     : convolve<double>(f, nout, G, Dn, spec, out, q);
}

extern "C" int p3mk_divergence(p3mk_fft *f, const double *G, const double *Dn, void *const in[3],
                               void *out, p3mk_queue *q) {
    return f->g.fp32 ? divergence<float>(f, G, Dn, in, out, q)
                     : divergence<double>(f, G, Dn, in, out, q);
}

template <typename T> static int fft3d(p3mk_fft *f, void *data, int sign, p3mk_queue *q) {
    using V = c2_t<T>;
    const int M = f->M;
    const int inv = sign > 0;
    const Three<V *> d = {{(V *)data, nullptr, nullptr}};
    LineMap z = {M, 1, 1, M, (long)M * M};
    LineMap y = {M, M, M, (long)M * M, (long)M * M};
    LineMap x = {M, (long)M * M, (long)M * M, 0, (long)M * M};
    P3MK_TRY(pass<T>(f, d, 1, z, inv, true, q));
    P3MK_TRY(pass<T>(f, d, 1, y, inv, false, q));
    return pass<T>(f, d, 1, x, inv, false, q);
}

extern "C" int p3mk_fft3d(p3mk_fft *f, void *data, int sign, p3mk_queue *q) {
    return f->g.fp32 ? fft3d<float>(f, data, sign, q) : fft3d<double>(f, data, sign, q);
}
