// Kernels and launchers of the two-factor FFT passes (fft_two.hpp) for one
// element type; each of k_fft_two_f32.hip / _f64.hip (one mesh) and
// k_bfft_two_f32.hip / _f64.hip (a batch) instantiates its half.
#pragma once

#ifndef P3M_FFT_TWO_SINGLE
#include "batch_desc.hpp"
#endif
#include "fft_two.hpp"
#include "k_internal.hpp"

namespace p3m {
namespace fft {

// ---- one mesh (defined in k_fft_two_f32 / _f64) -----------------------------
template <typename T>
int two_pass(const TwoPlan &p, Three<c2_t<T> *> data, int k, const LineMap &m, const double2 *tw, int inv,
             bool contig, hipStream_t st);
template <typename T>
int two_r2c(const TwoPlan &p, Three<const T *> in, Three<c2_t<T> *> out, int k, long nlines, const double2 *tw,
            hipStream_t st);
template <typename T>
int two_c2r(const TwoPlan &p, Three<const c2_t<T> *> in, Three<T *> out, int k, long nlines, const double2 *tw,
            hipStream_t st);
template <typename T>
int two_convolve(const TwoPlan &p, const c2_t<T> *in, c2_t<T> *const out[3], int nout, long nl, int W,
                 const double2 *tw, const double *G, const double *Dn, double twopi_L, hipStream_t st);
template <typename T>
int two_divergence(const TwoPlan &p, const c2_t<T> *const in[3], c2_t<T> *out, long nl, int W,
                   const double2 *tw, const double *G, const double *Dn, double twopi_L, hipStream_t st);

#ifndef P3M_FFT_TWO_SINGLE
// ---- a batch (defined in k_bfft_two_f32 / _f64) -------------------------------
template <typename T>
int btwo_pass(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int axis, int slot, int inv,
              int r2c, hipStream_t st);
template <typename T>
int btwo_r2c(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int in_slot, int out_slot,
             hipStream_t st);
template <typename T>
int btwo_c2r(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int in_slot, int out_slot,
             hipStream_t st);
template <typename T>
int btwo_convolve(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int nout, int in_slot,
                  int out_slot, int r2c, hipStream_t st);
#endif

// log2 of the lines per workgroup of a batched pass: as many as kThreads
// threads cover (lines x r2) within kBatchTilePoints points; -1 for a mesh
// without a two-factor split (batch_tile_lines then)
__host__ __device__ inline int btwo_lg(const TwoPlan &p) {
    if (p.r1 == 0)
        return -1;
    int lg = 0;
    while ((2 << lg) * p.r2 <= kThreads && (2 << lg) * p.r1 * p.r2 <= kBatchTilePoints)
        lg++;
    return lg;
}

}  // namespace fft
}  // namespace p3m

#ifdef P3M_FFT_TWO_SINGLE

namespace p3m {
namespace fft {
namespace {

template <typename T> size_t two_lds(const TwoPlan &p, int lg) {
    return sizeof(c2_t<T>) * (size_t)two_lds_points(p, 1 << lg);
}

// Lines per workgroup over one mesh: 16 (a strided row of 128 bytes in FP32,
// 256 in FP64), halved down to 4 while the launch would have fewer
// workgroups than the GPU has CUs, or while its LDS is above kLdsBudget, what
// a kernel gets without an attribute of its own (FP64 at 256 points: 69,632
// bytes with 16 lines).
template <typename T> int two_lg(const TwoPlan &p, long nlines) {
    int lg = 4;
    while (lg > 2 && (((nlines + (1 << lg) - 1) >> lg) < 256 || two_lds<T>(p, lg) > kLdsBudget))
        lg--;
    return lg;
}
inline unsigned two_blocks(long nlines, int lg) { return (unsigned)((nlines + (1 << lg) - 1) >> lg); }
inline unsigned two_block(const TwoPlan &p, int lg) { return (unsigned)((((p.r2 << lg) + 63) / 64) * 64); }

template <typename T, bool CONTIG>
__global__ void __launch_bounds__(kThreads)
k_two_pass(Three<c2_t<T> *> data, LineMap m, TwoPlan p, const double2 *__restrict__ tw, int inv, int lg) {
    extern __shared__ __align__(16) unsigned char smem[];
    two_pass_tile<T, CONTIG>(data.p[blockIdx.y], m, p, tw, inv, lg, (long)blockIdx.x << lg, smem);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_two_r2c(Three<const T *> in, Three<c2_t<T> *> out, long nlines, TwoPlan p,
          const double2 *__restrict__ tw, int lg) {
    extern __shared__ __align__(16) unsigned char smem[];
    two_r2c_tile<T>(in.p[blockIdx.y], out.p[blockIdx.y], nlines, p, tw, lg, (long)blockIdx.x << lg, smem);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_two_c2r(Three<const c2_t<T> *> in, Three<T *> out, long nlines, TwoPlan p,
          const double2 *__restrict__ tw, int lg) {
    extern __shared__ __align__(16) unsigned char smem[];
    two_c2r_tile<T>(in.p[blockIdx.y], out.p[blockIdx.y], nlines, p, tw, lg, (long)blockIdx.x << lg, smem);
}

template <int NOUT, typename T>
__global__ void __launch_bounds__(kThreads)
k_two_convolve(const c2_t<T> *in, c2_t<T> *out0, c2_t<T> *out1, c2_t<T> *out2, long nl, int W, TwoPlan p,
               const double2 *__restrict__ tw, const double *__restrict__ G, const double *__restrict__ Dn,
               double twopi_L, int lg) {
    extern __shared__ __align__(16) unsigned char smem[];
    two_convolve_tile<NOUT, T>(in, out0, out1, out2, nl, W, p, tw, G, Dn, twopi_L, lg, (long)blockIdx.x << lg,
                               smem);
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_two_divergence(const c2_t<T> *in0, const c2_t<T> *in1, const c2_t<T> *in2, c2_t<T> *out, long nl, int W,
                 TwoPlan p, const double2 *__restrict__ tw, const double *__restrict__ G,
                 const double *__restrict__ Dn, double twopi_L, int lg) {
    extern __shared__ __align__(16) unsigned char smem[];
    two_divergence_tile<T>(in0, in1, in2, out, nl, W, p, tw, G, Dn, twopi_L, lg, (long)blockIdx.x << lg, smem);
}

}  // namespace

template <typename T>
int two_pass(const TwoPlan &p, Three<c2_t<T> *> data, int k, const LineMap &m, const double2 *tw, int inv,
             bool contig, hipStream_t st) {
    const int lg = two_lg<T>(p, k * m.nlines);
    const dim3 grid(two_blocks(m.nlines, lg), (unsigned)k), block(two_block(p, lg));
    if (contig)
        hipLaunchKernelGGL((k_two_pass<T, true>), grid, block, two_lds<T>(p, lg), st, data, m, p, tw, inv, lg);
    else
        hipLaunchKernelGGL((k_two_pass<T, false>), grid, block, two_lds<T>(p, lg), st, data, m, p, tw, inv, lg);
    return p3mk_launch_check("fft pass");
}

template <typename T>
int two_r2c(const TwoPlan &p, Three<const T *> in, Three<c2_t<T> *> out, int k, long nlines, const double2 *tw,
            hipStream_t st) {
    const int lg = two_lg<T>(p, k * nlines);
    hipLaunchKernelGGL(k_two_r2c<T>, dim3(two_blocks(nlines, lg), (unsigned)k), dim3(two_block(p, lg)), two_lds<T>(p, lg), st,
                       in, out, nlines, p, tw, lg);
    return p3mk_launch_check("fft r2c");
}

template <typename T>
int two_c2r(const TwoPlan &p, Three<const c2_t<T> *> in, Three<T *> out, int k, long nlines, const double2 *tw,
            hipStream_t st) {
    const int lg = two_lg<T>(p, k * nlines);
    hipLaunchKernelGGL(k_two_c2r<T>, dim3(two_blocks(nlines, lg), (unsigned)k), dim3(two_block(p, lg)), two_lds<T>(p, lg), st,
                       in, out, nlines, p, tw, lg);
    return p3mk_launch_check("fft c2r");
}

template <typename T>
int two_convolve(const TwoPlan &p, const c2_t<T> *in, c2_t<T> *const out[3], int nout, long nl, int W,
                 const double2 *tw, const double *G, const double *Dn, double twopi_L, hipStream_t st) {
    const int lg = two_lg<T>(p, nl);
    const dim3 grid(two_blocks(nl, lg)), block(two_block(p, lg));
    if (nout == 1)
        hipLaunchKernelGGL((k_two_convolve<1, T>), grid, block, two_lds<T>(p, lg), st, in, out[0], nullptr, nullptr,
                           nl, W, p, tw, G, Dn, twopi_L, lg);
    else
        hipLaunchKernelGGL((k_two_convolve<3, T>), grid, block, two_lds<T>(p, lg), st, in, out[0], out[1], out[2],
                           nl, W, p, tw, G, Dn, twopi_L, lg);
    return p3mk_launch_check("convolve");
}

template <typename T>
int two_divergence(const TwoPlan &p, const c2_t<T> *const in[3], c2_t<T> *out, long nl, int W,
                   const double2 *tw, const double *G, const double *Dn, double twopi_L, hipStream_t st) {
    const int lg = two_lg<T>(p, nl);
    hipLaunchKernelGGL(k_two_divergence<T>, dim3(two_blocks(nl, lg)), dim3(two_block(p, lg)), two_lds<T>(p, lg), st,
                       in[0], in[1], in[2], out, nl, W, p, tw, G, Dn, twopi_L, lg);
    return p3mk_launch_check("divergence");
}

#define P3M_INST(T)                                                                                        \
    template int two_pass<T>(const TwoPlan &, Three<c2_t<T> *>, int, const LineMap &, const double2 *, int, bool, \
                             hipStream_t);                                                                 \
    template int two_r2c<T>(const TwoPlan &, Three<const T *>, Three<c2_t<T> *>, int, long, const double2 *, \
                            hipStream_t);                                                                  \
    template int two_c2r<T>(const TwoPlan &, Three<const c2_t<T> *>, Three<T *>, int, long, const double2 *, \
                            hipStream_t);                                                                  \
    template int two_convolve<T>(const TwoPlan &, const c2_t<T> *, c2_t<T> *const[3], int, long, int,      \
                                 const double2 *, const double *, const double *, double, hipStream_t);    \
    template int two_divergence<T>(const TwoPlan &, const c2_t<T> *const[3], c2_t<T> *, long, int,         \
                                   const double2 *, const double *, const double *, double, hipStream_t);

}  // namespace fft
}  // namespace p3m
#endif

#ifdef P3M_FFT_TWO_BATCH

// Block b belongs to the system s with blk[s] <= b < blk[s + 1]; its tile
// starts at line (b - blk[s]) times the system's lines per tile.  Systems
// without a two-factor split take the per-radix passes of fft_tiles.hpp.
namespace p3m {
namespace fft {
namespace {

template <typename T, bool CONTIG>
__global__ void __launch_bounds__(kThreads)
k_btwo_pass(const BSys *__restrict__ sys, const long *__restrict__ blk, int nsys, int slot, int inv, int r2c) {
    extern __shared__ __align__(16) unsigned char smem[];
    using V = c2_t<T>;
    const int s = prefix_slot(blk, nsys, (long)blockIdx.x);
    const BSys &S = sys[s];
    const int M = S.M, W = r2c ? M / 2 + 1 : M;
    LineMap m;
    if (CONTIG)
        m = {M, 1, 1, M, (long)M * M};
    else
        m = {M, W, W, (long)M * W, (long)M * W};
    const long tile = (long)(blockIdx.x - blk[s]);
    const int lg = btwo_lg(S.two);
    if (lg >= 0) {
        two_pass_tile<T, CONTIG>((V *)S.buf[slot], m, S.two, S.tw64, inv, lg, tile << lg, smem);
    } else {
        const int lt = batch_tile_lines<T>(M, 2);
        fft_pass_tile<T>((V *)S.buf[slot], m, S.rp, (const V *)S.tw, inv, lt, CONTIG ? 1 : 0, tile * lt, smem);
    }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_btwo_r2c(const BSys *__restrict__ sys, const long *__restrict__ blk, int nsys, int in_slot, int out_slot) {
    extern __shared__ __align__(16) unsigned char smem[];
    using V = c2_t<T>;
    const int s = prefix_slot(blk, nsys, (long)blockIdx.x);
    const BSys &S = sys[s];
    const int M = S.M;
    const long tile = (long)(blockIdx.x - blk[s]);
    const int lg = btwo_lg(S.two);
    if (lg >= 0) {
        two_r2c_tile<T>((const T *)S.buf[in_slot], (V *)S.buf[out_slot], (long)M * M, S.two, S.tw64, lg,
                        tile << lg, smem);
    } else {
        const int lt = batch_tile_lines<T>(M, 2);
        fft_r2c_z_tile<T>((const T *)S.buf[in_slot], (V *)S.buf[out_slot], (long)M * M, M, S.rp,
                          (const V *)S.tw, lt, tile * lt, smem);
    }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
k_btwo_c2r(const BSys *__restrict__ sys, const long *__restrict__ blk, int nsys, int in_slot, int out_slot) {
    extern __shared__ __align__(16) unsigned char smem[];
    using V = c2_t<T>;
    const int s = prefix_slot(blk, nsys, (long)blockIdx.x);
    const BSys &S = sys[s];
    const int M = S.M;
    const long tile = (long)(blockIdx.x - blk[s]);
    const int lg = btwo_lg(S.two);
    if (lg >= 0) {
        two_c2r_tile<T>((const V *)S.buf[in_slot], (T *)S.buf[out_slot], (long)M * M, S.two, S.tw64, lg,
                        tile << lg, smem);
    } else {
        const int lt = batch_tile_lines<T>(M, 2);
        fft_c2r_z_tile<T>((const V *)S.buf[in_slot], (T *)S.buf[out_slot], (long)M * M, M, S.rp,
                          (const V *)S.tw, lt, tile * lt, smem);
    }
}

template <int NOUT, typename T>
__global__ void __launch_bounds__(kThreads)
k_btwo_convolve(const BSys *__restrict__ sys, const long *__restrict__ blk, int nsys, int in_slot, int out_slot,
                int r2c) {
    extern __shared__ __align__(16) unsigned char smem[];
    using V = c2_t<T>;
    const int s = prefix_slot(blk, nsys, (long)blockIdx.x);
    const BSys &S = sys[s];
    const int M = S.M, W = r2c ? M / 2 + 1 : M;
    const long nl = (long)M * W;
    V *o0 = (V *)S.buf[out_slot];
    V *o1 = NOUT == 3 ? (V *)S.buf[out_slot + 1] : nullptr;
    V *o2 = NOUT == 3 ? (V *)S.buf[out_slot + 2] : nullptr;
    const double twopi_L = 2.0 * 3.14159265358979323846 / S.L;
    const long tile = (long)(blockIdx.x - blk[s]);
    const int lg = btwo_lg(S.two);
    if (lg >= 0) {
        two_convolve_tile<NOUT, T>((const V *)S.buf[in_slot], o0, o1, o2, nl, W, S.two, S.tw64, S.G, S.Dn,
                                   twopi_L, lg, tile << lg, smem);
    } else {
        const LineMap m = {M, nl, nl, 0, nl};
        const int lt = batch_tile_lines<T>(M, NOUT == 3 ? 3 : 2);
        convolve_x_tile<T>((const V *)S.buf[in_slot], o0, o1, o2, m, W, S.rp, (const V *)S.tw, S.G, S.Dn, twopi_L,
                           NOUT, lt, tile * lt, smem);
    }
}

}  // namespace

template <typename T>
int btwo_pass(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int axis, int slot, int inv,
              int r2c, hipStream_t st) {
    if (axis == kPassZ)
        hipLaunchKernelGGL((k_btwo_pass<T, true>), dim3((unsigned)nblocks), dim3(kThreads), lds, st, sys, blk,
                           nsys, slot, inv, r2c);
    else
        hipLaunchKernelGGL((k_btwo_pass<T, false>), dim3((unsigned)nblocks), dim3(kThreads), lds, st, sys, blk,
                           nsys, slot, inv, r2c);
    return p3mk_launch_check("batched fft pass");
}

template <typename T>
int btwo_r2c(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int in_slot, int out_slot,
             hipStream_t st) {
    hipLaunchKernelGGL(k_btwo_r2c<T>, dim3((unsigned)nblocks), dim3(kThreads), lds, st, sys, blk, nsys, in_slot,
                       out_slot);
    return p3mk_launch_check("batched fft r2c");
}

template <typename T>
int btwo_c2r(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int in_slot, int out_slot,
             hipStream_t st) {
    hipLaunchKernelGGL(k_btwo_c2r<T>, dim3((unsigned)nblocks), dim3(kThreads), lds, st, sys, blk, nsys, in_slot,
                       out_slot);
    return p3mk_launch_check("batched fft c2r");
}

template <typename T>
int btwo_convolve(const BSys *sys, const long *blk, int nsys, long nblocks, size_t lds, int nout, int in_slot,
                  int out_slot, int r2c, hipStream_t st) {
    if (nout == 1)
        hipLaunchKernelGGL((k_btwo_convolve<1, T>), dim3((unsigned)nblocks), dim3(kThreads), lds, st, sys, blk,
                           nsys, in_slot, out_slot, r2c);
    else
        hipLaunchKernelGGL((k_btwo_convolve<3, T>), dim3((unsigned)nblocks), dim3(kThreads), lds, st, sys, blk,
                           nsys, in_slot, out_slot, r2c);
    return p3mk_launch_check("batched convolve");
}

#define P3M_INST(T)                                                                                       \
    template int btwo_pass<T>(const BSys *, const long *, int, long, size_t, int, int, int, int,          \
                              hipStream_t);                                                               \
    template int btwo_r2c<T>(const BSys *, const long *, int, long, size_t, int, int, hipStream_t);       \
    template int btwo_c2r<T>(const BSys *, const long *, int, long, size_t, int, int, hipStream_t);       \
    template int btwo_convolve<T>(const BSys *, const long *, int, long, size_t, int, int, int, int,      \
                                  hipStream_t);

}  // namespace fft
}  // namespace p3m
#endif
