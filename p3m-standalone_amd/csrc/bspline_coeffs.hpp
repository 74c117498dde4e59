/* Generated by gen_bspline.py -- do not edit.
 * Cardinal B-spline charge-assignment weights of order P (cao):
 *   w[j]  = W_j(x)  = B_P(x - j + (P-1)/2),  x in [-1/2, 1/2]
 *   dw[j] = W'_j(x),  d2w[j] = W''_j(x)
 * each times u D_P, D_P = 2^(P-1) (P-1)!: integer-coefficient Horner
 * polynomials.  u is 1 in FP64 and in FP32 one over the largest power of two
 * up to D_P, so that the coefficients are exact in both and FP32 sums of mesh
 * values times weights stay in the range of the mesh values (the scaled
 * coefficients in FP64 too: k_collect 1045 -> 1253 us at order 7, fewer of
 * them are inline constants).  The caller multiplies the product of three by
 * norm^3 (stencil_norm) in FP64, once per particle: a rounded FP32 1/D_P in
 * every weight scales all of them by the same error. */
#pragma once

namespace p3m {

template <int P, typename T> struct Bspline;

template <typename T> struct Bspline<1, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 1;
  static constexpr double norm = 1.0 / (u * 1);
  __host__ __device__ static inline void w(T x, T *o) {
    (void)x;
    o[0] = (T(u * 1));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    (void)x;
    o[0] = T(0.0);
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    (void)x;
    o[0] = T(0.0);
  }
};

template <typename T> struct Bspline<2, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 2;
  static constexpr double norm = 1.0 / (u * 2);
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(u * 1) + x * (T(u * -2)));
    o[1] = (T(u * 1) + x * (T(u * 2)));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    (void)x;
    o[0] = (T(u * -2));
    o[1] = (T(u * 2));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    (void)x;
    o[0] = T(0.0);
    o[1] = T(0.0);
  }
};

template <typename T> struct Bspline<3, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 8;
  static constexpr double norm = 1.0 / (u * 8);
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(u * 1) + x * (T(u * -4) + x * (T(u * 4))));
    o[1] = (T(u * 6) + x * (T(u * 0) + x * (T(u * -8))));
    o[2] = (T(u * 1) + x * (T(u * 4) + x * (T(u * 4))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(u * -4) + x * (T(u * 8)));
    o[1] = (T(u * 0) + x * (T(u * -16)));
    o[2] = (T(u * 4) + x * (T(u * 8)));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    (void)x;
    o[0] = (T(u * 8));
    o[1] = (T(u * -16));
    o[2] = (T(u * 8));
  }
};

template <typename T> struct Bspline<4, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 32;
  static constexpr double norm = 1.0 / (u * 48);
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(u * 1) + x * (T(u * -6) + x * (T(u * 12) + x * (T(u * -8)))));
    o[1] = (T(u * 23) + x * (T(u * -30) + x * (T(u * -12) + x * (T(u * 24)))));
    o[2] = (T(u * 23) + x * (T(u * 30) + x * (T(u * -12) + x * (T(u * -24)))));
    o[3] = (T(u * 1) + x * (T(u * 6) + x * (T(u * 12) + x * (T(u * 8)))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(u * -6) + x * (T(u * 24) + x * (T(u * -24))));
    o[1] = (T(u * -30) + x * (T(u * -24) + x * (T(u * 72))));
    o[2] = (T(u * 30) + x * (T(u * -24) + x * (T(u * -72))));
    o[3] = (T(u * 6) + x * (T(u * 24) + x * (T(u * 24))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(u * 24) + x * (T(u * -48)));
    o[1] = (T(u * -24) + x * (T(u * 144)));
    o[2] = (T(u * -24) + x * (T(u * -144)));
    o[3] = (T(u * 24) + x * (T(u * 48)));
  }
};

template <typename T> struct Bspline<5, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 256;
  static constexpr double norm = 1.0 / (u * 384);
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(u * 1) + x * (T(u * -8) + x * (T(u * 24) + x * (T(u * -32) + x * (T(u * 16))))));
    o[1] = (T(u * 76) + x * (T(u * -176) + x * (T(u * 96) + x * (T(u * 64) + x * (T(u * -64))))));
    o[2] = (T(u * 230) + x * (T(u * 0) + x * (T(u * -240) + x * (T(u * 0) + x * (T(u * 96))))));
    o[3] = (T(u * 76) + x * (T(u * 176) + x * (T(u * 96) + x * (T(u * -64) + x * (T(u * -64))))));
    o[4] = (T(u * 1) + x * (T(u * 8) + x * (T(u * 24) + x * (T(u * 32) + x * (T(u * 16))))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(u * -8) + x * (T(u * 48) + x * (T(u * -96) + x * (T(u * 64)))));
    o[1] = (T(u * -176) + x * (T(u * 192) + x * (T(u * 192) + x * (T(u * -256)))));
    o[2] = (T(u * 0) + x * (T(u * -480) + x * (T(u * 0) + x * (T(u * 384)))));
    o[3] = (T(u * 176) + x * (T(u * 192) + x * (T(u * -192) + x * (T(u * -256)))));
    o[4] = (T(u * 8) + x * (T(u * 48) + x * (T(u * 96) + x * (T(u * 64)))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(u * 48) + x * (T(u * -192) + x * (T(u * 192))));
    o[1] = (T(u * 192) + x * (T(u * 384) + x * (T(u * -768))));
    o[2] = (T(u * -480) + x * (T(u * 0) + x * (T(u * 1152))));
    o[3] = (T(u * 192) + x * (T(u * -384) + x * (T(u * -768))));
    o[4] = (T(u * 48) + x * (T(u * 192) + x * (T(u * 192))));
  }
};

template <typename T> struct Bspline<6, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 2048;
  static constexpr double norm = 1.0 / (u * 3840);
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(u * 1) + x * (T(u * -10) + x * (T(u * 40) + x * (T(u * -80) + x * (T(u * 80) + x * (T(u * -32)))))));
    o[1] = (T(u * 237) + x * (T(u * -750) + x * (T(u * 840) + x * (T(u * -240) + x * (T(u * -240) + x * (T(u * 160)))))));
    o[2] = (T(u * 1682) + x * (T(u * -1540) + x * (T(u * -880) + x * (T(u * 1120) + x * (T(u * 160) + x * (T(u * -320)))))));
    o[3] = (T(u * 1682) + x * (T(u * 1540) + x * (T(u * -880) + x * (T(u * -1120) + x * (T(u * 160) + x * (T(u * 320)))))));
    o[4] = (T(u * 237) + x * (T(u * 750) + x * (T(u * 840) + x * (T(u * 240) + x * (T(u * -240) + x * (T(u * -160)))))));
    o[5] = (T(u * 1) + x * (T(u * 10) + x * (T(u * 40) + x * (T(u * 80) + x * (T(u * 80) + x * (T(u * 32)))))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(u * -10) + x * (T(u * 80) + x * (T(u * -240) + x * (T(u * 320) + x * (T(u * -160))))));
    o[1] = (T(u * -750) + x * (T(u * 1680) + x * (T(u * -720) + x * (T(u * -960) + x * (T(u * 800))))));
    o[2] = (T(u * -1540) + x * (T(u * -1760) + x * (T(u * 3360) + x * (T(u * 640) + x * (T(u * -1600))))));
    o[3] = (T(u * 1540) + x * (T(u * -1760) + x * (T(u * -3360) + x * (T(u * 640) + x * (T(u * 1600))))));
    o[4] = (T(u * 750) + x * (T(u * 1680) + x * (T(u * 720) + x * (T(u * -960) + x * (T(u * -800))))));
    o[5] = (T(u * 10) + x * (T(u * 80) + x * (T(u * 240) + x * (T(u * 320) + x * (T(u * 160))))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(u * 80) + x * (T(u * -480) + x * (T(u * 960) + x * (T(u * -640)))));
    o[1] = (T(u * 1680) + x * (T(u * -1440) + x * (T(u * -2880) + x * (T(u * 3200)))));
    o[2] = (T(u * -1760) + x * (T(u * 6720) + x * (T(u * 1920) + x * (T(u * -6400)))));
    o[3] = (T(u * -1760) + x * (T(u * -6720) + x * (T(u * 1920) + x * (T(u * 6400)))));
    o[4] = (T(u * 1680) + x * (T(u * 1440) + x * (T(u * -2880) + x * (T(u * -3200)))));
    o[5] = (T(u * 80) + x * (T(u * 480) + x * (T(u * 960) + x * (T(u * 640)))));
  }
};

template <typename T> struct Bspline<7, T> {
  static constexpr double u = sizeof(T) == 8 ? 1.0 : 1.0 / 32768;
  static constexpr double norm = 1.0 / (u * 46080);
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(u * 1) + x * (T(u * -12) + x * (T(u * 60) + x * (T(u * -160) + x * (T(u * 240) + x * (T(u * -192) + x * (T(u * 64))))))));
    o[1] = (T(u * 722) + x * (T(u * -2832) + x * (T(u * 4440) + x * (T(u * -3200) + x * (T(u * 480) + x * (T(u * 768) + x * (T(u * -384))))))));
    o[2] = (T(u * 10543) + x * (T(u * -17340) + x * (T(u * 4740) + x * (T(u * 6880) + x * (T(u * -4080) + x * (T(u * -960) + x * (T(u * 960))))))));
    o[3] = (T(u * 23548) + x * (T(u * 0) + x * (T(u * -18480) + x * (T(u * 0) + x * (T(u * 6720) + x * (T(u * 0) + x * (T(u * -1280))))))));
    o[4] = (T(u * 10543) + x * (T(u * 17340) + x * (T(u * 4740) + x * (T(u * -6880) + x * (T(u * -4080) + x * (T(u * 960) + x * (T(u * 960))))))));
    o[5] = (T(u * 722) + x * (T(u * 2832) + x * (T(u * 4440) + x * (T(u * 3200) + x * (T(u * 480) + x * (T(u * -768) + x * (T(u * -384))))))));
    o[6] = (T(u * 1) + x * (T(u * 12) + x * (T(u * 60) + x * (T(u * 160) + x * (T(u * 240) + x * (T(u * 192) + x * (T(u * 64))))))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(u * -12) + x * (T(u * 120) + x * (T(u * -480) + x * (T(u * 960) + x * (T(u * -960) + x * (T(u * 384)))))));
    o[1] = (T(u * -2832) + x * (T(u * 8880) + x * (T(u * -9600) + x * (T(u * 1920) + x * (T(u * 3840) + x * (T(u * -2304)))))));
    o[2] = (T(u * -17340) + x * (T(u * 9480) + x * (T(u * 20640) + x * (T(u * -16320) + x * (T(u * -4800) + x * (T(u * 5760)))))));
    o[3] = (T(u * 0) + x * (T(u * -36960) + x * (T(u * 0) + x * (T(u * 26880) + x * (T(u * 0) + x * (T(u * -7680)))))));
    o[4] = (T(u * 17340) + x * (T(u * 9480) + x * (T(u * -20640) + x * (T(u * -16320) + x * (T(u * 4800) + x * (T(u * 5760)))))));
    o[5] = (T(u * 2832) + x * (T(u * 8880) + x * (T(u * 9600) + x * (T(u * 1920) + x * (T(u * -3840) + x * (T(u * -2304)))))));
    o[6] = (T(u * 12) + x * (T(u * 120) + x * (T(u * 480) + x * (T(u * 960) + x * (T(u * 960) + x * (T(u * 384)))))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(u * 120) + x * (T(u * -960) + x * (T(u * 2880) + x * (T(u * -3840) + x * (T(u * 1920))))));
    o[1] = (T(u * 8880) + x * (T(u * -19200) + x * (T(u * 5760) + x * (T(u * 15360) + x * (T(u * -11520))))));
    o[2] = (T(u * 9480) + x * (T(u * 41280) + x * (T(u * -48960) + x * (T(u * -19200) + x * (T(u * 28800))))));
    o[3] = (T(u * -36960) + x * (T(u * 0) + x * (T(u * 80640) + x * (T(u * 0) + x * (T(u * -38400))))));
    o[4] = (T(u * 9480) + x * (T(u * -41280) + x * (T(u * -48960) + x * (T(u * 19200) + x * (T(u * 28800))))));
    o[5] = (T(u * 8880) + x * (T(u * 19200) + x * (T(u * 5760) + x * (T(u * -15360) + x * (T(u * -11520))))));
    o[6] = (T(u * 120) + x * (T(u * 960) + x * (T(u * 2880) + x * (T(u * 3840) + x * (T(u * 1920))))));
  }
};

// the norm of a product of three weights
template <int P, typename T> constexpr double stencil_norm =
    Bspline<P, T>::norm * Bspline<P, T>::norm * Bspline<P, T>::norm;

}  // namespace p3m
