/* Generated by gen_bspline.py -- do not edit.
 * Cardinal B-spline charge-assignment weights of order P (cao):
 *   w[j]  = W_j(x)  = B_P(x - j + (P-1)/2),  x in [-1/2, 1/2]
 *   dw[j] = W'_j(x),  d2w[j] = W''_j(x)
 * each times D_P = 2^(P-1) (P-1)!: integer-coefficient Horner polynomials.
 * The caller multiplies the product of three by inv_den^3 (stencil_norm)
 * in FP64, once per particle: a rounded FP32 1/D_P in every weight scales
 * all of them by the same error. */
#pragma once

namespace p3m {

template <int P, typename T> struct Bspline;

template <typename T> struct Bspline<1, T> {
  static constexpr double inv_den = 1.0 / 1.0;
  __host__ __device__ static inline void w(T x, T *o) {
    (void)x;
    o[0] = (T(1.0));
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
  static constexpr double inv_den = 1.0 / 2.0;
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(1.0) + x * (T(-2.0)));
    o[1] = (T(1.0) + x * (T(2.0)));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    (void)x;
    o[0] = (T(-2.0));
    o[1] = (T(2.0));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    (void)x;
    o[0] = T(0.0);
    o[1] = T(0.0);
  }
};

template <typename T> struct Bspline<3, T> {
  static constexpr double inv_den = 1.0 / 8.0;
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(1.0) + x * (T(-4.0) + x * (T(4.0))));
    o[1] = (T(6.0) + x * (T(0.0) + x * (T(-8.0))));
    o[2] = (T(1.0) + x * (T(4.0) + x * (T(4.0))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(-4.0) + x * (T(8.0)));
    o[1] = (T(0.0) + x * (T(-16.0)));
    o[2] = (T(4.0) + x * (T(8.0)));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    (void)x;
    o[0] = (T(8.0));
    o[1] = (T(-16.0));
    o[2] = (T(8.0));
  }
};

template <typename T> struct Bspline<4, T> {
  static constexpr double inv_den = 1.0 / 48.0;
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(1.0) + x * (T(-6.0) + x * (T(12.0) + x * (T(-8.0)))));
    o[1] = (T(23.0) + x * (T(-30.0) + x * (T(-12.0) + x * (T(24.0)))));
    o[2] = (T(23.0) + x * (T(30.0) + x * (T(-12.0) + x * (T(-24.0)))));
    o[3] = (T(1.0) + x * (T(6.0) + x * (T(12.0) + x * (T(8.0)))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(-6.0) + x * (T(24.0) + x * (T(-24.0))));
    o[1] = (T(-30.0) + x * (T(-24.0) + x * (T(72.0))));
    o[2] = (T(30.0) + x * (T(-24.0) + x * (T(-72.0))));
    o[3] = (T(6.0) + x * (T(24.0) + x * (T(24.0))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(24.0) + x * (T(-48.0)));
    o[1] = (T(-24.0) + x * (T(144.0)));
    o[2] = (T(-24.0) + x * (T(-144.0)));
    o[3] = (T(24.0) + x * (T(48.0)));
  }
};

template <typename T> struct Bspline<5, T> {
  static constexpr double inv_den = 1.0 / 384.0;
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(1.0) + x * (T(-8.0) + x * (T(24.0) + x * (T(-32.0) + x * (T(16.0))))));
    o[1] = (T(76.0) + x * (T(-176.0) + x * (T(96.0) + x * (T(64.0) + x * (T(-64.0))))));
    o[2] = (T(230.0) + x * (T(0.0) + x * (T(-240.0) + x * (T(0.0) + x * (T(96.0))))));
    o[3] = (T(76.0) + x * (T(176.0) + x * (T(96.0) + x * (T(-64.0) + x * (T(-64.0))))));
    o[4] = (T(1.0) + x * (T(8.0) + x * (T(24.0) + x * (T(32.0) + x * (T(16.0))))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(-8.0) + x * (T(48.0) + x * (T(-96.0) + x * (T(64.0)))));
    o[1] = (T(-176.0) + x * (T(192.0) + x * (T(192.0) + x * (T(-256.0)))));
    o[2] = (T(0.0) + x * (T(-480.0) + x * (T(0.0) + x * (T(384.0)))));
    o[3] = (T(176.0) + x * (T(192.0) + x * (T(-192.0) + x * (T(-256.0)))));
    o[4] = (T(8.0) + x * (T(48.0) + x * (T(96.0) + x * (T(64.0)))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(48.0) + x * (T(-192.0) + x * (T(192.0))));
    o[1] = (T(192.0) + x * (T(384.0) + x * (T(-768.0))));
    o[2] = (T(-480.0) + x * (T(0.0) + x * (T(1152.0))));
    o[3] = (T(192.0) + x * (T(-384.0) + x * (T(-768.0))));
    o[4] = (T(48.0) + x * (T(192.0) + x * (T(192.0))));
  }
};

template <typename T> struct Bspline<6, T> {
  static constexpr double inv_den = 1.0 / 3840.0;
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(1.0) + x * (T(-10.0) + x * (T(40.0) + x * (T(-80.0) + x * (T(80.0) + x * (T(-32.0)))))));
    o[1] = (T(237.0) + x * (T(-750.0) + x * (T(840.0) + x * (T(-240.0) + x * (T(-240.0) + x * (T(160.0)))))));
    o[2] = (T(1682.0) + x * (T(-1540.0) + x * (T(-880.0) + x * (T(1120.0) + x * (T(160.0) + x * (T(-320.0)))))));
    o[3] = (T(1682.0) + x * (T(1540.0) + x * (T(-880.0) + x * (T(-1120.0) + x * (T(160.0) + x * (T(320.0)))))));
    o[4] = (T(237.0) + x * (T(750.0) + x * (T(840.0) + x * (T(240.0) + x * (T(-240.0) + x * (T(-160.0)))))));
    o[5] = (T(1.0) + x * (T(10.0) + x * (T(40.0) + x * (T(80.0) + x * (T(80.0) + x * (T(32.0)))))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(-10.0) + x * (T(80.0) + x * (T(-240.0) + x * (T(320.0) + x * (T(-160.0))))));
    o[1] = (T(-750.0) + x * (T(1680.0) + x * (T(-720.0) + x * (T(-960.0) + x * (T(800.0))))));
    o[2] = (T(-1540.0) + x * (T(-1760.0) + x * (T(3360.0) + x * (T(640.0) + x * (T(-1600.0))))));
    o[3] = (T(1540.0) + x * (T(-1760.0) + x * (T(-3360.0) + x * (T(640.0) + x * (T(1600.0))))));
    o[4] = (T(750.0) + x * (T(1680.0) + x * (T(720.0) + x * (T(-960.0) + x * (T(-800.0))))));
    o[5] = (T(10.0) + x * (T(80.0) + x * (T(240.0) + x * (T(320.0) + x * (T(160.0))))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(80.0) + x * (T(-480.0) + x * (T(960.0) + x * (T(-640.0)))));
    o[1] = (T(1680.0) + x * (T(-1440.0) + x * (T(-2880.0) + x * (T(3200.0)))));
    o[2] = (T(-1760.0) + x * (T(6720.0) + x * (T(1920.0) + x * (T(-6400.0)))));
    o[3] = (T(-1760.0) + x * (T(-6720.0) + x * (T(1920.0) + x * (T(6400.0)))));
    o[4] = (T(1680.0) + x * (T(1440.0) + x * (T(-2880.0) + x * (T(-3200.0)))));
    o[5] = (T(80.0) + x * (T(480.0) + x * (T(960.0) + x * (T(640.0)))));
  }
};

template <typename T> struct Bspline<7, T> {
  static constexpr double inv_den = 1.0 / 46080.0;
  __host__ __device__ static inline void w(T x, T *o) {
    o[0] = (T(1.0) + x * (T(-12.0) + x * (T(60.0) + x * (T(-160.0) + x * (T(240.0) + x * (T(-192.0) + x * (T(64.0))))))));
    o[1] = (T(722.0) + x * (T(-2832.0) + x * (T(4440.0) + x * (T(-3200.0) + x * (T(480.0) + x * (T(768.0) + x * (T(-384.0))))))));
    o[2] = (T(10543.0) + x * (T(-17340.0) + x * (T(4740.0) + x * (T(6880.0) + x * (T(-4080.0) + x * (T(-960.0) + x * (T(960.0))))))));
    o[3] = (T(23548.0) + x * (T(0.0) + x * (T(-18480.0) + x * (T(0.0) + x * (T(6720.0) + x * (T(0.0) + x * (T(-1280.0))))))));
    o[4] = (T(10543.0) + x * (T(17340.0) + x * (T(4740.0) + x * (T(-6880.0) + x * (T(-4080.0) + x * (T(960.0) + x * (T(960.0))))))));
    o[5] = (T(722.0) + x * (T(2832.0) + x * (T(4440.0) + x * (T(3200.0) + x * (T(480.0) + x * (T(-768.0) + x * (T(-384.0))))))));
    o[6] = (T(1.0) + x * (T(12.0) + x * (T(60.0) + x * (T(160.0) + x * (T(240.0) + x * (T(192.0) + x * (T(64.0))))))));
  }
  __host__ __device__ static inline void dw(T x, T *o) {
    o[0] = (T(-12.0) + x * (T(120.0) + x * (T(-480.0) + x * (T(960.0) + x * (T(-960.0) + x * (T(384.0)))))));
    o[1] = (T(-2832.0) + x * (T(8880.0) + x * (T(-9600.0) + x * (T(1920.0) + x * (T(3840.0) + x * (T(-2304.0)))))));
    o[2] = (T(-17340.0) + x * (T(9480.0) + x * (T(20640.0) + x * (T(-16320.0) + x * (T(-4800.0) + x * (T(5760.0)))))));
    o[3] = (T(0.0) + x * (T(-36960.0) + x * (T(0.0) + x * (T(26880.0) + x * (T(0.0) + x * (T(-7680.0)))))));
    o[4] = (T(17340.0) + x * (T(9480.0) + x * (T(-20640.0) + x * (T(-16320.0) + x * (T(4800.0) + x * (T(5760.0)))))));
    o[5] = (T(2832.0) + x * (T(8880.0) + x * (T(9600.0) + x * (T(1920.0) + x * (T(-3840.0) + x * (T(-2304.0)))))));
    o[6] = (T(12.0) + x * (T(120.0) + x * (T(480.0) + x * (T(960.0) + x * (T(960.0) + x * (T(384.0)))))));
  }
  __host__ __device__ static inline void d2w(T x, T *o) {
    o[0] = (T(120.0) + x * (T(-960.0) + x * (T(2880.0) + x * (T(-3840.0) + x * (T(1920.0))))));
    o[1] = (T(8880.0) + x * (T(-19200.0) + x * (T(5760.0) + x * (T(15360.0) + x * (T(-11520.0))))));
    o[2] = (T(9480.0) + x * (T(41280.0) + x * (T(-48960.0) + x * (T(-19200.0) + x * (T(28800.0))))));
    o[3] = (T(-36960.0) + x * (T(0.0) + x * (T(80640.0) + x * (T(0.0) + x * (T(-38400.0))))));
    o[4] = (T(9480.0) + x * (T(-41280.0) + x * (T(-48960.0) + x * (T(19200.0) + x * (T(28800.0))))));
    o[5] = (T(8880.0) + x * (T(19200.0) + x * (T(5760.0) + x * (T(-15360.0) + x * (T(-11520.0))))));
    o[6] = (T(120.0) + x * (T(960.0) + x * (T(2880.0) + x * (T(3840.0) + x * (T(1920.0))))));
  }
};

// 1/D_P^3, the norm of a product of three weights
template <int P> constexpr double stencil_norm =
    Bspline<P, double>::inv_den * Bspline<P, double>::inv_den * Bspline<P, double>::inv_den;

}  // namespace p3m
