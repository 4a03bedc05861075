// One neighbour pair's radial functions, angular damping and real harmonics by a
// few lanes of a wavefront.
#pragma once
#include "tgx_internal.h"

namespace {

template <class T> __device__ __forceinline__ T w_exp(T x);
template <> __device__ __forceinline__ double w_exp<double>(double x) { return exp(x); }
template <> __device__ __forceinline__ float w_exp<float>(float x) { return __expf(x); }
template <class T> __device__ __forceinline__ T w_pow(T x, T y);
template <> __device__ __forceinline__ double w_pow<double>(double x, double y) { return pow(x, y); }
template <> __device__ __forceinline__ float w_pow<float>(float x, float y) { return powf(x, y); }
template <class T> __device__ __forceinline__ T w_sqrt(T x);
template <> __device__ __forceinline__ double w_sqrt<double>(double x) { return sqrt(x); }
template <> __device__ __forceinline__ float w_sqrt<float>(float x) { return sqrtf(x); }

// Sum over the LPP consecutive lanes that share a pair, by DPP on the VALU; the
// same on all of them.
template <int CTRL> __device__ __forceinline__ float dpp_of(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double dpp_of(double x) {
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true));
}
template <int LPP, class T> __device__ __forceinline__ T lanes_sum(T v) {
  static_assert(LPP == 4 || LPP == 8 || LPP == 16, "groups of 4, 8 or 16 lanes");
  v += dpp_of<0xB1>(v);                     // quad_perm [1, 0, 3, 2]
  v += dpp_of<0x4E>(v);                     // quad_perm [2, 3, 0, 1]
  if constexpr (LPP >= 8) v += dpp_of<0x141>(v);   // row_half_mirror: the other quad of the eight
  if constexpr (LPP >= 16) v += dpp_of<0x140>(v);  // row_mirror: the other eight of the row
  return v;
}

// Radial projections of one pair by LPP lanes: R[n] and, when GRAD, dR[n]/dr,
// complete on every lane, from the species' nodes xq[q] and basis Bt[q][NB]. Lane
// sub takes the nodes sub, sub + LPP, ...: a lane per pair left three quarters of
// the wavefront-per-site kernels' lanes idle (16 pairs a pass) through the
// Gaussians, the largest part of both.
template <class T, bool GRAD, int LPP, int NB>
__device__ __forceinline__ void radial_lanes(const SpeciesParams& sp, const T* xq, const T* Bt, int sub, T r,
                                             T (&R)[NB], T (&dR)[NB]) {
  const T inv_rc = (T)sp.inv_rc;
  const T x = r * inv_rc;
  const T sig = (T)sp.sig_r * ((T)1 + (T)sp.sig_r_sc * r) * inv_rc;
  const T dsig = (T)(sp.sig_r * sp.sig_r_sc) * inv_rc;
  const T inv_s2 = (T)1 / (sig * sig);
  const T d1 = inv_s2 * inv_rc, d2 = inv_s2 / sig * dsig, ex = -(T)0.5 * inv_s2;
#pragma unroll
  for (int n = 0; n < NB; ++n) { R[n] = 0; dR[n] = 0; }
  const int nb = sp.nb;
  for (int q = sub; q < sp.nq; q += LPP) {
    const T dx = xq[q] - x;
    const T g = w_exp<T>(dx * dx * ex);
    T dg = 0;
    if (GRAD) dg = g * (dx * d1 + dx * dx * d2);
    const T* b = Bt + q * NB;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      if (n < nb) {
        R[n] += b[n] * g;
        if (GRAD) dR[n] += b[n] * dg;
      }
    }
  }
  const T a = (T)sp.amp_a;
  const T Pp = (T)1 + (T)2 * x * x * x - (T)3 * x * x;
  const T dPp = ((T)6 * x * x - (T)6 * x) * inv_rc;
  T amp, damp;
  if (a == (T)0) {
    amp = (T)1 / sig;
    damp = -dsig / (sig * sig);
  } else if (Pp <= (T)1.0e-10) {
    amp = 0;
    damp = 0;
  } else {
    const T Pa = a == (T)1 ? Pp : w_pow<T>(Pp, a);  // x^1 = x and x^0 = 1 exactly
    amp = Pa / sig;
    damp = a * (a == (T)1 ? (T)1 : w_pow<T>(Pp, a - (T)1)) * dPp / sig - Pa * dsig / (sig * sig);
  }
  amp *= (T)sp.gs;
  damp *= (T)sp.gs;
#pragma unroll
  for (int n = 0; n < NB; ++n) {
    if (n < nb) {
      const T I = lanes_sum<LPP>(R[n]);
      R[n] = amp * I;
      if (GRAD) dR[n] = damp * I + amp * lanes_sum<LPP>(dR[n]);
    }
  }
}

// Angular damping A_l = exp(-l(l+1) kk): A_l = prod_{k <= l} e2^k with e2 =
// exp(-2 kk); -A_l'/A_l = l(l+1) dk.
template <class T> struct Damp {
  T e2, dk;
  __device__ void init(const SpeciesParams& sp, T r) {
    const T st = (T)sp.sig_t * ((T)1 + (T)sp.sig_t_sc * r);
    const T dst = (T)(sp.sig_t * sp.sig_t_sc);
    dk = st * st / (r * r * r) - st * dst / (r * r);
    const T e1 = w_exp<T>(-(st * st / ((T)2 * r * r)));
    e2 = e1 * e1;
  }
};

// The real harmonics at u (and the gradient of the solid harmonic when GRAD) of
// one pair by LPP lanes, to f(l, lm, A_l, Y, gx, gy, gz). Lane sub takes the orders
// m = sub, 2 LPP - 1 - sub, 2 LPP + sub, ...: for l_max = 8 at most 15 degrees for
// four lanes and 10 for eight, against 45 for a lane on its own, the lanes
// stepping through their degrees together. The order's cos and sin factors c + i s = (ux + i
// uy)^m, their gradient (m (c', s') of order m - 1) and A_m come from the powers
// up to m.
template <class T, bool GRAD, int LPP, class F>
__device__ __forceinline__ void ylm_lanes(int L, const T* ynorm, int sub, T ux, T uy, T uz, T e2, F&& f) {
  T c = (T)1, s = (T)0, cp = (T)0, sp = (T)0, pw0 = (T)1, A0 = (T)1;
  int k = 0;
  for (int t = 0; LPP * t <= L; ++t) {
    const int m = 2 * LPP * (t >> 1) + ((t & 1) ? 2 * LPP - 1 - sub : sub);
    for (; k < m && k < L; ++k) {
      cp = c;
      sp = s;
      c = cp * ux - sp * uy;
      s = cp * uy + sp * ux;
      pw0 *= e2;
      A0 *= pw0;
    }
    const T dm = (T)m;
    const T cx = dm * cp, cy = -dm * sp, sx = dm * sp, sy = dm * cp;
    T q = (T)1, qx = (T)0, qy = (T)0, qz = (T)0, p = (T)0, px = (T)0, py = (T)0, pz = (T)0;
    T Al = A0, pw = pw0;
    for (int i = 0; i <= L; ++i) {
      const int l = m + i;
      if (l > L) break;
      if (i == 1) {
        p = q; px = qx; py = qy; pz = qz;
        qz = (T)2 * dm + (T)1;
        q = qz * uz;
        qx = (T)0; qy = (T)0;
      } else if (i > 1) {
        const T inv = (T)1 / (T)i, a = ((T)2 * dm + (T)(2 * i - 1)) * inv,
                     b = ((T)2 * dm + (T)(i - 1)) * inv;
        const T nq = a * uz * q - b * p;
        if (GRAD) {
          const T nqx = a * uz * qx - b * ((T)2 * ux * p + px);
          const T nqy = a * uz * qy - b * ((T)2 * uy * p + py);
          const T nqz = a * (q + uz * qz) - b * ((T)2 * uz * p + pz);
          px = qx; py = qy; pz = qz;
          qx = nqx; qy = nqy; qz = nqz;
        }
        p = q;
        q = nq;
      }
      if (i > 0) {
        pw *= e2;
        Al *= pw;
      }
      const int base = l * l + l;
      const T N = ynorm[base + m];
      f(l, base + m, Al, N * q * c, N * (qx * c + q * cx), N * (qy * c + q * cy), N * qz * c);
      if (m > 0) f(l, base - m, Al, N * q * s, N * (qx * s + q * sx), N * (qy * s + q * sy), N * qz * s);
    }
  }
}

}  // namespace
