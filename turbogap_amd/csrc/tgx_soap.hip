// SOAP descriptor kernels: radial (poly3/poly3gauss by fixed Gauss-Legendre
// projection) and real-spherical-harmonic expansion, power spectrum,
// normalisation, and the two force routes:
//   plain   — dq_i/dr_j written for every pair, (3, D, P) like soap_cart_der
//             (src/gap_interface.f90:312-317), then contracted by k_plain_force;
//   adjoint — dE/dq back-propagated to dE/dc_nlm per site and contracted with
//             dc_nlm/dr_j recomputed per pair; dq/dr is never stored.
// The conventions (basis, density, amplitude, angular damping, ordering,
// multiplicity sqrt(2), normalisation, self pair = -sum) are the ones the
// FP64 oracle states; soap_turbo's own source is not available to follow.
//
// One workgroup (256 threads, 4 wavefronts) per central site. The site's
// expansion coefficients c(n, lm) live in LDS; lanes of a wavefront split the
// quadrature nodes, the (l, m) harmonics and the (n, l) channel sums of a pair;
// the power spectrum and its derivative are split over threads by component.
#include "tgx_internal.h"
#include "tgx_soap_lanes.h"

int tgx_desc_wave(tgx_ctx* ctx, tgx_model_t* m, bool fp64, const int* d_sites, int n_rows, void* q_out, void* pn_out);
int tgx_adjoint_wave(tgx_ctx* ctx, tgx_model_t* m, bool fp64);
int tgx_desc_f32(tgx_ctx* ctx, tgx_model_t* m);
int tgx_adjoint_f32(tgx_ctx* ctx, tgx_model_t* m);

namespace {

constexpr int WG = 256;

template <class T> __device__ __forceinline__ T t_exp(T x);
template <> __device__ __forceinline__ double t_exp<double>(double x) { return exp(x); }
template <> __device__ __forceinline__ float t_exp<float>(float x) { return __expf(x); }
template <class T> __device__ __forceinline__ T t_sqrt(T x);
template <> __device__ __forceinline__ double t_sqrt<double>(double x) { return sqrt(x); }
template <> __device__ __forceinline__ float t_sqrt<float>(float x) { return sqrtf(x); }
template <class T> __device__ __forceinline__ T t_pow(T x, T y);
template <> __device__ __forceinline__ double t_pow<double>(double x, double y) { return pow(x, y); }
template <> __device__ __forceinline__ float t_pow<float>(float x, float y) { return powf(x, y); }

// Real spherical harmonic Y_lm(u) (orthonormal, Condon-Shortley phase) and the
// gradient of the homogeneous solid harmonic r^l Y_lm at the unit vector u.
// nrm is the tabulated constant sqrt((2l+1)/(4 pi) (l-|m|)!/(l+|m|)!)
// (-1)^|m| (2|m|-1)!! (times sqrt 2 for m != 0).
template <class T>
__device__ void ylm_one(int l, int m, T nrm, T ux, T uy, T uz, T& Y, T& gx, T& gy, T& gz) {
  const int am = m < 0 ? -m : m;
  // (x + i y)^am and its x, y derivatives
  T c = 1, cx = 0, cy = 0, s = 0, sx = 0, sy = 0;
  for (int k = 0; k < am; ++k) {
    T nc = c * ux - s * uy, ncx = cx * ux + c - sx * uy, ncy = cy * ux - sy * uy - s;
    T ns = c * uy + s * ux, nsx = cx * uy + sx * ux + s, nsy = cy * uy + c + sy * ux;
    c = nc; cx = ncx; cy = ncy; s = ns; sx = nsx; sy = nsy;
  }
  // Q_l^am(z, r^2) with Q_am^am = 1 (the constant is in nrm)
  T q = 1, qx = 0, qy = 0, qz = 0;        // Q_{l'}
  T p = 0, px = 0, py = 0, pz = 0;        // Q_{l'-1}
  if (l > am) {
    p = q; px = qx; py = qy; pz = qz;
    q = (T)(2 * am + 1) * uz; qx = 0; qy = 0; qz = (T)(2 * am + 1);
    for (int lp = am + 2; lp <= l; ++lp) {
      const T a = (T)(2 * lp - 1), b = (T)(lp + am - 1), inv = (T)1 / (T)(lp - am);
      // r^2 = 1 at the unit vector, d(r^2) = 2u
      T nq = (a * uz * q - b * p) * inv;
      T nqx = (a * uz * qx - b * ((T)2 * ux * p + px)) * inv;
      T nqy = (a * uz * qy - b * ((T)2 * uy * p + py)) * inv;
      T nqz = (a * (q + uz * qz) - b * ((T)2 * uz * p + pz)) * inv;
      p = q; px = qx; py = qy; pz = qz;
      q = nq; qx = nqx; qy = nqy; qz = nqz;
    }
  }
  const T N = nrm;
  if (m == 0) {
    Y = N * q; gx = N * qx; gy = N * qy; gz = N * qz;
  } else if (m > 0) {
    Y = N * q * c; gx = N * (qx * c + q * cx); gy = N * (qy * c + q * cy); gz = N * qz * c;
  } else {
    Y = N * q * s; gx = N * (qx * s + q * sx); gy = N * (qy * s + q * sy); gz = N * qz * s;
  }
}

__device__ __forceinline__ int lm_l(int lm) {
  int l = (int)sqrtf((float)lm + 0.5f);
  return l * l > lm ? l - 1 : l;
}

// Scratch of one pair in LDS.
template <class T> struct PairScratch {
  T* G;   // [MAX_Q]
  T* dG;  // [MAX_Q]
  T* R;   // [MAX_NB]
  T* dR;  // [MAX_NB]
  T* A;   // [L+1]
  T* dA;  // [L+1]
  T* Y;   // [NLM]
  T* gY;  // [3 NLM]  gradient of the solid harmonic
  static constexpr int size(int L, int NLM) { return 2 * TGX_MAX_Q + 2 * TGX_MAX_NB + 2 * (L + 1) + 4 * NLM; }
  __device__ void bind(T* base, int L, int NLM) {
    G = base; dG = G + TGX_MAX_Q; R = dG + TGX_MAX_Q; dR = R + TGX_MAX_NB; A = dR + TGX_MAX_NB; dA = A + (L + 1);
    Y = dA + (L + 1); gY = Y + NLM;
  }
};

// Gaussians at the quadrature nodes (threads t < nq of nthr) and the angular
// damping A_l (thread nthr - 1) of one pair.
template <class T>
__device__ __forceinline__ void pair_gauss(const SoapParams& P, int s, T r, int t, int nthr, PairScratch<T>& ps,
                                           bool need_grad) {
  const SpeciesParams& sp = P.sp[s];
  const T inv_rc = (T)sp.inv_rc;
  const T x = r * inv_rc;
  const T sig = (T)sp.sig_r * ((T)1 + (T)sp.sig_r_sc * r) * inv_rc;
  const T dsig = (T)(sp.sig_r * sp.sig_r_sc) * inv_rc;
  const T inv_s2 = (T)1 / (sig * sig);
  const double* xq = P.xq + s * TGX_MAX_Q;
  for (int q = t; q < sp.nq; q += nthr) {
    const T dx = (T)xq[q] - x;
    const T g = t_exp<T>(-(T)0.5 * dx * dx * inv_s2);
    ps.G[q] = g;
    if (need_grad) ps.dG[q] = g * (dx * inv_s2 * inv_rc + dx * dx * inv_s2 / sig * dsig);
  }
  if (t == nthr - 1) {
    // A_l = exp(-l(l+1) k), k = st^2/(2 r^2): one exponential, A_l = A_{l-1} e^(2l) with e = exp(-k)
    const T st = (T)sp.sig_t * ((T)1 + (T)sp.sig_t_sc * r);
    const T dst = (T)(sp.sig_t * sp.sig_t_sc);
    const T kk = st * st / ((T)2 * r * r);
    const T dk = st * st / (r * r * r) - st * dst / (r * r);  // -dk/dr
    const T e1 = t_exp<T>(-kk), e2 = e1 * e1;
    T Al = 1, pw = 1;
    for (int l = 0; l <= P.L; ++l) {
      if (l > 0) { pw *= e2; Al *= pw; }
      const T ll = (T)(l * (l + 1));
      ps.A[l] = Al;
      ps.dA[l] = Al * ll * dk;
    }
  }
}

// Step 1 of a pair, by `nthr` threads with local index t: Gaussians at the
// quadrature nodes, harmonics, angular damping.
template <class T>
__device__ void pair_step1(const SoapParams& P, int s, T r, T ux, T uy, T uz, int t, int nthr, PairScratch<T>& ps,
                           bool need_grad) {
  pair_gauss<T>(P, s, r, t, nthr, ps, true);
  for (int lm = t; lm < P.NLM; lm += nthr) {
    const int l = lm_l(lm), m = lm - l * l - l;
    T Y, gx, gy, gz;
    ylm_one<T>(l, m, (T)P.ynorm[lm], ux, uy, uz, Y, gx, gy, gz);
    ps.Y[lm] = Y;
    if (need_grad) { ps.gY[3 * lm] = gx; ps.gY[3 * lm + 1] = gy; ps.gY[3 * lm + 2] = gz; }
  }
}

// Step 2: radial functions of the pair's species block and their r-derivatives.
template <class T>
__device__ void pair_step2(const SoapParams& P, int s, T r, int t, int nthr, PairScratch<T>& ps) {
  const SpeciesParams& sp = P.sp[s];
  const T inv_rc = (T)sp.inv_rc;
  const T x = r * inv_rc;
  const T sig = (T)sp.sig_r * ((T)1 + (T)sp.sig_r_sc * r) * inv_rc;
  const T dsig = (T)(sp.sig_r * sp.sig_r_sc) * inv_rc;
  const T a = (T)sp.amp_a;
  const T Pp = (T)1 + (T)2 * x * x * x - (T)3 * x * x;
  const T dPp = ((T)6 * x * x - (T)6 * x) * inv_rc;
  T amp, damp;
  if (a == (T)0) {
    amp = (T)1 / sig;
    damp = -dsig / (sig * sig);
  } else if (Pp <= (T)1.0e-10) {
    amp = 0; damp = 0;
  } else {
    const T Pa = t_pow<T>(Pp, a);
    amp = Pa / sig;
    damp = a * t_pow<T>(Pp, a - (T)1) * dPp / sig - Pa * dsig / (sig * sig);
  }
  amp *= (T)sp.gs;
  damp *= (T)sp.gs;
  const double* B = P.B + (size_t)s * TGX_MAX_NB * TGX_MAX_Q;
  if (nthr == 64) {
    // 64 lanes = nb groups x (64/nb) node slices (nb <= 16 divides into 4-lane slices at least)
    const int parts = sp.nb <= 8 ? 8 : 4;
    const int n = t / parts, part = t - n * parts;
    T I = 0, dI = 0;
    if (n < sp.nb) {
      const double* Bn = B + n * TGX_MAX_Q;
      for (int q = part; q < sp.nq; q += parts) {
        const T b = (T)Bn[q];
        I += b * ps.G[q];
        dI += b * ps.dG[q];
      }
    }
    for (int o = 1; o < parts; o <<= 1) {
      I += __shfl_xor(I, o);
      dI += __shfl_xor(dI, o);
    }
    if (n < sp.nb && part == 0) {
      ps.R[n] = amp * I;
      ps.dR[n] = damp * I + amp * dI;
    }
    return;
  }
  for (int n = t; n < sp.nb; n += nthr) {
    T I = 0, dI = 0;
    const double* Bn = B + n * TGX_MAX_Q;
    for (int q = 0; q < sp.nq; ++q) {
      const T b = (T)Bn[q];
      I += b * ps.G[q];
      dI += b * ps.dG[q];
    }
    ps.R[n] = amp * I;
    ps.dR[n] = damp * I + amp * dI;
  }
}

struct SiteArgs {
  const int* site_atom;
  const int64_t* site_beg;
  const int* pr_spec;
  const double* pr_r;
  const double* pr_xyz;
  const int64_t* pr_gidx;
};

// Phase A: expansion coefficients c(n, lm) of one site into LDS.
template <class T>
__device__ void site_coefficients(const SoapParams& P, const SiteArgs& a, int64_t b0, int nn, T* c, T* wscr) {
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int NLM = P.NLM, L = P.L;
  for (int e = tid; e < P.N * NLM; e += WG) c[e] = 0;
  PairScratch<T> ps;
  ps.bind(wscr + w * PairScratch<T>::size(L, NLM), L, NLM);
  __syncthreads();
  // central atom (self pair, first of the site): its own species block, l = 0
  {
    const int s = a.pr_spec[b0];
    if (s >= 0)
      for (int n = tid; n < P.sp[s].nb; n += WG) c[(P.sp[s].off + n) * NLM] += (T)P.cen[s * TGX_MAX_NB + n];
  }
  __syncthreads();
  for (int g = 1; g < nn; g += 4) {
    const int k = g + w;
    int s = -1;
    T r = 0, ux = 0, uy = 0, uz = 0;
    if (k < nn) {
      s = a.pr_spec[b0 + k];
      r = (T)a.pr_r[b0 + k];
      if (s >= 0 && !(a.pr_r[b0 + k] < P.sp[s].rc)) s = -1;
      if (s >= 0) {
        const T inv = (T)1 / r;
        ux = (T)a.pr_xyz[3 * (b0 + k)] * inv;
        uy = (T)a.pr_xyz[3 * (b0 + k) + 1] * inv;
        uz = (T)a.pr_xyz[3 * (b0 + k) + 2] * inv;
      }
    }
    if (s >= 0) pair_step1<T>(P, s, r, ux, uy, uz, lane, 64, ps, false);
    __syncthreads();
    if (s >= 0) pair_step2<T>(P, s, r, lane, 64, ps);
    __syncthreads();
    // accumulate the (up to) four pairs of this group in pair order
    for (int ww = 0; ww < 4; ++ww) {
      const int kk = g + ww;
      if (kk >= nn) break;
      int ss = a.pr_spec[b0 + kk];
      if (ss < 0 || !(a.pr_r[b0 + kk] < P.sp[ss].rc)) continue;
      PairScratch<T> po;
      po.bind(wscr + ww * PairScratch<T>::size(L, NLM), L, NLM);
      const int nb = P.sp[ss].nb, off = P.sp[ss].off;
      for (int e = tid; e < nb * NLM; e += WG) {
        const int n = e / NLM, lm = e - n * NLM;
        c[(off + n) * NLM + lm] += po.R[n] * po.A[lm_l(lm)] * po.Y[lm];
      }
    }
    __syncthreads();
  }
}

// Phase B: power spectrum into X[0..D), |p| returned to every thread; X is
// normalised in place to q.
template <class T>
__device__ T power_spectrum(const SoapParams& P, const T* c, T* X, T* red) {
  const int tid = threadIdx.x;
  const int NLM = P.NLM;
  T acc = 0;
  for (int d = tid; d < P.D; d += WG) {
    const int code = P.dtab[d];
    const int n = code & 0xff, np = (code >> 8) & 0xff, l = code >> 16;
    const T* c1 = c + n * NLM + l * l;
    const T* c2 = c + np * NLM + l * l;
    T s = 0;
    for (int m = 0; m < 2 * l + 1; ++m) s += c1[m] * c2[m];
    if (n != np) s *= (T)M_SQRT2;
    X[d] = s;
    acc += s * s;
  }
  red[tid] = acc;
  __syncthreads();
  for (int o = WG / 2; o > 0; o >>= 1) {
    if (tid < o) red[tid] += red[tid + o];
    __syncthreads();
  }
  const T nrm = t_sqrt<T>(red[0]);
  __syncthreads();
  const T inv = nrm > (T)0 ? (T)1 / nrm : (T)0;
  for (int d = tid; d < P.D; d += WG) X[d] *= inv;
  __syncthreads();
  return nrm;
}

// H(n, lm) = sum_n' S(n, n', l) c(n', lm) with S = sqrt2 V(n,n',l) off the
// diagonal and 2 V(n,n,l) on it: the gradient of V . p with respect to c.
template <class T>
__device__ void contract_channel(const SoapParams& P, const T* V, const T* c, T* H) {
  const int NLM = P.NLM, N = P.N, L1 = P.L + 1;
  for (int e = threadIdx.x; e < N * NLM; e += WG) {
    const int n = e / NLM, lm = e - n * NLM, l = lm_l(lm);
    T h = 0;
    for (int np = 0; np < N; ++np) {
      const int a = n < np ? n : np, b = n < np ? np : n;
      const int pidx = a * N - a * (a - 1) / 2 + (b - a);
      const T v = V[pidx * L1 + l];
      h += (n == np ? (T)2 : (T)M_SQRT2) * v * c[np * NLM + lm];
    }
    H[e] = h;
  }
}

// Mode 0: descriptors only. Mode 1: descriptors and dq/dr (plain path, FP64).
template <class T, int MODE, int KMAX>
__global__ __launch_bounds__(WG) void k_soap_site(SoapParams P, SiteArgs a, int n_sites, T* __restrict__ q_out,
                                                  T* __restrict__ pnorm_out, double* __restrict__ der_out,
                                                  const int* __restrict__ site_list) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* sm = reinterpret_cast<T*>(smem_raw);
  if ((int)blockIdx.x >= n_sites) return;
  // with a site list (descriptors only), row blockIdx.x of the output holds site_list[blockIdx.x]
  const int site = site_list ? site_list[blockIdx.x] : (int)blockIdx.x;
  const int orow = blockIdx.x;
  const int tid = threadIdx.x;
  const int NLM = P.NLM, N = P.N, L = P.L, L1 = L + 1, D = P.D;
  T* c = sm;                                   // N*NLM
  T* X = c + N * NLM;                          // D (p then q)
  T* red = X + D;                              // WG
  T* H = red + WG;                             // N*NLM (mode 1)
  T* wscr = H + (MODE == 1 ? N * NLM : 0);     // 4 pair scratches / phase D scratch
  const int64_t b0 = a.site_beg[site];
  const int nn = (int)(a.site_beg[site + 1] - b0);
  site_coefficients<T>(P, a, b0, nn, c, wscr);
  const T nrm = power_spectrum<T>(P, c, X, red);
  T* qrow = q_out + (size_t)orow * P.Dpad;
  for (int d = tid; d < P.Dpad; d += WG) qrow[d] = d < D ? X[d] : (T)0;
  if (tid == 0) pnorm_out[orow] = nrm;
  if (MODE == 0) return;
  // ---- dq/dr for every pair of the site (MODE 1) ----
  contract_channel<T>(P, X, c, H);
  __syncthreads();
  PairScratch<T> ps;
  ps.bind(wscr, L, NLM);
  T* s_nl = wscr + PairScratch<T>::size(L, NLM);  // N*L1
  T* vg_nl = s_nl + N * L1;                       // 3*N*L1 (becomes v)
  T* E_nl = vg_nl + 3 * N * L1;                   // N*L1
  T* Dd_nl = E_nl + N * L1;                       // N*L1
  T* sH = Dd_nl + N * L1;                         // MAX_NB*L1
  T* vgH = sH + TGX_MAX_NB * L1;                  // 3*MAX_NB*L1
  T* qd = vgH + 3 * TGX_MAX_NB * L1;              // 3 + pad
  // component ownership: d = tid + WG*k, k < KMAX (KMAX*WG >= D)
  T self_acc[KMAX][3];
  T qreg[KMAX];
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    self_acc[k][0] = self_acc[k][1] = self_acc[k][2] = 0;
    const int d = tid + WG * k;
    qreg[k] = d < D ? X[d] : (T)0;
  }
  const T inv_n = nrm > (T)0 ? (T)1 / nrm : (T)0;
  for (int k = 1; k < nn; ++k) {
    const int64_t p = b0 + k;
    int s = a.pr_spec[p];
    const double rr = a.pr_r[p];
    if (s >= 0 && !(rr < P.sp[s].rc)) s = -1;
    double* out = der_out + (size_t)p * 3 * D;
    if (s < 0 || nrm == (T)0) {
      // a pair the descriptor does not see: q does not depend on it
      for (int e = tid; e < 3 * D; e += WG) out[e] = 0.0;
      continue;
    }
    const T r = (T)rr, inv_r = (T)1 / r;
    const T ux = (T)a.pr_xyz[3 * p] * inv_r, uy = (T)a.pr_xyz[3 * p + 1] * inv_r, uz = (T)a.pr_xyz[3 * p + 2] * inv_r;
    pair_step1<T>(P, s, r, ux, uy, uz, tid, WG, ps, true);
    __syncthreads();
    const int nb = P.sp[s].nb, off = P.sp[s].off;
    if (tid < 64) {
      pair_step2<T>(P, s, r, tid, 64, ps);
    } else {
      // channel sums over m: s(n,l) = sum_m Y c, vg(n,l) = sum_m gY c, and the
      // same against H for the pair's block
      const int tasks = N * L1 + nb * L1;
      for (int task = tid - 64; task < tasks; task += WG - 64) {
        const bool withH = task >= N * L1;
        const int tt = withH ? task - N * L1 : task;
        const int n = tt / L1, l = tt - n * L1;
        const T* src = withH ? H + (off + n) * NLM : c + n * NLM;
        T s0 = 0, g0 = 0, g1 = 0, g2 = 0;
        for (int lm = l * l; lm < (l + 1) * (l + 1); ++lm) {
          const T v = src[lm];
          s0 += ps.Y[lm] * v;
          g0 += ps.gY[3 * lm] * v;
          g1 += ps.gY[3 * lm + 1] * v;
          g2 += ps.gY[3 * lm + 2] * v;
        }
        if (withH) {
          sH[tt] = s0; vgH[3 * tt] = g0; vgH[3 * tt + 1] = g1; vgH[3 * tt + 2] = g2;
        } else {
          s_nl[tt] = s0; vg_nl[3 * tt] = g0; vg_nl[3 * tt + 1] = g1; vg_nl[3 * tt + 2] = g2;
        }
      }
    }
    __syncthreads();
    // E = R A, Dd = (R A)', v = (vg - l s u)/r; zero outside the block
    for (int e = tid; e < N * L1; e += WG) {
      const int n = e / L1, l = e - n * L1;
      const T sv = s_nl[e];
      const T lf = (T)l;
      vg_nl[3 * e] = (vg_nl[3 * e] - lf * sv * ux) * inv_r;
      vg_nl[3 * e + 1] = (vg_nl[3 * e + 1] - lf * sv * uy) * inv_r;
      vg_nl[3 * e + 2] = (vg_nl[3 * e + 2] - lf * sv * uz) * inv_r;
      const int nl = n - off;
      if (nl >= 0 && nl < nb) {
        E_nl[e] = ps.R[nl] * ps.A[l];
        Dd_nl[e] = ps.dR[nl] * ps.A[l] + ps.R[nl] * ps.dA[l];
      } else {
        E_nl[e] = 0;
        Dd_nl[e] = 0;
      }
    }
    // q . dp: sum over the block's channels (one wavefront, fixed order)
    if (tid < 64) {
      T a0 = 0, a1 = 0, a2 = 0;
      for (int tt = tid; tt < nb * L1; tt += 64) {
        const int n = tt / L1, l = tt - n * L1;
        const T E = ps.R[n] * ps.A[l];
        const T Dd = ps.dR[n] * ps.A[l] + ps.R[n] * ps.dA[l];
        const T sh = sH[tt], lf = (T)l;
        a0 += Dd * sh * ux + E * (vgH[3 * tt] - lf * sh * ux) * inv_r;
        a1 += Dd * sh * uy + E * (vgH[3 * tt + 1] - lf * sh * uy) * inv_r;
        a2 += Dd * sh * uz + E * (vgH[3 * tt + 2] - lf * sh * uz) * inv_r;
      }
      for (int o = 32; o > 0; o >>= 1) {
        a0 += __shfl_xor(a0, o);
        a1 += __shfl_xor(a1, o);
        a2 += __shfl_xor(a2, o);
      }
      if (tid == 0) { qd[0] = a0; qd[1] = a1; qd[2] = a2; }
    }
    __syncthreads();
    const T q0 = qd[0], q1 = qd[1], q2 = qd[2];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      const int d = tid + WG * k;
      if (d >= D) break;
      const int code = P.dtab[d];
      const int n = code & 0xff, np = (code >> 8) & 0xff, l = code >> 16;
      const int i1 = n * L1 + l, i2 = np * L1 + l;
      const T w = n == np ? (T)1 : (T)M_SQRT2;
      const T rad = Dd_nl[i1] * s_nl[i2] + Dd_nl[i2] * s_nl[i1];
      const T E1 = E_nl[i1], E2 = E_nl[i2];
      const T dp0 = w * (rad * ux + E1 * vg_nl[3 * i2] + E2 * vg_nl[3 * i1]);
      const T dp1 = w * (rad * uy + E1 * vg_nl[3 * i2 + 1] + E2 * vg_nl[3 * i1 + 1]);
      const T dp2 = w * (rad * uz + E1 * vg_nl[3 * i2 + 2] + E2 * vg_nl[3 * i1 + 2]);
      const T o0 = (dp0 - qreg[k] * q0) * inv_n;
      const T o1 = (dp1 - qreg[k] * q1) * inv_n;
      const T o2 = (dp2 - qreg[k] * q2) * inv_n;
      out[3 * d] = (double)o0;
      out[3 * d + 1] = (double)o1;
      out[3 * d + 2] = (double)o2;
      self_acc[k][0] -= o0;
      self_acc[k][1] -= o1;
      self_acc[k][2] -= o2;
    }
    __syncthreads();
  }
  double* out = der_out + (size_t)b0 * 3 * D;
#pragma unroll
  for (int k = 0; k < KMAX; ++k) {
    const int d = tid + WG * k;
    if (d >= D) break;
    out[3 * d] = (double)self_acc[k][0];
    out[3 * d + 1] = (double)self_acc[k][1];
    out[3 * d + 2] = (double)self_acc[k][2];
  }
}

// Workgroup barrier that orders LDS only: it waits for this wavefront's LDS
// operations, not for its global stores, so streamed output stays in flight
// across the barrier (no thread of a workgroup reads another's global output).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ void der_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Per-pair channel tables of the plain dq/dr kernel, one slot per wavefront:
//   s(n,l) = sum_m Y_lm c(n,lm)
//   v_k(n,l) = (sum_m dY_lm/du_k c(n,lm) - l s u_k) / r     (k = x, y, z)
//   E(n,l) = R_n A_l, Dd(n,l) = (R_n A_l)'   (zero outside the pair's block)
// and misc = { q.dp_x, q.dp_y, q.dp_z, u_x, u_y, u_z, valid }.
struct DerSlot {
  static __host__ __device__ int size(int NL, int L, int NLM) {
    return 6 * NL + 8 + PairScratch<double>::size(L, NLM);
  }
};

// One wavefront reduces pair p of the site to its channel tables in `slot`.
__device__ void der_pair_tables(const SoapParams& P, const SiteArgs& a, int64_t p, bool site_ok, const double* c,
                                const double* H, double* slot) {
  const int lane = threadIdx.x & 63;
  const int NLM = P.NLM, L = P.L, L1 = L + 1, NL = P.N * L1;
  double* s_t = slot;
  double* v_t = s_t + NL;
  double* E_t = v_t + 3 * NL;
  double* Dd_t = E_t + NL;
  double* misc = Dd_t + NL;
  int s = a.pr_spec[p];
  const double rr = a.pr_r[p];
  if (!site_ok || s < 0 || !(rr < P.sp[s].rc)) {
    if (lane == 0) misc[6] = 0.0;
    return;
  }
  PairScratch<double> ps;
  ps.bind(misc + 8, L, NLM);
  const double r = rr, inv_r = 1.0 / r;
  const double ux = a.pr_xyz[3 * p] * inv_r, uy = a.pr_xyz[3 * p + 1] * inv_r, uz = a.pr_xyz[3 * p + 2] * inv_r;
  pair_step1<double>(P, s, r, ux, uy, uz, lane, 64, ps, true);
  der_wave_sync();
  pair_step2<double>(P, s, r, lane, 64, ps);
  der_wave_sync();
  const int nb = P.sp[s].nb, off = P.sp[s].off;
  double a0 = 0.0, a1 = 0.0, a2 = 0.0;
  for (int t = lane; t < NL; t += 64) {
    const int n = t / L1, l = t - n * L1;
    const int nl = n - off;
    const bool inb = nl >= 0 && nl < nb;
    const double* cr = c + n * NLM;
    const double* hr = H + n * NLM;
    double s0 = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0;
    double h = 0.0, h0 = 0.0, h1 = 0.0, h2 = 0.0;
    for (int lm = l * l; lm < (l + 1) * (l + 1); ++lm) {
      const double Y = ps.Y[lm], gx = ps.gY[3 * lm], gy = ps.gY[3 * lm + 1], gz = ps.gY[3 * lm + 2];
      const double v = cr[lm];
      s0 += Y * v;
      g0 += gx * v;
      g1 += gy * v;
      g2 += gz * v;
      if (inb) {
        const double hv = hr[lm];
        h += Y * hv;
        h0 += gx * hv;
        h1 += gy * hv;
        h2 += gz * hv;
      }
    }
    const double lf = (double)l;
    s_t[t] = s0;
    v_t[t] = (g0 - lf * s0 * ux) * inv_r;
    v_t[NL + t] = (g1 - lf * s0 * uy) * inv_r;
    v_t[2 * NL + t] = (g2 - lf * s0 * uz) * inv_r;
    double E = 0.0, Dd = 0.0;
    if (inb) {
      E = ps.R[nl] * ps.A[l];
      Dd = ps.dR[nl] * ps.A[l] + ps.R[nl] * ps.dA[l];
      a0 += Dd * h * ux + E * (h0 - lf * h * ux) * inv_r;
      a1 += Dd * h * uy + E * (h1 - lf * h * uy) * inv_r;
      a2 += Dd * h * uz + E * (h2 - lf * h * uz) * inv_r;
    }
    E_t[t] = E;
    Dd_t[t] = Dd;
  }
  for (int o = 32; o > 0; o >>= 1) {
    a0 += __shfl_xor(a0, o);
    a1 += __shfl_xor(a1, o);
    a2 += __shfl_xor(a2, o);
  }
  if (lane == 0) {
    misc[0] = a0; misc[1] = a1; misc[2] = a2;
    misc[3] = ux; misc[4] = uy; misc[5] = uz;
    misc[6] = 1.0;
  }
}

// Plain-path dq/dr in FP64, (3, D) per pair like soap_cart_der
// (src/gap_interface.f90:312-317), the self pair holding -sum of the others
// (src/gap.f90:275-277). One workgroup per site. The site's coefficients c,
// its power spectrum and H = d(q . p)/dc stay in LDS; the pairs go four at a
// time: each wavefront reduces one pair to its channel tables, then the 256
// threads stream the four slabs. Thread t owns elements e = t + 256 j of a
// slab (e = 3 d + k, k the Cartesian component), so each store instruction
// writes 2 KB of consecutive doubles, and it keeps the self-pair sums of its
// elements in registers. J * 256 >= 3 D.
template <int J>
__global__ __launch_bounds__(WG, 2) void k_soap_der(SoapParams P, SiteArgs a, int n_sites, double* __restrict__ q_out,
                                                    double* __restrict__ pnorm_out, double* __restrict__ der_out) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  double* sm = reinterpret_cast<double*>(smem_raw);
  const int site = blockIdx.x;
  if (site >= n_sites) return;
  const int tid = threadIdx.x, w = tid >> 6;
  const int NLM = P.NLM, N = P.N, L1 = P.L + 1, D = P.D, D3 = 3 * D, NL = N * L1;
  double* c = sm;
  double* H = c + N * NLM;
  double* X = H + N * NLM;  // p, then q: kept for the whole site
  double* U = X + D;
  double* red = U;
  double* wscr = red + WG;
  const int64_t b0 = a.site_beg[site];
  const int nn = (int)(a.site_beg[site + 1] - b0);
  site_coefficients<double>(P, a, b0, nn, c, wscr);
  const double nrm = power_spectrum<double>(P, c, X, red);
  double* qrow = q_out + (size_t)site * P.Dpad;
  for (int d = tid; d < P.Dpad; d += WG) qrow[d] = d < D ? X[d] : 0.0;
  if (tid == 0) pnorm_out[site] = nrm;
  contract_channel<double>(P, X, c, H);
  // element codes: i1 = n L1 + l | i2 = n' L1 + l << 8 | k << 16 | (n == n') << 18 | d << 19
  int code[J];
  double self[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int e = tid + WG * j;
    code[j] = -1;
    self[j] = 0.0;
    if (e < D3) {
      const int d = e / 3, k = e - 3 * d;
      const int cd = P.dtab[d];
      const int n = cd & 0xff, np = (cd >> 8) & 0xff, l = cd >> 16;
      code[j] = (n * L1 + l) | ((np * L1 + l) << 8) | (k << 16) | ((n == np ? 1 : 0) << 18) | (d << 19);
    }
  }
  const double inv_n = nrm > 0.0 ? 1.0 / nrm : 0.0;
  const bool site_ok = nrm > 0.0;
  const int SL = DerSlot::size(NL, P.L, NLM);
  __syncthreads();  // red and the coefficient scratch are dead: the slots overlay them
  for (int g = 1; g < nn; g += 4) {
    if (g + w < nn) der_pair_tables(P, a, b0 + g + w, site_ok, c, H, U + w * SL);
    lds_barrier();
    const int cnt = min(4, nn - g);
    double* out = der_out + (size_t)(b0 + g) * D3 + tid;
    // element-major: an element's decoded indices are live only while its four pairs are written
#pragma unroll
    for (int j = 0; j < J; ++j) {
      int cj = code[j];
      if (cj < 0) continue;
      // opaque to the optimiser: the decoded fields are not hoisted out of the pair loop, where
      // they would stay live (16 elements' worth) across the table phase
      asm volatile("" : "+v"(cj));
      const int i1 = cj & 0xff, i2 = (cj >> 8) & 0xff, k = (cj >> 16) & 3;
      const double wgt = ((cj >> 18) & 1) ? 1.0 : M_SQRT2;
      const double qd = X[cj >> 19];
      for (int ww = 0; ww < cnt; ++ww) {
        const double* s_t = U + ww * SL;
        const double* v_t = s_t + NL;
        const double* E_t = v_t + 3 * NL;
        const double* Dd_t = E_t + NL;
        const double* misc = Dd_t + NL;
        double o = 0.0;  // zero for a pair the descriptor does not see: q does not depend on it
        if (misc[6] != 0.0) {
          const double rad = Dd_t[i1] * s_t[i2] + Dd_t[i2] * s_t[i1];
          const double dp = wgt * (rad * misc[3 + k] + E_t[i1] * v_t[k * NL + i2] + E_t[i2] * v_t[k * NL + i1]);
          o = (dp - qd * misc[k]) * inv_n;
        }
        out[(size_t)ww * D3 + WG * j] = o;
        self[j] -= o;
      }
    }
    lds_barrier();
  }
  double* out = der_out + (size_t)b0 * D3;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (code[j] >= 0) out[tid + WG * j] = self[j];
}

// ---- The same dq/dr, and FP64 descriptors and adjoint forces, for l_max = 8 and at
// most two species of at most eight radial functions each (16 stacked rows). LL
// names the 8 in sizes and indexes; the degree sets of der_lm, the calls of
// der_channel and the (l, m) tiles of l_channel are laid out for it alone.

template <int LL> struct DerL {
  static constexpr int L1 = LL + 1, NLM = L1 * L1, NL = 16 * L1, D = 16 * 17 / 2 * L1;
  static constexpr int CHK = 32;             // pairs prepared together, eight lanes each
  static constexpr int TABS = 2 * TGX_MAX_Q * 9;  // the species' nodes and basis [q][8]
  static constexpr int ST = 33;              // one pair's record, see der_prepare
  static constexpr int CP = 17;              // row of c or H at one (l, m), padded
  static constexpr int SL = 6 * NL;          // one pair's channel tables
  static constexpr int SPW = sizeof(SpeciesParams) / 8;     // doubles of a species' parameters
  static_assert(sizeof(SpeciesParams) % 8 == 0, "copied to LDS in doubles");
  static constexpr int HEAD = NLM + CHK * ST + 8 + 2 * SPW;
  static constexpr int HEADP = HEAD + (HEAD & 1);
  static constexpr int U1 = TABS + CHK * NLM;               // expansion: tables and W
  static constexpr int U2 = NLM * CP + 1 + D;               // c, then H, and the spectrum
  static constexpr int HG = 16;                             // pairs whose harmonics are kept
  static constexpr int U3 = 4 * SL + HG * 4 * NLM + 48;     // four pairs' tables, harmonics, q . dp
  static constexpr int U = U1 > U2 ? (U1 > U3 ? U1 : U3) : (U2 > U3 ? U2 : U3);
  static constexpr size_t LDS = sizeof(double) * (HEADP + U);
  static constexpr size_t LDS_DESC = sizeof(double) * (HEADP + (U1 > U2 ? U1 : U2));
  static constexpr int U4 = HG * 4 * NLM + 4 * HG * 3;  // adjoint: harmonics, partials
  static constexpr size_t LDS_ADJ = sizeof(double) * (HEADP + (U1 > U2 ? (U1 > U4 ? U1 : U4) : (U2 > U4 ? U2 : U4)));
};

typedef double f64x4_t __attribute__((ext_vector_type(4)));

// The species' nodes and basis (at most two species, eight functions) on their way
// from memory to LDS, xq[s][q] and Bt[s][q][8]: loaded in registers at the kernel's
// start, before anything that waits on the site's own offsets.
struct DerTabs {
  double x, b[4];
  __device__ __forceinline__ void load(const double* xq, const double* B, int S) {
    const int t = threadIdx.x;
    x = t < S * TGX_MAX_Q ? xq[t] : 0.0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = t + WG * u, sn = i / TGX_MAX_Q, q = i % TGX_MAX_Q;
      b[u] = sn < 8 * S ? B[((size_t)(sn >> 3) * TGX_MAX_NB + (sn & 7)) * TGX_MAX_Q + q] : 0.0;
    }
  }
  __device__ __forceinline__ void store(double* tabs) const {
    const int t = threadIdx.x;
    if (t < 2 * TGX_MAX_Q) tabs[t] = x;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = t + WG * u, sn = i / TGX_MAX_Q, q = i % TGX_MAX_Q;
      tabs[2 * TGX_MAX_Q + ((sn >> 3) * TGX_MAX_Q + q) * 8 + (sn & 7)] = b[u];
    }
  }
};

// Records of the site's pairs k0 + 1 .. k0 + cnt, eight lanes each (cnt <= CHK), from
// the species' parameters spl and tables tabs in LDS:
//   R[8] | dR[8] | A[9] | -A'/(A l (l + 1)) | 1/r | u | seen (1 or 0) | first row, row count
// (R, dR rows of the pair's own species block) and, with W, A_l Y_lm of every pair.
template <int LL, bool W>
__device__ __forceinline__ void der_prepare(const SpeciesParams* spl, const int* pr_spec, const double* pr_r,
                                            const double* pr_xyz, int64_t b0, int k0, int cnt, const double* ynorm,
                                            double* rec, const double* tabs, double* w) {
  using G = DerL<LL>;
  const double* xq = tabs;
  const double* Bt = tabs + 2 * TGX_MAX_Q;
  const int j = threadIdx.x >> 3, sub = threadIdx.x & 7;
  int s = -1;
  double r = 1.0, ux = 0.0, uy = 0.0, uz = 0.0;
  if (j < cnt) {
    const int64_t p = b0 + k0 + 1 + j;
    s = pr_spec[p];
    r = pr_r[p];
    const double inv = 1.0 / r;
    ux = pr_xyz[3 * p] * inv;
    uy = pr_xyz[3 * p + 1] * inv;
    uz = pr_xyz[3 * p + 2] * inv;
  }
  lds_barrier();
  if (j >= cnt) return;
  const SpeciesParams sp = spl[max(s, 0)];
  if (s >= 0 && !(r < sp.rc)) s = -1;
  double* st = rec + j * G::ST;
  if (s >= 0) {
    double R[8], dR[8];
    radial_lanes<double, true, 8, 8>(sp, xq + s * TGX_MAX_Q, Bt + s * TGX_MAX_Q * 8, sub, r, R, dR);
    Damp<double> dmp;
    dmp.init(sp, r);
    if (sub == 0) {
#pragma unroll
      for (int n = 0; n < 8; ++n) st[n] = R[n];
#pragma unroll
      for (int n = 0; n < 8; ++n) st[8 + n] = dR[n];
      double Al = 1.0, pw = 1.0;
      st[16] = 1.0;
#pragma unroll
      for (int l = 1; l <= LL; ++l) {
        pw *= dmp.e2;
        Al *= pw;
        st[16 + l] = Al;
      }
      st[25] = dmp.dk;
      st[26] = 1.0 / r;
      st[27] = ux;
      st[28] = uy;
      st[29] = uz;
      st[30] = 1.0;
      st[31] = (double)sp.off;
      st[32] = (double)sp.nb;
    }
    if (W)
      ylm_lanes<double, false, 8>(LL, ynorm, sub, ux, uy, uz, dmp.e2,
                                  [&](int, int lm, double Al, double Y, double, double, double) {
                                    w[j * G::NLM + lm] = Al * Y;
                                  });
  } else {
    for (int i = sub; i < G::ST; i += 8) st[i] = 0.0;
    if (W)
      for (int lm = sub; lm < G::NLM; lm += 8) w[j * G::NLM + lm] = 0.0;
  }
}

// The records of a later chunk of a site with more than CHK pairs, tables included.
// Not inlined: its registers would push the pair loop's, live across it, into
// scratch for every site (9.41 -> 9.64 ms at 65,536 atoms, 50 -> 54 us at 216).
template <int LL>
__device__ __attribute__((noinline)) void der_prepare_again(const SpeciesParams* spl, const double* xq, const double* B,
                                                            int S, const int* pr_spec, const double* pr_r,
                                                            const double* pr_xyz, int64_t b0, int k0, int cnt,
                                                            double* rec, double* tabs) {
  lds_barrier();
  DerTabs t;
  t.load(xq, B, S);
  t.store(tabs);
  der_prepare<LL, false>(spl, pr_spec, pr_r, pr_xyz, b0, k0, cnt, nullptr, rec, tabs, nullptr);
}

// The wavefront's degrees of the channel tables, 20 or 21 (l, m) in all: {8, 0, 1},
// {7, 2}, {6, 3} or {5, 4}; the i-th (l, m) of wavefront w.
template <int LL> __device__ __forceinline__ int der_lm(int w, int i) {
  static_assert(LL == 8, "degree sets are laid out for l_max = 8");
  const int l = LL - w, k = 2 * l + 1;
  return i < k ? l * l + i : (w == 0 ? i - k : (w + 1) * (w + 1) + min(i - k, 2 * w + 2));
}

struct DerLane {
  double R, dR, dk, inv_r, ux, uy, uz;
  bool ok;
};

// Entries (n, l) of one pair's channel tables, six doubles (s, E, v_x, v_y, v_z, Dd)
// at 6 (n L1 + l), read back as three 16-byte loads:
//   s(n,l) = sum_m Y c(n,lm),  v_k(n,l) = (sum_m dY_k c(n,lm) - l s u_k) / r,
//   E(n,l) = R_n A_l,  Dd(n,l) = dR_n A_l + R_n A_l'  (rows of the pair's block),
// and the row's part of q . dp_k, Dd h u_k + E (h_k - l h u_k) / r with
// h = sum_m Y H(n,lm), h_k = sum_m dY_k H(n,lm). c and H of the row's (l, m) come in
// registers I0, I0 + 1, ...; y holds the pair's (Y, gx, gy, gz).
template <int LL, int l, int I0>
__device__ __forceinline__ void der_channel(const DerLane& p, const double* y, const double* A, const double (&c)[21],
                                            const double (&H)[21], double* slot, double& qx, double& qy, double& qz) {
  double s0 = 0.0, gx = 0.0, gy = 0.0, gz = 0.0, h0 = 0.0, hx = 0.0, hy = 0.0, hz = 0.0;
  if (p.ok) {
#pragma unroll
    for (int i = 0; i < 2 * l + 1; ++i) {
      const double2* y4 = reinterpret_cast<const double2*>(y + 4 * (l * l + i));
      const double2 ya = y4[0], yb = y4[1];
      const double cv = c[I0 + i], hv = H[I0 + i];
      s0 += ya.x * cv;
      gx += ya.y * cv;
      gy += yb.x * cv;
      gz += yb.y * cv;
      h0 += ya.x * hv;
      hx += ya.y * hv;
      hy += yb.x * hv;
      hz += yb.y * hv;
    }
  }
  const double lf = (double)l, Al = A[l];
  const double E = p.R * Al;
  const double Dd = p.dR * Al + p.R * (Al * (lf * (lf + 1.0)) * p.dk);
  double2* t = reinterpret_cast<double2*>(slot + 6 * l);
  t[0] = make_double2(s0, E);
  t[1] = make_double2((gx - lf * s0 * p.ux) * p.inv_r, (gy - lf * s0 * p.uy) * p.inv_r);
  t[2] = make_double2((gz - lf * s0 * p.uz) * p.inv_r, Dd);
  qx += Dd * h0 * p.ux + E * (hx - lf * h0 * p.ux) * p.inv_r;
  qy += Dd * h0 * p.uy + E * (hy - lf * h0 * p.uy) * p.inv_r;
  qz += Dd * h0 * p.uz + E * (hz - lf * h0 * p.uz) * p.inv_r;
}

// What the three kernels of a site share. LDS: ynorm [NLM], CHK pair records, red [8],
// the species' parameters, then U (its use differs).
template <int LL> struct LSite {
  using G = DerL<LL>;
  double *ynorm, *rec, *red, *U;
  SpeciesParams* spl;
  int tid, w, lane, li, lg;
  int64_t b0;
  int np1;
  __device__ __forceinline__ LSite(const SiteArgs& a, double* sm, int site) {
    tid = threadIdx.x;
    w = __builtin_amdgcn_readfirstlane(tid >> 6);
    lane = tid & 63;
    li = lane & 15;
    lg = lane >> 4;
    ynorm = sm;
    rec = ynorm + G::NLM;
    red = rec + G::CHK * G::ST;
    spl = reinterpret_cast<SpeciesParams*>(red + 8);
    U = sm + G::HEADP;
    b0 = a.site_beg[site];
    np1 = (int)(a.site_beg[site + 1] - b0) - 1;
  }
};

// c(n, lm) of the site into CH = U ([NLM][CP]), (l, m) tiles w and w + 4.
template <int LL>
__device__ __forceinline__ void l_expand(const SoapParams& P, const SiteArgs& a, const LSite<LL>& S) {
  using G = DerL<LL>;
  constexpr int NLM = G::NLM, CHK = G::CHK, ST = G::ST, CP = G::CP;
  constexpr int NT = (NLM + 15) / 16;
  static_assert(NT <= 8 && LL <= 8, "two tiles a wavefront, a degree's (l, m) in at most two tiles");
  const int w = S.w, li = S.li, lg = S.lg, tid = S.tid;
  double* CH = S.U;
  DerTabs tabs;
  tabs.load(P.xq, P.B, P.n_species);
  const double yn = tid < NLM ? P.ynorm[tid] : 0.0;
  const int sself = a.pr_spec[S.b0];
  if (tid < NLM) S.ynorm[tid] = yn;
  if (tid < 2 * G::SPW) (S.red + 8)[tid] = reinterpret_cast<const double*>(P.sp)[tid];
  tabs.store(S.U);
  double* W = S.U + G::TABS;         // [CHK][NLM]
  f64x4_t acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
  for (int k0 = 0; k0 < S.np1; k0 += CHK) {
    const int cnt = min(CHK, S.np1 - k0);
    der_prepare<LL, true>(S.spl, a.pr_spec, a.pr_r, a.pr_xyz, S.b0, k0, cnt, S.ynorm, S.rec, S.U, W);
    lds_barrier();
    for (int j0 = 0; j0 < cnt; j0 += 4) {
      const int j = j0 + lg;
      const bool ok = j < cnt;
      const double* st = S.rec + j * ST;
      const int nl = ok ? li - (int)st[31] : -1;
      const double av = ok && nl >= 0 && nl < (int)st[32] ? st[nl] : 0.0;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int lm = 16 * (w + 4 * t) + li;
        if (w + 4 * t < NT) {
          const double bv = ok && lm < NLM ? W[j * NLM + lm] : 0.0;
          acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc[t], 0, 0, 0);
        }
      }
    }
    lds_barrier();
  }
  if (S.np1 <= 0) lds_barrier();  // the parameters, which the preparation's barrier covers otherwise
  if (w == 0 && li == 0 && sself >= 0) {  // central atom (self pair): its own species block, l = 0
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int nl = 4 * r + lg - S.spl[sself].off;
      if (nl >= 0 && nl < S.spl[sself].nb) acc[0][r] += P.cen[sself * TGX_MAX_NB + nl];
    }
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int lm = 16 * (w + 4 * t) + li;
    if (w + 4 * t < NT && lm < NLM)
#pragma unroll
      for (int r = 0; r < 4; ++r) CH[lm * CP + 4 * r + lg] = acc[t][r];
  }
  lds_barrier();
}

// Power spectrum of CH into X [D], its norm, and this thread's components d = tid + WG j
// of q = p / |p| (zero past D), also written to q_out's row; X holds p.
template <int LL, int J>
__device__ __forceinline__ double l_spectrum(const SoapParams& P, const LSite<LL>& S, double* X, double (&qd)[J],
                                             double* qrow, double* pnorm) {
  using G = DerL<LL>;
  constexpr int L1 = G::L1, CP = G::CP;
  const int w = S.w, lane = S.lane, li = S.li, lg = S.lg, tid = S.tid, N = P.N, D = P.D;
  const double* CH = S.U;
  double* red = S.red;
  // degrees w, w + 4, w + 8
  for (int l = w; l < L1; l += 4) {
    const int K = 2 * l + 1;
    f64x4_t g = {0.0, 0.0, 0.0, 0.0};
    double v[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      const int k = 4 * q + lg;
      v[q] = k < K ? CH[(l * l + k) * CP + li] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 5; ++q)
      if (4 * q < K) g = __builtin_amdgcn_mfma_f64_16x16x4f64(v[q], v[q], g, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 4 * r + lg, np = li;
      if (n <= np && np < N) X[(n * N - n * (n - 1) / 2 + (np - n)) * L1 + l] = n == np ? g[r] : M_SQRT2 * g[r];
    }
  }
  lds_barrier();
  double nrm;
  {
    double s2 = 0.0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int d = tid + WG * j;
      qd[j] = d < D ? X[d] : 0.0;
      s2 += qd[j] * qd[j];
    }
    for (int o = 32; o > 0; o >>= 1) s2 += __shfl_xor(s2, o);
    if (lane == 0) red[w] = s2;
    lds_barrier();
    nrm = sqrt((red[0] + red[1]) + (red[2] + red[3]));
  }
  const double inv_n = nrm > 0.0 ? 1.0 / nrm : 0.0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int d = tid + WG * j;
    qd[j] *= inv_n;
    if (d < P.Dpad) qrow[d] = qd[j];
  }
  for (int d = tid + WG * J; d < P.Dpad; d += WG) qrow[d] = 0.0;
  if (tid == 0) *pnorm = nrm;
  return nrm;
}

// H_l = S_l c_l in place of c, S(n, n') = 2 X or sqrt 2 X off the diagonal: l = 0..7, then
// (l, m) 64..79 and 80 of l = 8.
template <int LL>
__device__ __forceinline__ void l_channel(const SoapParams& P, const LSite<LL>& S, const double* X) {
  static_assert(LL == 8, "degree 8 takes two tiles, the others one");
  using G = DerL<LL>;
  constexpr int L1 = G::L1, CP = G::CP;
  const int w = S.w, li = S.li, lg = S.lg, N = P.N;
  double* CH = S.U;
  for (int ht = w; ht < LL + 2; ht += 4) {
    const int l = min(ht, LL);
    const int base = ht <= LL ? l * l : l * l + 16;
    const int width = ht < LL ? 2 * l + 1 : (ht == LL ? 16 : 2 * LL - 15);
    f64x4_t h = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int n = li, np = 4 * s + lg;
      const int u = min(n, np), v = max(n, np);
      const double av =
          v < N ? (n == np ? 2.0 : M_SQRT2) * X[(u * N - u * (u - 1) / 2 + (v - u)) * L1 + l] : 0.0;
      const double bv = li < width ? CH[(base + li) * CP + np] : 0.0;
      h = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, h, 0, 0, 0);
    }
    if (li < width)
#pragma unroll
      for (int r = 0; r < 4; ++r) CH[(base + li) * CP + 4 * r + lg] = h[r];
  }
  lds_barrier();
}

// Harmonics with gradients, (Y, gx, gy, gz) per lm, of the records g .. g + 15 (< cnt), a
// row of lanes each.
template <int LL>
__device__ __forceinline__ void l_harmonics(const LSite<LL>& S, int g, int cnt, double* Yb) {
  using G = DerL<LL>;
  const int hj = S.tid >> 4;
  const double* st = S.rec + min(g + hj, cnt - 1) * G::ST;
  if (g + hj < cnt && st[30] != 0.0) {
    double2* y = reinterpret_cast<double2*>(Yb + hj * 4 * G::NLM);
    ylm_lanes<double, true, 16>(LL, S.ynorm, S.li, st[27], st[28], st[29], 1.0,
                                [&](int, int lm, double, double Y, double gx, double gy, double gz) {
                                  y[2 * lm] = make_double2(Y, gx);
                                  y[2 * lm + 1] = make_double2(gy, gz);
                                });
  }
}

// Plain-path dq/dr for l_max = 8 (the output and element layout of
// k_soap_der), one workgroup per site.
//   * Pairs are prepared 32 at a time, eight lanes each (der_prepare), and their
//     harmonics 16 at a time, a row of lanes each: with a wavefront per pair, five or
//     six pairs in turn, a preparation took 13,000 cycles, nearly all of them the
//     chain of exponentials, divisions and recurrences with 15 to 40 of 64 lanes idle.
//   * The expansion c = sum_j R_j W_j, the power spectrum p_l = c_l c_l^T and
//     H_l = S_l c_l are products on the FP64 matrix cores (16 rows n, the (l, m)
//     or pairs of one degree as the other sides).
//   * Each lane (n, p) keeps c and H of its row n at its wavefront's (l, m) in
//     registers for the channel tables of four pairs at a time (der_channel); with
//     neither in LDS the harmonics of 16 pairs fit beside two workgroups a CU
//     (79 KB each; three of 48 KB with four pairs' harmonics spill at 168
//     registers, 15.4 ms).
//   * Each thread writes whole components d = tid + WG j (its three Cartesian
//     entries) of every pair of the group and keeps the self-pair sums of its
//     components in registers. J >= D / WG.
// Bound by the 42 GB it writes at 65,536 atoms of two species (1.42 million pairs of
// 1,224 components, two blocks): 15.0 -> 9.3 ms, 4.5 TB/s where a plain fill reaches
// 6.3; at 4,096 atoms 1.15 -> 0.61 ms, at 216 atoms of one species, a workgroup a CU,
// 110 -> 50 us. Stores staged through LDS to be contiguous (10.5 -> 11.6 ms) and
// non-temporal stores (10.6) lost, as did the component codes read before the
// expansion (0.61 -> 0.64 ms at 4,096 atoms).
template <int LL, int J>
__global__ __launch_bounds__(WG, 2) void k_soap_der_l(SoapParams P, SiteArgs a, int n_sites,
                                                      double* __restrict__ q_out, double* __restrict__ pnorm_out,
                                                      double* __restrict__ der_out) {
  using G = DerL<LL>;
  constexpr int L1 = G::L1, NLM = G::NLM, SL = G::SL, CHK = G::CHK, ST = G::ST, CP = G::CP;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int site = blockIdx.x;
  if (site >= n_sites) return;
  const LSite<LL> S(a, reinterpret_cast<double*>(smem_raw), site);
  const int tid = S.tid, w = S.w, li = S.li, lg = S.lg, np1 = S.np1;
  const int D = P.D, D3 = 3 * D;
  const int64_t b0 = S.b0;
  double *U = S.U, *rec = S.rec;
  l_expand<LL>(P, a, S);
  const double* CH = U;
  double* X = U + NLM * CP + 1;      // [D]: p, then q
  double cc[21], hh[21], qd[J];
#pragma unroll
  for (int i = 0; i < 21; ++i) cc[i] = CH[der_lm<LL>(w, i) * CP + li];
  const double nrm =
      l_spectrum<LL, J>(P, S, X, qd, q_out + (size_t)site * P.Dpad, pnorm_out + site);
  const double inv_n = nrm > 0.0 ? 1.0 / nrm : 0.0;
  const bool site_ok = nrm > 0.0;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if (tid + WG * j < D) X[tid + WG * j] = qd[j];
  lds_barrier();
  l_channel<LL>(P, S, X);
#pragma unroll
  for (int i = 0; i < 21; ++i) hh[i] = CH[der_lm<LL>(w, i) * CP + li];
  lds_barrier();
  // components d = tid + WG j of this thread: row offsets of (n, l) and (n', l)
  // in the tables, n == n'
  int code[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int cd = P.dtab[min(tid + WG * j, D - 1)];
    const int n = cd & 0xff, np = (cd >> 8) & 0xff, l = cd >> 16;
    code[j] = (n * L1 + l) | ((np * L1 + l) << 8) | ((n == np ? 1 : 0) << 16);
  }
  // ---- pairs, four at a time
  double* Yb = U + 4 * SL;              // [HG][NLM][4]
  double* qpart = Yb + G::HG * 4 * NLM;     // [wave][pair][k] partial q . dp
  double self[J][3];
#pragma unroll
  for (int j = 0; j < J; ++j) self[j][0] = self[j][1] = self[j][2] = 0.0;
  for (int k0 = 0; k0 < np1; k0 += CHK) {
    const int cntc = min(CHK, np1 - k0);
    if (np1 > CHK)  // the records hold the expansion's last pairs: this chunk's again
      der_prepare_again<LL>(S.spl, P.xq, P.B, P.n_species, a.pr_spec, a.pr_r, a.pr_xyz, b0, k0, cntc, rec, U);
    for (int g = 0; g < cntc; g += 4) {
      lds_barrier();
      if (g % G::HG == 0) {
        l_harmonics<LL>(S, g, cntc, Yb);
        lds_barrier();
      }
      {
        DerLane p;
        const bool have = g + lg < cntc;
        const double* st = rec + min(g + lg, cntc - 1) * ST;
        p.ok = have && st[30] != 0.0 && site_ok;
        const int nl = li - (int)st[31];
        const bool inb = p.ok && nl >= 0 && nl < (int)st[32];
        p.R = inb ? st[nl] : 0.0;
        p.dR = inb ? st[8 + nl] : 0.0;
        p.dk = st[25];
        p.inv_r = st[26];
        p.ux = st[27];
        p.uy = st[28];
        p.uz = st[29];
        const double* y = Yb + (g % G::HG + lg) * 4 * NLM;
        double* slot = U + lg * SL + 6 * li * L1;
        double qx = 0.0, qy = 0.0, qz = 0.0;
        if (w == 0) {
          der_channel<LL, 8, 0>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
          der_channel<LL, 0, 17>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
          der_channel<LL, 1, 18>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
        } else if (w == 1) {
          der_channel<LL, 7, 0>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
          der_channel<LL, 2, 15>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
        } else if (w == 2) {
          der_channel<LL, 6, 0>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
          der_channel<LL, 3, 13>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
        } else {
          der_channel<LL, 5, 0>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
          der_channel<LL, 4, 11>(p, y, st + 16, cc, hh, slot, qx, qy, qz);
        }
        qx = lanes_sum<16>(qx);
        qy = lanes_sum<16>(qy);
        qz = lanes_sum<16>(qz);
        if (li == 0) {
          double* q = qpart + (w * 4 + lg) * 3;
          q[0] = qx;
          q[1] = qy;
          q[2] = qz;
        }
      }
      lds_barrier();
      const int cnt = min(4, cntc - g);
      for (int pp = 0; pp < cnt; ++pp) {
        const double* slot = U + pp * SL;
        const double* st = rec + (g + pp) * ST;
        const double* qp = qpart + 3 * pp;
        const double q0 = ((qp[0] + qp[12]) + qp[24]) + qp[36];
        const double q1 = ((qp[1] + qp[13]) + qp[25]) + qp[37];
        const double q2 = ((qp[2] + qp[14]) + qp[26]) + qp[38];
        const double ux = st[27], uy = st[28], uz = st[29];
        double* out = der_out + (size_t)(b0 + 1 + k0 + g + pp) * D3;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int d = tid + WG * j;
          if (d >= D) continue;
          const int cj = code[j];
          const int i1 = cj & 0xff, i2 = (cj >> 8) & 0xff;
          const double wgt = (cj >> 16) ? 1.0 : M_SQRT2;
          const double2* t1 = reinterpret_cast<const double2*>(slot + 6 * i1);
          const double2* t2 = reinterpret_cast<const double2*>(slot + 6 * i2);
          const double2 a1 = t1[0], b1 = t1[1], c1 = t1[2];  // (s, E), (v_x, v_y), (v_z, Dd)
          const double2 a2 = t2[0], b2 = t2[1], c2 = t2[2];
          const double rad = c1.y * a2.x + c2.y * a1.x;
          const double ox = (wgt * (rad * ux + a1.y * b2.x + a2.y * b1.x) - qd[j] * q0) * inv_n;
          const double oy = (wgt * (rad * uy + a1.y * b2.y + a2.y * b1.y) - qd[j] * q1) * inv_n;
          const double oz = (wgt * (rad * uz + a1.y * c2.x + a2.y * c1.x) - qd[j] * q2) * inv_n;
          out[3 * d] = ox;
          out[3 * d + 1] = oy;
          out[3 * d + 2] = oz;
          self[j][0] -= ox;
          self[j][1] -= oy;
          self[j][2] -= oz;
        }
      }
    }
  }
  double* out = der_out + (size_t)b0 * D3;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int d = tid + WG * j;
    if (d < D) {
      out[3 * d] = self[j][0];
      out[3 * d + 1] = self[j][1];
      out[3 * d + 2] = self[j][2];
    }
  }
}

// FP64 descriptors for l_max = 8 by the first half of k_soap_der_l, one workgroup
// per site (listed or in order): a wavefront per site prepared its pairs 16 at a
// time with four lanes each and formed the rest in loops over LDS. Bound by the
// preparation's chains at three workgroups a CU (its floor, the pairs read and the
// descriptors written, is 0.05 ms): 892 -> 342 us at 16,001 atoms of two species.
template <int LL, int J>
__global__ __launch_bounds__(WG, 3) void k_desc_l(SoapParams P, SiteArgs a, int n_sites, double* __restrict__ q_out,
                                                  double* __restrict__ pnorm_out, const int* __restrict__ site_list) {
  using G = DerL<LL>;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int row = blockIdx.x;
  if (row >= n_sites) return;
  const LSite<LL> S(a, reinterpret_cast<double*>(smem_raw), site_list ? site_list[row] : row);
  l_expand<LL>(P, a, S);
  double qd[J];
  l_spectrum<LL, J>(P, S, S.U + G::NLM * G::CP + 1, qd, q_out + (size_t)row * P.Dpad, pnorm_out + row);
}

// FP64 adjoint pair forces for l_max = 8, one workgroup per site: c as above, H from
// g = (Qss - (Qss . q) q) / |p|, then sixteen pairs at a time: x = sum_n R_n H(n, lm) and
// y = sum_n R_n' H(n, lm) of all of them on the FP64 matrix cores, one (l, m) tile after
// the other, and
//   f_j = sum_lm [ (A' x + A y) Y u + A x (grad Y - l Y u) / r ]
// summed by the lane that holds x and y of (j, lm), over the row's lanes, and over the
// wavefronts (tiles w, w + 4) in order. A wavefront per site held H in registers and
// walked x and y through LDS: 1,915 -> 752 us at 16,001 atoms of two species, bound as
// the descriptors (c is formed again: reading it back would cost 10 KB a site).
template <int LL, int J>
__global__ __launch_bounds__(WG, 3) void k_adjoint_l(SoapParams P, SiteArgs a, int n_sites,
                                                     const double* __restrict__ q_in,
                                                     const double* __restrict__ pnorm_in,
                                                     const double* __restrict__ qss, double* __restrict__ fglob) {
  using G = DerL<LL>;
  constexpr int NLM = G::NLM, CHK = G::CHK, ST = G::ST, CP = G::CP, HG = G::HG;
  constexpr int NT = (NLM + 15) / 16;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int site = blockIdx.x;
  if (site >= n_sites) return;
  const LSite<LL> S(a, reinterpret_cast<double*>(smem_raw), site);
  const int tid = S.tid, w = S.w, lane = S.lane, li = S.li, lg = S.lg, np1 = S.np1, D = P.D;
  const int64_t b0 = S.b0;
  double qd[J], sd[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int d = tid + WG * j;
    qd[j] = d < D ? q_in[(size_t)site * P.Dpad + d] : 0.0;
    sd[j] = d < D ? qss[(size_t)site * P.Dpad + d] : 0.0;
  }
  const double nrm = pnorm_in[site];
  l_expand<LL>(P, a, S);
  double* X = S.U + NLM * CP + 1;  // g
  {
    double sq = 0.0;
#pragma unroll
    for (int j = 0; j < J; ++j) sq += sd[j] * qd[j];
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_xor(sq, o);
    if (lane == 0) S.red[w] = sq;
    lds_barrier();
    sq = (S.red[0] + S.red[1]) + (S.red[2] + S.red[3]);
    const double inv_n = nrm > 0.0 ? 1.0 / nrm : 0.0;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int d = tid + WG * j;
      if (d < D) X[d] = (sd[j] - sq * qd[j]) * inv_n;
    }
  }
  lds_barrier();
  l_channel<LL>(P, S, X);
  double hreg[2][4];  // H(4 s + lg, lm) of this wavefront's tiles
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int lm = 16 * (w + 4 * t) + li;
      hreg[t][s] = lm < NLM ? S.U[lm * CP + 4 * s + lg] : 0.0;
    }
  lds_barrier();
  double* Yb = S.U;                    // [HG][NLM][4]
  double* part = Yb + HG * 4 * NLM;    // [wave][pair][k]
  const int oj = tid / 3, ok = tid - 3 * oj;  // pair and component of the thread's output (oj < HG)
  double self = 0.0;
  for (int k0 = 0; k0 < np1; k0 += CHK) {
    const int cntc = min(CHK, np1 - k0);
    if (np1 > CHK)  // the records hold the expansion's last pairs: this chunk's again
      der_prepare_again<LL>(S.spl, P.xq, P.B, P.n_species, a.pr_spec, a.pr_r, a.pr_xyz, b0, k0, cntc, S.rec, S.U);
    for (int g = 0; g < cntc; g += HG) {
      lds_barrier();
      l_harmonics<LL>(S, g, cntc, Yb);
      const bool mine = oj < HG && g + oj < cntc;
      const int64_t gi = mine ? a.pr_gidx[b0 + 1 + k0 + g + oj] : 0;
      double ra[4], da[4];
      {
        const double* st = S.rec + min(g + li, cntc - 1) * ST;
        const int off = (int)st[31], nb = (int)st[32];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int nl = 4 * s + lg - off;
          const bool in = g + li < cntc && nl >= 0 && nl < nb;
          ra[s] = in ? st[nl] : 0.0;
          da[s] = in ? st[8 + nl] : 0.0;
        }
      }
      lds_barrier();
      double tu[4], fx[4], fy[4], fz[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) tu[r] = fx[r] = fy[r] = fz[r] = 0.0;
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (w + 4 * t >= NT) break;
        f64x4_t x = {0.0, 0.0, 0.0, 0.0}, y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          x = __builtin_amdgcn_mfma_f64_16x16x4f64(ra[s], hreg[t][s], x, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f64_16x16x4f64(da[s], hreg[t][s], y, 0, 0, 0);
        }
        const int lm = 16 * (w + 4 * t) + li;
        if (lm < NLM) {
          const int l = lm_l(lm);
          const double lf = (double)l, ll = lf * (lf + 1.0);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int j = 4 * r + lg;  // pairs past the end or unseen: dropped below
            const double* st = S.rec + min(g + j, cntc - 1) * ST;
            const double2* yv = reinterpret_cast<const double2*>(Yb + j * 4 * NLM + 4 * lm);
            const double2 ya = yv[0], yb = yv[1];
            const double A = st[16 + l], Ax = A * x[r], ang = Ax * st[26];
            tu[r] += (Ax * (ll * st[25]) + A * y[r] - ang * lf) * ya.x;
            fx[r] += ang * ya.y;
            fy[r] += ang * yb.x;
            fz[r] += ang * yb.y;
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 4 * r + lg;
        const double* st = S.rec + min(g + j, cntc - 1) * ST;
        const double tt = lanes_sum<16>(tu[r]);
        const double vx = lanes_sum<16>(fx[r]) + tt * st[27], vy = lanes_sum<16>(fy[r]) + tt * st[28],
                     vz = lanes_sum<16>(fz[r]) + tt * st[29];
        if (li == 0) {
          double* o = part + (w * HG + j) * 3;
          o[0] = vx;
          o[1] = vy;
          o[2] = vz;
        }
      }
      lds_barrier();
      if (mine && S.rec[(g + oj) * ST + 30] != 0.0) {
        const double* o = part + 3 * oj + ok;
        const double f = ((o[0] + o[3 * HG]) + o[6 * HG]) + o[9 * HG];
        fglob[3 * gi + ok] += f;
        self += f;
      }
    }
  }
  // the self entry: minus the sum of the others, over the sixteen pairs' threads in order
  lds_barrier();
  if (oj < HG) part[tid] = self;
  lds_barrier();
  if (tid < 3) {
    double v = 0.0;
    for (int j = 0; j < HG; ++j) v += part[3 * j + tid];
    fglob[3 * a.pr_gidx[b0] + tid] -= v;
  }
}

// Plain-path pair force: f_p = Qss_i . soap_cart_der(:, :, p), one wavefront per
// pair, streamed over the (3, D) slab. This is the scatter of src/gap.f90:206-224.
__global__ __launch_bounds__(256) void k_plain_force(int n_sites, const int64_t* __restrict__ site_beg, int D,
                                                    int Dpad, const double* __restrict__ qss,
                                                    const double* __restrict__ der,
                                                    const int64_t* __restrict__ pr_gidx, int64_t n_pairs,
                                                    const int* __restrict__ pair_site, double* __restrict__ fglob) {
  const int lane = threadIdx.x & 63;
  const int64_t p = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= n_pairs) return;
  const int i = pair_site[p];
  if (i < 0) return;  // a pair no site claims (caller-supplied offsets)
  const double* s = qss + (size_t)i * Dpad;
  const double* g = der + (size_t)p * 3 * D;
  double a0 = 0, a1 = 0, a2 = 0;
  for (int d = lane; d < D; d += 64) {
    const double sv = s[d];
    a0 += sv * g[3 * d];
    a1 += sv * g[3 * d + 1];
    a2 += sv * g[3 * d + 2];
  }
  for (int o = 32; o > 0; o >>= 1) {
    a0 += __shfl_xor(a0, o);
    a1 += __shfl_xor(a1, o);
    a2 += __shfl_xor(a2, o);
  }
  if (lane == 0) {
    const int64_t gi = pr_gidx ? pr_gidx[p] : p;
    fglob[3 * gi] += a0;
    fglob[3 * gi + 1] += a1;
    fglob[3 * gi + 2] += a2;
  }
}

// local_property_predict (src/local_properties.f90:174-297) from the block's
// GAP contraction: V_s = max(0, E_s) (the model's e0 is V0), and per pair
// V_der = dV_i/dq . dq/dr = -Qss_i . soap_cart_der(:, :, p) (Qss here is
// -dE/dq), zero for a centre whose V is 0. One wavefront per pair.
__global__ __launch_bounds__(256) void k_local_property(int n_sites, int D, int Dpad, const double* __restrict__ e_site,
                                                         const double* __restrict__ qss, const double* __restrict__ der,
                                                         int64_t n_pairs, const int* __restrict__ pair_site,
                                                         double* __restrict__ V, double* __restrict__ vder) {
  const int lane = threadIdx.x & 63;
  const int64_t p = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p < n_sites && lane == 0) V[p] = e_site[p] < 0.0 ? 0.0 : e_site[p];
  if (p >= n_pairs || !vder) return;
  const int i = pair_site[p];
  double a0 = 0, a1 = 0, a2 = 0;
  if (e_site[i] > 0.0) {
    const double* s = qss + (size_t)i * Dpad;
    const double* g = der + (size_t)p * 3 * D;
    for (int d = lane; d < D; d += 64) {
      const double sv = s[d];
      a0 += sv * g[3 * d];
      a1 += sv * g[3 * d + 1];
      a2 += sv * g[3 * d + 2];
    }
    for (int o = 32; o > 0; o >>= 1) {
      a0 += __shfl_xor(a0, o);
      a1 += __shfl_xor(a1, o);
      a2 += __shfl_xor(a2, o);
    }
  }
  if (lane == 0) {
    vder[3 * p] = -a0;
    vder[3 * p + 1] = -a1;
    vder[3 * p + 2] = -a2;
  }
}

__global__ void k_pair_site(int n_sites, const int64_t* __restrict__ site_beg, int* __restrict__ pair_site) {
  const int i = blockIdx.x;
  if (i >= n_sites) return;
  for (int64_t p = site_beg[i] + threadIdx.x; p < site_beg[i + 1]; p += blockDim.x) pair_site[p] = i;
}

// k_pair_site for offsets the caller supplied: entries at or beyond n_pairs
// (offsets summing past it) are not written.
__global__ void k_pair_site_clip(int n_sites, const int64_t* __restrict__ site_beg, int64_t n_pairs,
                                 int* __restrict__ pair_site) {
  const int i = blockIdx.x;
  if (i >= n_sites) return;
  const int64_t e = site_beg[i + 1] < n_pairs ? site_beg[i + 1] : n_pairs;
  for (int64_t p = site_beg[i] + threadIdx.x; p < e; p += blockDim.x) pair_site[p] = i;
}

}  // namespace

// LDS bytes of the site kernels.
static size_t soap_lds_bytes(const SoapParams& P, int mode, size_t elt) {
  const int N = P.N, NLM = P.NLM, L1 = P.L + 1;
  const size_t ps = (size_t)(2 * TGX_MAX_Q + 2 * TGX_MAX_NB + 2 * L1 + 4 * NLM);
  size_t n = (size_t)N * NLM + P.D + WG;
  if (mode == 0) n += 4 * ps;
  if (mode == 1) {
    n += (size_t)N * NLM;
    size_t d_scr = ps + (size_t)N * L1 * 6 + (size_t)TGX_MAX_NB * L1 * 4 + 4;
    n += d_scr > 4 * ps ? d_scr : 4 * ps;
  }
  return n * elt;
}

static SiteArgs site_args(tgx_model_t* m) {
  SiteArgs a;
  a.site_atom = m->site_atom.as<int>();
  a.site_beg = m->site_beg.as<int64_t>();
  a.pr_spec = m->pr_spec.as<int>();
  a.pr_r = m->pr_r.as<double>();
  a.pr_xyz = m->pr_xyz.as<double>();
  a.pr_gidx = m->pr_gidx.as<int64_t>();
  return a;
}

static int check_lds(size_t bytes) {
  TGX_REQUIRE(bytes <= 160 * 1024, "SOAP kernel needs %zu bytes of LDS (more than 160 KiB): reduce n_max or l_max",
              bytes);
  return TGX_OK;
}

// Blocks that the kernels for l_max = 8 take: at most two species of at most eight
// radial functions, the sizes their degree sets, pair records and 16-row tiles are
// laid out for. At 16,001 atoms 1.09 ms for descriptors and adjoint together, 2.81
// for the wavefront-per-site kernels, which take every other block.
static bool l_kernels(const SoapParams& P) {
  bool ok = P.L == 8 && P.N <= 16 && P.n_species <= 2;
  for (int s = 0; s < P.n_species; ++s) ok = ok && P.sp[s].nb <= 8;
  return ok;
}

// FP64 descriptors of the block's (or the listed) sites.
static int desc_f64(tgx_ctx* ctx, tgx_model_t* m, const int* d_sites, int n_rows, double* q_out, double* pn_out) {
  const SoapParams& P = m->P;
  if (!l_kernels(P)) return tgx_desc_wave(ctx, m, true, d_sites, n_rows, q_out, pn_out);
  if (n_rows == 0) return TGX_OK;
  SiteArgs a = site_args(m);
  const char* name = d_sites ? "soap_desc_list_f64" : "soap_desc_f64";
  if (P.D <= 2 * WG)
    TGX_LAUNCH(ctx, name, (k_desc_l<8, 2>), dim3(n_rows), dim3(WG), DerL<8>::LDS_DESC, P, a, n_rows, q_out, pn_out,
               d_sites);
  else
    TGX_LAUNCH(ctx, name, (k_desc_l<8, 5>), dim3(n_rows), dim3(WG), DerL<8>::LDS_DESC, P, a, n_rows, q_out, pn_out,
               d_sites);
  return TGX_OK;
}

int tgx_soap_descriptors(tgx_ctx* ctx, tgx_model_t* m, int path, bool with_der) {
  m->der_whole = false;  // set again by a whole-block FP64 plain evaluation
  const int ns = m->n_sites_b;
  if (ns == 0) return TGX_OK;
  TGX_REQUIRE(m->P.D <= 24 * WG, "descriptor size %d exceeds this build's limit %d", m->P.D, 24 * WG);
  const size_t nsp = (size_t)tgx_round_up(ns, 128);
  TGX_TRY(m->pnorm.ensure(sizeof(double) * nsp));
  SiteArgs a = site_args(m);
  TGX_REQUIRE(!m->compress || path == TGX_PATH_FP64_PLAIN || path == TGX_PATH_FP64_ADJOINT,
              "compressed SOAP blocks run on the FP64 paths only");
  if (path == TGX_PATH_FP64_PLAIN || path == TGX_PATH_FP64_ADJOINT) {
    // a compressed block's kernels write the full descriptors, compressed below
    dbuf& qout = m->compress ? m->qf64 : m->q64;
    dbuf& dout = m->compress ? m->derf : m->soap_der;
    TGX_TRY(qout.ensure(sizeof(double) * nsp * m->P.Dpad));
    if (with_der) {
      TGX_TRY(dout.ensure(sizeof(double) * (size_t)(m->n_pairs_b > 0 ? m->n_pairs_b : 1) * 3 * m->P.D));
      const SoapParams& P = m->P;
      const int NL = P.N * (P.L + 1);
      const int j_need = (3 * P.D + WG - 1) / WG;
      if (l_kernels(P)) {
        constexpr size_t lds = DerL<8>::LDS;
#define TGX_SOAP_DER(J)                                                                                     \
  TGX_LAUNCH(ctx, "soap_site_der_f64", (k_soap_der_l<8, J>), dim3(ns), dim3(WG), lds, m->P, a, ns, \
             qout.as<double>(), m->pnorm.as<double>(), dout.as<double>())
        if (P.D <= 2 * WG) TGX_SOAP_DER(2);
        else TGX_SOAP_DER(5);
#undef TGX_SOAP_DER
      } else if (j_need <= 16 && NL <= 255 && P.D < 4096) {
        // coefficient, H and four pair slots; the slots overlay the spectrum and pair scratch
        const size_t head = 2 * (size_t)P.N * P.NLM + P.D;
        const size_t ps = (size_t)(2 * TGX_MAX_Q + 2 * TGX_MAX_NB + 2 * (P.L + 1) + 4 * P.NLM);
        const size_t u1 = (size_t)WG + 4 * ps;
        const size_t u2 = 4 * (size_t)(6 * NL + 8 + ps);
        const size_t lds = sizeof(double) * (head + (u1 > u2 ? u1 : u2));
        TGX_TRY(check_lds(lds));
#define TGX_SOAP_DER(J)                                                                                           \
  TGX_LAUNCH(ctx, "soap_site_der_f64", (k_soap_der<J>), dim3(ns), dim3(WG), lds, m->P, a, ns, qout.as<double>(), \
             m->pnorm.as<double>(), dout.as<double>())
        if (j_need <= 4) TGX_SOAP_DER(4);
        else if (j_need <= 8) TGX_SOAP_DER(8);
        else if (j_need <= 12) TGX_SOAP_DER(12);
        else TGX_SOAP_DER(16);
#undef TGX_SOAP_DER
      } else {
        const size_t lds = soap_lds_bytes(m->P, 1, sizeof(double));
        TGX_TRY(check_lds(lds));
        const int kmax = (m->P.D + WG - 1) / WG;
#define TGX_SOAP_DER(K)                                                                                 \
  TGX_LAUNCH(ctx, "soap_site_der_f64", (k_soap_site<double, 1, K>), dim3(ns), dim3(WG), lds, m->P, a, ns, \
             qout.as<double>(), m->pnorm.as<double>(), dout.as<double>(), (const int*)nullptr)
        if (kmax <= 8) TGX_SOAP_DER(8);
        else if (kmax <= 12) TGX_SOAP_DER(12);
        else TGX_SOAP_DER(24);
#undef TGX_SOAP_DER
      }
    } else {
      TGX_TRY(desc_f64(ctx, m, nullptr, ns, qout.as<double>(), m->pnorm.as<double>()));
    }
    if (m->compress) TGX_TRY(tgx_compress_descriptors(ctx, m, with_der));
  } else {
    TGX_TRY(m->q32.ensure(sizeof(float) * nsp * m->Dpad));
    if (m->P.N <= 16) {
      TGX_TRY(tgx_desc_f32(ctx, m));  // writes the BF16 copy as well
    } else {
      TGX_TRY(tgx_desc_wave(ctx, m, false, nullptr, ns, m->q32.p, m->pnorm.p));
      TGX_TRY(m->qbf.ensure(sizeof(__bf16) * (size_t)tgx_rows_bf16(ns) * m->Dpad));
      TGX_TRY(tgx_f32_to_bf16(ctx, m->q32.as<float>(), m->qbf.as<__bf16>(), (int64_t)nsp * m->Dpad));
    }
  }
  return TGX_OK;
}

int tgx_adjoint_pair_forces(tgx_ctx* ctx, tgx_model_t* m, int path) {
  const bool fp64 = path == TGX_PATH_FP64_ADJOINT || path == TGX_PATH_FP64_PLAIN;
  TGX_REQUIRE(!m->compress || fp64, "compressed SOAP blocks run on the FP64 paths only");
  if (m->compress) TGX_TRY(tgx_compress_gradient(ctx, m));
  if (!fp64 && m->P.N <= 16) return tgx_adjoint_f32(ctx, m);
  const SoapParams& P = m->P;
  if (fp64 && l_kernels(P)) {
    const int ns = m->n_sites_b;
    if (ns == 0) return TGX_OK;
    SiteArgs a = site_args(m);
    // a compressed block contracts the full-size gradient with the full descriptors
    const double* q = (m->compress ? m->qf64 : m->q64).as<double>();
    const double* g = (m->compress ? m->qssf64 : m->qss64).as<double>();
    if (P.D <= 2 * WG)
      TGX_LAUNCH(ctx, "soap_adjoint_f64", (k_adjoint_l<8, 2>), dim3(ns), dim3(WG), DerL<8>::LDS_ADJ, P, a, ns, q,
                 m->pnorm.as<double>(), g, ctx->fglob.as<double>());
    else
      TGX_LAUNCH(ctx, "soap_adjoint_f64", (k_adjoint_l<8, 5>), dim3(ns), dim3(WG), DerL<8>::LDS_ADJ, P, a, ns, q,
                 m->pnorm.as<double>(), g, ctx->fglob.as<double>());
    return TGX_OK;
  }
  return tgx_adjoint_wave(ctx, m, fp64);
}

int tgx_plain_pair_forces(tgx_ctx* ctx, tgx_model_t* m) { return tgx_plain_pair_forces_q(ctx, m, m->qss64.as<double>()); }

int tgx_plain_pair_forces_q(tgx_ctx* ctx, tgx_model_t* m, const double* qss) {
  const int ns = m->n_sites_b;
  const int64_t np = m->n_pairs_b;
  if (ns == 0 || np == 0) return TGX_OK;
  TGX_TRY(m->pair_site.ensure(sizeof(int) * (size_t)np));
  int* pair_site = m->pair_site.as<int>();
  TGX_LAUNCH(ctx, "pair_site", k_pair_site, dim3(ns), dim3(64), 0, ns, m->site_beg.as<int64_t>(), pair_site);
  TGX_LAUNCH(ctx, "plain_force", k_plain_force, dim3((unsigned)((np + 3) / 4)), dim3(256), 0, ns,
             m->site_beg.as<int64_t>(), m->D, m->Dpad, qss, m->soap_der.as<double>(), m->pr_gidx.as<int64_t>(), np,
             pair_site, ctx->fglob.as<double>());
  return TGX_OK;
}

// The plain pair forces on caller-supplied buffers: fpair (3, n_pairs) +=
// Qss_i . der(:, :, p) for the pairs p of every site i (offsets site_beg, which
// may sum past n_pairs: those entries are skipped), pair_site a work array of
// n_pairs ints. No allocation.
int tgx_plain_pair_forces_raw(tgx_ctx* ctx, int ns, const int64_t* site_beg, int64_t np, int D, int Dpad,
                              const double* qss, const double* der, int* pair_site, double* fpair) {
  if (ns == 0 || np == 0) return TGX_OK;
  TGX_LAUNCH(ctx, "pair_site", k_pair_site_clip, dim3(ns), dim3(64), 0, ns, site_beg, np, pair_site);
  TGX_LAUNCH(ctx, "plain_force", k_plain_force, dim3((unsigned)((np + 3) / 4)), dim3(256), 0, ns, site_beg, D, Dpad,
             qss, der, (const int64_t*)nullptr, np, (const int*)pair_site, fpair);
  return TGX_OK;
}

// V (n_sites_b) and, with derivatives, V_der (3, n_pairs_b) on the device
// (ctx->scratch) after the FP64 plain descriptors and contraction of the block.
int tgx_local_property_finish(tgx_ctx* ctx, tgx_model_t* m, bool with_der, double** d_V, double** d_vder) {
  const int ns = m->n_sites_b;
  const int64_t np = with_der ? m->n_pairs_b : 0;
  TGX_TRY(ctx->scratch.ensure(sizeof(double) * ((size_t)ns + 3 * (size_t)np) + sizeof(int) * (size_t)np + 64));
  double* V = ctx->scratch.as<double>();
  double* vder = V + ns;
  int* pair_site = reinterpret_cast<int*>(vder + 3 * np);
  if (np > 0)
    TGX_LAUNCH(ctx, "pair_site", k_pair_site, dim3(ns), dim3(64), 0, ns, m->site_beg.as<int64_t>(), pair_site);
  const int64_t rows = np > ns ? np : ns;
  if (rows > 0)
    TGX_LAUNCH(ctx, "local_property", k_local_property, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, ns, m->D,
               m->Dpad, m->e_site.as<double>(), np > 0 ? m->qss64.as<double>() : nullptr,
               np > 0 ? m->soap_der.as<double>() : nullptr, np, pair_site, V, np > 0 ? vder : nullptr);
  *d_V = V;
  *d_vder = vder;
  return TGX_OK;
}

// FP64 descriptors of the listed sites of the current block, row r of q_out
// holding site d_sites[r] (used to re-evaluate gated sites with the GAP).
int tgx_soap_descriptors_sites(tgx_ctx* ctx, tgx_model_t* m, const int* d_sites, int n_list, double* q_out,
                               double* pnorm_out) {
  return desc_f64(ctx, m, d_sites, n_list, q_out, pnorm_out);
}
