// Wavefront-per-site SOAP kernels (descriptor and adjoint forces).
//
// One wavefront owns one central site and synchronises only with itself, so a
// workgroup's four wavefronts run four sites independently. Within a site
// quads of lanes take the neighbour pairs (16 per pass):
//   * a quad of lanes computes its pair's radial projections R_n (n in the pair's
//     species block) from the Gaussian at the fixed quadrature nodes, a quarter
//     of the nodes each, and streams all real spherical harmonics from
//     recurrences in m and l, a quarter of the orders m each;
//   * the expansion c(n, lm) = sum_j R_n(j) A_l(j) Y_lm(j) is then a small
//     product of the staged R and W = A Y, with lanes over (n, lm) outputs;
//   * the adjoint contracts H(n, lm) = d(g . p)/dc with dc/dr_j on the fly:
//     f_j = sum_lm [ (A' x + A y) Y u + A x (grad Y - l Y u)/r ], with
//     x = sum_n R_n H(n, lm), y = sum_n R_n' H(n, lm), so no per-pair table
//     of harmonics is kept.
// Same conventions and results as the workgroup-per-site kernels (the plain
// dq/dr kernel keeps that form).
#include "tgx_internal.h"
#include "tgx_soap_lanes.h"

namespace {

constexpr int WAVES = 4;

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <class T> __device__ __forceinline__ T wave_sum(T v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

struct WaveArgs {
  const int64_t* site_beg;
  const int* pr_spec;
  const double* pr_r;
  const double* pr_xyz;
  const int64_t* pr_gidx;
};

// Per-workgroup tables staged in LDS: harmonic constants, nodes, B transposed to [q][n].
template <class T> struct Tables {
  T* ynorm;  // [NLM]
  T* xq;     // [S][MAX_Q]
  T* Bt;     // [S][MAX_Q][MAX_NB]
  static __host__ __device__ int size(int S, int NLM) { return NLM + S * TGX_MAX_Q + S * TGX_MAX_Q * TGX_MAX_NB; }
  __device__ void load(const SoapParams& P, T* base) {
    ynorm = base;
    xq = ynorm + P.NLM;
    Bt = xq + P.n_species * TGX_MAX_Q;
    for (int i = threadIdx.x; i < P.NLM; i += blockDim.x) ynorm[i] = (T)P.ynorm[i];
    for (int i = threadIdx.x; i < P.n_species * TGX_MAX_Q; i += blockDim.x) xq[i] = (T)P.xq[i];
    for (int i = threadIdx.x; i < P.n_species * TGX_MAX_Q * TGX_MAX_NB; i += blockDim.x) {
      const int s = i / (TGX_MAX_Q * TGX_MAX_NB), rem = i - s * TGX_MAX_Q * TGX_MAX_NB;
      const int q = rem / TGX_MAX_NB, n = rem - q * TGX_MAX_NB;
      Bt[i] = (T)P.B[((size_t)s * TGX_MAX_NB + n) * TGX_MAX_Q + q];
    }
  }
};

// Expansion coefficients of one site into C (LDS, [N][NLM]) by one wavefront.
// Pass over chunks of CH pairs: quads of lanes stage Rf[j][n] (stacked radial index,
// zero outside the pair's species block) and W[j][lm] = A_l Y_lm in LDS; then
// lanes over lm accumulate C[n][lm] += sum_j Rf[j][n] W[j][lm] with the n
// column in registers and Rf rows read as LDS broadcasts.
template <class T, int CH, int NMAX>
__device__ void wave_coefficients(const SoapParams& P, const Tables<T>& tb, const WaveArgs& a, int64_t b0, int nn, T* C,
                                  T* W, T* Rf) {
  const int lane = threadIdx.x & 63, pj = lane >> 2, sub = lane & 3;  // a quad of lanes per pair
  static_assert(CH <= 16, "a pass holds a pair per quad");
  const int NLM = P.NLM, N = P.N, L = P.L;
  T acc[2][NMAX];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int n = 0; n < NMAX; ++n) acc[h][n] = 0;
  {
    const int s = a.pr_spec[b0];
    if (s >= 0) {
      // central atom: l = m = 0 of its own block
#pragma unroll
      for (int n = 0; n < NMAX; ++n) {
        const int nl = n - P.sp[s].off;
        if (lane == 0 && nl >= 0 && nl < P.sp[s].nb) acc[0][n] = (T)P.cen[s * TGX_MAX_NB + nl];
      }
    }
  }
  for (int k0 = 1; k0 < nn; k0 += CH) {
    const int cnt = min(CH, nn - k0);
    wave_sync();
    if (pj < cnt) {
      const int64_t p = b0 + k0 + pj;
      int s = a.pr_spec[p];
      const double rr = a.pr_r[p];
      if (s >= 0 && !(rr < P.sp[s].rc)) s = -1;
      T* rf = Rf + pj * NMAX;
      for (int n = sub; n < NMAX; n += 4) rf[n] = 0;
      T* w = W + pj * NLM;
      if (s >= 0) {
        const T r = (T)rr, inv = (T)1 / r;
        const T ux = (T)a.pr_xyz[3 * p] * inv, uy = (T)a.pr_xyz[3 * p + 1] * inv, uz = (T)a.pr_xyz[3 * p + 2] * inv;
        T R[TGX_MAX_NB], dR[TGX_MAX_NB];
        radial_lanes<T, false, 4, TGX_MAX_NB>(P.sp[s], tb.xq + s * TGX_MAX_Q, tb.Bt + s * TGX_MAX_Q * TGX_MAX_NB, sub, r,
                                                R, dR);
        const int off = P.sp[s].off, nb = P.sp[s].nb;
        wave_sync();  // the quad's zeros before its values
        if (sub == 0)
#pragma unroll
          for (int n = 0; n < TGX_MAX_NB; ++n)
            if (n < nb) rf[off + n] = R[n];
        Damp<T> dmp;
        dmp.init(P.sp[s], r);
        ylm_lanes<T, false, 4>(L, tb.ynorm, sub, ux, uy, uz, dmp.e2,
                           [&](int l, int lm, T Al, T Y, T, T, T) { w[lm] = Al * Y; });
      } else {
        for (int lm = sub; lm < NLM; lm += 4) w[lm] = 0;
      }
    }
    wave_sync();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int lm = lane + 64 * h;
      if (lm < NLM) {
        for (int j = 0; j < cnt; ++j) {
          const T wv = W[j * NLM + lm];
          const T* rf = Rf + j * NMAX;
#pragma unroll
          for (int n = 0; n < NMAX; ++n) acc[h][n] += rf[n] * wv;
        }
      }
    }
  }
  wave_sync();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int lm = lane + 64 * h;
    if (lm < NLM)
#pragma unroll
      for (int n = 0; n < NMAX; ++n)
        if (n < N) C[n * NLM + lm] = acc[h][n];
  }
  wave_sync();
}

// Power spectrum of C into X[0..D), returns |p| (X normalised to q in place).
template <class T>
__device__ T wave_power(const SoapParams& P, const T* C, T* X) {
  const int lane = threadIdx.x & 63;
  const int NLM = P.NLM;
  T acc = 0;
  for (int d = lane; d < P.D; d += 64) {
    const int code = P.dtab[d];
    const int n = code & 0xff, np = (code >> 8) & 0xff, l = code >> 16;
    const T* c1 = C + n * NLM + l * l;
    const T* c2 = C + np * NLM + l * l;
    T s0 = 0, s1 = 0;
#pragma unroll
    for (int m = 0; m < 2 * TGX_MAX_L + 1; m += 2) {
      if (m < 2 * l + 1) s0 += c1[m] * c2[m];
      if (m + 1 < 2 * l + 1) s1 += c1[m + 1] * c2[m + 1];
    }
    T s = s0 + s1;
    if (n != np) s *= (T)M_SQRT2;
    X[d] = s;
    acc += s * s;
  }
  const T nrm = w_sqrt<T>(wave_sum<T>(acc));
  const T inv = nrm > (T)0 ? (T)1 / nrm : (T)0;
  for (int d = lane; d < P.D; d += 64) X[d] *= inv;
  wave_sync();
  return nrm;
}

template <class T> struct WaveLayout {
  // per-wavefront LDS (elements of T):
  //   descriptor: C [N NLM] | U = max(W [CH NLM] + Rf [CH NMAX], X [D])
  //   adjoint:    C | H [N NLM] | U = max(W + Rf, X, pair chunk - N NLM)
  //   where the pair chunk (Xa, Xb [CH NLM], R, dR [CH NMAX]) overlays C and U.
  static __host__ __device__ int coef_chunk(int CH, int NLM, int NMAX) { return CH * NLM + CH * NMAX; }
  static __host__ __device__ int pair_chunk(int CH, int NLM, int NMAX) { return 2 * CH * NLM + 2 * CH * NMAX; }
  static __host__ __device__ int per_wave(int CH, int NMAX, const SoapParams& P, bool adjoint) {
    const int cn = P.N * P.NLM;
    int u = coef_chunk(CH, P.NLM, NMAX);
    if (P.D > u) u = P.D;
    if (!adjoint) return cn + u;
    const int pc = pair_chunk(CH, P.NLM, NMAX) - cn;
    if (pc > u) u = pc;
    return 2 * cn + u;
  }
};

template <class T, int CH, int NMAX>
__global__ __launch_bounds__(64 * WAVES) void k_desc_wave(SoapParams P, WaveArgs a, int n_sites, T* __restrict__ q_out,
                                                          T* __restrict__ pnorm_out, const int* __restrict__ site_list) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* sm = reinterpret_cast<T*>(smem_raw);
  Tables<T> tb;
  tb.load(P, sm);
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int orow = blockIdx.x * WAVES + w;
  if (orow >= n_sites) return;
  const int site = site_list ? site_list[orow] : orow;
  T* base = sm + Tables<T>::size(P.n_species, P.NLM) + w * WaveLayout<T>::per_wave(CH, NMAX, P, false);
  T* C = base;
  T* U = C + P.N * P.NLM;
  const int64_t b0 = a.site_beg[site];
  const int nn = (int)(a.site_beg[site + 1] - b0);
  wave_coefficients<T, CH, NMAX>(P, tb, a, b0, nn, C, U, U + CH * P.NLM);
  T* X = U;  // reuses the chunk scratch
  const T nrm = wave_power<T>(P, C, X);
  T* qrow = q_out + (size_t)orow * P.Dpad;
  for (int d = lane; d < P.Dpad; d += 64) qrow[d] = d < P.D ? X[d] : (T)0;
  if (lane == 0) pnorm_out[orow] = nrm;
}

template <class T, int CH, int NMAX>
__global__ __launch_bounds__(64 * WAVES) void k_adjoint_wave(SoapParams P, WaveArgs a, int n_sites,
                                                             const T* __restrict__ q_in, const T* __restrict__ pnorm_in,
                                                             const T* __restrict__ qss, double* __restrict__ fglob) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* sm = reinterpret_cast<T*>(smem_raw);
  Tables<T> tb;
  tb.load(P, sm);
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, pj = lane >> 2, sub = lane & 3;
  const int site = blockIdx.x * WAVES + w;
  if (site >= n_sites) return;
  const int NLM = P.NLM, N = P.N, L = P.L, D = P.D, CN = N * NLM;
  T* base = sm + Tables<T>::size(P.n_species, NLM) + w * WaveLayout<T>::per_wave(CH, NMAX, P, true);
  T* C = base;
  T* H = C + CN;
  T* U = H + CN;
  const int64_t b0 = a.site_beg[site];
  const int nn = (int)(a.site_beg[site + 1] - b0);
  wave_coefficients<T, CH, NMAX>(P, tb, a, b0, nn, C, U, U + CH * NLM);
  // g = (Qss - (Qss . q) q) / |p|
  T* X = U;
  const T* qrow = q_in + (size_t)site * P.Dpad;
  const T* srow = qss + (size_t)site * P.Dpad;
  T acc = 0;
  for (int d = lane; d < D; d += 64) acc += srow[d] * qrow[d];
  const T sq = wave_sum<T>(acc);
  const T nrm = pnorm_in[site];
  const T inv_n = nrm > (T)0 ? (T)1 / nrm : (T)0;
  for (int d = lane; d < D; d += 64) X[d] = (srow[d] - sq * qrow[d]) * inv_n;
  wave_sync();
  // H(n, lm) = sum_n' S(n, n', l) C(n', lm): lanes over lm, C column in registers
  const int L1 = L + 1;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int lm = lane + 64 * h;
    if (lm < NLM) {
      int l = (int)sqrtf((float)lm + 0.5f);
      if (l * l > lm) --l;
      T cc[NMAX];
#pragma unroll
      for (int n = 0; n < NMAX; ++n) cc[n] = n < N ? C[n * NLM + lm] : (T)0;
#pragma unroll
      for (int n = 0; n < NMAX; ++n) {
        if (n >= N) break;
        T hsum = 0;
#pragma unroll
        for (int np = 0; np < NMAX; ++np) {
          if (np >= N) break;
          const int lo = n < np ? n : np, hi = n < np ? np : n;
          const int pidx = lo * N - lo * (lo - 1) / 2 + (hi - lo);
          hsum += (n == np ? (T)2 : (T)M_SQRT2) * X[pidx * L1 + l] * cc[np];
        }
        H[n * NLM + lm] = hsum;
      }
    }
  }
  wave_sync();
  // pair chunks: Xa[j][lm] = sum_n R_n(j) H(n, lm), Xb[j][lm] = sum_n R_n'(j) H(n, lm)
  T* Xa = C;                       // overlays C and the start of U (C is dead now)
  T* Xb = Xa + CH * NLM;
  T* Rr = Xb + CH * NLM;           // [CH][NMAX] stacked radial values, zero outside the block
  T* dRr = Rr + CH * NMAX;
  T hreg[2][NMAX];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int lm = lane + 64 * h;
#pragma unroll
    for (int n = 0; n < NMAX; ++n) hreg[h][n] = (lm < NLM && n < N) ? H[n * NLM + lm] : (T)0;
  }
  T s0 = 0, s1 = 0, s2 = 0;
  for (int k0 = 1; k0 < nn; k0 += CH) {
    const int cnt = min(CH, nn - k0);
    // 1) pair quads: radial values and derivatives
    int s = -1;
    T r = 0, ux = 0, uy = 0, uz = 0;
    int64_t p = 0;
    wave_sync();
    if (pj < cnt) {
      p = b0 + k0 + pj;
      s = a.pr_spec[p];
      const double rr = a.pr_r[p];
      if (s >= 0 && !(rr < P.sp[s].rc)) s = -1;
      T* rr_ = Rr + pj * NMAX;
      T* dr_ = dRr + pj * NMAX;
      for (int n = sub; n < NMAX; n += 4) { rr_[n] = 0; dr_[n] = 0; }
      if (s >= 0) {
        r = (T)rr;
        const T inv = (T)1 / r;
        ux = (T)a.pr_xyz[3 * p] * inv; uy = (T)a.pr_xyz[3 * p + 1] * inv; uz = (T)a.pr_xyz[3 * p + 2] * inv;
        T R[TGX_MAX_NB], dR[TGX_MAX_NB];
        radial_lanes<T, true, 4, TGX_MAX_NB>(P.sp[s], tb.xq + s * TGX_MAX_Q, tb.Bt + s * TGX_MAX_Q * TGX_MAX_NB, sub, r,
                                             R, dR);
        const int off = P.sp[s].off, nb = P.sp[s].nb;
        wave_sync();  // the quad's zeros before its values
        if (sub == 0)
#pragma unroll
          for (int n = 0; n < TGX_MAX_NB; ++n)
            if (n < nb) { rr_[off + n] = R[n]; dr_[off + n] = dR[n]; }
      }
    }
    wave_sync();
    // 2) lm lanes: Xa, Xb for every pair of the chunk
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int lm = lane + 64 * h;
      if (lm < NLM)
        for (int j = 0; j < cnt; ++j) {
          const T* rj = Rr + j * NMAX;
          const T* dj = dRr + j * NMAX;
          T xa = 0, xb = 0;
#pragma unroll
          for (int n = 0; n < NMAX; ++n) {
            xa += rj[n] * hreg[h][n];
            xb += dj[n] * hreg[h][n];
          }
          Xa[j * NLM + lm] = xa;
          Xb[j * NLM + lm] = xb;
        }
    }
    wave_sync();
    // 3) pair quads: contract with the harmonics and their gradients
    T f0 = 0, f1 = 0, f2 = 0;
    if (pj < cnt && s >= 0) {
      const T inv_r = (T)1 / r;
      Damp<T> dmp;
      dmp.init(P.sp[s], r);
      const T* xa = Xa + pj * NLM;
      const T* xb = Xb + pj * NLM;
      ylm_lanes<T, true, 4>(L, tb.ynorm, sub, ux, uy, uz, dmp.e2, [&](int l, int lm, T A, T Y, T gx, T gy, T gz) {
        const T x = xa[lm], y = xb[lm];
        const T Ax = A * x, lf = (T)l;
        const T ang = Ax * inv_r;
        // rad Y u + ang (grad - l Y u), rad = A' x + A y
        const T t = (Ax * (lf * (lf + (T)1) * dmp.dk) + A * y - ang * lf) * Y;
        f0 += t * ux + ang * gx;
        f1 += t * uy + ang * gy;
        f2 += t * uz + ang * gz;
      });
      f0 = lanes_sum<4>(f0);
      f1 = lanes_sum<4>(f1);
      f2 = lanes_sum<4>(f2);
    }
    if (pj < cnt && sub == 0) {
      const int64_t gi = a.pr_gidx[p];
      fglob[3 * gi] += (double)f0;
      fglob[3 * gi + 1] += (double)f1;
      fglob[3 * gi + 2] += (double)f2;
    } else {
      f0 = f1 = f2 = 0;  // one lane of a quad carries the pair into the self entry's sum
    }
    s0 += f0;
    s1 += f1;
    s2 += f2;
  }
  const double d0 = wave_sum<double>((double)s0), d1 = wave_sum<double>((double)s1), d2 = wave_sum<double>((double)s2);
  if (lane == 0) {
    const int64_t gi = a.pr_gidx[b0];
    fglob[3 * gi] -= d0;
    fglob[3 * gi + 1] -= d1;
    fglob[3 * gi + 2] -= d2;
  }
}

}  // namespace

static WaveArgs wave_args(tgx_model_t* m) {
  WaveArgs a;
  a.site_beg = m->site_beg.as<int64_t>();
  a.pr_spec = m->pr_spec.as<int>();
  a.pr_r = m->pr_r.as<double>();
  a.pr_xyz = m->pr_xyz.as<double>();
  a.pr_gidx = m->pr_gidx.as<int64_t>();
  return a;
}

template <class T> static size_t wave_lds(const SoapParams& P, int CH, int NMAX, bool adjoint) {
  return sizeof(T) * ((size_t)Tables<T>::size(P.n_species, P.NLM) +
                      (size_t)WAVES * WaveLayout<T>::per_wave(CH, NMAX, P, adjoint)) + 64;
}

// CH pairs per pass: 16. NMAX (stacked radial functions held per lane) is the
// smallest of 8, 16, 32 that covers N.
template <class T, int NMAX>
static int launch_desc(tgx_ctx* ctx, tgx_model_t* m, const int* d_sites, int n_rows, void* q_out, void* pn_out,
                       const char* name) {
  WaveArgs a = wave_args(m);
  const size_t lds = wave_lds<T>(m->P, 16, NMAX, false);
  TGX_REQUIRE(lds <= 160 * 1024, "descriptor kernel needs %zu bytes of LDS", lds);
  TGX_LAUNCH(ctx, name, (k_desc_wave<T, 16, NMAX>), dim3((n_rows + WAVES - 1) / WAVES), dim3(64 * WAVES), lds, m->P,
             a, n_rows, (T*)q_out, (T*)pn_out, d_sites);
  return TGX_OK;
}

template <class T, int NMAX>
static int launch_adj(tgx_ctx* ctx, tgx_model_t* m, const T* q, const T* pn, const T* qss, const char* name) {
  WaveArgs a = wave_args(m);
  const int ns = m->n_sites_b;
  const size_t lds = wave_lds<T>(m->P, 16, NMAX, true);
  TGX_REQUIRE(lds <= 160 * 1024, "adjoint kernel needs %zu bytes of LDS", lds);
  TGX_LAUNCH(ctx, name, (k_adjoint_wave<T, 16, NMAX>), dim3((ns + WAVES - 1) / WAVES), dim3(64 * WAVES), lds, m->P, a,
             ns, q, pn, qss, ctx->fglob.as<double>());
  return TGX_OK;
}

int tgx_desc_wave(tgx_ctx* ctx, tgx_model_t* m, bool fp64, const int* d_sites, int n_rows, void* q_out, void* pn_out) {
  if (n_rows == 0) return TGX_OK;
  const int N = m->P.N;
  if (fp64) {
    const char* nm = d_sites ? "soap_desc_list_f64" : "soap_desc_f64";
    if (N <= 8) return launch_desc<double, 8>(ctx, m, d_sites, n_rows, q_out, pn_out, nm);
    if (N <= 16) return launch_desc<double, 16>(ctx, m, d_sites, n_rows, q_out, pn_out, nm);
    return launch_desc<double, 32>(ctx, m, d_sites, n_rows, q_out, pn_out, nm);
  }
  if (N <= 8) return launch_desc<float, 8>(ctx, m, d_sites, n_rows, q_out, pn_out, "soap_desc_f32");
  if (N <= 16) return launch_desc<float, 16>(ctx, m, d_sites, n_rows, q_out, pn_out, "soap_desc_f32");
  return launch_desc<float, 32>(ctx, m, d_sites, n_rows, q_out, pn_out, "soap_desc_f32");
}

int tgx_adjoint_wave(tgx_ctx* ctx, tgx_model_t* m, bool fp64) {
  if (m->n_sites_b == 0) return TGX_OK;
  const int N = m->P.N;
  if (fp64) {
    // a compressed block contracts the full-size gradient with the full descriptors
    const double* q = (m->compress ? m->qf64 : m->q64).as<double>();
    const double* g = (m->compress ? m->qssf64 : m->qss64).as<double>();
    const double* pn = m->pnorm.as<double>();
    if (N <= 8) return launch_adj<double, 8>(ctx, m, q, pn, g, "soap_adjoint_f64");
    if (N <= 16) return launch_adj<double, 16>(ctx, m, q, pn, g, "soap_adjoint_f64");
    return launch_adj<double, 32>(ctx, m, q, pn, g, "soap_adjoint_f64");
  }
  const float *q = m->q32.as<float>(), *pn = m->pnorm.as<float>(), *g = m->qss32.as<float>();
  if (N <= 8) return launch_adj<float, 8>(ctx, m, q, pn, g, "soap_adjoint_f32");
  if (N <= 16) return launch_adj<float, 16>(ctx, m, q, pn, g, "soap_adjoint_f32");
  return launch_adj<float, 32>(ctx, m, q, pn, g, "soap_adjoint_f32");
}
