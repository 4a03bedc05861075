// GAP kernel contraction on the matrix cores (src/gap.f90:115-186):
//   K    = q . Qs^T                       (n_sites x n_sparse, k = D)
//   E_i  = delta^2 sum_s alpha_s K_is^zeta + e0
//   Kd   = -zeta delta^2 K^(zeta-1) o alpha
//   Qss  = Kd . Qs                        (n_sites x D, k = n_sparse)  = -dE/dq
// Both products are "NT" GEMMs (both operands contiguous along k): Qs is kept
// as [S][D] for the first and transposed [D][S] for the second, uploaded once.
//
// FP64: v_mfma_f64_16x16x4f64. BF16: v_mfma_f32_16x16x32_bf16 with FP32
// accumulation; the epilogue keeps the energy row sums in FP64.
// Workgroup tile 128x128, four wavefronts of 64x64 (4x4 MFMA tiles each).
// Tiles are handed out XCD-aware: the eight XCDs each walk a contiguous run of
// tiles in groups of eight tile rows, column by column inside a group, so that
// the tiles one XCD has in flight share their A and B panels in its L2.
#include "tgx_internal.h"

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int BM = 128, BN = 128;
constexpr int TILE_GM = 8;  // tile rows per group of the GEMM tile order (tile_of)

enum { EPI_STORE = TGX_EPI_STORE_F32, EPI_GAP = 1, EPI_SILU = TGX_EPI_SILU, EPI_SCALE_AUX = TGX_EPI_SCALE_AUX,
       EPI_ACT2 = TGX_EPI_ACT2 };

struct EpiArgs {
  double pref;           // -zeta delta^2 (EPI_GAP) / output scale (EPI_STORE, EPI_SCALE_AUX)
  double zeta;
  int zeta_int;          // >= 0 when zeta is an integer
  const double* alpha;   // [N] (FP64 path)
  const float* alpha_f;  // [N] (BF16 path)
  void* out;             // Kd, Qss or the MLP output
  int ldo;
  double* epart;         // [M][n_tiles] (EPI_GAP)
  int n_tiles;
  const float* bias;     // [N] (EPI_SILU)
  float* aux;            // silu'(v) written by EPI_SILU, read by EPI_SCALE_AUX
  int ldaux;
  int64_t sA, sB, sOut, sAux, sBias;  // per-blockIdx.z element strides
  const float* zscale;   // per-z scale (EPI_SCALE_AUX), or null for pref
  const float* w3;       // [N] output weights (EPI_ACT2)
  int64_t sW3, sEpart;   // per-blockIdx.z strides of w3 and epart
};

// GM > 1: inside its range an XCD walks groups of GM tile rows column by
// column, so that the tiles it has in flight at once share their A and B
// panels GM ways each (instead of one row of tiles sharing A only).
template <int GM = 1>
__device__ __forceinline__ void tile_of(int& tm, int& tn) {
  const int ntn = gridDim.x, ntm = gridDim.y;
  const int total = ntn * ntm;
  const int lin = blockIdx.x + ntn * blockIdx.y;
  const int xcd = lin & 7, local = lin >> 3;
  // tiles with lin % 8 == x go to XCD x; give each XCD a contiguous range
  const int base = total / 8, rem = total % 8;
  const int start = xcd * base + (xcd < rem ? xcd : rem);
  const int tile = start + local;
  if (GM == 1) {
    tm = tile / ntn;
    tn = tile - tm * ntn;
  } else {
    const int group = tile / (GM * ntn), first = group * GM;
    const int gm = min(ntm - first, GM), in = tile - first * ntn;
    tm = first + in % gm;
    tn = in / gm;
  }
}

template <class T, bool ZINT>
__device__ __forceinline__ void kpow(T k, double zeta, int zi, T& kz, T& kzm1) {
  if (ZINT) {
    T p = 1;
    for (int i = 0; i < zi - 1; ++i) p *= k;
    kzm1 = p;
    kz = p * k;
  } else {
    kzm1 = (T)pow((double)k, zeta - 1.0);
    kz = (T)pow((double)k, zeta);
  }
}

// FP64 epilogue. acc holds, for tile (ti, tj) and register r, the element
// (row0 + ti*16 + 4*r + lane/16, col0 + tj*16 + lane%16) (the register-major
// layout of v_mfma_f64_16x16x4f64, checked against a host GEMM on the device).
__device__ __forceinline__ int tile_row(int lane, int r) { return 4 * r + (lane >> 4); }

// TI x TJ MFMA tiles of 16 x 16 per wavefront (a WM x WN wave tile), the
// workgroup tile BMT rows tall with two wavefronts along N.
template <int EPI, bool ZINT, int TI, int TJ, int WM, int WN, int BMT>
__device__ __forceinline__ void epilogue_f64(const f64x4 (&acc)[TI][TJ], int m0, int n0, int tn, int wm, int wn,
                                             const EpiArgs& e, double* sE) {
  const int lane = threadIdx.x & 63;
  const int rbase = m0 + wm * WM;
  const int cbase = n0 + wn * WN + (lane & 15);
  double* out = reinterpret_cast<double*>(e.out);
  if (EPI == EPI_STORE) {
#pragma unroll
    for (int ti = 0; ti < TI; ++ti)
#pragma unroll
      for (int tj = 0; tj < TJ; ++tj)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[(size_t)(rbase + ti * 16 + tile_row(lane, r)) * e.ldo + cbase + tj * 16] = e.pref * acc[ti][tj][r];
    return;
  }
  // one 16-row slab at a time keeps only four row partials live
#pragma unroll
  for (int ti = 0; ti < TI; ++ti) {
    double er[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int tj = 0; tj < TJ; ++tj) {
      const int col = cbase + tj * 16;
      const double al = e.alpha[col];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double kz, kzm1;
        kpow<double, ZINT>(acc[ti][tj][r], e.zeta, e.zeta_int, kz, kzm1);
        out[(size_t)(rbase + ti * 16 + tile_row(lane, r)) * e.ldo + col] = e.pref * kzm1 * al;
        er[r] += al * kz;
      }
    }
    // reduce over the 16 lanes that share rows
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double v = er[r];
      v += __shfl_xor(v, 1);
      v += __shfl_xor(v, 2);
      v += __shfl_xor(v, 4);
      v += __shfl_xor(v, 8);
      if ((lane & 15) == 0) sE[wn * BMT + wm * WM + ti * 16 + tile_row(lane, r)] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x < BMT) {
    const int row = m0 + threadIdx.x;
    e.epart[(size_t)row * e.n_tiles + tn] = sE[threadIdx.x] + sE[BMT + threadIdx.x];
  }
}

// BF16 epilogues (FP32 accumulators), in two layouts.
// Straight, v_mfma(A, B): register r of tile (ti, tj) is the element (row0 + ti*16
// + 4*(lane/16) + r, col0 + tj*16 + lane%16), so that a store instruction writes
// 64-byte runs of FP32; for the epilogues with an FP32 output or factor.
// Exchanged, v_mfma(B, A): a lane's four registers are four consecutive columns
// of one row, row0 + ti*16 + lane%16, columns col0 + tj*16 + 4*(lane/16) + r; for
// the epilogues that write BF16 only and sum rows: 8-byte stores instead of four
// 2-byte ones and two shuffles a row sum instead of four a register (GAP product
// 32,768 x 4,096 x 1,280: 0.431 -> 0.402 ms; exchanged, the FP32 stores of the
// 32,768 x 1,280 x 768 product cost 0.095 ms against 0.082).
template <int EPI> constexpr bool exchanged() { return EPI == EPI_GAP || EPI == EPI_ACT2; }

template <int EPI>
__device__ __forceinline__ f32x4 mfma_bf16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
  return exchanged<EPI>() ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0)
                          : __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// TI x 4 MFMA tiles per wavefront (a WM x 64 wave tile), the workgroup tile BMT
// rows tall with two wavefronts along N.
template <int EPI, class OutT, bool ZINT, int TI, int WM, int BMT>
__device__ __forceinline__ void epilogue_bf16(const f32x4 (&acc)[TI][4], int m0, int n0, int tn, int wm, int wn,
                                              const EpiArgs& e, double* sE) {
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  OutT* out = reinterpret_cast<OutT*>(e.out);
  const float pref = (float)e.pref;
  if constexpr (!exchanged<EPI>()) {
    const int rbase = m0 + wm * WM + 4 * lg, cbase = n0 + wn * 64 + li;
#pragma unroll
    for (int ti = 0; ti < TI; ++ti)
#pragma unroll
      for (int tj = 0; tj < 4; ++tj) {
        const int col = cbase + tj * 16;
        const float b = EPI == EPI_SILU ? e.bias[col] : 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const size_t row = (size_t)(rbase + ti * 16 + r);
          const float x = acc[ti][tj][r];
          if constexpr (EPI == EPI_SILU) {
            out[row * e.ldo + col] = (OutT)tgx_silu(x + b);
            e.aux[row * e.ldaux + col] = tgx_silu1(x + b);
          } else if constexpr (EPI == EPI_SCALE_AUX) {
            out[row * e.ldo + col] = (OutT)(x * e.aux[row * e.ldaux + col] * pref);
          } else {
            out[row * e.ldo + col] = (OutT)(pref * x);
          }
        }
      }
    return;
  } else {
    const int cbase = n0 + wn * 64 + 4 * lg;
#pragma unroll
    for (int ti = 0; ti < TI; ++ti) {
      const int trow = wm * WM + ti * 16 + li;
      const size_t row = (size_t)(m0 + trow);
      double er = 0.0;
#pragma unroll
      for (int tj = 0; tj < 4; ++tj) {
        const int col = cbase + tj * 16;
        const f32x4 x = acc[ti][tj];
        bf16x4 o;
        if constexpr (EPI == EPI_ACT2) {
          // a2 = w3 silu'(v) out, and the row sums of w3 silu(v) over the tile's
          // columns as partial energies (as the GAP epilogue's)
          const f32x4 b = load4(e.bias + col), w3 = load4(e.w3 + col);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float v = x[r] + b[r];
            o[r] = (__bf16)(w3[r] * tgx_silu1(v));
            er += (double)(w3[r] * tgx_silu(v));
          }
        } else {
          const f32x4 al = load4(e.alpha_f + col);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            float kz, kzm1;
            kpow<float, ZINT>(x[r], e.zeta, e.zeta_int, kz, kzm1);
            o[r] = (__bf16)(pref * kzm1 * al[r]);
            er += (double)(al[r] * kz);
          }
        }
        *reinterpret_cast<bf16x4*>(out + row * e.ldo + col) = o;
      }
      er += __shfl_xor(er, 16);
      er += __shfl_xor(er, 32);
      if (lane < 16) sE[wn * BMT + trow] = er;
    }
    __syncthreads();
    if (threadIdx.x < BMT) {
      const int row = m0 + threadIdx.x;
      e.epart[(size_t)row * e.n_tiles + tn] = sE[threadIdx.x] + sE[BMT + threadIdx.x];
    }
  }
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 16, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x3F70 | N);  // vmcnt(N); expcnt and lgkmcnt not waited on
}

// The same, and every LDS read of this wavefront is done.
template <int N>
__device__ __forceinline__ void wait_vmcnt_lds() {
  static_assert(N >= 0 && N < 16, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt(0x0070 | N);
}

// FP64 NT GEMM fed by direct global-to-LDS loads: workgroup tile (32 TI) x
// (32 TJ), four wavefronts of (16 TI) x (16 TJ), BK = 16 in a two-slot ring. A
// stage is 32 (TI + TJ) rows of 128 bytes (the A rows, then the B rows); the
// eight 16-byte chunks of row r sit at chunk c ^ (r & 7), so that a 16-byte
// fragment read spreads over all banks. One load instruction fills eight rows.
// A lane's chunk holds two consecutive k, which go to two MFMAs: the k of both
// operands are permuted alike, so the product is the same. Each half stage's
// fragments are read into registers while the other half's MFMAs run, and the
// one barrier a stage sits between the halves: without it, the two workgroups
// of a CU reach their fragment waits and barriers together and the matrix
// cores idle. Bound by the FP64 MFMA rate.
// M a multiple of 32 TI, N of 32 TJ, K of 16.
__host__ __device__ constexpr int f64_stage_bytes(int ti, int tj) { return 32 * (ti + tj) * 128; }
__host__ __device__ constexpr int f64_lds_bytes(int ti, int tj) { return 2 * f64_stage_bytes(ti, tj) + 2 * 32 * ti * 8; }

template <int TI, int TJ>
__device__ __forceinline__ void f64_read(const unsigned char* sb, int aoff, int boff, int cpos, double2 (&a)[TI],
                                         double2 (&b)[TJ]) {
#pragma unroll
  for (int i = 0; i < TI; ++i) a[i] = *reinterpret_cast<const double2*>(sb + aoff + i * 16 * 128 + cpos);
#pragma unroll
  for (int j = 0; j < TJ; ++j) b[j] = *reinterpret_cast<const double2*>(sb + boff + j * 16 * 128 + cpos);
}

template <int TI, int TJ>
__device__ __forceinline__ void f64_mfma(f64x4 (&acc)[TI][TJ], const double2 (&a)[TI], const double2 (&b)[TJ]) {
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].x, b[j].x, acc[i][j], 0, 0, 0);
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i].y, b[j].y, acc[i][j], 0, 0, 0);
}

template <int EPI, bool ZINT, int TI, int TJ, int OCC>
__global__ __launch_bounds__(256, OCC) void k_gemm_f64(int K, const double* __restrict__ A, int lda,
                                                       const double* __restrict__ B, int ldb, EpiArgs e) {
  constexpr int BK = 16, SB = f64_stage_bytes(TI, TJ);
  constexpr int NBA = 4 * TI, P = TI + TJ;  // load blocks of eight rows: A's, and per wavefront
  extern __shared__ __align__(16) unsigned char dsm[];
  double* sE = reinterpret_cast<double*>(dsm + 2 * SB);
  int tm, tn;
  tile_of<TILE_GM>(tm, tn);
  const int m0 = tm * 32 * TI, n0 = tn * 32 * TJ;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
  const double* src[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int b = w + 4 * j;
    src[j] = b < NBA ? A + (size_t)(m0 + 8 * b + lrow) * lda + 2 * lchunk
                     : B + (size_t)(n0 + 8 * (b - NBA) + lrow) * ldb + 2 * lchunk;
  }
  auto issue = [&](int st, int slot) {
#pragma unroll
    for (int j = 0; j < P; ++j)
      __builtin_amdgcn_global_load_lds(const_cast<double*>(src[j] + st * BK), dsm + slot * SB + (w + 4 * j) * 1024, 16,
                                       0, 0);
  };
  const int li = lane & 15, lg = lane >> 4;
  const int aoff = (wm * 16 * TI + li) * 128, boff = (32 * TI + wn * 16 * TJ + li) * 128;
  const int c0 = (lg ^ (li & 7)) << 4, c1 = ((lg + 4) ^ (li & 7)) << 4;
  f64x4 acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = (f64x4){0, 0, 0, 0};
  const int n_stages = K / BK;
  issue(0, 0);
  wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  issue(min(1, n_stages - 1), 1);
  double2 a0[TI], b0[TJ], a1[TI], b1[TJ];
  f64_read<TI, TJ>(dsm, aoff, boff, c0, a0, b0);
  for (int st = 0; st < n_stages; ++st) {
    const int slot = st & 1;
    f64_read<TI, TJ>(dsm + slot * SB, aoff, boff, c1, a1, b1);
    __builtin_amdgcn_sched_barrier(0);
    f64_mfma<TI, TJ>(acc, a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    // this wavefront's part of stage st + 1 has landed and its reads of stage st are done
    wait_vmcnt_lds<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    issue(min(st + 2, n_stages - 1), slot);  // an in-bounds repeat past the end
    f64_read<TI, TJ>(dsm + (slot ^ 1) * SB, aoff, boff, c0, a0, b0);
    __builtin_amdgcn_sched_barrier(0);
    f64_mfma<TI, TJ>(acc, a1, b1);
  }
  wait_vmcnt<0>();  // the loads issued past the last stage land before the LDS is released
  __builtin_amdgcn_sched_barrier(0);
  epilogue_f64<EPI, ZINT, TI, TJ, 16 * TI, 16 * TJ, 32 * TI>(acc, m0, n0, tn, wm, wn, e, sE);
}

// FP64 NT GEMM for few rows: workgroup tile 32 x (32 NC), NC x KS wavefronts of
// 32 x 32 that each take a K / KS range straight from global memory (nothing is
// shared, so nothing is staged), and the KS partials are added through LDS in
// order. A handful of 128 x 128 tiles would each walk the whole K alone: the
// reduction is what fills the chip there. M a multiple of 32, N of 32 NC, K of
// 16 KS.
template <int EPI, bool ZINT, int NC, int KS>
__global__ __launch_bounds__(64 * NC * KS) void k_gemm_f64_few(int K, const double* __restrict__ A, int lda,
                                                               const double* __restrict__ B, int ldb, EpiArgs e) {
  extern __shared__ __align__(16) unsigned char dsm[];
  double* part = reinterpret_cast<double*>(dsm);  // [KS][32][32 NC]
  constexpr int W = 32 * NC;
  int tm, tn;
  tile_of<TILE_GM>(tm, tn);
  const int m0 = tm * 32, n0 = tn * W;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wc = w % NC, wk = w / NC, kr = K / KS;
  const int li = lane & 15, lg = lane >> 4;
  const double* Ap = A + (size_t)(m0 + li) * lda + wk * kr + 2 * lg;
  const double* Bp = B + (size_t)(n0 + 32 * wc + li) * ldb + wk * kr + 2 * lg;
  const size_t a16 = (size_t)16 * lda, b16 = (size_t)16 * ldb;
  f64x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f64x4){0, 0, 0, 0};
  // DEPTH rounds of 16 k in flight: two waves per SIMD do not cover a load's latency
  constexpr int DEPTH = 4;
  double2 a[DEPTH][2][2], b[DEPTH][2][2];
  const int rounds = kr / 16;
  auto load = [&](int it, double2(&ra)[2][2], double2(&rb)[2][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = 16 * it + 8 * h;
      ra[h][0] = *reinterpret_cast<const double2*>(Ap + k);
      ra[h][1] = *reinterpret_cast<const double2*>(Ap + a16 + k);
      rb[h][0] = *reinterpret_cast<const double2*>(Bp + k);
      rb[h][1] = *reinterpret_cast<const double2*>(Bp + b16 + k);
    }
  };
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) load(min(u, rounds - 1), a[u], b[u]);
  for (int it = 0; it < rounds; it += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      if (it + u < rounds) {
        f64_mfma<2, 2>(acc, a[u][0], b[u][0]);
        f64_mfma<2, 2>(acc, a[u][1], b[u][1]);
      }
      load(min(it + u + DEPTH, rounds - 1), a[u], b[u]);  // in bounds past the end
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        part[(wk * 32 + i * 16 + tile_row(lane, r)) * W + 32 * wc + j * 16 + li] = acc[i][j][r];
  __syncthreads();
  // thread: row tid / TR, columns tid % TR + TR c
  constexpr int TR = 2 * NC * KS, CP = W / TR;
  static_assert(W % TR == 0 && TR <= 64, "columns per thread");
  const int row = tid / TR, c0 = tid % TR;
  double er = 0.0;
#pragma unroll
  for (int c = 0; c < CP; ++c) {
    const int col = c0 + c * TR;
    double v = part[row * W + col];
#pragma unroll
    for (int k = 1; k < KS; ++k) v += part[(k * 32 + row) * W + col];
    double* o = reinterpret_cast<double*>(e.out) + (size_t)(m0 + row) * e.ldo + n0 + col;
    if (EPI == EPI_GAP) {
      const double al = e.alpha[n0 + col];
      double kz, kzm1;
      kpow<double, ZINT>(v, e.zeta, e.zeta_int, kz, kzm1);
      *o = e.pref * kzm1 * al;
      er += al * kz;
    } else {
      *o = e.pref * v;
    }
  }
  if (EPI == EPI_GAP) {
#pragma unroll
    for (int x = 1; x < TR; x <<= 1) er += __shfl_xor(er, x);
    if (c0 == 0) e.epart[(size_t)(m0 + row) * e.n_tiles + tn] = er;
  }
}

// BF16 NT GEMM with FP32 accumulation. M, N multiples of 128; K multiple of 64.
// Two LDS stages: the global loads of stage k+1 are in flight while the MFMAs
// of stage k run, and one barrier per stage separates the LDS write of k+1
// from the reads of k. Each thread moves four 16-byte chunks per operand and
// stage: chunk t%8 of rows t/8 + 32 j, so a wavefront reads eight full 128-byte
// row segments per load. The next-stage offset is clamped to the last stage
// (a redundant, in-bounds reload) so the staging registers are written on
// every iteration and never demoted to private memory.
template <int EPI, class OutT, bool ZINT>
__global__ __launch_bounds__(256) void k_gemm_bf16(int K, const __bf16* __restrict__ A, int lda,
                                                   const __bf16* __restrict__ B, int ldb, EpiArgs e) {
  constexpr int BK = 64, LDS_STRIDE = BK + 8;  // 144-byte row pitch: conflict-free 16-byte reads
  __shared__ __align__(16) __bf16 As[2][BM * LDS_STRIDE];
  __shared__ __align__(16) __bf16 Bs[2][BN * LDS_STRIDE];
  __shared__ double sE[2 * BM];
  int tm, tn;
  tile_of<TILE_GM>(tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int lr = tid >> 3, lc = (tid & 7) * 8;
  {
    const int z = blockIdx.z;  // batch member: offset every operand
    A += z * e.sA;
    B += z * e.sB;
    e.out = reinterpret_cast<OutT*>(e.out) + z * e.sOut;
    if (e.aux) e.aux += z * e.sAux;
    if (e.bias) e.bias += z * e.sBias;
    if (e.w3) e.w3 += z * e.sW3;
    if (e.epart) e.epart += z * e.sEpart;
    if (e.zscale) e.pref = e.zscale[z];
  }
  const __bf16* Ag = A + (size_t)(m0 + lr) * lda + lc;
  const __bf16* Bg = B + (size_t)(n0 + lr) * ldb + lc;
  const size_t a32 = (size_t)32 * lda, b32 = (size_t)32 * ldb;
  // The scaled epilogue's factors are read before the main loop, so that their
  // latency overlaps it (a short K leaves the epilogue most of the time; the
  // 64 registers fit in the two waves per SIMD that the LDS allows)
  float auxv[4][4][4];
  if constexpr (EPI == EPI_SCALE_AUX) {
    const int rb = m0 + wm * 64 + 4 * (lane >> 4), cb = n0 + wn * 64 + (lane & 15);
#pragma unroll
    for (int tj = 0; tj < 4; ++tj)
#pragma unroll
      for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) auxv[ti][tj][r] = e.aux[(size_t)(rb + ti * 16 + r) * e.ldaux + cb + tj * 16];
  }
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0, 0, 0, 0};
  uint4 ra0, ra1, ra2, ra3, rb0, rb1, rb2, rb3;
  auto gload = [&](int k) {
    ra0 = *reinterpret_cast<const uint4*>(Ag + k);
    ra1 = *reinterpret_cast<const uint4*>(Ag + a32 + k);
    ra2 = *reinterpret_cast<const uint4*>(Ag + 2 * a32 + k);
    ra3 = *reinterpret_cast<const uint4*>(Ag + 3 * a32 + k);
    rb0 = *reinterpret_cast<const uint4*>(Bg + k);
    rb1 = *reinterpret_cast<const uint4*>(Bg + b32 + k);
    rb2 = *reinterpret_cast<const uint4*>(Bg + 2 * b32 + k);
    rb3 = *reinterpret_cast<const uint4*>(Bg + 3 * b32 + k);
  };
  auto lstore = [&](int buf) {
    __bf16* as = &As[buf][lr * LDS_STRIDE + lc];
    __bf16* bs = &Bs[buf][lr * LDS_STRIDE + lc];
    *reinterpret_cast<uint4*>(as) = ra0;
    *reinterpret_cast<uint4*>(as + 32 * LDS_STRIDE) = ra1;
    *reinterpret_cast<uint4*>(as + 64 * LDS_STRIDE) = ra2;
    *reinterpret_cast<uint4*>(as + 96 * LDS_STRIDE) = ra3;
    *reinterpret_cast<uint4*>(bs) = rb0;
    *reinterpret_cast<uint4*>(bs + 32 * LDS_STRIDE) = rb1;
    *reinterpret_cast<uint4*>(bs + 64 * LDS_STRIDE) = rb2;
    *reinterpret_cast<uint4*>(bs + 96 * LDS_STRIDE) = rb3;
  };
  gload(0);
  lstore(0);
  __syncthreads();
  const int n_stages = K / BK;
  for (int st = 0; st < n_stages; ++st) {
    const int buf = st & 1;
    const int kn = min(st + 1, n_stages - 1) * BK;
    gload(kn);
    __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the MFMAs they overlap
    const __bf16* as = &As[buf][(wm * 64 + (lane & 15)) * LDS_STRIDE + 8 * (lane >> 4)];
    const __bf16* bs = &Bs[buf][(wn * 64 + (lane & 15)) * LDS_STRIDE + 8 * (lane >> 4)];
#pragma unroll
    for (int ks = 0; ks < BK / 32; ++ks) {
      bf16x8 a[4], b[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        a[t] = *reinterpret_cast<const bf16x8*>(as + t * 16 * LDS_STRIDE + ks * 32);
        b[t] = *reinterpret_cast<const bf16x8*>(bs + t * 16 * LDS_STRIDE + ks * 32);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma_bf16<EPI>(a[i], b[j], acc[i][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    lstore(buf ^ 1);
    __syncthreads();
  }
  if constexpr (EPI == EPI_SCALE_AUX) {
    OutT* out = reinterpret_cast<OutT*>(e.out);
    const int rb = m0 + wm * 64 + 4 * (lane >> 4), cb = n0 + wn * 64 + (lane & 15);
#pragma unroll
    for (int tj = 0; tj < 4; ++tj)
#pragma unroll
      for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          out[(size_t)(rb + ti * 16 + r) * e.ldo + cb + tj * 16] =
              (OutT)(acc[ti][tj][r] * auxv[ti][tj][r] * (float)e.pref);
  } else {
    epilogue_bf16<EPI, OutT, ZINT, 4, 64, BM>(acc, m0, n0, tn, wm, wn, e, sE);
  }
}

// BF16 NT GEMM fed by direct global-to-LDS loads (global_load_lds_dwordx4):
// workgroup tile TM x 128, four wavefronts of (TM / 2) x 64, BK = 32, an
// NS-slot ring of LDS stages. A stage is TM + 128 rows of 64 bytes (the A
// rows, then the B rows); the four 16-byte chunks of row r sit at chunk
// c ^ ((r >> 1) & 3), so that the eight rows a 16-byte fragment read serves
// per cycle cover all 32 banks. One load instruction fills 16 rows (lane l
// writes chunk l & 3 of row l >> 2 and fetches the chunk that belongs there);
// nothing is staged through registers. The fragments of each stage are held
// in registers, double-buffered: stage s + 1's fragments are read while stage
// s's MFMAs run, so a ring slot is free as soon as every wavefront has read it
// and stage s + NS is loaded into stage s's slot right after the barrier of
// iteration s (NS stages in flight). Iteration s: the MFMAs of the first half
// of the tile rows, then (vmcnt: this wavefront's part of stage s + 1 landed)
// the barrier, the loads of stage s + NS and the fragment reads of stage
// s + 1, then the second half of the MFMAs, which cover the reads' latency.
// M a multiple of TM, N of 128, K of 32.
constexpr int DK = 32;                      // k per stage
constexpr int DROW = DK * 2;                // bytes per staged row
__host__ __device__ constexpr int dma_stage_bytes(int tm) { return (tm + BN) * DROW; }
__host__ __device__ constexpr int dma_lds_bytes(int tm, int ns) { return ns * dma_stage_bytes(tm) + 2 * tm * 8; }

// One stage's loads of a wavefront: its P blocks of 16 rows, block b of the
// stage into bytes [1024 b, 1024 b + 1024) of the stage buffer.
template <int P>
__device__ __forceinline__ void dma_issue(const __bf16* const (&src)[P], int k0, unsigned char* stage, int w) {
#pragma unroll
  for (int j = 0; j < P; ++j)
    __builtin_amdgcn_global_load_lds(const_cast<__bf16*>(src[j] + k0), stage + (w + 4 * j) * 1024, 16, 0, 0);
}

template <int TI>
__device__ __forceinline__ void pf_read(const unsigned char* sb, int aoff, int boff, bf16x8 (&a)[TI], bf16x8 (&b)[4]) {
#pragma unroll
  for (int t = 0; t < 4; ++t) b[t] = *reinterpret_cast<const bf16x8*>(sb + boff + t * 16 * DROW);
#pragma unroll
  for (int i = 0; i < TI; ++i) a[i] = *reinterpret_cast<const bf16x8*>(sb + aoff + i * 16 * DROW);
}

template <int EPI, int TI, int I0, int I1>
__device__ __forceinline__ void pf_mfma(f32x4 (&acc)[TI][4], const bf16x8 (&a)[TI], const bf16x8 (&b)[4]) {
#pragma unroll
  for (int i = I0; i < I1; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = mfma_bf16<EPI>(a[i], b[j], acc[i][j]);
}

template <int EPI, int TI, int P, int NS, int SB>
__device__ __forceinline__ void pf_stage(f32x4 (&acc)[TI][4], const bf16x8 (&a)[TI], const bf16x8 (&b)[4],
                                         bf16x8 (&an)[TI], bf16x8 (&bn)[4], const __bf16* const (&src)[P],
                                         unsigned char* dsm, int st, int n_stages, int& slot, int aoff, int boff,
                                         int w) {
  pf_mfma<EPI, TI, 0, TI / 2>(acc, a, b);
  __builtin_amdgcn_sched_barrier(0);
  // this wavefront's part of the next stage has landed, and its reads of this one are done: the
  // products above need only the first half of a
  wait_vmcnt_lds<(NS - 2) * P>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  // every wavefront has read this stage's slot: it takes stage st + NS (an in-bounds repeat past the end)
  dma_issue<P>(src, min(st + NS, n_stages - 1) * DK, dsm + slot * SB, w);
  slot = slot + 1 == NS ? 0 : slot + 1;
  pf_read<TI>(dsm + slot * SB, aoff, boff, an, bn);
  __builtin_amdgcn_sched_barrier(0);
  pf_mfma<EPI, TI, TI / 2, TI>(acc, a, b);
}

template <int EPI, class OutT, bool ZINT, int TM, int NS, int OCC>
__global__ __launch_bounds__(256, OCC) void k_gemm_bf16_pf(int K, const __bf16* __restrict__ A, int lda,
                                                          const __bf16* __restrict__ B, int ldb, EpiArgs e) {
  constexpr int TI = TM / 32;
  constexpr int NBA = TM / 16, NBB = BN / 16;
  constexpr int P = (NBA + NBB) / 4;
  static_assert((NBA + NBB) % 4 == 0, "load blocks per wavefront");
  static_assert(NS >= 3 && (NS - 1) * P < 16, "vmcnt range");
  constexpr int SB = dma_stage_bytes(TM);
  extern __shared__ __align__(16) unsigned char dsm[];
  double* sE = reinterpret_cast<double*>(dsm + NS * SB);
  int tm, tn;
  tile_of<TILE_GM>(tm, tn);
  const int m0 = tm * TM, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  {
    const int z = blockIdx.z;
    A += z * e.sA;
    B += z * e.sB;
    e.out = reinterpret_cast<OutT*>(e.out) + z * e.sOut;
    if (e.aux) e.aux += z * e.sAux;
    if (e.bias) e.bias += z * e.sBias;
    if (e.w3) e.w3 += z * e.sW3;
    if (e.epart) e.epart += z * e.sEpart;
    if (e.zscale) e.pref = e.zscale[z];
  }
  const int lrow = lane >> 2, lchunk = (lane & 3) ^ ((lane >> 3) & 3);
  const __bf16* src[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int b = w + 4 * j;
    src[j] = b < NBA ? A + (size_t)(m0 + 16 * b + lrow) * lda + 8 * lchunk
                     : B + (size_t)(n0 + 16 * (b - NBA) + lrow) * ldb + 8 * lchunk;
  }
  const int li = lane & 15, lg = lane >> 4;
  const int foff = li * DROW + ((lg ^ ((li >> 1) & 3)) << 4);
  const int aoff = wm * (TM / 2) * DROW + foff, boff = TM * DROW + wn * 64 * DROW + foff;
  f32x4 acc[TI][4];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0, 0, 0, 0};
  const int n_stages = K / DK;
#pragma unroll
  for (int s = 0; s < NS; ++s) dma_issue<P>(src, min(s, n_stages - 1) * DK, dsm + s * SB, w);
  wait_vmcnt<(NS - 1) * P>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  bf16x8 a0[TI], b0[4], a1[TI], b1[4];
  pf_read<TI>(dsm, aoff, boff, a0, b0);
  int slot = 0, st = 0;
  for (; st + 1 < n_stages; st += 2) {
    pf_stage<EPI, TI, P, NS, SB>(acc, a0, b0, a1, b1, src, dsm, st, n_stages, slot, aoff, boff, w);
    pf_stage<EPI, TI, P, NS, SB>(acc, a1, b1, a0, b0, src, dsm, st + 1, n_stages, slot, aoff, boff, w);
  }
  if (st < n_stages) pf_stage<EPI, TI, P, NS, SB>(acc, a0, b0, a1, b1, src, dsm, st, n_stages, slot, aoff, boff, w);
  // the loads issued past the last stage land before the workgroup's LDS is released
  wait_vmcnt<0>();
  __builtin_amdgcn_sched_barrier(0);
  epilogue_bf16<EPI, OutT, ZINT, TI, TM / 2, TM>(acc, m0, n0, tn, wm, wn, e, sE);
}

// BF16 NT GEMM for few tiles: workgroup tile (32 TI) x 128, four wavefronts of
// (16 TI) x 64, BK = 64 in a three-slot ring of direct global-to-LDS loads (two
// stages in flight), stages laid out as in k_gemm_f64: rows of 128 bytes with
// chunk c of row r at c ^ (r & 7). Small systems leave 128 x 128 tiles on a
// fraction of the 256 CUs, each walking the whole K alone. M a multiple of 32 TI,
// N of 128, K of 64.
__host__ __device__ constexpr int few_stage_bytes(int ti) { return (32 * ti + BN) * 128; }
__host__ __device__ constexpr int few_lds_bytes(int ti) { return 3 * few_stage_bytes(ti) + 2 * 32 * ti * 8; }

template <int EPI, class OutT, bool ZINT, int TI>
__global__ __launch_bounds__(256, 2) void k_gemm_bf16_few(int K, const __bf16* __restrict__ A, int lda,
                                                          const __bf16* __restrict__ B, int ldb, EpiArgs e) {
  constexpr int SB = few_stage_bytes(TI), NS = 3, P = TI + 4, NBA = 4 * TI;
  extern __shared__ __align__(16) unsigned char dsm[];
  double* sE = reinterpret_cast<double*>(dsm + NS * SB);
  int tm, tn;
  tile_of<TILE_GM>(tm, tn);
  const int m0 = tm * 32 * TI, n0 = tn * BN;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wm = w >> 1, wn = w & 1;
  {
    const int z = blockIdx.z;
    A += z * e.sA;
    B += z * e.sB;
    e.out = reinterpret_cast<OutT*>(e.out) + z * e.sOut;
    if (e.aux) e.aux += z * e.sAux;
    if (e.bias) e.bias += z * e.sBias;
    if (e.w3) e.w3 += z * e.sW3;
    if (e.epart) e.epart += z * e.sEpart;
    if (e.zscale) e.pref = e.zscale[z];
  }
  const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
  const __bf16* src[P];
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int b = w + 4 * j;
    src[j] = b < NBA ? A + (size_t)(m0 + 8 * b + lrow) * lda + 8 * lchunk
                     : B + (size_t)(n0 + 8 * (b - NBA) + lrow) * ldb + 8 * lchunk;
  }
  const int n_stages = K / 64;
  auto issue = [&](int st, int slot) {
    const int k0 = min(st, n_stages - 1) * 64;  // an in-bounds repeat past the end
#pragma unroll
    for (int j = 0; j < P; ++j)
      __builtin_amdgcn_global_load_lds(const_cast<__bf16*>(src[j] + k0), dsm + slot * SB + (w + 4 * j) * 1024, 16, 0, 0);
  };
  const int li = lane & 15, lg = lane >> 4;
  const int aoff = (wm * 16 * TI + li) * 128, boff = (32 * TI + wn * 64 + li) * 128;
  f32x4 acc[TI][4];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4){0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) issue(s, s);
  int slot = 0, fill = NS - 1;
  for (int st = 0; st < n_stages; ++st) {
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<(NS - 2) * P>();  // this wavefront's part of stage st has landed
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    issue(st + NS - 1, fill);  // into the slot that every wavefront read in the last round
    fill = fill + 1 == NS ? 0 : fill + 1;
    const unsigned char* sb = dsm + slot * SB;
    slot = slot + 1 == NS ? 0 : slot + 1;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int cp = ((4 * ks + lg) ^ (li & 7)) << 4;
      bf16x8 a[TI], b[4];
#pragma unroll
      for (int t = 0; t < TI; ++t) a[t] = *reinterpret_cast<const bf16x8*>(sb + aoff + t * 16 * 128 + cp);
#pragma unroll
      for (int t = 0; t < 4; ++t) b[t] = *reinterpret_cast<const bf16x8*>(sb + boff + t * 16 * 128 + cp);
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mfma_bf16<EPI>(a[i], b[j], acc[i][j]);
    }
  }
  wait_vmcnt<0>();  // the loads issued past the last stage land before the LDS is released
  __builtin_amdgcn_sched_barrier(0);
  epilogue_bf16<EPI, OutT, ZINT, TI, 16 * TI, 32 * TI>(acc, m0, n0, tn, wm, wn, e, sE);
}

// E_i = delta^2 sum_t epart[i][t] + e0. 16 lanes a row, lane t adding partials
// t, t + 16, ... in order, then a fixed xor butterfly (one thread a row read its
// 32 partials one line after another: 26 us at 2,048 rows, this 5).
__global__ void k_energy_finalize(int n, const double* __restrict__ epart, int n_tiles, double d2, double e0,
                                  double* __restrict__ e_site) {
  const int t = threadIdx.x & 15;
  const int i = (blockIdx.x * blockDim.x + threadIdx.x) >> 4;
  double s = 0.0;
  if (i < n)
    for (int k = t; k < n_tiles; k += 16) s += epart[(size_t)i * n_tiles + k];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (i < n && t == 0) e_site[i] = d2 * s + e0;
}

__global__ void k_f32_to_bf16(int64_t n, const float* __restrict__ x, __bf16* __restrict__ y) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) y[i] = (__bf16)x[i];
}

}  // namespace

static EpiArgs gap_epi(const tgx_model_t* m) {
  EpiArgs e{};
  const double z = m->zeta;
  const bool zint = std::fabs(z - (double)(int)z) < 1.0e-5;
  e.zeta_int = zint ? (int)z : 0;
  e.zeta = zint ? (double)(int)z : z;
  e.pref = -e.zeta * m->delta * m->delta;
  return e;
}

template <int EPI, class OutT, bool ZINT, int TM, int NS, int OCC>
static int launch_pf(tgx_ctx* ctx, const char* name, int M, int N, int K, int batch, const __bf16* A, int lda,
                     const __bf16* B, int ldb, EpiArgs e) {
  TGX_LAUNCH(ctx, name, (k_gemm_bf16_pf<EPI, OutT, ZINT, TM, NS, OCC>), dim3(N / BN, M / TM, batch), dim3(256),
             dma_lds_bytes(TM, NS), K, A, lda, B, ldb, e);
  return TGX_OK;
}

template <int EPI, class OutT, bool ZINT, int TI>
static int launch_few(tgx_ctx* ctx, const char* name, int M, int N, int K, int batch, const __bf16* A, int lda,
                      const __bf16* B, int ldb, EpiArgs e) {
  TGX_LAUNCH(ctx, name, (k_gemm_bf16_few<EPI, OutT, ZINT, TI>), dim3(N / BN, M / (32 * TI), batch), dim3(256),
             few_lds_bytes(TI), K, A, lda, B, ldb, e);
  return TGX_OK;
}

// BF16 NT GEMM launch, by the number of 128 x 128 tiles t (256 CUs, two or three
// workgroups each), all times alone on the card:
//   t <= 96    32-row tiles (512 x 768 x 1,280, 24 tiles: 0.012 ms, 128-row tiles 0.017-0.023)
//   t < 384    64-row tiles (1,024 x 4,096 x 1,280, 256 tiles: 0.020 against 0.026); plain products with a long
//              K up to 1,023 (8,192 x 1,280 x 4,096, 640 tiles: 0.104 against 0.106-0.117)
//   M a multiple of 256, t >= 1,024: the 256-row direct-load kernel for plain and GAP epilogues (32,768 x 1,280 x
//              4,096: 0.356 ms, 128-row tiles 0.412; GAP 32,768 x 4,096 x 1,280: 0.392 against 0.501)
//   else       the 128-row direct-load kernel for plain, GAP and second-layer epilogues, and the register-staged
//              one for the two that read or write an FP32 factor (32,768 x 256 x 256 x 3 alike at 0.041 ms; beside
//              the other block the 256-row SiLU kernel, faster alone, is not: 0.239 against 0.232)
// The GAP and second-layer epilogues write one energy partial per row and
// 128-column tile whatever the rule.
template <int EPI, class OutT, bool ZINT>
static int launch_bf16(tgx_ctx* ctx, const char* name, int M, int N, int K, int batch, const __bf16* A, int lda,
                       const __bf16* B, int ldb, EpiArgs e) {
  TGX_REQUIRE(M % BM == 0 && N % BN == 0 && K % 64 == 0 && lda % 8 == 0 && ldb % 8 == 0,
              "gemm_bf16 %s: unpadded shape %d x %d x %d", name, M, N, K);
  if constexpr (exchanged<EPI>())  // four columns at a time
    TGX_REQUIRE(e.ldo % 4 == 0 && e.sOut % 4 == 0 && e.sBias % 4 == 0 && e.sW3 % 4 == 0 && (uintptr_t)e.out % 8 == 0 &&
                    ((uintptr_t)e.bias | (uintptr_t)e.w3 | (uintptr_t)e.alpha_f) % 16 == 0,
                "gemm_bf16 %s: misaligned epilogue operands", name);
  const int64_t t = (int64_t)(M / BM) * (N / BN) * batch;
  if (t <= 96) return launch_few<EPI, OutT, ZINT, 1>(ctx, name, M, N, K, batch, A, lda, B, ldb, e);
  if (t < 384 || (EPI == EPI_STORE && K >= 2048 && t < 1024))
    return launch_few<EPI, OutT, ZINT, 2>(ctx, name, M, N, K, batch, A, lda, B, ldb, e);
  if constexpr (EPI == EPI_STORE || EPI == EPI_GAP) {
    if (M % 256 == 0 && t >= 1024)
      return launch_pf<EPI, OutT, ZINT, 256, 3, 2>(ctx, name, M, N, K, batch, A, lda, B, ldb, e);
  }
  if constexpr (EPI == EPI_STORE || EPI == EPI_GAP || EPI == EPI_ACT2) {
    return launch_pf<EPI, OutT, ZINT, 128, 3, 3>(ctx, name, M, N, K, batch, A, lda, B, ldb, e);
  } else {
    TGX_LAUNCH(ctx, name, (k_gemm_bf16<EPI, OutT, ZINT>), dim3(N / BN, M / BM, batch), dim3(256), 0, K, A, lda, B, ldb,
               e);
    return TGX_OK;
  }
}

template <int EPI, bool ZINT, int TI, int TJ, int OCC>
static int launch_f64_tile(tgx_ctx* ctx, const char* name, int M, int N, int K, const double* A, int lda,
                           const double* B, int ldb, EpiArgs e) {
  TGX_LAUNCH(ctx, name, (k_gemm_f64<EPI, ZINT, TI, TJ, OCC>), dim3(N / (32 * TJ), M / (32 * TI)), dim3(256),
             f64_lds_bytes(TI, TJ), K, A, lda, B, ldb, e);
  return TGX_OK;
}

template <int EPI, bool ZINT, int NC, int KS>
static int launch_f64_few(tgx_ctx* ctx, const char* name, int M, int N, int K, const double* A, int lda,
                          const double* B, int ldb, EpiArgs e) {
  TGX_LAUNCH(ctx, name, (k_gemm_f64_few<EPI, ZINT, NC, KS>), dim3(N / (32 * NC), M / 32), dim3(64 * NC * KS),
             sizeof(double) * 32 * 32 * NC * KS, K, A, lda, B, ldb, e);
  return TGX_OK;
}

// FP64 NT GEMM launch. 128 x 128 tiles while they fill the 256 CUs twice over
// (32,768 x 1,280 x 4,096: 5.2 ms, 66 TFLOP/s; the half-tall tile 5.8), smaller
// ones below (2,048 x 1,280 x 4,096: 0.60 ms on 160 tiles of 128 x 128, 0.41 on
// 64 x 64; 1,024 x 2,048 x 384: 0.073 -> 0.047 on 64 x 128), and the kernel that
// splits K between the wavefronts when even those leave most CUs empty (256 x
// 384 x 2,048: 0.28 ms on 128 x 128, 0.12 on 64 x 64, 0.04 split). The lines lie
// where the two sides measured alike. The energy partials of the GAP epilogue
// are per 128 columns whatever the tile, so their layout does not depend on the
// rule. shared: another block's kernels run beside this one and take the CUs a
// last round leaves idle, so that the wide tile pays earlier (two blocks of
// 8,000 centres, FP64 adjoint step: 11.33 ms with 64 x 64 tiles, 11.08 with 128 x
// 128, although alone the latter's 630 tiles take 2.06 ms against 1.39). The tiles
// of 64 and 128 rows add an element's products in the same order, so that results
// do not depend on which of them, or on shared; the kernel that splits K adds its
// wavefronts' partial sums, another order, so they change in the last bits with the
// row count at its line.
template <int EPI, bool ZINT>
static int launch_f64(tgx_ctx* ctx, bool shared, int M, int N, int K, const double* A, int lda, const double* B,
                      int ldb, EpiArgs e, const char* name) {
  TGX_REQUIRE(M % BM == 0 && N % BN == 0 && K % BN == 0, "gemm_f64: unpadded shape %d x %d x %d", M, N, K);
  const int64_t tiles = (int64_t)(M / BM) * (N / BN);
  if constexpr (EPI == EPI_GAP) {
    if (tiles >= 512) return launch_f64_tile<EPI, ZINT, 4, 4, 2>(ctx, name, M, N, K, A, lda, B, ldb, e);
    if (tiles >= 96) return launch_f64_tile<EPI, ZINT, 2, 4, 3>(ctx, name, M, N, K, A, lda, B, ldb, e);
    return launch_f64_few<EPI, ZINT, 4, 2>(ctx, name, M, N, K, A, lda, B, ldb, e);
  } else {
    if (tiles >= (shared ? 512 : 1024))
      return launch_f64_tile<EPI, ZINT, 4, 4, 2>(ctx, name, M, N, K, A, lda, B, ldb, e);
    if (tiles >= 48) return launch_f64_tile<EPI, ZINT, 2, 2, 4>(ctx, name, M, N, K, A, lda, B, ldb, e);
    return launch_f64_few<EPI, ZINT, 1, 8>(ctx, name, M, N, K, A, lda, B, ldb, e);
  }
}

int tgx_gap_contract_f64(tgx_ctx* ctx, const tgx_model_t* m, int ns, const double* q, double* kd, double* epart,
                         double* e_site, double* qss) {
  if (ns == 0) return TGX_OK;
  const int Mp = (int)tgx_round_up(ns, BM);
  const int Sp = m->Spad, Dp = m->Dpad;
  const int n_tiles = Sp / BN;
  const bool shared = m->stream && ctx->stream == m->stream;  // blocks run concurrently
  EpiArgs e = gap_epi(m);
  e.epart = epart;
  e.n_tiles = n_tiles;
  e.alpha = m->alpha.as<double>();
  e.out = kd;
  e.ldo = Sp;
  if (e.zeta_int >= 1)
    TGX_TRY((launch_f64<EPI_GAP, true>(ctx, shared, Mp, Sp, Dp, q, Dp, m->Qs.as<double>(), Dp, e, "gemm_kernel_f64")));
  else
    TGX_TRY((launch_f64<EPI_GAP, false>(ctx, shared, Mp, Sp, Dp, q, Dp, m->Qs.as<double>(), Dp, e, "gemm_kernel_f64")));
  TGX_LAUNCH(ctx, "energy_finalize", k_energy_finalize, dim3((ns + 15) / 16), dim3(256), 0, ns, epart, n_tiles,
             m->delta * m->delta, m->e0, e_site);
  if (!qss) return TGX_OK;
  EpiArgs s{};
  s.pref = 1.0;
  s.out = qss;
  s.ldo = Dp;
  return launch_f64<EPI_STORE, true>(ctx, shared, Mp, Dp, Sp, kd, Sp, m->QsT.as<double>(), Sp, s, "gemm_qss_f64");
}

int tgx_gap_contract(tgx_ctx* ctx, tgx_model_t* m, int path, bool do_forces) {
  const int ns = m->n_sites_b;
  if (ns == 0) return TGX_OK;
  const int Sp = m->Spad, Dp = m->Dpad;
  const int n_tiles = Sp / BN;
  if (path == TGX_PATH_FP64_PLAIN || path == TGX_PATH_FP64_ADJOINT) {
    const int Mp = (int)tgx_round_up(ns, BM);
    TGX_TRY(m->epart.ensure(sizeof(double) * (size_t)Mp * n_tiles));
    TGX_TRY(m->e_site.ensure(sizeof(double) * (size_t)Mp));
    TGX_TRY(m->kd64.ensure(sizeof(double) * (size_t)Mp * Sp));
    if (do_forces) TGX_TRY(m->qss64.ensure(sizeof(double) * (size_t)Mp * Dp));
    return tgx_gap_contract_f64(ctx, m, ns, m->q64.as<double>(), m->kd64.as<double>(), m->epart.as<double>(),
                                m->e_site.as<double>(), do_forces ? m->qss64.as<double>() : nullptr);
  }
  // mixed path: qbf (BF16 descriptors) comes from the FP32 descriptor pass
  const int Mp = tgx_rows_bf16(ns);
  TGX_TRY(m->epart.ensure(sizeof(double) * (size_t)Mp * n_tiles));
  TGX_TRY(m->e_site.ensure(sizeof(double) * (size_t)Mp));
  EpiArgs e = gap_epi(m);
  e.epart = m->epart.as<double>();
  e.n_tiles = n_tiles;
  TGX_REQUIRE(m->qbf.bytes >= sizeof(__bf16) * (size_t)Mp * Dp, "gemm_bf16: BF16 descriptors missing");
  TGX_TRY(m->kdbf.ensure(sizeof(__bf16) * (size_t)Mp * Sp));
  e.alpha_f = m->alpha_f.as<float>();
  e.out = m->kdbf.p;
  e.ldo = Sp;
  if (e.zeta_int >= 1)
    TGX_TRY((launch_bf16<EPI_GAP, __bf16, true>(ctx, "gemm_kernel_bf16", Mp, Sp, Dp, 1, m->qbf.as<__bf16>(), Dp,
                                                 m->Qs_bf.as<__bf16>(), Dp, e)));
  else
    TGX_TRY((launch_bf16<EPI_GAP, __bf16, false>(ctx, "gemm_kernel_bf16", Mp, Sp, Dp, 1, m->qbf.as<__bf16>(), Dp,
                                                  m->Qs_bf.as<__bf16>(), Dp, e)));
  TGX_LAUNCH(ctx, "energy_finalize", k_energy_finalize, dim3((ns + 15) / 16), dim3(256), 0, ns,
             m->epart.as<double>(), n_tiles, m->delta * m->delta, m->e0, m->e_site.as<double>());
  if (!do_forces) return TGX_OK;
  EpiArgs s{};
  s.pref = 1.0;
  TGX_TRY(m->qss32.ensure(sizeof(float) * (size_t)Mp * Dp));
  s.out = m->qss32.p;
  s.ldo = Dp;
  return launch_bf16<EPI_STORE, float, true>(ctx, "gemm_qss_bf16", Mp, Dp, Sp, 1, m->kdbf.as<__bf16>(), Sp,
                                             m->QsT_bf.as<__bf16>(), Sp, s);
}

// C[M][N] (FP32) = scale * A[M][K] . B[N][K]^T in BF16 with FP32 accumulation.
// M, N multiples of 128, K a multiple of 64, leading dimensions in elements.
int tgx_gemm_bf16_nt(tgx_ctx* ctx, const char* name, int M, int N, int K, const __bf16* A, int lda, const __bf16* B,
                     int ldb, float* C, int ldc, double scale) {
  EpiArgs s{};
  s.pref = scale;
  s.out = C;
  s.ldo = ldc;
  return launch_bf16<EPI_STORE, float, true>(ctx, name, M, N, K, 1, A, lda, B, ldb, s);
}

int tgx_gemm_bf16(tgx_ctx* ctx, const char* name, const tgx_gemm_desc& d) {
  TGX_REQUIRE(d.M % BM == 0 && d.N % BN == 0 && d.K % 64 == 0 && d.lda % 8 == 0 && d.ldb % 8 == 0 && d.sA % 8 == 0 &&
                  d.sB % 8 == 0 && d.batch >= 1 && d.batch <= 65535,
              "gemm_bf16 %s: unpadded shape %d x %d x %d (batch %d)", name, d.M, d.N, d.K, d.batch);
  TGX_REQUIRE(d.epi != TGX_EPI_SILU || (d.bias && d.aux), "gemm_bf16 %s: SiLU epilogue needs bias and aux", name);
  TGX_REQUIRE(d.epi != TGX_EPI_SCALE_AUX || d.aux, "gemm_bf16 %s: scaled epilogue needs aux", name);
  TGX_REQUIRE(d.epi != TGX_EPI_ACT2 || (d.bias && d.w3 && d.epart), "gemm_bf16 %s: ACT2 needs bias, w3, epart",
              name);
  EpiArgs e{};
  e.pref = d.scale;
  e.out = d.C;
  e.ldo = d.ldc;
  e.bias = d.bias;
  e.aux = d.aux;
  e.ldaux = d.ldaux;
  e.sA = d.sA;
  e.sB = d.sB;
  e.sOut = d.sC;
  e.sAux = d.sAux;
  e.sBias = d.sBias;
  e.zscale = d.zscale;
  e.w3 = d.w3;
  e.sW3 = d.sW3;
  e.epart = d.epart;
  e.sEpart = d.sEpart;
  e.n_tiles = d.N / BN;
  switch (d.epi) {
    case TGX_EPI_STORE_F32:
      return launch_bf16<EPI_STORE, float, true>(ctx, name, d.M, d.N, d.K, d.batch, d.A, d.lda, d.B, d.ldb, e);
    case TGX_EPI_SILU:
      return launch_bf16<EPI_SILU, __bf16, true>(ctx, name, d.M, d.N, d.K, d.batch, d.A, d.lda, d.B, d.ldb, e);
    case TGX_EPI_SCALE_AUX:
      return launch_bf16<EPI_SCALE_AUX, __bf16, true>(ctx, name, d.M, d.N, d.K, d.batch, d.A, d.lda, d.B, d.ldb, e);
    case TGX_EPI_ACT2:
      return launch_bf16<EPI_ACT2, __bf16, true>(ctx, name, d.M, d.N, d.K, d.batch, d.A, d.lda, d.B, d.ldb, e);
    default:
      TGX_REQUIRE(false, "gemm_bf16 %s: unknown epilogue %d", name, d.epi);
  }
}

int tgx_f32_to_bf16(tgx_ctx* ctx, const float* x, __bf16* y, int64_t n) {
  TGX_LAUNCH(ctx, "to_bf16", k_f32_to_bf16, dim3(1024), dim3(256), 0, n, x, y);
  return TGX_OK;
}
