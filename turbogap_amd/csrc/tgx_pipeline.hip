// Per-block marshal (src/gap_interface.f90:204-309), per-atom force gather and
// virial/energy reductions (src/gap.f90:206-224, src/turbogap.f90:1352-1373,
// 1941-1954).
//
// Forces are gathered, not scattered with atomics: every pair force lives at its
// global pair index, and atom j sums the entries of the pairs that point at it
// by walking its own list through the reverse-pair index, in list order. The
// result is the same bits on every run.
#include <algorithm>

#include "tgx_internal.h"
#include "tgx_util.h"

namespace {

struct SpeciesMap {
  int n;
  int code[TGX_MAX_SPECIES];
  __device__ int index(int c) const {
    for (int s = 0; s < n; ++s)
      if (code[s] == c) return s;
    return -1;
  }
};

// A site is a centre of the block when its species is the block's central
// species (or the block takes every atom); a pair is kept when it lies inside
// the block's largest cutoff and the block sees the neighbour's species.
// Only atoms in [lo, hi) can be centres (a batch of the block's sites). Two
// atoms per wavefront, 32 lanes each, as the fill (one thread walking its
// atom's list took 18 us, 37 at 53 neighbours; this takes 5).
// One block per blockIdx.y.
struct SelectTask {
  SpeciesMap sm;
  int lo, hi, central;
  double rcut;
  int* flag;
  int* npairs;
};
constexpr int SELECT_TASKS = TGX_SCAN_TASKS / 2;
struct SelectTasks {
  SelectTask t[SELECT_TASKS];
};

__global__ __launch_bounds__(256) void k_select_count(int n, SelectTasks ts, const int* __restrict__ n_neigh,
                                                    const int64_t* __restrict__ off, const int* __restrict__ species,
                                                    const double* __restrict__ rjs, const int* __restrict__ nspec) {
  const SelectTask& t = ts.t[blockIdx.y];
  const int lane = threadIdx.x & 63, sub = lane & 31;
  const uint64_t half = (lane < 32 ? 0xffffffffull : 0xffffffff00000000ull);
  const int i = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 2 + (lane >> 5);
  if (i >= n) return;
  const int sc = t.sm.index(species[i]);
  const int nn = n_neigh[i];
  const bool sel = i >= t.lo && i < t.hi && nn > 0 && sc >= 0 && (t.central == 0 || sc == t.central - 1);
  int cnt = 0;
  if (sel) {
    const int64_t b = off[i];
    for (int base = 0; base < nn; base += 32) {
      const int k = base + sub;
      const bool keep = k < nn && rjs[b + k] < t.rcut && t.sm.index(nspec[b + k]) >= 0;
      cnt += __popcll(__ballot(keep) & half);
    }
  }
  if (sub == 0) {
    t.flag[i] = sel ? 1 : 0;
    t.npairs[i] = cnt;
  }
}

__global__ __launch_bounds__(256) void k_select_fill(int n, SpeciesMap sm, double rcut, const int* __restrict__ flag,
                                                   const int64_t* __restrict__ site_idx,
                                                   const int64_t* __restrict__ pair_off,
                                                   const int* __restrict__ n_neigh, const int64_t* __restrict__ off,
                                                   const int* __restrict__ nlist, const double* __restrict__ rjs,
                                                   const double* __restrict__ xyz, const int* __restrict__ nspec,
                                                   int* __restrict__ site_atom, int64_t* __restrict__ site_beg,
                                                   int64_t* __restrict__ pr_gidx, int* __restrict__ pr_nbr,
                                                   int* __restrict__ pr_spec, double* __restrict__ pr_r,
                                                   double* __restrict__ pr_xyz) {
  if (blockIdx.x == 0 && threadIdx.x == 0) site_beg[site_idx[n]] = pair_off[n];
  // two atoms per wavefront, 32 lanes each (lists average about 22 entries);
  // each half's ballot bits are masked to its own lanes
  const int lane = threadIdx.x & 63, sub = lane & 31;
  const uint64_t half = (lane < 32 ? 0xffffffffull : 0xffffffff00000000ull);
  const int i = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 2 + (lane >> 5);
  if (i >= n || !flag[i]) return;
  const int64_t s = site_idx[i];
  const int64_t o = pair_off[i];
  if (sub == 0) { site_atom[s] = i; site_beg[s] = o; }
  const int64_t b = off[i];
  const int nn = n_neigh[i];
  int kept = 0;
  for (int base = 0; base < nn; base += 32) {
    const int k = base + sub;
    bool keep = false;
    int sp = -1;
    if (k < nn) {
      sp = sm.index(nspec[b + k]);
      keep = rjs[b + k] < rcut && sp >= 0;
    }
    const uint64_t mask = __ballot(keep) & half;
    if (keep) {
      const int64_t p = o + kept + __popcll(mask & ((1ull << lane) - 1ull));
      const int64_t g = b + k;
      const int j = (nlist[g] - 1) % n;
      pr_gidx[p] = g;
      pr_nbr[p] = j;
      pr_spec[p] = sp;
      pr_r[p] = rjs[g];
      pr_xyz[3 * p] = xyz[3 * g];
      pr_xyz[3 * p + 1] = xyz[3 * g + 1];
      pr_xyz[3 * p + 2] = xyz[3 * g + 2];
    }
    kept += __popcll(mask);
  }
}

// The end of a force evaluation in one launch: workgroups [0, n_gather) gather
// forces, the next n_vir sum the virial, the rest the energies. The partials and
// the missing-reverse flag go straight to pinned host memory, so that the step
// ends with one kernel and one wait (five launches and a copy before: 25 us of
// gaps and small kernels).
//
// F_j = sum over j's list entries q of fglob[rev[q]], in list order.
// GATHER_LANES lanes per atom: lane t sums entries t, t + GATHER_LANES, ... in
// order, then the lanes' sums combine by a fixed xor butterfly, so every run
// adds in the same order. Virial: 0.5 (f x^T + x f^T) summed over a fixed slice
// of pairs per workgroup (column-major 3x3). Energies: a fixed slice per
// workgroup in a fixed tree.
constexpr int GATHER_LANES = 16;
constexpr int VIRIAL_PARTS = 512;

struct FinishArgs {
  int n;
  int64_t P;
  const int* n_neigh;
  const int64_t* off;
  const int64_t* rev;
  const double* fglob;
  const double* xyz;
  const double* energies;
  double* F;
  double* vpart;  // pinned: [n_vir][9]
  double* epart;  // pinned: [n_e]
  int* bad;       // pinned, set when a pair has no reverse entry
  int n_gather, n_vir, n_e;
};

__global__ __launch_bounds__(256) void k_finish(FinishArgs a) {
  __shared__ double sh[9][256];
  int blk = blockIdx.x;
  if (blk < a.n_gather) {
    const int t = threadIdx.x % GATHER_LANES;
    const int j = (blk * 256 + (int)threadIdx.x) / GATHER_LANES;
    const bool live = j < a.n;
    double f0 = 0, f1 = 0, f2 = 0;
    if (live) {
      const int64_t b = a.off[j];
      const int nn = a.n_neigh[j];
      for (int k = t; k < nn; k += GATHER_LANES) {
        const int64_t r = a.rev[b + k];
        if (r < 0) { *a.bad = 1; continue; }
        f0 += a.fglob[3 * r];
        f1 += a.fglob[3 * r + 1];
        f2 += a.fglob[3 * r + 2];
      }
    }
#pragma unroll
    for (int o = GATHER_LANES / 2; o > 0; o >>= 1) {  // every lane of the wavefront takes part
      f0 += __shfl_xor(f0, o);
      f1 += __shfl_xor(f1, o);
      f2 += __shfl_xor(f2, o);
    }
    if (live && t == 0) {
      a.F[3 * (size_t)j] = f0;
      a.F[3 * (size_t)j + 1] = f1;
      a.F[3 * (size_t)j + 2] = f2;
    }
    return;
  }
  blk -= a.n_gather;
  const bool vir = blk < a.n_vir;
  const int nv = vir ? 9 : 1;
  double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (vir) {
    const int64_t per = (a.P + a.n_vir - 1) / a.n_vir;
    const int64_t b = (int64_t)blk * per, e = b + per < a.P ? b + per : a.P;
    for (int64_t p = b + threadIdx.x; p < e; p += 256) {
      const double f[3] = {a.fglob[3 * p], a.fglob[3 * p + 1], a.fglob[3 * p + 2]};
      const double x[3] = {a.xyz[3 * p], a.xyz[3 * p + 1], a.xyz[3 * p + 2]};
#pragma unroll
      for (int k1 = 0; k1 < 3; ++k1)
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) v[3 * k2 + k1] += 0.5 * (f[k1] * x[k2] + f[k2] * x[k1]);
    }
  } else {
    blk -= a.n_vir;
    const int per = (a.n + a.n_e - 1) / a.n_e;
    const int b = blk * per, e = b + per < a.n ? b + per : a.n;
    for (int i = b + (int)threadIdx.x; i < e; i += 256) v[0] += a.energies[i];
  }
#pragma unroll
  for (int k = 0; k < 9; ++k)
    if (k < nv) sh[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if (threadIdx.x < o)
      for (int k = 0; k < nv; ++k) sh[k][threadIdx.x] += sh[k][threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x < nv) {
    if (vir) a.vpart[9 * blk + threadIdx.x] = sh[threadIdx.x][0];
    else a.epart[blk] = sh[0][0];
  }
}

// Centre energies into their atoms, one block per blockIdx.y (blocks of one launch
// have no centre in common).
struct ScatterTasks {
  int ns[SELECT_TASKS];
  const int* atom[SELECT_TASKS];
  const double* e[SELECT_TASKS];
};

__global__ void k_energy_scatter(ScatterTasks t, double* __restrict__ energies) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
  if (s < t.ns[k]) energies[t.atom[k][s]] += t.e[k][s];
}

}  // namespace

static SpeciesMap species_map(const tgx_model_t* m) {
  SpeciesMap sm{};
  sm.n = m->n_species;
  for (int s = 0; s < m->n_species; ++s) sm.code[s] = m->species_types[s];
  return sm;
}

// Block selection in two halves: the count and scans, which leave the two totals
// in pinned host memory (no wait), then, once the caller has synchronised the
// stream, the allocation and the fill. Several blocks can have their counts in
// flight before one wait.
struct SelectView {
  int* flag;
  int* npairs;
  int64_t* site_idx;
  int64_t* pair_off;
};

static SelectView select_view(tgx_model_t* m, int n) {
  SelectView v;
  v.flag = m->sel_scratch.as<int>();
  v.npairs = v.flag + n;
  v.site_idx = reinterpret_cast<int64_t*>(m->sel_scratch.as<char>() + tgx_round_up(sizeof(int) * 2 * (size_t)n, 16));
  v.pair_off = v.site_idx + tgx_round_up(n + 1, 2);  // 16-byte aligned for the scan
  return v;
}

int tgx_blocks_select_count(tgx_ctx* ctx, tgx_model_t* const* models, int count) {
  TGX_REQUIRE(ctx->have_list, "no neighbour list: call tgx_build_neighbors_list first");
  const int n = ctx->n_sites;
  for (int k0 = 0; k0 < count; k0 += SELECT_TASKS) {
    const int cnt = std::min(SELECT_TASKS, count - k0);
    SelectTasks st{};
    tgx_scan_tasks sc{};
    for (int k = 0; k < cnt; ++k) {
      tgx_model_t* m = models[k0 + k];
      // the block's own scratch: blocks may be selected while another block's kernels still run
      TGX_TRY(m->sel_scratch.ensure(sizeof(int) * 2 * (size_t)n + sizeof(int64_t) * 2 * (size_t)(n + 1) + 256));
      if (!m->sel_host) TGX_TRY(ctx->pinned.take(&m->sel_host, 2));
      const SelectView v = select_view(m, n);
      const int lo = m->sel_lo > 0 ? m->sel_lo : 0, hi = (m->sel_hi >= 0 && m->sel_hi < n) ? m->sel_hi : n;
      st.t[k] = SelectTask{species_map(m), lo, hi, m->central_species, m->rcut_max, v.flag, v.npairs};
      sc.t[2 * k] = tgx_scan_task{v.flag, v.site_idx, m->sel_host};
      sc.t[2 * k + 1] = tgx_scan_task{v.npairs, v.pair_off, m->sel_host + 1};
    }
    TGX_LAUNCH(ctx, "select_count", k_select_count, dim3((n + 7) / 8, cnt), dim3(256), 0, n, st, ctx->n_neigh.as<int>(),
               ctx->nl_off.as<int64_t>(), ctx->species_sc.as<int>(), ctx->rjs.as<double>(), ctx->nspec.as<int>());
    TGX_TRY(tgx_scan_many(ctx, sc, 2 * cnt, n, &models[k0]->scan_tmp));
  }
  return TGX_OK;
}

int tgx_block_select_count(tgx_ctx* ctx, tgx_model_t* m) { return tgx_blocks_select_count(ctx, &m, 1); }

int tgx_block_select_counts_host(tgx_ctx* ctx, tgx_model_t* m, std::vector<int>& flag, std::vector<int64_t>& pair_off) {
  const int n = ctx->n_sites;
  const SelectView v = select_view(m, n);
  flag.resize((size_t)n);
  pair_off.resize((size_t)n + 1);
  TGX_CHECK_HIP(hipMemcpyAsync(flag.data(), v.flag, sizeof(int) * (size_t)n, hipMemcpyDeviceToHost, ctx->stream));
  TGX_CHECK_HIP(hipMemcpyAsync(pair_off.data(), v.pair_off, sizeof(int64_t) * ((size_t)n + 1), hipMemcpyDeviceToHost,
                               ctx->stream));
  TGX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  return TGX_OK;
}

int tgx_block_select_fill(tgx_ctx* ctx, tgx_model_t* m) {
  const int n = ctx->n_sites;
  const SelectView v = select_view(m, n);
  SpeciesMap sm = species_map(m);
  const int64_t ns = m->sel_host[0], np = m->sel_host[1];
  m->n_sites_b = (int)ns;
  m->n_pairs_b = np;
  const size_t npz = (size_t)(np > 0 ? np : 1);
  TGX_TRY(m->site_atom.ensure(sizeof(int) * (size_t)(ns + 1)));
  TGX_TRY(m->site_beg.ensure(sizeof(int64_t) * (size_t)(ns + 1)));
  TGX_TRY(m->pr_gidx.ensure(sizeof(int64_t) * npz));
  TGX_TRY(m->pr_nbr.ensure(sizeof(int) * npz));
  TGX_TRY(m->pr_spec.ensure(sizeof(int) * npz));
  TGX_TRY(m->pr_r.ensure(sizeof(double) * npz));
  TGX_TRY(m->pr_xyz.ensure(sizeof(double) * 3 * npz));
  TGX_LAUNCH(ctx, "select_fill", k_select_fill, dim3((n + 7) / 8), dim3(256), 0, n, sm, m->rcut_max, v.flag,
             v.site_idx, v.pair_off, ctx->n_neigh.as<int>(), ctx->nl_off.as<int64_t>(), ctx->nlist.as<int>(),
             ctx->rjs.as<double>(), ctx->xyz.as<double>(), ctx->nspec.as<int>(), m->site_atom.as<int>(),
             m->site_beg.as<int64_t>(), m->pr_gidx.as<int64_t>(), m->pr_nbr.as<int>(), m->pr_spec.as<int>(),
             m->pr_r.as<double>(), m->pr_xyz.as<double>());
  return TGX_OK;
}

int tgx_block_select(tgx_ctx* ctx, tgx_model_t* m) {
  TGX_TRY(tgx_block_select_count(ctx, m));
  TGX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  return tgx_block_select_fill(ctx, m);
}

// Forces and virial from the accumulated pair forces; adds every model's site
// energies was done by the caller. energy_out/virial_out may be NULL.
int tgx_gather_forces(tgx_ctx* ctx, double* energy_out, double* virial_out) {
  TGX_TRY(ctx->forces.ensure(sizeof(double) * 3 * (size_t)ctx->n_sites));
  return tgx_gather_pair_forces(ctx, ctx->fglob.as<double>(), ctx->forces.as<double>(), virial_out,
                                ctx->energies.as<double>(), energy_out);
}

// ctx->red_host: VIRIAL_PARTS x 9 virial partials, TGX_SUM_PARTS energy partials,
// the missing-reverse flag.
int tgx_red_host(tgx_ctx* ctx) {
  if (ctx->red_host) return TGX_OK;
  return ctx->pinned.take(&ctx->red_host, 9 * (size_t)VIRIAL_PARTS + TGX_SUM_PARTS + 1);
}

static int gather_launch(tgx_ctx* ctx, const double* fglob, double* F, bool with_virial, const double* d_energies) {
  TGX_TRY(tgx_red_host(ctx));
  FinishArgs a;
  a.n = ctx->n_sites;
  a.P = ctx->n_pairs;
  a.n_neigh = ctx->n_neigh.as<int>();
  a.off = ctx->nl_off.as<int64_t>();
  a.rev = ctx->rev.as<int64_t>();
  a.fglob = fglob;
  a.xyz = ctx->xyz.as<double>();
  a.energies = d_energies;
  a.F = F;
  a.vpart = ctx->red_host;
  a.epart = a.vpart + 9 * VIRIAL_PARTS;
  a.bad = reinterpret_cast<int*>(a.epart + TGX_SUM_PARTS);
  *a.bad = 0;  // every use of the buffer ends with a wait: no kernel holds it now
  // about 2,048 pairs or atoms a partial, so that a small system writes few of them
  auto parts = [](int64_t n, int most) { return (int)std::min<int64_t>(most, std::max<int64_t>(1, (n + 2047) / 2048)); };
  a.n_gather = (int)(((int64_t)a.n * GATHER_LANES + 255) / 256);
  a.n_vir = with_virial ? parts(a.P, VIRIAL_PARTS) : 0;
  a.n_e = d_energies ? parts(a.n, TGX_SUM_PARTS) : 0;
  ctx->gather_parts[0] = a.n_vir;
  ctx->gather_parts[1] = a.n_e;
  TGX_LAUNCH(ctx, "force_gather", k_finish, dim3((unsigned)(a.n_gather + a.n_vir + a.n_e)), dim3(256), 0, a);
  return TGX_OK;
}

int tgx_gather_collect(tgx_ctx* ctx, double* virial_out, double* energy_out) {
  const double* vp = ctx->red_host;
  const double* ep = vp + 9 * VIRIAL_PARTS;
  if (*reinterpret_cast<const int*>(ep + TGX_SUM_PARTS)) {
    tgx_set_error("force gather: a pair has no reverse entry (an atom without its own list); build with do_list = all");
    return TGX_ERR_UNSUPPORTED;
  }
  if (virial_out) {
    for (int k = 0; k < 9; ++k) virial_out[k] = 0.0;
    for (int b = 0; b < ctx->gather_parts[0]; ++b)
      for (int k = 0; k < 9; ++k) virial_out[k] += vp[9 * b + k];
  }
  if (energy_out && ctx->gather_parts[1] > 0) {
    double e = 0.0;
    for (int i = 0; i < ctx->gather_parts[1]; ++i) e += ep[i];
    *energy_out = e;
  }
  return TGX_OK;
}

int tgx_gather_forces_launch(tgx_ctx* ctx) {
  TGX_TRY(ctx->forces.ensure(sizeof(double) * 3 * (size_t)ctx->n_sites));
  return gather_launch(ctx, ctx->fglob.as<double>(), ctx->forces.as<double>(), true, nullptr);
}

int tgx_gather_pair_forces(tgx_ctx* ctx, const double* fglob, double* F, double* virial_out,
                           const double* d_energies, double* energy_out) {
  TGX_TRY(gather_launch(ctx, fglob, F, virial_out != nullptr, energy_out ? d_energies : nullptr));
  TGX_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  return tgx_gather_collect(ctx, virial_out, energy_out);
}

int tgx_energy_scatter_blocks(tgx_ctx* ctx, tgx_model_t* const* models, int count) {
  for (int k0 = 0; k0 < count; k0 += SELECT_TASKS) {
    const int cnt = std::min(SELECT_TASKS, count - k0);
    ScatterTasks t{};
    int most = 0;
    for (int k = 0; k < cnt; ++k) {
      tgx_model_t* m = models[k0 + k];
      t.ns[k] = m->n_sites_b;
      t.atom[k] = m->site_atom.as<int>();
      t.e[k] = m->e_site.as<double>();
      most = std::max(most, m->n_sites_b);
    }
    if (most == 0) continue;
    TGX_LAUNCH(ctx, "energy_scatter", k_energy_scatter, dim3((most + 255) / 256, cnt), dim3(256), 0, t,
               ctx->energies.as<double>());
  }
  return TGX_OK;
}

int tgx_energy_scatter(tgx_ctx* ctx, tgx_model_t* m) { return tgx_energy_scatter_blocks(ctx, &m, 1); }

// get_gap_soap's results pass through pinned memory, fold_host, for n atoms: forces
// [n][3], the centres' energies [n] and atoms [n] in the order of the sites, and a
// mark for every atom a pair reaches [n]. The centres are listed, not marked: the
// host's test of a mark that one atom in two has cost 2 to 3 ns an atom (energies
// of 300,000 atoms, half of them centres: 2.64 ms with marks, 1.72 listed).

// A batch of ns sites into the list from site `first` on, and marks (mark not null)
// of the atoms of its np pairs, each centre's self entry among them.
__global__ void k_mark_seen(int64_t np, int ns, const int* __restrict__ pr_nbr, const int* __restrict__ site_atom,
                            const double* __restrict__ e_site, int* __restrict__ mark, double* __restrict__ e_out,
                            int* __restrict__ atom_out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (mark && p < np) mark[pr_nbr[p]] = 1;
  if (p < ns) {
    e_out[p] = e_site[p];
    atom_out[p] = site_atom[p];
  }
}

int tgx_fold_sites(tgx_ctx* ctx, tgx_model_t* m, int first, int* d_mark) {
  const int64_t np = std::max<int64_t>(d_mark ? m->n_pairs_b : 0, m->n_sites_b);
  if (np == 0) return TGX_OK;
  const size_t n = (size_t)ctx->n_sites;
  double* e = ctx->fold_host + 3 * n;
  TGX_LAUNCH(ctx, "mark_seen", k_mark_seen, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, m->n_pairs_b,
             m->n_sites_b, m->pr_nbr.as<int>(), m->site_atom.as<int>(), (const double*)m->e_site.as<double>(), d_mark,
             e + first, reinterpret_cast<int*>(e + n) + first);
  return TGX_OK;
}

// Forces of every atom into fold_host, with the marks (get_gap_soap) or the atoms'
// energies (get_results; in the energies' place).
__global__ void k_fold_out(int n, const double* __restrict__ F, const double* __restrict__ energies,
                           const int* __restrict__ mark, double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[3 * (size_t)i] = F[3 * (size_t)i];
  out[3 * (size_t)i + 1] = F[3 * (size_t)i + 1];
  out[3 * (size_t)i + 2] = F[3 * (size_t)i + 2];
  if (energies) out[3 * (size_t)n + i] = energies[i];
  if (mark) reinterpret_cast<int*>(out + 4 * (size_t)n)[n + i] = mark[i];
}

int tgx_fold_out(tgx_ctx* ctx, const double* energies, const int* d_mark) {
  const int n = ctx->n_sites;
  TGX_LAUNCH(ctx, "fold_out", k_fold_out, dim3((n + 255) / 256), dim3(256), 0, n, (const double*)ctx->forces.as<double>(),
             energies, d_mark, ctx->fold_host);
  return TGX_OK;
}

// fold_host for the system's atoms.
int tgx_fold_ensure(tgx_ctx* ctx) {
  const int n = ctx->n_sites;
  constexpr size_t row = sizeof(double) * 4 + sizeof(int) * 2;
  if (ctx->fold_n < n && n <= TGX_FOLD_POOL) {
    TGX_TRY(ctx->pinned.take(reinterpret_cast<char**>(&ctx->fold_host), row * TGX_FOLD_POOL));
    ctx->fold_n = TGX_FOLD_POOL;
  } else if (ctx->fold_n < n) {
    // a size that rises again gets 25% headroom, as the device buffers: releasing it costs 250 us
    int want = ctx->fold_own ? n + n / 4 : n;
    if (ctx->fold_own) (void)hipHostFree(ctx->fold_own);
    ctx->fold_own = ctx->fold_host = nullptr;
    ctx->fold_n = 0;
    if (want > n && hipHostMalloc(&ctx->fold_own, row * (size_t)want, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      ctx->fold_own = nullptr;
      want = n;
    }
    if (!ctx->fold_own) TGX_CHECK_HIP(hipHostMalloc(&ctx->fold_own, row * (size_t)n, hipHostMallocDefault));
    ctx->fold_host = static_cast<double*>(ctx->fold_own);
    ctx->fold_n = want;
  }
  return TGX_OK;
}
