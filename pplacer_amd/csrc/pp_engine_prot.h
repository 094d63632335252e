// Master/worker three-taxon engine for 20-state (protein) models.
//
// Same command protocol and control as the nucleotide engine
// (pp_engine_mw.h, pp_engine_ctl.h), with the evolves taken in the
// eigenbasis of Q.  P_r(t)[i][j] = sum_k x[i][k] e_r[k] xit[j][k] with
// e_r[k] = exp(rate_r * t * l_k) (Diagd.multi_exp, diagd.ml:79-100), so
//
//   evolved row  y_i = sum_k x[i][k] * e_r[k] * a_k,   a_k = sum_j xit[j][k] * src_j
//   pendant row  z_i = sum_k x[i][k] * e_r[k] * L[c][k], L[c][k] = sum_j xit[j][k] * lv[c][j]
//   util = sum_r sum_i ((pi_i x_i) y_i) z_i = sum_r sum_k e_pend,r[k] * G_r[k],
//          G_r[k] = L[c][k] * sum_i ((pi_i x_i) y_i) x[i][k].
//
// A probe therefore needs only the 20 R exponentials per changed branch
// length, which the master computes; no P matrix is formed.  Work item = one
// (masked site, rate) pair; the R pairs of a site sit in consecutive lanes
// and their utils are summed across those lanes.  The eigen coordinates a of
// the distal and proximal rows (set at each gather, read by distal probes)
// live in a per-workgroup region of a global scratch buffer laid out in tiles
// of 64 pairs, [k][64]; G (set at each distal probe, read by every probe) in the worker's
// registers, and in the scratch for the pairs beyond them.
//
// This is the same likelihood as ten_log_like3_c (linear_c.c:367-424) on
// the same GLVs; the sums are grouped differently from the stubs' explicit
// P(t) * GLV products, so results agree to rounding (~1e-14 relative).
#pragma once

#include <climits>
#include <type_traits>

#include "pp_engine.h"
#include "pp_engine_ctl.h"
#include "pp_engine_mw.h"

namespace pp {

constexpr int kProtS = 20;
constexpr int kProtBlock = 512;                     // lanes of a workgroup (master + workers)
constexpr int kProtWorkers = kProtBlock / 64 - 1;   // worker waves

struct ProtShared {
  double x[kProtS * kProtS], xit[kProtS * kProtS];  // [i][k], [j][k]
  double lt[kMaxCodes * kProtS];                    // L[c][k]
  double l[kProtS], statd[kProtS], rates[kMaxRates];
  // exp(rate_r * bl * l_k) at [r][k] for the proximal, distal, pendant lengths
  double ep[kMaxRates * kProtS], ed[kMaxRates * kProtS], en[kMaxRates * kProtS];
  int op, M, q, loc;
  // FP32 form: which transition tables a probe rebuilds (bit 0: proximal and
  // distal, bit 1: pendant), and the number of character codes
  int tflags, n_codes;
  int tile_next;  // FP32 form: the next 64-pair tile a worker wave takes
  double part[kProtWorkers];      // per-worker-wave sums of site logs
  long long ipart[kProtWorkers];  // per-worker-wave sums of site exponents
};

struct ProtLayout {
  static constexpr size_t head = (sizeof(ProtShared) + 15) & ~size_t(15);
  // shared header, masked-site list
  static __host__ __device__ size_t bytes(int N) { return head + sizeof(int) * (size_t)N; }
  static __device__ int *sidx(char *s) { return reinterpret_cast<int *>(s + head); }
  static __host__ __device__ size_t align(size_t v) { return (v + 15) & ~size_t(15); }
  // Reals of per-pair scratch per workgroup: a(dist), a(prox), G, each [cap / 64][20][64]
  static __host__ __device__ size_t scratch_reals(int cap_pairs) { return (size_t)3 * kProtS * cap_pairs; }
};

__device__ __forceinline__ void prot_copy_model(ProtShared *sh, const DevModel *dm) {
  constexpr int S = kProtS;
  for (int t = threadIdx.x; t < S * S; t += blockDim.x) { sh->x[t] = dm->x[t]; sh->xit[t] = dm->xit[t]; }
  for (int t = threadIdx.x; t < S; t += blockDim.x) { sh->l[t] = dm->l[t]; sh->statd[t] = dm->statd[t]; }
  for (int t = threadIdx.x; t < kMaxRates; t += blockDim.x) sh->rates[t] = dm->rates[t];
  for (int t = threadIdx.x; t < dm->n_codes * S; t += blockDim.x) {
    const int c = t / S, k = t % S;
    double acc = dm->xit[k] * dm->lv[c * S];
    for (int j = 1; j < S; j++) acc = acc + dm->xit[j * S + k] * dm->lv[c * S + j];
    sh->lt[t] = acc;
  }
}

// The eigenbasis contractions use fused multiply-adds:
// this grouping of the likelihood already differs from the stubs' rounding.
__device__ __forceinline__ double emadd(double acc, double a, double b) { return fma(a, b, acc); }

// ---------------------------------------------------------------------------
// worker waves
// ---------------------------------------------------------------------------

// The model's x and xit where the workers read them: constant memory, so that
// a row is scalar loads and an operand of the multiply-adds, not 10 LDS reads
// per row and wave.
typedef const double __attribute__((address_space(4))) *ProtRows;

// A workgroup's scratch in tiles of 64 pairs, [20][64] each, through buffer
// loads and stores: lane l's entry k of a tile is one vector offset (8 l), a
// scalar one (the tile's) and an immediate.  (With 64-bit addresses per lane
// the compiler kept one for every entry, and spilled.)
struct ProtScratch {
  __amdgpu_buffer_rsrc_t rs;
  unsigned lane8;
  __device__ __forceinline__ ProtScratch(double *scr, size_t reals)
      : rs(__builtin_amdgcn_make_buffer_rsrc(scr, (short)0, (int)(reals * 8), 0x00020000)),
        lane8((threadIdx.x & 63) * 8) {}
  static __device__ __forceinline__ unsigned tile_bytes() { return kProtS * 64 * 8; }
  __device__ __forceinline__ double get(unsigned tile, int k) const {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, lane8 + (k & 7) * 512, tile + (k >> 3) * 4096, 0));
  }
  __device__ __forceinline__ void put(unsigned tile, int k, double v) const {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), rs, lane8 + (k & 7) * 512, tile + (k >> 3) * 4096, 0);
  }
};

// Eigen coordinates of one pair's row: a_k = sum over j of xit[j][k] v[j], in
// order of j, to the tile at `out`.
__device__ __forceinline__ void prot_coords(ProtRows xit, const double *v, const ProtScratch &scr, unsigned out) {
  constexpr int S = kProtS;
  double row[S], acc[S];
#pragma unroll
  for (int j = 0; j < S; j++) row[j] = v[j];
  asm volatile("" ::: "memory");  // the whole row in flight at once
#pragma unroll
  for (int k = 0; k < S; k++) acc[k] = xit[k] * row[0];
#pragma unroll
  for (int j = 1; j < S; j++)
#pragma unroll
    for (int k = 0; k < S; k++) acc[k] = emadd(acc[k], xit[j * S + k], row[j]);
#pragma unroll
  for (int k = 0; k < S; k++) scr.put(out, k, acc[k]);
}

// One pair of a distal probe: g[k] = L[c][k] sum_i ((pi_i x_i) y_i) x[i][k]
// with x_i, y_i the evolved proximal and distal entries (ep, ed: the pair's
// exponentials, ap, ad: its coordinates' tiles, lt: L's row of its code).
__device__ __forceinline__ void prot_pair(ProtRows x, ProtRows statd, const double *ep, const double *ed,
                                          const ProtScratch &scr, unsigned ap, unsigned ad, const double *lt,
                                          double (&g)[kProtS]) {
  constexpr int S = kProtS;
  double bd[S], bp[S];
  // The pair's 40 loads in flight at once, none kept from pair to pair (the
  // compiler's own order waited for each of them in turn, or spilled)
  asm volatile("" ::: "memory");
#pragma unroll
  for (int k = 0; k < S; k++) {
    bd[k] = scr.get(ad, k);
    bp[k] = scr.get(ap, k);
  }
  asm volatile("" ::: "memory");
#pragma unroll
  for (int k = 0; k < S; k++) {
    bd[k] = ed[k] * bd[k];
    bp[k] = ep[k] * bp[k];
    g[k] = 0.;  // fma(w, x, 0) is w x up to the sign of a zero, which no later operation can observe
  }
#pragma unroll 1
  for (int i = 0; i < S; i++) {
    ProtRows xr = x + i * S;
    double xi = xr[0] * bp[0], yi = xr[0] * bd[0];
#pragma unroll
    for (int k = 1; k < S; k++) {
      xi = emadd(xi, xr[k], bp[k]);
      yi = emadd(yi, xr[k], bd[k]);
    }
    const double wi = (statd[i] * xi) * yi;
#pragma unroll
    for (int k = 0; k < S; k++) g[k] = emadd(g[k], wi, xr[k]);
  }
#pragma unroll
  for (int k = 0; k < S; k++) g[k] = lt[k] * g[k];
}

// A lane's pairs are p = its index + k * (worker lanes), k its rounds.  G
// stays on the CU from a distal probe to the pendant-only ones after it (7 of
// 10 probes): that of rounds 0 and 1 in registers, of round 2 in LDS where the
// workgroup has room for it (lds_g), of later ones (masked lengths beyond 336
// at four rates) in the scratch.  With every G in the scratch the workgroups'
// working set (165 MB at 230 sites) was streamed from beyond the L2 at each
// probe: 21,100 cycles a pendant and 97,200 a distal probe.
//
// site_cat: Price-CAT (R == 1), the exponential tables of site s are those of
// its category site_cat[s]; nullptr: the tables of rate r.
constexpr int kProtRegRounds = 2;

// LDS bytes of one round's G for a workgroup's worker lanes: [wave][20][64].
constexpr size_t prot_round_bytes(int worker_lanes) { return sizeof(double) * kProtS * (size_t)worker_lanes; }

template <int R>
__device__ __forceinline__ void prot_worker(char *smem, double *scratch, int cap, int N, const uint8_t *codes,
                                            const double *darr, const double *parr, const int *darr_e,
                                            const int *parr_e, const int *site_cat, const DevModel *dm,
                                            double *lds_g) {
  constexpr int S = kProtS, RS = R * S, KR = kProtRegRounds;
  ProtShared *sh = reinterpret_cast<ProtShared *>(smem);
  const int *sidx = ProtLayout::sidx(smem);
  const ProtRows x = (ProtRows)(uintptr_t)dm->x, xit = (ProtRows)(uintptr_t)dm->xit;
  const ProtRows statd = (ProtRows)(uintptr_t)dm->statd;
  const int lane = threadIdx.x & 63;
  const int wv = wave_id() - 1;
  const int stride = (int)blockDim.x - 64;  // worker lanes, a multiple of 64
  const int my = wv * 64 + lane;
  const int r = my % R;  // of every pair of the lane
  const ProtScratch scr(scratch, ProtLayout::scratch_reals(cap));
  // the tile of the wave's round k in the a(dist), a(prox) or G part
  enum { AD = 0, AP = 1, GS = 2 };
  const auto tile = [&](int part, int k) {
    return (unsigned)(part * (cap >> 6) + wv + k * (stride >> 6)) * ProtScratch::tile_bytes();
  };
  // The command stream is QUERY (GATHER PROBE*)* ... EXIT (see pp_engine_mw.h).
  __syncthreads();  // A
  int op = sh->op;
  while (op == CMD_QUERY) {
    const int n_pairs = sh->M * R;
    // rounds in which the wave has a pair; a round's sites have all R pairs
    const int rounds = n_pairs > wv * 64 ? (n_pairs - wv * 64 + stride - 1) / stride : 0;
    const uint8_t *qc = codes + (size_t)sh->q * N;
    int lt_at[KR + 1];  // L's row of the pair's code
#pragma unroll
    for (int k = 0; k < KR + 1; k++) {
      const int p = my + k * stride;
      lt_at[k] = p < n_pairs ? qc[sidx[p / R]] * S : 0;
    }
    __syncthreads();  // B
    __syncthreads();  // A
    op = sh->op;
    while (op == CMD_GATHER) {
      const int loc = sh->loc;
      long long es = 0;
      for (int k = 0; k < rounds; k++) {
        const int p = my + k * stride;
        if (p < n_pairs) {
          const size_t row = (size_t)loc * N + sidx[p / R];
          prot_coords(xit, darr + row * RS + r * S, scr, tile(AD, k));
          prot_coords(xit, parr + row * RS + r * S, scr, tile(AP, k));
          if (r == 0) es += (long long)darr_e[row] + (long long)parr_e[row];
        }
      }
      es = wave_sum_ll(es);
      if (lane == 0) sh->ipart[wv] = es;
      __syncthreads();  // B
      __syncthreads();  // A
      op = sh->op;
      double G[KR][S];
#pragma unroll
      for (int k = 0; k < KR; k++)
#pragma unroll
        for (int kk = 0; kk < S; kk++) G[k][kk] = 0.;
      while (op == CMD_PROBE || op == CMD_PROBE_DIST) {
        const bool nd = op == CMD_PROBE_DIST;
        double lsum = 0.0;
        // util of round k's pair from its G, summed over its site's rates (the
        // four lanes of a quad, which all get the sum)
        const auto site_util = [&](int k, const double (&g)[S]) {
          const int p = my + k * stride;
          const int er = (R == 1 && site_cat) ? site_cat[sidx[p < n_pairs ? p : 0]] : r;
          const double *en = sh->en + er * S;
          double u = en[0] * g[0];
#pragma unroll
          for (int kk = 1; kk < S; kk++) u = emadd(u, en[kk], g[kk]);
          u = p < n_pairs ? u : 0.0;
          if (R == 4) {
            u += dpp_f64<0xB1>(u);  // lane ^ 1
            u += dpp_f64<0x4E>(u);  // lane ^ 2
          }
          return u;
        };
        // (lanes past the query's pairs compute on what their scratch holds;
        // site_util and the log sum leave them out)
        const auto distal = [&](int k, int lt, double (&g)[S]) {
          const int p = my + k * stride;
          const int er = (R == 1 && site_cat) ? site_cat[sidx[p < n_pairs ? p : 0]] : r;
          prot_pair(x, statd, sh->ep + er * S, sh->ed + er * S, scr, tile(AP, k), tile(AD, k), sh->lt + lt, g);
        };
        // Rounds 0 to 2; with four rates lane r of a quad takes the log of
        // round r's sum, and lane 0 adds them in order.
        double hold = 1.0;
        const auto first_rounds = [&](int k, double u) {
          if (R == 4) hold = r == k ? u : hold;
          else if (my + k * stride < n_pairs) lsum += log(u);
        };
        double *at = lds_g + (size_t)wv * S * 64 + lane;
        const bool in_lds = lds_g && rounds > KR;  // round KR
        if (nd) {
          if (in_lds) {
            double g[S];
            distal(KR, lt_at[KR], g);
#pragma unroll
            for (int kk = 0; kk < S; kk++) at[64 * kk] = g[kk];
          }
#pragma unroll
          for (int k = 0; k < KR; k++)
            if (k < rounds) distal(k, lt_at[k], G[k]);
        }
#pragma unroll
        for (int k = 0; k < KR; k++)
          if (k < rounds) first_rounds(k, site_util(k, G[k]));
        if (in_lds) {
          double g[S];
#pragma unroll
          for (int kk = 0; kk < S; kk++) g[kk] = at[64 * kk];
          first_rounds(KR, site_util(KR, g));
        }
        const int done = in_lds ? KR + 1 : KR;
        if (R == 4) {
          const double l = log(hold);
          const double l0 = dpp_f64<0x00>(l), l1 = dpp_f64<0x55>(l), l2 = dpp_f64<0xAA>(l);
          if (r == 0) {
            if (my < n_pairs) lsum += l0;
            if (my + stride < n_pairs) lsum += l1;
            if (in_lds && my + 2 * stride < n_pairs) lsum += l2;
          }
        }
#pragma unroll 1
        for (int k = done; k < rounds; k++) {
          const int p = my + k * stride;
          double g[S];
          if (nd) {
            distal(k, qc[sidx[(p < n_pairs ? p : 0) / R]] * S, g);
#pragma unroll
            for (int kk = 0; kk < S; kk++) scr.put(tile(GS, k), kk, g[kk]);
          } else {
#pragma unroll
            for (int kk = 0; kk < S; kk++) g[kk] = scr.get(tile(GS, k), kk);
          }
          const double u = site_util(k, g);
          if (p < n_pairs && r == 0) lsum += log(u);
        }
        lsum = wave_sum(lsum);
        if (lane == 0) sh->part[wv] = lsum;
        __syncthreads();  // B
        __syncthreads();  // A
        op = sh->op;
      }
    }
  }
  // op == CMD_EXIT
}

// ---------------------------------------------------------------------------
// master wave
// ---------------------------------------------------------------------------
template <typename Real, int R>
struct ProtMaster : ThreeTaxControl<ProtMaster<Real, R>> {
  using Ctl = ThreeTaxControl<ProtMaster<Real, R>>;
  using Ctl::M;
  using Ctl::pend_bl;
  using Ctl::dist_bl;
  using Ctl::prox_bl;
  using Ctl::c_pend;
  using Ctl::c_dist;
  using Ctl::c_prox;
  using Ctl::esum;
  using Ctl::last_ll;
  using Ctl::have_last;
  using Ctl::n_calls;
  using Ctl::n_probes;
  using Ctl::n_dist_probes;
  static constexpr int S = kProtS;
  // FP32 form: state-basis MFMA workers (pp_engine_prot32.h)
  static constexpr bool kF32 = std::is_same<Real, float>::value;
  ProtShared *sh;
  int *sidx;
  int lane, cap_sites, n_inf, n_sl;
  double log_R;

  __device__ __forceinline__ void init(char *smem, const DevModel *dm, int cap_pairs) {
    n_sl = dm->n_sl;
    sh = reinterpret_cast<ProtShared *>(smem);
    sidx = ProtLayout::sidx(smem);
    lane = threadIdx.x & 63;
    cap_sites = cap_pairs / R;
    n_inf = dm->n_inf;
    log_R = dm->log_R;
    c_pend = c_dist = c_prox = __builtin_nan("");
  }

  __device__ __forceinline__ void command(int op) {
    if (lane == 0) sh->op = op;
    __syncthreads();  // A
    if (op == CMD_EXIT) return;
    if constexpr (kF32) {
      if (op == CMD_PROBE || op == CMD_PROBE_DIST) __syncthreads();  // C: the workers built the FP32 tables
    }
    __syncthreads();  // B
  }

  // mask_reindex of the query's informative sites (core.ml:25-28,146-156),
  // then CMD_QUERY.  Returns M.
  __device__ __forceinline__ int load_query(const uint8_t *codes, int N, int q) {
    unsigned present = 0;
    const int total = mask_sites(codes, N, n_inf, N, sidx, present);
    if (lane == 0) {
      sh->M = total;
      sh->q = q;
    }
    M = total;
    if (total > 0 && total <= cap_sites) command(CMD_QUERY);
    return total;
  }

  // Glv.mask_into of darr[loc] / parr[loc] and their exponent totals.
  __device__ __forceinline__ void gather(int loc) {
    if (lane == 0) sh->loc = loc;
    command(CMD_GATHER);
    const long long es = wave_sum_ll(lane < kProtWorkers ? sh->ipart[lane] : 0);
    esum = scalar((double)es);
    c_dist = c_prox = __builtin_nan("");
    have_last = false;
  }

  // The exponentials of Diagd.multi_exp for the changed branch lengths.
  __device__ __forceinline__ void tables(bool new_pend, bool new_dist) {
    const int lane = fresh_lane();
    // one table per transition-matrix slice: rate (gamma) or category (CAT)
    if (new_dist) {
      for (int t = lane; t < 2 * n_sl * S; t += 64) {
        const int which = t / (n_sl * S), rem = t % (n_sl * S), r = rem / S, k = rem % S;
        const double e = exp((sh->rates[r] * (which ? dist_bl : prox_bl)) * sh->l[k]);
        (which ? sh->ed : sh->ep)[rem] = e;
      }
    }
    if (new_pend) {
      for (int t = lane; t < n_sl * S; t += 64) {
        const int r = t / S, k = t % S;
        sh->en[t] = exp((sh->rates[r] * pend_bl) * sh->l[k]);
      }
    }
  }

  // One likelihood probe (Model.log_like3 at the current three-taxon state).
  __device__ __forceinline__ double log_like() {
    const bool new_pend = wave_true(!(pend_bl == c_pend));
    const bool new_dist = wave_true(!(dist_bl == c_dist && prox_bl == c_prox));
    tables(new_pend, new_dist);
    if (lane == 0) {
      sh->tflags = (new_dist ? 1 : 0) | (new_pend ? 2 : 0);
      sh->tile_next = 0;
    }
    command(new_dist ? CMD_PROBE_DIST : CMD_PROBE);
    const double tot = sum_parts<kProtWorkers>(sh->part);  // in wave order
    c_pend = scalar(pend_bl);
    c_dist = scalar(dist_bl);
    c_prox = scalar(prox_bl);
    n_calls++;
    n_probes++;
    n_dist_probes += new_dist;
    const double ll = (tot - (double)M * log_R) + PP_LOG2 * (esum + 0.0);
    last_ll = scalar(ll);
    have_last = true;
    return ll;
  }
};

}  // namespace pp
