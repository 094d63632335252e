// Master/worker three-taxon engine (nucleotide models, S = 4).
//
// A workgroup is one master wave (wave 0) plus W worker waves.  The master
// runs pplacer's sequential control -- baseball (core.ml:283-320),
// Three_tax.optimize (three_tax.ml:70-83), Minimization.brent with the GSL
// Brent minimiser (minimization.ml:11-100) -- on wave-uniform registers, and
// builds each probe's transition matrices and evolved pendant rows with its 64
// lanes (Diagd.multi_exp, diagd.ml:79-100; gemmish_c, linear_c.c:29-90).  Lane
// j of worker wave w holds, in registers, the distal and proximal GLV rows of
// the current edge (Glv.mask_into, gmix_model.ml:121-141) at its masked
// sites; the cached (pi*prox_ev)*dist_ev products of ten_log_like3_c
// (linear_c.c:367-424) are kept in LDS.  Each command is one LDS word and two
// barriers:
//
//   master: [tables, command] -> barrier A -> .............................. -> barrier B -> [sum]
//   worker: ..................   barrier A -> [site work, wave partial sum] -> barrier B
//
// (Price-CAT: every wave builds a share of the tables behind barrier A, with a
// barrier C before the site work.)
//
// With SPL sites per lane, worker lane j of wave w holds masked sites
// 64*(w-1)+j + k*64*W for k < SPL.  Queries longer than the registers and LDS
// of a workgroup hold take the streaming form (SPL = 0): a worker lane walks
// its sites 64*(w-1)+j + k*64*W for every k, re-reads the rows from the
// resident GLV arrays at each distal probe and keeps the cached products in a
// per-workgroup global scratch, so any masked length fits.
//
// Control state and site data live in different waves, so the register
// allocator sizes the kernel for max(control, data) rather than their sum;
// that sets how many queries a CU holds at once.
//
// Arithmetic order is the C stubs': each evolved entry is a sequential sum
// over j of P[i][j]*src[j]; each site's util the sequential (rate, state) sum
// of ((pi*prox)*dist)*pend; P entries the sequential sum over k of
// (exp(rate*bl*l_k)*x[i][k])*xit[j][k].  The FP64 form rounds every product
// and sum separately (-ffp-contract=off) and sums the per-site logs as the
// stub does, sequentially in masked-site order (linear_c.c:416-419): workers
// leave each site's log in LDS and, behind barrier B, the master wave
// reproduces that sum bit for bit (wave_sequential_sum).  The FP32 form uses
// FMAs and sums the logs (in FP64) per wave, then in wave order.
#pragma once

#include <climits>
#include <type_traits>

#include "pp_engine.h"
#include "pp_engine_ctl.h"
#include "pp_exact_sum.h"

namespace pp {

// CMD_PROBE_DIST: a probe whose proximal/distal lengths changed (re-evolve)
enum { CMD_EXIT = 0, CMD_QUERY = 1, CMD_GATHER = 2, CMD_PROBE = 3, CMD_PROBE_DIST = 4 };

struct MWShared {
  double x[16], l[4], xit[16], statd[4], rates[kMaxRates];
  double lv[kNucCodes * 4];
  int op, n_slots, M, q, loc;
  // character code -> pendant row of this query; the one-hot characters
  // (codes 0-3) always use rows 0-3
  int code_slot[kNucCodes];
  int slot_code[kNucCodes];
  // Price-CAT: the proximal, distal and pendant lengths whose tables a probe
  // builds (tflags bit 0: the first two, bit 1: the third)
  double bl[3];
  int tflags;
  double part[16];           // per-worker-wave sums of site logs, 0.0 past the workers
  long long ipart[16];       // per-worker-wave sums of site exponents
};

// LDS of one workgroup: shared header, pendant rows [n_tsl][kTable], P(prox)
// and P(dist) [n_sl][kP], then per masked site (cap = the longest masked length the launch takes): the
// site's log of a probe (FP64 form, rounded up to whole blocks of 64), its
// column (the masked-site list) and in the streaming form its pendant row.
// Gamma model: n_tsl = 1, n_sl = R (rate r uses slice r); Price-CAT: R = 1
// and n_tsl = n_sl = n_cats (a site uses its category's).
template <typename Real, int R, bool STRICT>
struct MWLayout {
  static constexpr int RS = R * 4;
  static constexpr size_t head = (sizeof(MWShared) + 15) & ~size_t(15);
  // Reals from one pendant row, one transition-matrix slice to the next: 16
  // bytes of padding keep the rows that a wave's lanes read at once (one per
  // character, one per rate or category) in different banks
  static constexpr int kPad = 16 / (int)sizeof(Real);
  static constexpr int kT = RS + (R == 4 ? kPad : 0), kP = 16 + kPad;
  static constexpr int kTable = kNucCodes * kT + (R == 4 ? 0 : 4);  // one category's pendant rows
  static constexpr bool strict = STRICT;  // site logs summed in site order
  int n_tsl, n_sl, cap;
  bool stream;
  MWLayout() = default;
  __host__ __device__ MWLayout(int n_tsl_, int n_sl_, int cap_, bool stream_)
      : n_tsl(n_tsl_), n_sl(n_sl_), cap(cap_), stream(stream_) {}
  __host__ __device__ size_t tbytes() const { return sizeof(Real) * (size_t)n_tsl * kTable; }
  __host__ __device__ size_t pbytes() const { return sizeof(Real) * (size_t)n_sl * kP; }
  __host__ __device__ size_t off_slog() const { return head + tbytes() + 2 * pbytes(); }
  __host__ __device__ size_t off_sidx() const {
    return off_slog() + (strict ? sizeof(double) * (size_t)((cap + 63) & ~63) : 0);
  }
  __host__ __device__ size_t bytes() const { return off_sidx() + sizeof(int) * (size_t)cap * (stream ? 2 : 1); }
  __device__ Real *T(char *s) const { return reinterpret_cast<Real *>(s + head); }
  __device__ Real *Pp(char *s) const { return reinterpret_cast<Real *>(s + head + tbytes()); }
  __device__ Real *Pd(char *s) const { return reinterpret_cast<Real *>(s + head + tbytes() + pbytes()); }
  __device__ double *slog(char *s) const { return reinterpret_cast<double *>(s + off_slog()); }
  __device__ int *sidx(char *s) const { return reinterpret_cast<int *>(s + off_sidx()); }
  __device__ int *sslot(char *s) const { return reinterpret_cast<int *>(s + off_sidx()) + cap; }
  static __host__ __device__ size_t align(size_t off) { return (off + 15) & ~size_t(15); }
};

template <typename Real, int R, bool STRICT>
__device__ __forceinline__ MWLayout<Real, R, STRICT> mw_layout(const DevModel *dm, int cap, bool stream) {
  return MWLayout<Real, R, STRICT>(dm->cat ? dm->n_sl : 1, dm->n_sl, cap, stream);
}

// Wave-uniform branch on the wave index (wave 0 = master).
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ __forceinline__ void mw_copy_model(MWShared *sh, const DevModel *dm) {
  for (int t = threadIdx.x; t < 16; t += blockDim.x) { sh->x[t] = dm->x[t]; sh->xit[t] = dm->xit[t]; }
  for (int t = threadIdx.x; t < 4; t += blockDim.x) { sh->l[t] = dm->l[t]; sh->statd[t] = dm->statd[t]; }
  for (int t = threadIdx.x; t < kMaxRates; t += blockDim.x) sh->rates[t] = dm->rates[t];
  for (int t = threadIdx.x; t < 16; t += blockDim.x) sh->part[t] = 0.0;
  for (int t = threadIdx.x; t < min(dm->n_codes, kNucCodes) * 4; t += blockDim.x) sh->lv[t] = dm->lv[t];
}

// One lane's entry of P(t) from its quad's exponentials e (lane k holds that of
// eigenvalue k) and its rows of x and xit: the sum over k in order.
__device__ __forceinline__ double p_entry(double e, const double (&mx)[4], const double (&mxit)[4]) {
  double acc = 0.0;
  acc = acc + (dpp_f64<0x00>(e) * mx[0]) * mxit[0];
  acc = acc + (dpp_f64<0x55>(e) * mx[1]) * mxit[1];
  acc = acc + (dpp_f64<0xAA>(e) * mx[2]) * mxit[2];
  acc = acc + (dpp_f64<0xFF>(e) * mx[3]) * mxit[3];
  return acc;
}

// Ambiguity codes present in the query: entry (r, i) of rows 4.. by the
// stub's sum over the row's P entries p, which a quad's lanes hold; lane j
// takes every fourth row.  The whole wave calls; `at` is row 0's entry, rows
// `stride` apart.
template <typename Real>
__device__ __forceinline__ void ambiguity_rows(const MWShared *sh, int n_amb, double p, bool active, Real *at,
                                               int stride) {
  const double p0 = dpp_f64<0x00>(p), p1 = dpp_f64<0x55>(p), p2 = dpp_f64<0xAA>(p), p3 = dpp_f64<0xFF>(p);
  if (active)
    for (int slot = 4 + (fresh_lane() & 3); slot < 4 + n_amb; slot += 4) {
      const double *lv = sh->lv + sh->slot_code[slot] * 4;
      double acc = 0.0;
      acc = acc + p0 * lv[0];
      acc = acc + p1 * lv[1];
      acc = acc + p2 * lv[2];
      acc = acc + p3 * lv[3];
      at[slot * stride] = (Real)acc;
    }
}

// The exponentials of P(t): correctly rounded where the site logs are
// summed in site order (the FP64 form), as the stubs' libm returns them;
// the library's otherwise.
template <bool STRICT>
__device__ __forceinline__ double table_exp(double v) {
  if constexpr (STRICT) return cr::exp(v);
  else return exp(v);
}

// A wave's share of a Price-CAT probe's tables (sh->bl, sh->tflags): the
// slices of categories 4 w .. 4 w + 3, then every 4 waves' further, lane
// (category mod 4) 16 + 4 i + j taking entry (i, j) as the gamma model's does.
// With up to 20 categories every wave of a five-wave workgroup builds at most
// one group, in 1,900 cycles with the barrier; by the control wave alone, with
// the others waiting, the tables took 4,280 of a probe's 10,250 cycles (2,000
// 16S reads 14.7 -> 11.9 ms).
template <typename Real, bool STRICT>
__device__ __forceinline__ void cat_tables(const MWShared *sh, const MWLayout<Real, 1, STRICT> &lay, char *smem) {
  using L = MWLayout<Real, 1, STRICT>;
  const int lane = fresh_lane(), fl = __builtin_amdgcn_readfirstlane(sh->tflags);
  const int n_sl = lay.n_sl, n_amb = __builtin_amdgcn_readfirstlane(sh->n_slots) - 4;
  const int i = (lane >> 2) & 3, j = lane & 3;
  const double m_l = sh->l[j];
  double mx[4], mxit[4];  // the lane's row of x and of xit
#pragma unroll
  for (int k = 0; k < 4; k++) {
    mx[k] = sh->x[i * 4 + k];
    mxit[k] = sh->xit[j * 4 + k];
  }
  // (whole waves: quads exchange exponentials and entries)
#pragma unroll 1
  for (int s0 = 4 * wave_id(); s0 < n_sl; s0 += (int)blockDim.x >> 4) {
    const int s = s0 + (lane >> 4);
    const bool in = s < n_sl;
    const double rate = sh->rates[in ? s : 0];
    if (fl & 1) {
      const double p = p_entry(table_exp<STRICT>((rate * sh->bl[0]) * m_l), mx, mxit);
      const double d = p_entry(table_exp<STRICT>((rate * sh->bl[1]) * m_l), mx, mxit);
      if (in) {
        lay.Pp(smem)[s * L::kP + (lane & 15)] = (Real)p;
        lay.Pd(smem)[s * L::kP + (lane & 15)] = (Real)d;
      }
    }
    if (fl & 2) {
      const double p = p_entry(table_exp<STRICT>((rate * sh->bl[2]) * m_l), mx, mxit);
      Real *t = lay.T(smem) + s * L::kTable;
      if (in) t[j * 4 + i] = (Real)p;  // one-hot row j, entry i
      if (n_amb > 0) ambiguity_rows<Real>(sh, n_amb, (double)(Real)p, in, t + i, L::kT);
    }
  }
}

// ---------------------------------------------------------------------------
// worker waves
// ---------------------------------------------------------------------------

// The cached products of masked site i live in LDS in groups of four sites:
// byte (i/4)*kGroupBytes + t*4*sizeof(Real) + (i%4)*sizeof(Real).  Each lane's
// sixteen products are immediate offsets from one address, and the 32-byte pad
// per group spreads a wave's accesses over all banks.
template <typename Real, int RS>
struct MWProducts {
  static constexpr int kGroupBytes = RS * 4 * (int)sizeof(Real) + 32;
  static __host__ __device__ size_t bytes(int sites) { return (size_t)((sites + 3) / 4) * kGroupBytes; }
  static __device__ __forceinline__ int base(int i) { return (i >> 2) * kGroupBytes + (i & 3) * (int)sizeof(Real); }
  static __device__ __forceinline__ Real &at(char *wl, int base, int t) {
    return *reinterpret_cast<Real *>(wl + base + t * 4 * (int)sizeof(Real));
  }
};

// One masked site of a CMD_PROBE_DIST: evolve the proximal and distal rows
// by P(prox) and P(dist) (sequential sums over j), form each (rate, state)
// product ((pi*prox_ev)*dist_ev), hand it to keep(t, value) and accumulate
// util = sum over (rate, state) of product*pend in that order.  pp / pd are
// the site's P slices (for Price-CAT, where R is 1, its category's; else rate
// r's slice is pp + P r), z its evolved pendant row.
template <typename Real, int R, int P, class Keep>
__device__ __forceinline__ Real site_dist_util(const Real *pp, const Real *pd, const Real *z,
                                               const double *statd, const Real (&pO)[R * 4],
                                               const Real (&dO)[R * 4], Keep &&keep) {
  using Ops = RealOps<Real>;
  Real util = 0;
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const Real *ppr = pp + r * P + i * 4, *pdr = pd + r * P + i * 4;
      const Real pi = (Real)statd[i];
      const int t = r * 4 + i;
      Real xv = ppr[0] * pO[r * 4], yv = pdr[0] * dO[r * 4];
#pragma unroll
      for (int j = 1; j < 4; j++) {
        xv = Ops::madd(xv, ppr[j], pO[r * 4 + j]);
        yv = Ops::madd(yv, pdr[j], dO[r * 4 + j]);
      }
      const Real w = (pi * xv) * yv;
      keep(t, w);
      // sums start from their first product: 0 + p == p up to the sign of a
      // zero, which no later operation can observe
      util = t == 0 ? w * z[t] : Ops::madd(util, w, z[t]);
    }
  return util;
}

// part[0] + part[1] + ... + part[N-1], N the workers of the launch class: a
// chain of N additions of values read at once, where a loop over the waves
// there are took two lane reads and a wait for each (40 cycles; 1,500 proteins
// in FP64 33.8 -> 32.9 ms).
template <int N>
__device__ __forceinline__ double sum_parts(const double *part) {
  double v[N];
#pragma unroll
  for (int w = 0; w < N; w++) v[w] = part[w];
  double tot = v[0];
#pragma unroll
  for (int w = 1; w < N; w++) tot += v[w];
  return tot;
}

// Orders one wave's LDS writes before its later LDS reads of other lanes'
// entries (LDS executes a wave's operations in order).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// CAT: Price-CAT, R == 1, site k uses P slice and pendant table sl[k] = its
// category (site_cat); otherwise slice r for rate r and pendant table 0.
// FP64 (strict): each site's log goes to slog (0.0 past the query's sites),
// where the master adds them as the stub does, in site order with one
// rounding per term (wave_sequential_sum); FP32: the lane's logs are summed
// and reduced per wave.
template <typename Real, int R, int SPL, bool CAT, bool STRICT>
__device__ __forceinline__ void mw_worker(char *smem, const MWLayout<Real, R, STRICT> &lay, char *wl, int N,
                                          const uint8_t *codes, const Real *darr, const Real *parr,
                                          const int *darr_e, const int *parr_e, const int *site_cat) {
  constexpr int RS = R * 4;
  constexpr bool strict = STRICT;
  static_assert(R == 1, "one rate; four rates take mw_worker_rates");
  static_assert(SPL >= 1, "register-resident form");
  using L = MWLayout<Real, R, STRICT>;
  using W = MWProducts<Real, RS>;
  using Ops = RealOps<Real>;
  MWShared *sh = reinterpret_cast<MWShared *>(smem);
  const Real *sT = lay.T(smem), *sPp = lay.Pp(smem), *sPd = lay.Pd(smem);
  const int *sidx = lay.sidx(smem);
  double *slog = lay.slog(smem);
  const int lane = threadIdx.x & 63;
  const int wv = wave_id() - 1;
  const int stride = (int)blockDim.x - 64;  // worker lanes
  const int my = wv * 64 + lane;
  int site[SPL], slot[SPL], wb[SPL], sl[SPL];
  bool active[SPL];
#pragma unroll
  for (int k = 0; k < SPL; k++) wb[k] = W::base(my + k * stride);
  // The command stream is QUERY (GATHER PROBE*)* ... EXIT; the nested loops
  // follow it, so each edge's rows are defined once per GATHER and stay in
  // place through that edge's probes.
  __syncthreads();  // A
  int op = sh->op;
  while (op == CMD_QUERY) {
#pragma unroll
    for (int k = 0; k < SPL; k++) {
      const int i = my + k * stride;
      active[k] = i < sh->M;
      site[k] = active[k] ? sidx[i] : 0;
      sl[k] = CAT ? site_cat[site[k]] : 0;
      // pendant row of the site: table sl, character slot
      slot[k] = sl[k] * L::kTable + (active[k] ? sh->code_slot[codes[(size_t)sh->q * N + site[k]]] : 0) * L::kT;
    }
    __syncthreads();  // B
    __syncthreads();  // A
    op = sh->op;
    while (op == CMD_GATHER) {
      // Inactive slots load row 0 (any valid row).
      Real dO[SPL][RS], pO[SPL][RS];
      long long es = 0;
#pragma unroll
      for (int k = 0; k < SPL; k++) {
        const size_t row = active[k] ? (size_t)sh->loc * N + site[k] : 0;
        const Real *d = darr + row * RS;
        const Real *p = parr + row * RS;
#pragma unroll
        for (int t = 0; t < RS; t++) { dO[k][t] = d[t]; pO[k][t] = p[t]; }
        if (active[k]) es += (long long)darr_e[row] + (long long)parr_e[row];
      }
      es = wave_sum_ll(es);
      if (lane == 0) sh->ipart[wv] = es;
      __syncthreads();  // B
      __syncthreads();  // A
      op = sh->op;
      while (op == CMD_PROBE || op == CMD_PROBE_DIST) {
        if constexpr (CAT) {
          cat_tables<Real, STRICT>(sh, lay, smem);
          __syncthreads();  // C
        }
        Real util[SPL];
        if (op == CMD_PROBE_DIST) {
#pragma unroll
          for (int k = 0; k < SPL; k++) {
            const int o = CAT ? sl[k] * L::kP : 0;
            util[k] = site_dist_util<Real, R, L::kP>(sPp + o, sPd + o, sT + slot[k], sh->statd, pO[k], dO[k],
                                                   [&](int t, Real w) { W::at(wl, wb[k], t) = w; });
          }
        } else {
#pragma unroll
          for (int t = 0; t < RS; t++)
#pragma unroll
            for (int k = 0; k < SPL; k++) {
              const Real w = W::at(wl, wb[k], t), z = sT[slot[k] + t];
              util[k] = t == 0 ? w * z : Ops::madd(util[k], w, z);
            }
        }
        if constexpr (strict) {
#pragma unroll
          for (int k = 0; k < SPL; k++)
            slog[my + k * stride] = active[k] ? Ops::logs(util[k]) : 0.0;
        } else {
          double lsum = 0.0;
#pragma unroll
          for (int k = 0; k < SPL; k++)
            if (active[k]) lsum += Ops::logd(util[k]);
          lsum = wave_sum(lsum);
          if (lane == 0) sh->part[wv] = lsum;
        }
        __syncthreads();  // B
        __syncthreads();  // A
        op = sh->op;
      }
    }
  }
  // op == CMD_EXIT
}

// The worker of the four-rate gamma model.  Two layouts of a wave's 64 SPL
// sites:
//  * evolves (CMD_PROBE_DIST): lane 4 q + r holds rate r of sites 16 k + q, k <
//    4 SPL.  The R quarters of a 128-byte (FP64) row sit in one quad, so a
//    gather reads whole rows from consecutive lanes, and an entry of P is read
//    from LDS once for 4 SPL sites instead of once per site, whose sums are
//    independent chains.  With a lane per site the gather touched 64 lines per
//    load and the evolve waited for LDS at each of its 16 (rate, state) pairs.
//  * util and log: lane j owns site j (+ 64), as the sum over (rate, state) is
//    sequential in a site.  The products pass through LDS, where they are kept
//    for the pendant-only probes (three quarters of all) in any case.
template <typename Real, int SPL, bool STRICT>
__device__ __forceinline__ void mw_worker_rates(char *smem, const MWLayout<Real, 4, STRICT> &lay, char *wl, int N,
                                                const uint8_t *codes, const Real *darr, const Real *parr,
                                                const int *darr_e, const int *parr_e) {
  constexpr int RS = 16, K = 4 * SPL, KW = 8 / SPL;
  using L = MWLayout<Real, 4, STRICT>;
  using W = MWProducts<Real, RS>;
  using Ops = RealOps<Real>;
  MWShared *sh = reinterpret_cast<MWShared *>(smem);
  const int *sidx = lay.sidx(smem);
  double *slog = lay.slog(smem);
  const int lane = threadIdx.x & 63;
  const int wv = wave_id() - 1;
  const int first = wv * 64 * SPL;  // the wave's first site
  const int r = lane & 3, q = lane >> 2;
  const Real *sPp = lay.Pp(smem) + r * L::kP, *sPd = lay.Pd(smem) + r * L::kP;
  const Real *z[SPL];
  Real pi[4];
#pragma unroll
  for (int i = 0; i < 4; i++) pi[i] = (Real)scalar(sh->statd[i]);
  // products of site first + 16 k + q: this address + 16 k sites (four groups)
  char *wq = wl + W::base(first + q) + r * 16 * (int)sizeof(Real);
  __syncthreads();  // A
  int op = sh->op;
  while (op == CMD_QUERY) {
    const int M = sh->M;
#pragma unroll
    for (int k = 0; k < SPL; k++) {
      const int i = first + 64 * k + lane;
      z[k] = lay.T(smem) + (i < M ? sh->code_slot[codes[(size_t)sh->q * N + sidx[i]]] : 0) * L::kT;
    }
    __syncthreads();  // B
    __syncthreads();  // A
    op = sh->op;
    while (op == CMD_GATHER) {
      const size_t row0 = (size_t)sh->loc * N;
      Real dO[K][4], pO[K][4];
      // sites past the query's read the row of column 0 (any valid row)
#pragma unroll
      for (int k = 0; k < K; k++) {
        const int i = first + 16 * k + q;
        const size_t at = (row0 + (i < M ? sidx[i] : 0)) * RS + r * 4;
#pragma unroll
        for (int j = 0; j < 4; j++) { dO[k][j] = darr[at + j]; pO[k][j] = parr[at + j]; }
      }
      long long es = 0;
#pragma unroll
      for (int k = 0; k < SPL; k++) {
        const int i = first + 64 * k + lane;
        if (i < M) es += (long long)darr_e[row0 + sidx[i]] + (long long)parr_e[row0 + sidx[i]];
      }
      es = wave_sum_ll(es);
      if (lane == 0) sh->ipart[wv] = es;
      __syncthreads();  // B
      __syncthreads();  // A
      op = sh->op;
      // The first products and pendant entries are asked for together with the
      // command (a distal probe makes the products anew): one LDS latency less
      // on a probe's path, one read 2.08 -> 2.05 ms
      Real w0[KW][SPL], z0[KW][SPL];
      const auto ask = [&] {
#pragma unroll
        for (int t = 0; t < KW; t++)
#pragma unroll
          for (int k = 0; k < SPL; k++) {
            w0[t][k] = W::at(wl + W::base(first + 64 * k + lane), 0, t);
            z0[t][k] = z[k][t];
          }
      };
      ask();
      while (op == CMD_PROBE || op == CMD_PROBE_DIST) {
        if (op == CMD_PROBE_DIST) {
#pragma unroll
          for (int i = 0; i < 4; i++) {
            Real pp[4], pd[4];
#pragma unroll
            for (int j = 0; j < 4; j++) { pp[j] = sPp[i * 4 + j]; pd[j] = sPd[i * 4 + j]; }
#pragma unroll
            for (int k = 0; k < K; k++) {
              Real xv = pp[0] * pO[k][0], yv = pd[0] * dO[k][0];
#pragma unroll
              for (int j = 1; j < 4; j++) {
                xv = Ops::madd(xv, pp[j], pO[k][j]);
                yv = Ops::madd(yv, pd[j], dO[k][j]);
              }
              W::at(wq + k * 4 * W::kGroupBytes, 0, i) = (pi[i] * xv) * yv;
            }
          }
          wave_lds_sync();  // a site's products come from its quad's lanes
#pragma unroll
          for (int t = 0; t < KW; t++)
#pragma unroll
            for (int k = 0; k < SPL; k++) w0[t][k] = W::at(wl + W::base(first + 64 * k + lane), 0, t);
        }
        Real util[SPL];
#pragma unroll
        for (int t = 0; t < RS; t++)
#pragma unroll
          for (int k = 0; k < SPL; k++) {
            const Real w = t < KW ? w0[t < KW ? t : 0][k] : W::at(wl + W::base(first + 64 * k + lane), 0, t);
            const Real zt = t < KW ? z0[t < KW ? t : 0][k] : z[k][t];
            // the sum starts from its first product: 0 + p == p up to the sign
            // of a zero, which no later operation can observe
            util[k] = t == 0 ? w * zt : Ops::madd(util[k], w, zt);
          }
        if constexpr (STRICT) {
#pragma unroll
          for (int k = 0; k < SPL; k++) {
            const int i = first + 64 * k + lane;
            slog[i] = i < M ? Ops::logs(util[k]) : 0.0;
          }
        } else {
          double lsum = 0.0;
#pragma unroll
          for (int k = 0; k < SPL; k++)
            if (first + 64 * k + lane < M) lsum += Ops::logd(util[k]);
          lsum = wave_sum(lsum);
          if (lane == 0) sh->part[wv] = lsum;
        }
        __syncthreads();  // B
        __syncthreads();  // A
        op = sh->op;
        ask();
      }
    }
  }
  // op == CMD_EXIT
}

// Streaming form of the worker for masked lengths beyond the register-resident
// form: lane j of worker wave w walks sites i = 64 (w-1) + j + k W64 for every
// k while i < M.  The distal and proximal rows are read from darr / parr at
// each distal probe (one 16-value row each), and the products cached for the
// pendant-only probes live in prod[t * cap + i] (per-workgroup global scratch,
// consecutive sites in consecutive addresses).  Same arithmetic as mw_worker.
template <typename Real, int R, bool CAT, bool STRICT>
__device__ __forceinline__ void mw_worker_stream(char *smem, const MWLayout<Real, R, STRICT> &lay, Real *prod, int cap,
                                                 int N, const uint8_t *codes, const Real *darr,
                                                 const Real *parr, const int *darr_e, const int *parr_e,
                                                 const int *site_cat) {
  constexpr int RS = R * 4;
  constexpr bool strict = STRICT;
  static_assert(!CAT || R == 1, "Price-CAT GLVs have no rate axis");
  using L = MWLayout<Real, R, STRICT>;
  using Ops = RealOps<Real>;
  MWShared *sh = reinterpret_cast<MWShared *>(smem);
  const Real *sT = lay.T(smem), *sPp = lay.Pp(smem), *sPd = lay.Pd(smem);
  const int *sidx = lay.sidx(smem);
  int *sslot = lay.sslot(smem);
  double *slog = lay.slog(smem);
  const int lane = threadIdx.x & 63;
  const int wv = wave_id() - 1;
  const int stride = (int)blockDim.x - 64;
  const int my = wv * 64 + lane;
  __syncthreads();  // A
  int op = sh->op;
  while (op == CMD_QUERY) {
    const int M = sh->M, q = sh->q;
    // the sum reads whole blocks of 64: zeros past the query's sites
    if constexpr (strict)
      if (my < 64 && M + my < ((M + 63) & ~63)) slog[M + my] = 0.0;
    for (int i = my; i < M; i += stride) {
      const int site = sidx[i];
      const int sl = CAT ? site_cat[site] : 0;
      sslot[i] = sl * L::kTable + sh->code_slot[codes[(size_t)q * N + site]] * L::kT;
    }
    __syncthreads();  // B
    __syncthreads();  // A
    op = sh->op;
    while (op == CMD_GATHER) {
      const size_t rowbase = (size_t)sh->loc * N;
      long long es = 0;
      for (int i = my; i < M; i += stride) {
        const size_t row = rowbase + sidx[i];
        es += (long long)darr_e[row] + (long long)parr_e[row];
      }
      es = wave_sum_ll(es);
      if (lane == 0) sh->ipart[wv] = es;
      __syncthreads();  // B
      __syncthreads();  // A
      op = sh->op;
      while (op == CMD_PROBE || op == CMD_PROBE_DIST) {
        if constexpr (CAT) {
          cat_tables<Real, STRICT>(sh, lay, smem);
          __syncthreads();  // C
        }
        double lsum = 0.0;
        for (int i = my; i < M; i += stride) {
          const int slot = sslot[i];
          const Real *z = sT + slot;
          Real util;
          if (op == CMD_PROBE_DIST) {
            const int site = sidx[i];
            const size_t row = rowbase + site;
            Real dO[RS], pO[RS];
#pragma unroll
            for (int t = 0; t < RS; t++) { dO[t] = darr[row * RS + t]; pO[t] = parr[row * RS + t]; }
            const int o = CAT ? (slot / L::kTable) * L::kP : 0;
            util = site_dist_util<Real, R, L::kP>(sPp + o, sPd + o, z, sh->statd, pO, dO,
                                                [&](int t, Real w) { prod[(size_t)t * cap + i] = w; });
          } else {
#pragma unroll
            for (int t = 0; t < RS; t++) {
              const Real w = prod[(size_t)t * cap + i];
              util = t == 0 ? w * z[t] : Ops::madd(util, w, z[t]);
            }
          }
          if constexpr (strict) slog[i] = Ops::logs(util);
          else lsum += Ops::logd(util);
        }
        if constexpr (!strict) {
          lsum = wave_sum(lsum);
          if (lane == 0) sh->part[wv] = lsum;
        }
        __syncthreads();  // B
        __syncthreads();  // A
        op = sh->op;
      }
    }
  }
  // op == CMD_EXIT
}

// The informative columns of a query in order, list[0 .. cap) of them, by one
// wave: 64 consecutive columns at a time, a column's place from the ballot of
// those before it, eight loads in flight.  Returns how many there are (beyond
// cap, too) and the lane's codes in `present`.
__device__ __forceinline__ int mask_sites(const uint8_t *codes, int N, int n_inf, int cap, int *list,
                                          unsigned &present) {
  const int lane = fresh_lane();
  int total = 0;
  for (int k0 = 0; k0 < N; k0 += 512) {
    int c[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int k = k0 + 64 * u + lane;
      c[u] = k < N ? (int)codes[k] : n_inf;
    }
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const bool in = c[u] < n_inf;
      const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
      if (in) {
        const int pos = total + (int)__builtin_popcountll(m & ~(~0ull << lane));
        if (pos < cap) list[pos] = k0 + 64 * u + lane;
        present |= 1u << c[u];
      }
      total += __builtin_popcountll(m);
    }
  }
  return total;
}

// ---------------------------------------------------------------------------
// master wave
// ---------------------------------------------------------------------------
template <typename Real, int R, int MAXBD, int SPL, bool CAT, bool STRICT>
struct MWMaster : ThreeTaxControl<MWMaster<Real, R, MAXBD, SPL, CAT, STRICT>> {
  using Ctl = ThreeTaxControl<MWMaster<Real, R, MAXBD, SPL, CAT, STRICT>>;
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
  using L = MWLayout<Real, R, STRICT>;
  static constexpr int RS = R * 4;
  MWShared *sh;
  Real *sT, *sPp, *sPd;
  const double *slog;
  int *sidx;
  int lane, n_workers, cap_sites, n_codes, n_inf, n_sl;
  int n_amb;  // ambiguity codes present in the query
  double log_R;
  char *smem;
  L lay;

  // cap: the longest masked length the launch takes (the layout's capacity)
  __device__ __forceinline__ void init(char *smem_, const DevModel *dm, int cap) {
    smem = smem_;
    lay = mw_layout<Real, R, STRICT>(dm, cap, SPL == 0);
    sh = reinterpret_cast<MWShared *>(smem);
    sT = lay.T(smem);
    sPp = lay.Pp(smem);
    sPd = lay.Pd(smem);
    slog = lay.slog(smem);
    sidx = lay.sidx(smem);
    n_sl = dm->n_sl;
    lane = threadIdx.x & 63;
    n_workers = (int)(blockDim.x >> 6) - 1;
    cap_sites = cap;
    n_codes = dm->n_codes;
    n_inf = dm->n_inf;
    log_R = dm->log_R;
    n_amb = 0;
    c_pend = c_dist = c_prox = __builtin_nan("");
  }

  __device__ __forceinline__ void command(int op) {
    if (lane == 0) sh->op = op;
    __syncthreads();  // A
    if (op == CMD_EXIT) return;
    if constexpr (CAT)
      if (op == CMD_PROBE || op == CMD_PROBE_DIST) {
        cat_tables<Real, STRICT>(sh, lay, smem);
        __syncthreads();  // C
      }
    __syncthreads();  // B
  }

  // mask_reindex of the query's informative sites (core.ml:25-28,146-156),
  // the set of characters present (their evolved rows are all a probe
  // needs), then CMD_QUERY.  Returns M.
  __device__ __forceinline__ int load_query(const uint8_t *codes, int N, int q) {
    unsigned present = 0;
    const int total = mask_sites(codes, N, n_inf, cap_sites, sidx, present);
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) present |= __shfl_xor(present, m, 64);
    if (lane == 0) {
      int ns = 4;
      for (int c = 0; c < n_codes; c++) {
        if (c < 4) { sh->code_slot[c] = c; sh->slot_code[c] = c; continue; }
        sh->code_slot[c] = (present >> c) & 1u ? ns : 0;
        if ((present >> c) & 1u) sh->slot_code[ns++] = c;
      }
      sh->n_slots = ns;
      sh->M = total;
      sh->q = q;
    }
    M = total;
    n_amb = __builtin_popcount(__builtin_amdgcn_readfirstlane(present) >> 4);
    c_pend = __builtin_nan("");  // the pendant rows are per query
    if (total > 0 && total <= cap_sites) command(CMD_QUERY);
    return total;
  }

  // Glv.mask_into of darr[loc] / parr[loc] and their exponent totals.
  __device__ __forceinline__ void gather(int loc) {
    if (lane == 0) sh->loc = loc;
    command(CMD_GATHER);
    const long long es = wave_sum_ll(fresh_lane() < n_workers ? sh->ipart[fresh_lane()] : 0);
    esum = scalar((double)es);
    c_dist = c_prox = __builtin_nan("");
    have_last = false;
  }

  // Diagd.multi_exp for the changed branch lengths and the evolved pendant
  // rows of the characters present, with the master's 64 lanes: lane r*16 +
  // i*4 + j owns entry (i, j) of rate r's matrices.  It takes the exponential
  // of k = j, and a quad's four exponentials reach its lanes through DPP, so
  // nothing is staged in LDS on the probe's critical path.
  __device__ __forceinline__ void tables(bool new_pend, bool new_dist) {
    if constexpr (CAT) {  // built by all waves once the command is out
      if (fresh_lane() == 0) {
        sh->bl[0] = prox_bl;
        sh->bl[1] = dist_bl;
        sh->bl[2] = pend_bl;
        sh->tflags = (new_dist ? 1 : 0) | (new_pend ? 2 : 0);
      }
      return;
    }
    const int lane = fresh_lane();
    const double m_rate = sh->rates[(lane >> 4) & (R - 1)], m_l = sh->l[lane & 3];
    double mx[4], mxit[4];  // the lane's row of x and of xit
#pragma unroll
    for (int k = 0; k < 4; k++) {
      mx[k] = sh->x[(lane & 12) + k];
      mxit[k] = sh->xit[(lane & 3) * 4 + k];
    }
    if (new_dist) {
      const double p = p_entry(table_exp<STRICT>((m_rate * prox_bl) * m_l), mx, mxit);
      const double d = p_entry(table_exp<STRICT>((m_rate * dist_bl) * m_l), mx, mxit);
      if (lane < R * 16) {
        sPp[(lane >> 4) * L::kP + (lane & 15)] = (Real)p;
        sPd[(lane >> 4) * L::kP + (lane & 15)] = (Real)d;
      }
    }
    if (new_pend) {
      const double p = p_entry(table_exp<STRICT>((m_rate * pend_bl) * m_l), mx, mxit);
      const int j = lane & 3, ri = (lane >> 2) & (R * 4 - 1);
      // One-hot characters: their evolved rows are columns of P (every other
      // product in gemmish_c is an exact zero), row j entry (r, i) = P[r][i][j].
      if (lane < R * 16) sT[j * L::kT + ri] = (Real)p;
      if (n_amb > 0) ambiguity_rows<Real>(sh, n_amb, p, lane < R * 16, sT + ri, L::kT);
    }
  }

  // One likelihood probe (Model.log_like3 at the current three-taxon state).
  __device__ __forceinline__ double log_like() {
    const bool new_pend = wave_true(!(pend_bl == c_pend));
    const bool new_dist = wave_true(!(dist_bl == c_dist && prox_bl == c_prox));
    tables(new_pend, new_dist);
    command(new_dist ? CMD_PROBE_DIST : CMD_PROBE);
    double tot;
    if constexpr (L::strict) {
      tot = wave_sequential_sum<SPL == 0 ? INT_MAX : SPL * (MAXBD - 64)>(slog, M);
    } else {
      tot = sum_parts<MAXBD / 64 - 1>(sh->part);
    }
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
