// Device walker engine: the reference's `EnergyMC::move_once`
// (src/mc/energy.rs:904-974), as a proposal and a visit, for a group of G lanes
// that share one walker.
//
// Layout.  Every lane of a group holds the walker's hot scalar state in
// registers (identical values: all lanes execute the same bookkeeping, so no
// broadcast is ever needed).  For LJ/WCA, lane l of the group owns atoms l,
// l+G, l+2G, ... (K slots); the positions of all N atoms are an SoA tile in LDS,
// so any lane can read the moved atom.  The energy
// difference of a move is a per-lane partial sum over the lane's atoms
// followed by an xor butterfly across the G lanes.  Ising uses one lane per
// walker (G = 1) with the N*N <= 64 spins bit-packed in one 64-bit register.
//
// Bins.  A walker's bins are a fixed window of `cap` records in HBM, split by
// use (HotBin, ColdBin, the arrays beside them).
// Logical bin i lives in physical slot base + i; the reference's front
// insertion (energy.rs:400-420) becomes base -= 1, and the slots outside the
// window are zero from allocation, which is exactly the value the reference
// inserts.  The current bin's record is held in registers; the record of a
// proposed bin is loaded once (one dependent memory round trip per move) and
// becomes the current record if the move lands there.  Indices that only
// change when the window or the SAD range changes (the current bin, the bins
// of too_lo and too_hi, and ln w at those two bins) are cached and refreshed
// exactly when their inputs change, so each move computes one bin index.
// Periodic checks (verify_energy, the fixed refresh, WCA pressure) use
// next-trigger counters instead of a 64-bit modulo per move.
#pragma once

#include "sadmc_common.h"
#include "sadmc_proposal.h"
#include "../../include/sadmc.h"

namespace sadmc {

enum { SYS_ISING = 0, SYS_LJ = 1, SYS_WCA = 2 };
// Method families compiled separately: SAD; SAMC; WL and 1/t-WL (which may
// switch to SAMC, energy.rs:747-756); canonical.
enum { M_SAD = 0, M_SAMC = 1, M_WL = 2, M_CAN = 3 };

struct PExtra {
  uint64_t count;
  double total;
};

// Bin records are split by who reads them.  The hot part (16 bytes) is what
// the accept/reject decision and the entropy reduction read; the cold part (32
// bytes, so that no record straddles a cache line) is what a visit updates;
// t_found is written on a bin's first visit only.  WL's own histogram lives
// in another array that only WL kernels touch.
struct HotBin {
  double lnw;
  uint64_t hist;
};
struct alignas(32) ColdBin {
  double etot, esq;
  uint64_t rt, vep;
};

// Arguments of one walker set, passed by value to the kernels (they live in
// scalar registers).
struct SetArgs {
  sadmc_walker_state *ws;
  double *pos;       // [W][3][npad]
  uint64_t *spins;   // [W]
  HotBin *hot;       // [W][cap]
  ColdBin *cold;     // [W][cap]
  uint64_t *tfound;  // [W][cap]
  uint64_t *wlh;     // [W][cap] WL histogram, or null
  PExtra *extra;     // [W][cap] (WCA pressure) or null
  int32_t *flag;     // set to 1 when any walker of the set stops with a status
  int64_t cap;
  uint64_t zone_n;     // Uniform::new(0, n) acceptance zone
  uint64_t zone_site;  // gen_range(0, N) acceptance zone (Ising)
  int32_t W, n, npad, G, K;
  int32_t method, move_plan, has_min_e, has_max_e, has_min_gamma;
  int32_t refresh, collect_pressure, precision, move_kind;
  double method_param, move_param, min_e, max_e, rc2, width, inv_width;
  double floor_e, ceil_e;  // min_e and max_e, or -inf and +inf without them
  const uint16_t *mlp;  // learned proposal: 1377 BF16 weights, or null
};

// Pending change of the single-walker plan/confirm entry points (for a
// learned LJ move, `dabse` carries ln H).
struct Pending {
  int32_t some, which;
  double tx, ty, tz, e, dabse;
};

// Cross-lane move of a double with a DPP pattern (both 32-bit halves).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  uint64_t b = __builtin_bit_cast(uint64_t, v);
  int lo = __builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xF, 0xF, false);
  int hi = __builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, false);
  return __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// Sum over the G lanes of a group, every lane ending with the same value.
// Steps 1-4 are DPP: quad_perm [1,0,3,2] (xor 1), quad_perm [2,3,0,1]
// (xor 2), row_half_mirror and row_mirror.  After steps 1-2 the four lanes of
// a quad hold one value, after step 3 the eight lanes of a half row do, so
// the mirrors pair each lane with a lane holding exactly the partial sum the
// xor-4 / xor-8 partner would hold: the result is bit-identical to an xor
// butterfly.  Wider groups finish with cross-row shuffles.
__device__ __forceinline__ double group_sum(double v, int G) {
  if (G >= 2) v = v + dpp_f64<0xB1>(v);
  if (G >= 4) v = v + dpp_f64<0x4E>(v);
  if (G >= 8) v = v + dpp_f64<0x141>(v);
  if (G >= 16) v = v + dpp_f64<0x140>(v);
  if (G >= 32) v = v + __shfl_xor(v, 16, 64);
  if (G >= 64) v = v + __shfl_xor(v, 32, 64);
  return v;
}

// rand 0.7 UniformInt sampling with a precomputed zone (lj.rs:368 /
// ising.rs:105 semantics; the zone is the only part that depends on n).
// The range fits 32 bits, so the 128-bit product takes two 32 x 32 + 64
// multiply-adds.
__device__ __forceinline__ uint32_t sample_zone(uint64_t &s0, uint64_t &s1, uint32_t range, uint64_t zone) {
  for (;;) {
    const uint64_t v = rng_next(s0, s1);
    const uint64_t a = (uint64_t)(uint32_t)v * range;
    const uint64_t b = (uint64_t)(uint32_t)(v >> 32) * range + (a >> 32);
    if (((b << 32) | (uint32_t)a) <= zone) return (uint32_t)(b >> 32);
  }
}


// MV = 1: the learned Gaussian move with its Hastings term (LJ only).
// GC > 0: the lanes per walker fixed at compile time (must equal the set's
// G), which folds the group sums, lane indices and atom-slot arithmetic.
// SH: a wave with few walkers, in which kShare = KMAX lanes stand for each of a
// group's G, all with the walker's whole state, and share its pair terms, one
// atom slot a lane.
template <int SYS, int KMAX, int PREC, int METH, int MV = 0, int GC = 0, bool SH = false>
struct Engine {
  static constexpr int kShare = SH ? KMAX : 1;
  SADMC_DF static int wave_lane() { return (int)(threadIdx.x & 63); }
  const SetArgs *Ap;  // kernel argument segment (uniform; read with scalar loads)
  SADMC_DF const SetArgs &args() const { return *Ap; }
  int lane, G, K, n;
  HotBin *H;
  ColdBin *Cb;
  uint64_t *WH;
  int wk;  // the walker's index in its set
  // system
  double *lx, *ly, *lz;
  // The positions stay in LDS (one tile per walker): copies of a lane's atoms
  // in registers cost 24 of them and 30 selects per accepted move, more than
  // the reads (1 to 4 % of the walker kernels).
  // The slots a pair loop runs without asking for K, so that their chains
  // interleave: K > KMAX/2 always, and up to 4 slots the one too many is
  // cheaper than a branch.
  static constexpr int kFirst = KMAX <= 4 ? KMAX : KMAX / 2 + 1;
  uint64_t spins;
  double R2, L, halfL;
  // EnergyMC scalars
  uint64_t s0, s1;
  double E, err;
  uint64_t moves, accepted;
  double tm;  // (double)moves, kept exact by +1.0 steps
  double acc_rate, tscale, usc;
  double bmin;
  int32_t base, len;
  double max_S;
  int32_t max_S_index;
  uint64_t epoch;
  int32_t bulk, status, method;
  double btop;  // bmin + width * len, the upper edge of the bins
  // SAD; rtF, rNs = 1 / tF, 1 / N_s and
  // gzero (gamma is 0) follow lam, tF and N_s, which change rarely; tl_now:
  // tL was set in this move; tmax: the largest t_found in the range.  What a
  // walker below too_lo needs each move is here too: one such walker, which
  // can stay there for a whole launch, holds up its wave and so the launch.
  // tL and WCA's has_pressure, only ever written, stay in the walker's record.
  double too_lo, too_hi, lam, min_T, rtF, rNs, lnw_lo, lnw_hi;
  uint64_t tF, Ns, tmax;
  bool gzero, tl_now;
  uint64_t highest;
  int32_t ilo, ihi;
  SADMC_DF sadmc_walker_state &rec() const { return args().ws[wk]; }
  SADMC_DF uint64_t *tfound() const { return args().tfound + (int64_t)wk * args().cap; }
  // SAMC / WL
  double t0, wl_gamma, wl_Ns, wl_min_e;
  uint64_t wl_lowest, wl_highest, wl_total;
  int32_t wl_len;
  // current bin (logical cur_i, physical cur_p): its whole record (and WL
  // count), written back when the walker leaves the bin; cur_p = -1: none
  int32_t cur_i, cur_p;
  double c_lnw;
  uint64_t c_hist, c_wlh;
  double c_etot, c_esq;
  uint64_t c_rt, c_vep;
  int32_t from_i;  // the bin this move started in
  // periodic triggers
  uint64_t next_check, next_press;
  // pending move
  int32_t pw;
  double ptx, pty, ptz, pe, pdabse;
  // learned move: weights and this walker's exchange row in LDS, ln H
  const float *PW;
  float *XC;
  double lnh;
  // this move's SAD gamma (computed again if the move changes lambda or N_s),
  // and the next uniform with the generator state after drawing it, computed
  // while the proposed bin's record loads
  double gpre, spec_u;
  uint64_t spec0, spec1;
  // SAD's gamma for the group's next G moves, one per lane; g_next counts the
  // moves served from it (G: none left)
  double g_lane;
  int32_t g_next;
  // sqrt(1 / moves) for the wave's next 64 moves, one per lane, while its
  // walkers all stand at one move number (rs_same; as they do unless they
  // were uploaded at different ones)
  double rs_wave;
  bool rs_same;

  // ---------------------------------------------------------------- setup
  SADMC_DF void load_system(const SetArgs &a, int walker, int lane_in_group, double *lds_group) {
    Ap = &a;
    lane = lane_in_group;
    G = GC ? GC : a.G;
    K = a.K;
    n = a.n;
    H = a.hot + (int64_t)walker * a.cap;
    Cb = a.cold + (int64_t)walker * a.cap;
    wk = walker;
    WH = METH == M_WL ? a.wlh + (int64_t)walker * a.cap : nullptr;
    cur_p = -1;
    if (SYS == SYS_ISING) {
      spins = a.spins[walker];
    } else {
      lx = lds_group;
      ly = lds_group + a.npad;
      lz = lds_group + 2 * a.npad;
      const double *P = a.pos + (int64_t)walker * 3 * a.npad;
#pragma unroll
      for (int k = 0; k < KMAX; k++) {
        if (k < K) {
          int j = lane + G * k;
          lx[j] = P[j];
          ly[j] = P[a.npad + j];
          lz[j] = P[2 * a.npad + j];
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
  }

  SADMC_DF void load(const SetArgs &a, int walker, int lane_in_group, double *lds_group) {
    load_system(a, walker, lane_in_group, lds_group);
    const sadmc_walker_state &w = a.ws[walker];
    s0 = w.rng[0];
    s1 = w.rng[1];
    E = w.E;
    err = w.error;
    moves = w.moves;
    tm = (double)moves;
    accepted = w.accepted_moves;
    acc_rate = w.acceptance_rate;
    tscale = w.translation_scale;
    bmin = w.bins_min;
    base = (int32_t)w.base;
    len = (int32_t)w.len;
    max_S = w.max_S;
    max_S_index = (int32_t)w.max_S_index;
    epoch = w.epoch;
    bulk = (int32_t)w.bulk_visited;
    status = w.status;
    method = w.method;
    if (METH == M_SAD) {
      too_lo = w.too_lo;
      too_hi = w.too_hi;
      lam = w.latest_parameter;
      min_T = w.min_T;
      tmax = w.tmax;
      tF = w.tF;
      Ns = w.num_states;
      highest = w.highest_hist;
    }
    if (METH == M_SAMC || METH == M_WL) t0 = w.t0;
    if (METH == M_WL) {
      wl_gamma = w.wl_gamma;
      wl_Ns = w.wl_num_states;
      wl_min_e = w.wl_min_energy;
      wl_lowest = w.wl_lowest_hist;
      wl_highest = w.wl_highest_hist;
      wl_total = w.wl_total_hist;
      wl_len = (int32_t)w.wl_len;
    }
    if (SYS != SYS_ISING) {
      if (SYS == SYS_LJ) R2 = w.geom * w.geom;
      L = w.geom;
      halfL = 0.5 * w.geom;
    }
    usc = SYS == SYS_ISING ? 0.0 : uniform_scale(-tscale, tscale);
    btop = bmin + args().width * (double)len;
    g_next = G;
    if (METH == M_SAD) gamma_changed();
    cur_p = -1;
    if (!status) {
      refresh_indices();
      reset_checks();
    }
  }

  // Write back the walker state; the fields that only from_params sets, or
  // that are kept in the record during a launch, are not here.
  SADMC_DF void store(int walker) {
    write_back();
    if (lane == 0) {
      sadmc_walker_state &w = args().ws[walker];
      if (METH == M_SAD) {
        w.too_lo = too_lo;
        w.too_hi = too_hi;
        w.latest_parameter = lam;
        w.tF = tF;
        w.num_states = Ns;
        w.highest_hist = highest;
        w.tmax = tmax;
      }
      if (METH == M_SAMC || METH == M_WL) w.t0 = t0;
      if (METH == M_WL) {
        w.wl_gamma = wl_gamma;
        w.wl_num_states = wl_Ns;
        w.wl_min_energy = wl_min_e;
        w.wl_lowest_hist = wl_lowest;
        w.wl_highest_hist = wl_highest;
        w.wl_total_hist = wl_total;
        w.wl_len = wl_len;
      }
    }
    store_common(walker);
  }
  SADMC_DF void store_common(int walker) {
    if (lane == 0) {
      sadmc_walker_state &w = args().ws[walker];
      w.rng[0] = s0;
      w.rng[1] = s1;
      w.E = E;
      w.error = err;
      w.moves = moves;
      w.accepted_moves = accepted;
      w.acceptance_rate = acc_rate;
      w.translation_scale = tscale;
      w.bins_min = bmin;
      w.bins_width = args().width;
      w.base = base;
      w.len = len;
      w.max_S = max_S;
      w.max_S_index = max_S_index;
      w.epoch = epoch;
      w.bulk_visited = (uint64_t)bulk;
      w.status = status;
      w.method = method;
      if (status) *args().flag = 1;
    }
    if (SYS == SYS_ISING) {
      args().spins[walker] = spins;
    } else {
      double *P = args().pos + (int64_t)walker * 3 * args().npad;
#pragma unroll
      for (int k = 0; k < KMAX; k++) {
        if (k < K) {
          int j = lane + G * k;
          P[j] = lx[j];
          P[args().npad + j] = ly[j];
          P[2 * args().npad + j] = lz[j];
        }
      }
    }
  }

  // --------------------------------------------------------------- bins
  // Bins::state_to_index (energy.rs:371-373); `as usize` saturates.
  // The quotient by the width is first formed with the reciprocal; only
  // when that lands within 1e-9 of an integer (where the two roundings could
  // truncate differently) or outside (0, 1e6) is the division itself computed.
  SADMC_DF int32_t e_index(double e) const {
    const double d = e - bmin;
    const double v = d * args().inv_width;
    if (__builtin_expect(!(fabs(__builtin_amdgcn_fract(v) - 0.5) < 0.5 - 1e-9 && fabs(v - 5.0e5) < 5.0e5), 0)) {
      const double q = d / args().width;
      if (!(q > 0.0)) return 0;
      if (q >= 2.0e9) return 0x7fffffff;
      return (int32_t)q;
    }
    return (int32_t)v;
  }
  SADMC_DF double i_energy(int32_t i) const { return bmin + ((double)i + 0.5) * args().width; }
  SADMC_DF bool idx_ok(int32_t i) {
    if (i < 0 || i >= len) {
      status = SADMC_WS_INDEX;
      return false;
    }
    return true;
  }
  SADMC_DF double lnw_at(int32_t p) const { return p == cur_p ? c_lnw : H[p].lnw; }
  SADMC_DF uint64_t hist_at(int32_t p) const { return p == cur_p ? c_hist : H[p].hist; }
  SADMC_DF uint64_t wlh_at(int32_t p) const { return p == cur_p ? c_wlh : WH[p]; }

  // The current bin's record goes back to memory when the walker leaves the
  // bin or the launch ends (every read in between takes the registers).
  SADMC_DF void write_back() {
    if (lane == 0 && cur_p >= 0) {
      HotBin hb;
      hb.lnw = c_lnw;
      hb.hist = c_hist;
      H[cur_p] = hb;
      ColdBin cb;
      cb.etot = c_etot;
      cb.esq = c_esq;
      cb.rt = c_rt;
      cb.vep = c_vep;
      Cb[cur_p] = cb;
    }
  }
  SADMC_DF void set_current(int32_t p, const HotBin &hb, const ColdBin &cb, uint64_t wlh) {
    write_back();
    cur_p = p;
    c_lnw = hb.lnw;
    c_hist = hb.hist;
    if (METH == M_WL) c_wlh = wlh;
    c_etot = cb.etot;
    c_esq = cb.esq;
    c_rt = cb.rt;
    c_vep = cb.vep;
  }
  SADMC_DF void load_current(int32_t p) {
    const HotBin hb = H[p];
    const ColdBin cb = Cb[p];
    set_current(p, hb, cb, METH == M_WL ? WH[p] : 0);
  }

  // Re-derive every cached index from its inputs (after init, resume or a
  // window change) and reload the values cached at those indices.  An index
  // past the bins is left for move_once to report where the reference would
  // index out of bounds.
  // plo, phi: the physical bins whose ln w lnw_lo and lnw_hi already hold (a
  // window that grew at the front moves the indices, not the records).
  SADMC_DF void refresh_indices(int32_t plo = -1, int32_t phi = -1) {
    int32_t i = e_index(E);
    cur_i = i;
    if (i < len) {
      int32_t p = base + i;
      if (p != cur_p) load_current(p);
    } else {
      write_back();
      cur_p = -1;
    }
    if (METH == M_SAD) {
      ilo = e_index(too_lo);
      ihi = e_index(too_hi);
      if (ilo >= len || base + ilo != plo) lnw_lo = ilo < len ? lnw_at(base + ilo) : 0.0;
      if (ihi >= len || base + ihi != phi) lnw_hi = ihi < len ? lnw_at(base + ihi) : 0.0;
    }
  }

  // True when every cached index is inside the bins.
  SADMC_DF bool indices_valid() const {
    if (cur_p < 0) return false;
    if (METH == M_SAD && (ilo >= len || ihi >= len)) return false;
    return true;
  }

  SADMC_DF void reset_checks() {
    if (SYS != SYS_ISING) {
      uint64_t P = args().refresh > 0 ? (uint64_t)args().refresh : (uint64_t)len * (uint64_t)len * 1000ULL;
      next_check = (moves / P + 1) * P;
      if (SYS == SYS_WCA) {
        uint64_t Q = (uint64_t)n * (uint64_t)n;
        next_press = (moves / Q + 1) * Q;
      }
    }
  }

  // energy.rs:400-434 (prepare_for_state) for every energy in [lo, hi]: the
  // bins grow to both ends.  New slots get have_visited = true (visit_epoch =
  // epoch) and round_trips = 1; every other field is already zero.
  // A window without room stops the walker.
  SADMC_DF void prepare_for_range(double lo, double hi) {
    bool front = false, grew = false;
    const int32_t plo = METH == M_SAD && ilo < len ? base + ilo : -1;
    const int32_t phi = METH == M_SAD && ihi < len ? base + ihi : -1;
    while (status == 0 && lo < bmin) {
      if (base == 0) {
        status = SADMC_WS_CAPACITY;
      } else {
        base -= 1;
        len += 1;
        Cb[base].rt = 1;
        Cb[base].vep = epoch;
        bmin -= args().width;
        front = true;
      }
    }
    while (status == 0 && hi >= bmin + args().width * (double)len) {
      const int32_t q = base + len;
      if (q >= args().cap) {
        status = SADMC_WS_CAPACITY;
      } else {
        Cb[q].rt = 1;
        Cb[q].vep = epoch;
        len += 1;
        grew = true;
      }
    }
    btop = bmin + args().width * (double)len;
    if (status == 0 && (front || (grew && !indices_valid()))) refresh_indices(plo, phi);
    if (status == 0 && (front || grew) && SYS != SYS_ISING && args().refresh <= 0) {
      uint64_t P = (uint64_t)len * (uint64_t)len * 1000ULL;
      next_check = (moves / P + 1) * P;
    }
  }

  // ------------------------------------------------------------ systems
  SADMC_DF int spin(int b) const { return ((spins >> b) & 1ULL) ? 1 : -1; }

  // Full FP64 energy in lane-group order: lane l sums pairs (i, j<i) for its
  // atoms i; the G partial sums meet in the butterfly.
  SADMC_DF double full_energy() {
    if (SYS == SYS_ISING) {
      int N = n;
      double e = 0.0;
      for (int i1 = 0; i1 < N; i1++)
        for (int j1 = 0; j1 < N; j1++) {
          int j2 = j1 + 1 == N ? 0 : j1 + 1;
          int i2 = i1 + 1 == N ? 0 : i1 + 1;
          int nt = spin(i1 + j2 * N) + spin(i2 + j1 * N);
          e += (double)nt * (double)spin(i1 + j1 * N);
        }
      return e;
    }
    // rare: one small loop instead of KMAX unrolled ones
    double acc = 0.0;
#pragma unroll 1
    for (int i = lane; i < n; i += G) {
      const double xi = lx[i], yi = ly[i], zi = lz[i];
#pragma unroll 1
      for (int j = 0; j < i; j++) {
        if (SYS == SYS_LJ) {
          acc += lj_pair(norm2(xi - lx[j], yi - ly[j], zi - lz[j]));
        } else {
          acc += wca_pair_fast(norm2(min_image(xi - lx[j], L, halfL), min_image(yi - ly[j], L, halfL),
                                     min_image(zi - lz[j], L, halfL)),
                               args().rc2);
        }
      }
    }
    return group_sum(acc, G);
  }

  // The full energy of the group that lane `leader` belongs to, by the whole
  // wave (all 64 lanes running, the tiles of the wave's groups side by side in
  // LDS): lane v of group c takes the pairs (i, j) with i = v, v + G, ... and
  // j = c, c + 64/G, ..., and each lane then adds the terms of its v in the
  // order of j, which is the order of full_energy, so the bits are the same.
  // A term left out (j >= i) adds +0, which changes no sum here (none is
  // -0: they start at +0).
  //
  // The walkers of a wave need a new energy one by one, when their own error
  // estimate trips (LJ every 10 N accepted moves, WCA every 10), and a group
  // alone runs through the N^2/2 pairs with 64 - G lanes idle.
  SADMC_DF double wave_full_energy(int leader) const {
    const int R = 64 / G, c = wave_lane() / G, GP = G * kShare;
    const double *X = lx + (leader / GP - wave_lane() / GP) * 3 * args().npad, *Y = X + args().npad, *Z = Y + args().npad;
    const double Lw = SYS == SYS_WCA ? __shfl(L, leader, 64) : 0.0, hw = 0.5 * Lw;
    constexpr int U = 4;  // terms in flight per lane
    double acc = 0.0;
#pragma unroll 1
    for (int i0 = 0; i0 < n; i0 += G) {
      const int i = i0 + lane;
      const int jend = i < n ? i : 0;  // this lane's pairs: j < jend
      const int jmax = i0 + G - 1 < n - 1 ? i0 + G - 1 : n - 1;
      const double xi = X[jend], yi = Y[jend], zi = Z[jend];
#pragma unroll 1
      for (int j0 = 0; j0 < jmax; j0 += R * U) {
        double t[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          const int j = j0 + u * R + c;
          const bool ok = j < jend;
          const int jj = ok ? j : 0;
          double v;
          if (SYS == SYS_LJ) {
            v = lj_pair_fast(norm2(xi - X[jj], yi - Y[jj], zi - Z[jj]));
          } else {
            v = wca_pair_fast(norm2(min_image(xi - X[jj], Lw, hw), min_image(yi - Y[jj], Lw, hw),
                                    min_image(zi - Z[jj], Lw, hw)),
                              args().rc2);
          }
          t[u] = ok ? v : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          if (j0 + u * R < jmax) {
            if (GC > 0) {
#pragma unroll
              for (int q = 0; q < R; q++) acc += __shfl(t[u], q * G + lane, 64);
            } else {
              for (int q = 0; q < R; q++) acc += __shfl(t[u], q * G + lane, 64);
            }
          }
        }
      }
    }
    return group_sum(acc, G);
  }

  // A group of lanes without a walker (the last wave's, or a wave that holds
  // fewer than it could): it runs no moves and helps in wave_full_energy.
  SADMC_DF void load_idle(const SetArgs &a, int lane_in_group, double *lds_group) {
    Ap = &a;
    lane = lane_in_group;
    G = GC ? GC : a.G;
    K = a.K;
    n = a.n;
    lx = lds_group;
    status = SADMC_WS_OK + 100;
    L = 0.0;
  }

  // Full energies for the walkers with `need`, each the value of
  // full_energy (NaN sums, where the fast reciprocal may differ, included).
  SADMC_DF void full_energies(bool need) {
    uint64_t todo = __ballot(need);
    if (!todo) return;
    bool serial = need;
    if (SYS != SYS_ISING && G < 64 && __ballot(1) == ~0ULL) {
      const int GP = G * kShare, mine = wave_lane() / GP;
      while (todo) {
        const int leader = (int)__builtin_ctzll(todo);
        todo &= ~((~0ULL >> (64 - GP)) << (leader / GP * GP));
        const double e = wave_full_energy(leader);
        if (leader / GP == mine) {
          E = e;
          serial = SYS == SYS_LJ && e != e;
        }
      }
    }
    if (__builtin_expect(serial, 0)) E = full_energy();
  }

  // wca.rs:202-218 virial, ordered pairs, lane-group order.
  SADMC_DF double pressure() {
    double acc = 0.0;
#pragma unroll 1
    for (int i = lane; i < n; i += G) {
      const double xi = lx[i], yi = ly[i], zi = lz[i];
#pragma unroll 1
      for (int j = 0; j < n; j++) {
        if (j == i) continue;
        acc += wca_pair_pressure(norm2(min_image(xi - lx[j], L, halfL), min_image(yi - ly[j], L, halfL),
                                       min_image(zi - lz[j], L, halfL)),
                                 args().rc2);
      }
    }
    double p = group_sum(acc, G);
    return p / (3.0 * (L * L * L));
  }

  // ising.rs:104-119.
  SADMC_DF bool ising_plan(double &e2) {
    const int N = n;
    // sample_zone twice, in one loop: the zone is conservative (it refuses
    // half of the draws at N = 8), and every walker of the wave waits for the
    // one with the most refusals, of both draws together here instead of of
    // each
    int i = 0, j = -1;
    bool first = true;
    do {
      const uint64_t v = rng_next(s0, s1);
      const uint64_t a = (uint64_t)(uint32_t)v * (uint32_t)N;
      const uint64_t b = (uint64_t)(uint32_t)(v >> 32) * (uint32_t)N + (a >> 32);
      const bool ok = ((b << 32) | (uint32_t)a) <= args().zone_site;
      const int site = (int)(b >> 32);
      j = (ok & !first) ? site : j;
      i = (ok & first) ? site : i;
      first = first & !ok;
    } while (j < 0);
    int jp = j + 1 == N ? 0 : j + 1;
    int jm = j == 0 ? N - 1 : j - 1;
    int ip = i + 1 == N ? 0 : i + 1;
    int im = i == 0 ? N - 1 : i - 1;
    int nt = spin(i + jp * N) + spin(i + jm * N) + spin(ip + j * N) + spin(im + j * N);
    double e = E - (double)nt * (double)spin(i + j * N) * 2.0;
    pw = i + j * N;
    pe = e;
    e2 = e;
    return true;
  }

  // lj.rs:365-374 / wca.rs:341-353 with the cube move (half-width d,
  // Uniform::new(-d, d) scale sc); lj.rs:86-105 and wca.rs:119-140 for the
  // energy difference.
  SADMC_DF bool particle_plan(double d, double sc, double &e2) {
    int w = (int)sample_zone(s0, s1, (uint32_t)n, args().zone_n);
    const double fx = lx[w], fy = ly[w], fz = lz[w];
    __builtin_amdgcn_sched_barrier(0);  // the LDS reads run under the draws
    double ux = uniform_sample(s0, s1, -d, sc);
    double uy = uniform_sample(s0, s1, -d, sc);
    double uz = uniform_sample(s0, s1, -d, sc);
    double tx, ty, tz;
    // a move past the wall still runs through the sums below: its wave does
    // so anyway while any of its walkers moves inside
    bool some = true;
    if (SYS == SYS_LJ) {
      tx = fx + ux;
      ty = fy + uy;
      tz = fz + uz;
      double r2to = norm2(tx, ty, tz), r2from = norm2(fx, fy, fz);
      some = !(r2to > R2 && r2to > r2from);
    } else {
      tx = put_in_cell_step(fx + ux, L);
      ty = put_in_cell_step(fy + uy, L);
      tz = put_in_cell_step(fz + uz, L);
    }
    double acc = 0.0, accabs = 0.0;
    if (SYS == SYS_LJ) {
      acc = lj_lane_diff(w, tx, ty, tz, fx, fy, fz);
    } else {
      double vn, vo;
      auto terms = [&](int jr) {
        const double xj = lx[jr], yj = ly[jr], zj = lz[jr];
        vn = wca_pair_fast(norm2(min_image(xj - tx, L, halfL), min_image(yj - ty, L, halfL),
                                 min_image(zj - tz, L, halfL)),
                           args().rc2);
        vo = wca_pair_fast(norm2(min_image(xj - fx, L, halfL), min_image(yj - fy, L, halfL),
                                 min_image(zj - fz, L, halfL)),
                           args().rc2);
      };
      if constexpr (SH) {
        const int j = lane + G * (wave_lane() / G & (KMAX - 1));
        const bool use = (j < n) & (j != w);
        terms(use ? j : 0);
        acc = shared_sum(use ? vn - vo : 0.0);
        accabs = shared_sum(use ? vn + vo : 0.0);
      } else {
        auto slot = [&](int k) {
          const int j = lane + G * k;
          const bool use = (j < n) & (j != w);
          terms(2 * k > KMAX && j >= n ? 0 : j);  // as in lj_lane_sum
          const double na = acc + (vn - vo), nb = accabs + (vn + vo);
          acc = use ? na : acc;
          accabs = use ? nb : accabs;
        };
#pragma unroll
        for (int k = 0; k < kFirst; k++) slot(k);
        if (kFirst < KMAX && K > kFirst) {
#pragma unroll
          for (int k = kFirst; k < KMAX; k++) slot(k);
        }
      }
    }
    double e = E + group_sum(acc, G);
    if (SYS == SYS_WCA) pdabse = group_sum(accabs, G);
    pw = w;
    ptx = tx;
    pty = ty;
    ptz = tz;
    pe = e;
    e2 = e;
    return some;
  }

  // Features of the group's atoms around (px, py, pz), skipping atom w.  The
  // slots run side by side, as the pair loops' do; a slot without an atom adds
  // +0 to sums that are never negative.
  SADMC_DF void features(double px, double py, double pz, int w, float *f) {
#pragma unroll
    for (int c = 0; c < kPropNF; c++) f[c] = 0.0f;
    auto slot = [&](int k) {
      const int j = lane + G * k;
      const bool use = (j < n) & (j != w);
      const int jr = 2 * k > KMAX && j >= n ? 0 : j;  // as in lj_lane_sum
      const float a = (float)(lx[jr] - px), b = (float)(ly[jr] - py), c = (float)(lz[jr] - pz);
      const float r = __builtin_amdgcn_sqrtf(a * a + b * b + c * c);
      feature_add(use ? r : kPropFar, f);
    };
#pragma unroll
    for (int k = 0; k < kFirst; k++) slot(k);
    if (kFirst < KMAX && K > kFirst) {
#pragma unroll
      for (int k = kFirst; k < KMAX; k++) slot(k);
    }
#pragma unroll
    for (int c = 0; c < kPropNF; c++) f[c] = group_sum_f32(f[c], G);
  }

  // The sum over a lane's slots of the terms its KMAX lanes hold, in slot
  // order.  A slot without a term holds +0, which changes no sum here (none
  // is -0).
  SADMC_DF double shared_sum(double t) const {
    const int src = (wave_lane() & ~(G * KMAX - 1)) + lane;
    double v[KMAX], acc = 0.0;
#pragma unroll
    for (int k = 0; k < KMAX; k++) v[k] = __shfl(t, src + k * G, 64);
#pragma unroll
    for (int k = 0; k < KMAX; k++) acc += v[k];
    return acc;
  }

  // This lane's sum of the pair-term differences V(|x_j - t|^2) -
  // V(|x_j - f|^2) over its atoms j != w (lj.rs:86-105; in the precision
  // variant binary32 terms accumulated in FP64), with the fast reciprocals.
  // Every slot computes its terms; the moved atom's own slot and the padding
  // slots (whose terms may be inf or NaN) are dropped by a select of the
  // accumulator, which keeps the sums those of the skipped form without a
  // divergent branch per atom.
  SADMC_DF double lj_lane_sum(int w, double tx, double ty, double tz, double fx, double fy, double fz) {
    double acc = 0.0;
    auto term = [&](int jr) {
      const double xj = lx[jr], yj = ly[jr], zj = lz[jr];
      if (PREC == 1) {
        const float an = (float)(xj - tx), bn = (float)(yj - ty), cn = (float)(zj - tz);
        const float ao = (float)(xj - fx), bo = (float)(yj - fy), co = (float)(zj - fz);
        return (double)lj_pair_f32_fast(an * an + bn * bn + cn * cn) -
               (double)lj_pair_f32_fast(ao * ao + bo * bo + co * co);
      }
      return lj_pair_fast(norm2(xj - tx, yj - ty, zj - tz)) - lj_pair_fast(norm2(xj - fx, yj - fy, zj - fz));
    };
    if constexpr (SH) {
      const int j = lane + G * (wave_lane() / G & (KMAX - 1));
      const bool use = (j < n) & (j != w);
      const double t = term(use ? j : 0);
      return shared_sum(use ? t : 0.0);
    }
    auto slot = [&](int k) {
      const int j = lane + G * k;
      const bool use = (j < n) & (j != w);
      // slots that K may not reach read atom 0 (and are dropped)
      const double na = acc + term(2 * k > KMAX && j >= n ? 0 : j);
      acc = use ? na : acc;
    };
#pragma unroll
    for (int k = 0; k < kFirst; k++) slot(k);
    if (kFirst < KMAX && K > kFirst) {
#pragma unroll
      for (int k = kFirst; k < KMAX; k++) slot(k);
    }
    return acc;
  }
  // The same with the divisions; hardly ever needed, so a small loop.
  SADMC_DF double lj_lane_sum_div(int w, double tx, double ty, double tz, double fx, double fy, double fz) {
    double acc = 0.0;
#pragma unroll 1
    for (int j = lane; j < n; j += G) {
      if (j == w) continue;
      const double xj = lx[j], yj = ly[j], zj = lz[j];
      if (PREC == 1) {
        const float an = (float)(xj - tx), bn = (float)(yj - ty), cn = (float)(zj - tz);
        const float ao = (float)(xj - fx), bo = (float)(yj - fy), co = (float)(zj - fz);
        acc += (double)lj_pair_f32(an * an + bn * bn + cn * cn) - (double)lj_pair_f32(ao * ao + bo * bo + co * co);
      } else {
        acc += lj_pair(norm2(xj - tx, yj - ty, zj - tz)) - lj_pair(norm2(xj - fx, yj - fy, zj - fz));
      }
    }
    return acc;
  }

  // lj_lane_sum with the fast reciprocals, equal to the divisions' sum bit
  // for bit.  Binary32: the two reciprocals agree on [2^-126, 2^126); below
  // 2^-126 1/r^2 exceeds 2^126, so s^6 overflows and the pair term is NaN
  // with either; from 2^126 up s^2 underflows and both terms are +0; at +inf
  // only the fast one is NaN.  Binary64: see recip_f64_fast.  So the fast sum
  // differs only where it is NaN, and then the lanes still running this code
  // recompute with the division.
  SADMC_DF double lj_lane_diff(int w, double tx, double ty, double tz, double fx, double fy, double fz) {
    double acc = lj_lane_sum(w, tx, ty, tz, fx, fy, fz);
    if (__builtin_expect(__any(acc != acc), 0)) acc = lj_lane_sum_div(w, tx, ty, tz, fx, fy, fz);
    return acc;
  }

  // Sum over the group of the pair-term differences for atom w moving from
  // f to t (lj.rs:86-105).
  SADMC_DF double lj_delta(int w, double tx, double ty, double tz, double fx, double fy, double fz) {
    return group_sum(lj_lane_diff(w, tx, ty, tz, fx, fy, fz), G);
  }

  // The learned move: sigma from the network at the old position, a
  // Gaussian step, sigma' at the new position for the Hastings term.
  SADMC_DF bool learned_plan(double &e2) {
    int w = (int)sample_zone(s0, s1, (uint32_t)n, args().zone_n);
    const double fx = lx[w], fy = ly[w], fz = lz[w];
    float f[kPropNF], xi[3];
    features(fx, fy, fz, w, f);
    const float s = mlp_eval(PW, XC, f, lane, G);
    gaussian3(s0, s1, xi);
    const float sig = expf(s);
    const double tx = fx + (double)(sig * xi[0]), ty = fy + (double)(sig * xi[1]), tz = fz + (double)(sig * xi[2]);
    const double r2to = norm2(tx, ty, tz), r2from = norm2(fx, fy, fz);
    // the wall's verdict waits until after the second evaluation, so that
    // the whole wave reaches it together (its result is then unused)
    const bool outside = r2to > R2 && r2to > r2from;
    features(tx, ty, tz, w, f);
    const float s2 = mlp_eval(PW, XC, f, lane, G);
    if (outside) return false;
    const double e = E + lj_delta(w, tx, ty, tz, fx, fy, fz);
    lnh = prop_lnh(s, s2, xi[0] * xi[0] + xi[1] * xi[1] + xi[2] * xi[2]);
    pw = w;
    ptx = tx;
    pty = ty;
    ptz = tz;
    pe = e;
    pdabse = lnh;
    e2 = e;
    return true;
  }

  // SAD ln w(e) with the clamped extension (energy.rs:445-463); false if e
  // has no bin.
  SADMC_DF bool sad_lnw(double e, double &out) {
    if (ilo < 0 || ilo >= len || ihi < 0 || ihi >= len) return false;
    if (e < too_lo) {
      out = lnw_lo + (e - too_lo) / min_T;
      return true;
    }
    if (e > too_hi) {
      out = lnw_hi;
      return true;
    }
    const int32_t i = e_index(e);
    if (i < 0 || i >= len) return false;
    out = lnw_at(base + i);
    return true;
  }

  // `count` training records: the features of a random atom and, per scale
  // of the grid, the mean of alpha |d|^2 over kPropR Gaussian steps, from the
  // probe stream seeded by `seed`.  Lane 0 writes out[count][24].
  SADMC_DF void probe(uint64_t seed, int count, float *out) {
    uint64_t q0, q1;
    rng_seed(seed, q0, q1);
    double lnw1 = 0.0;
    const bool have1 = status == 0 && sad_lnw(E, lnw1);
    for (int c = 0; c < count; c++) {
      float rec[kPropRec];
      const int w = (int)uniform_index(q0, q1, (uint64_t)n);
      const double fx = lx[w], fy = ly[w], fz = lz[w];
      features(fx, fy, fz, w, rec);
#pragma unroll
      for (int k = 0; k < kPropNS; k++) {
        const float sig = expf(kPropSMin + (float)k * ((kPropSMax - kPropSMin) / (float)(kPropNS - 1)));
        float jsum = 0.0f;
        for (int r = 0; r < kPropR; r++) {
          float xi[3];
          gaussian3(q0, q1, xi);
          const float dx = sig * xi[0], dy = sig * xi[1], dz = sig * xi[2];
          const double tx = fx + (double)dx, ty = fy + (double)dy, tz = fz + (double)dz;
          const double r2to = norm2(tx, ty, tz), r2from = norm2(fx, fy, fz);
          if (r2to > R2 && r2to > r2from) continue;
          const double e2 = E + lj_delta(w, tx, ty, tz, fx, fy, fz);
          if (args().has_max_e && e2 > args().max_e && e2 > E) continue;
          double lnw2;
          if (!have1 || !sad_lnw(e2, lnw2)) continue;
          const double lr = lnw1 - lnw2;
          const float al = lr >= 0.0 ? 1.0f : (float)exp(lr);
          jsum += al * (dx * dx + dy * dy + dz * dz);
        }
        rec[kPropNF + k] = jsum / (float)kPropR;
      }
      if (lane == 0) {
#pragma unroll
        for (int i = 0; i < kPropRec; i++) out[(int64_t)c * kPropRec + i] = rec[i];
      }
    }
  }

  SADMC_DF bool plan_move(double d, double sc, double &e2) {
    if (SYS == SYS_ISING) return ising_plan(e2);
    if (MV == 1 && SYS == SYS_LJ) return learned_plan(e2);
    return particle_plan(d, sc, e2);
  }

  // The initial descent of from_params always uses the cube move.
  SADMC_DF bool cube_plan(double d, double sc, double &e2) {
    if (SYS == SYS_ISING) return ising_plan(e2);
    return particle_plan(d, sc, e2);
  }

  // lj.rs:106-123 and wca.rs:164-180 for a walker with `acc`: the new energy
  // is taken over unless the running error estimate has grown past its bound,
  // which asks for a full recomputation (true).
  SADMC_DF bool take_energy(bool acc, double new_e, double dabse) {
    if (SYS == SYS_ISING || args().refresh > 0) {
      E = acc ? new_e : E;
      return false;
    }
    const double nn = (double)n, ae = fabs(new_e);
    double ne;
    bool trip;
    if (SYS == SYS_LJ) {
      ne = (ae > fabs(E) ? ae * 1e-15 * nn : fabs(E) * 1e-15 * nn) + err;
      trip = ne > ae * 1e-14 * nn * nn;
      ne = trip ? ne * 0.0 : ne;
    } else {
      const double single = dabse > ae ? 1e-14 * dabse * nn : 1e-14 * ae * nn;
      ne = err + single * nn;
      trip = ne > ae * 1e-13 * nn * nn;
    }
    err = acc ? ne : err;
    E = acc && !trip ? new_e : E;
    return acc && trip;
  }
  // After the recomputation (wca.rs:175-177).
  SADMC_DF void took_full_energy() {
    if (SYS == SYS_WCA) err = 1e-15 * E * (double)n;
  }
  // take_energy with the recomputations shared by the wave.
  SADMC_DF void settle_energy(bool acc, double new_e, double dabse) {
    const bool trip = take_energy(acc, new_e, dabse);
    if (__builtin_expect(__any(trip), 0)) {
      full_energies(trip);
      if (trip) took_full_energy();
    }
  }

  // The part of ConfirmSystem::confirm (ising.rs:94-101, lj.rs:338-358,
  // wca.rs:276-301) that moves the atom.
  SADMC_DF void confirm_system() {
    if (SYS == SYS_ISING) {
      spins ^= (1ULL << pw);
      return;
    }
    if (lane == 0) {
      lx[pw] = ptx;
      ly[pw] = pty;
      lz[pw] = ptz;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  // The whole of it, for callers whose groups confirm on their own.
  SADMC_DF void confirm() {
    confirm_system();
    if (take_energy(true, pe, pdabse)) {
      E = full_energy();
      took_full_energy();
    }
  }

  // lj.rs:249-261, wca.rs:237-250; `egood` is the recomputed energy.
  SADMC_DF void verify_energy() { verify_energy(full_energy()); }
  SADMC_DF void verify_energy(double egood) {
    double nn = (double)n;
    double expected = SYS == SYS_LJ ? fabs(E) * 1e-14 * nn * nn : fabs(E) * 1e-13 * nn * nn;
    if (fabs(egood - E) > expected) status = SADMC_WS_VERIFY;
  }

  // ------------------------------------------------------------- method
  // energy.rs:22-38 with t = moves, tF, N_s (energy.rs:799-813).  t / tF and
  // t / N_s come from the kept correctly rounded reciprocals y = RN(1/b):
  // RN(t y) is within two units of the quotient, the first residual step
  // brings it to a faithful one, and with a faithful quotient the second
  // gives the correctly rounded one (Markstein 1990), which is the division's.
  // The operands lie between 1/2 and 2^64 (b; otherwise gamma is 0), so nothing
  // over- or underflows.
  SADMC_DF static double quot(double a, double b, double y) {
    double q = a * y;
    q = __builtin_fma(__builtin_fma(-b, q, a), y, q);
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
  }
  SADMC_DF double sad_gamma(double t) const {
    const double q = quot(t, (double)tF, rtF);
    const double g = (lam + q) / (lam + quot(t, (double)Ns, rNs) * q);
    return gzero ? 0.0 : g;
  }
  // After a change of lam, tF or Ns (during move tm): the reciprocals, and
  // the gammas of the moves from tm on that the lanes hold.
  SADMC_DF void gamma_changed() {
    rtF = 1.0 / (double)tF;
    rNs = 1.0 / (double)Ns;
    gzero = lam * (double)tF * (double)Ns == 0.0;
    g_lane = sad_gamma(tm + (double)(lane - (g_next - 1)));
  }
  SADMC_DF double gamma_now() const { return G == 1 ? g_lane : __shfl(g_lane, g_next - 1, G); }

  // Draw the next uniform ahead of the test that may use it.
  SADMC_DF void spec_draw() {
    spec0 = s0;
    spec1 = s1;
    spec_u = gen_f64(spec0, spec1);
  }
  // `need && u > exp(x)`, consuming the uniform only when `need`.
  // The comparison is settled from a single-precision 2^(x log2 e) whenever
  // u lies outside that estimate's error band; only inside the band is the
  // double exp computed.  Band: t = x log2 e (double, relative error 2^-52)
  // rounds to float with |dt| <= |t| 2^-24, v_exp_f32 is within a few ulp
  // (2^-21), so the estimate is within |t| 2^-24 ln 2 + 2^-21 < 1e-7 |t| +
  // 1e-6 of exp(x), and of the correctly rounded double exp (2^-53 more);
  // the band is ten times that.  Below t = -125 exp(x) < 2^-125 and the
  // estimate (possibly flushed to 0) lie under every nonzero u (multiples of
  // 2^-53); u = 0 and NaN take the double path.  When `need` holds, x <= 0.
  SADMC_DF bool mh_test(bool need, double x) {
    s0 = need ? spec0 : s0;
    s1 = need ? spec1 : s1;
    double t = x * 1.4426950408889634;
    t = t < -1000.0 ? -1000.0 : t;  // the estimate is 0 from there on, and -inf would make the band NaN
    const double est = (double)__builtin_amdgcn_exp2f((float)t);
    const double band = est * (1e-5 - 1e-6 * t);
    bool rejected = spec_u > est + band;
    if (__builtin_expect(need & !rejected & !(spec_u < est - band), 0)) rejected = spec_u > exp(x);
    return need & rejected;
  }
  // tempering.rs:101-104: `bde < 0 || u < exp(-bde)`, the uniform drawn only
  // for bde not below 0 (and `some`); settled as in mh_test.
  SADMC_DF bool canonical_test(bool some, double bde) {
    const bool need = some & !(bde < 0.0);
    spec_draw();
    s0 = need ? spec0 : s0;
    s1 = need ? spec1 : s1;
    double t = bde * -1.4426950408889634;
    t = t < -1000.0 ? -1000.0 : t;
    const double est = (double)__builtin_amdgcn_exp2f((float)t);
    const double band = est * (1e-5 - 1e-6 * t);
    bool take = spec_u < est - band;
    if (__builtin_expect(need & !take & !(spec_u > est + band), 0)) take = spec_u < exp(-bde);
    return !need | take;
  }
  // Metropolis-Hastings test on the log acceptance ratio.
  SADMC_DF bool reject_lr(bool go, double lr) { return mh_test(go & (lr < 0.0), lr); }
  // ln w(e) with the SAD clamped extension (energy.rs:445-463); `inside` is
  // the bin's ln w.
  SADMC_DF double sad_lnw_ext(double e, double inside) const {
    double v = e > too_hi ? lnw_hi : inside;
    if (__builtin_expect(e < too_lo, 0)) v = lnw_lo + (e - too_lo) / min_T;
    return v;
  }

  // energy.rs:440-512 on l1 and l2, ln w at the two energies (with SAD's
  // extension outside its range), and the proposed bin's count; nothing
  // happens for a walker without a move to test (`go` false).  The learned
  // move adds ln H to the exponent (the tests are the reference's when
  // ln H = 0).
  SADMC_DF bool reject_move(bool go, double e1, double e2, double l1, double l2, uint64_t r2_hist) {
    bool rejected;
    if (METH == M_CAN) {
      if (MV == 1) return reject_lr(go, (e1 - e2) / args().method_param + lnh);
      return mh_test(go & (e1 < e2), (e1 - e2) / args().method_param);
    }
    if (MV == 1) {
      rejected = reject_lr(go, l1 - l2 + lnh);
    } else {
      rejected = mh_test(go & (l2 > l1), l1 - l2);
    }
    const bool found = go & !rejected & (r2_hist == 0);
    if (METH == M_SAD) {
      if (__builtin_expect(found, 0) && e2 < too_hi && e2 > too_lo) {
        lam = (too_hi - too_lo) / min_T;
        Ns += 1;
        set_tL();
        gamma_changed();
        gpre = gamma_now();
      }
    } else if (METH == M_WL) {
      if (found && method != SADMC_SAMC && wl_lowest > 0) wl_Ns += 1.0;
    }
    return rejected;
  }

  // Running max of t_found over logical bins [a, b].
  // (The scans over bins that SAD's range changes need are split over the
  // walker's G lanes: each lane takes every G-th bin, so the loads of one
  // scan are in flight together; integer sums and maxima are then combined
  // across the group, which leaves every result as the sequential one.)
  SADMC_DF uint64_t group_max_u64(uint64_t v) const {
    for (int d = 1; d < G; d <<= 1) {
      const uint64_t o = __shfl_xor(v, d, 64);
      v = o > v ? o : v;
    }
    return v;
  }
  SADMC_DF uint32_t group_sum_u32(uint32_t v) const {
    for (int d = 1; d < G; d <<= 1) v += __shfl_xor(v, d, 64);
    return v;
  }
  SADMC_DF void set_tL() {
    tl_now = true;
    rec().tL = moves;
  }
  SADMC_DF void tmax_scan(int32_t a, int32_t b) {
    const uint64_t *TF = tfound();
    uint64_t m = 0;
    for (int32_t j = a + lane; j <= b; j += G) {
      const uint64_t t = TF[base + j];
      m = t > m ? t : m;
    }
    m = group_max_u64(m);
    tmax = m > tmax ? m : tmax;
  }

  // energy.rs:514-636 for the current bin (logical i = cur_i).
  SADMC_DF void update_sad(double E_, int32_t i) {
    const double E = E_;
    const bool in = !((too_lo > too_hi) | (E < too_lo) | (E > too_hi));
    c_lnw = in ? c_lnw + gpre : c_lnw;
    lnw_lo = (in & (i == ilo)) ? c_lnw : lnw_lo;
    lnw_hi = (in & (i == ihi)) ? c_lnw : lnw_hi;
    if (__builtin_expect((c_hist > highest) | tl_now, 0)) update_sad_range(E, i);
  }
  // The part of update_sad that a new highest count or a new tL needs.
  SADMC_DF void update_sad_range(double E, int32_t i) {
    if (c_hist > highest) {
      highest = c_hist;
      // the cached ln w at too_lo / too_hi and N_s change here only when
      // the range grows; otherwise ln w at those bins changes only through
      // the current bin, which the increment above already tracks
      bool grew = false;
      if ((E > too_hi && ihi >= len) || (E < too_lo && ilo >= len)) {
        status = SADMC_WS_INDEX;
      } else if (E > too_hi) {
        grew = true;
        const double vhi = lnw_hi;
        int32_t jlo = ihi > 0 ? ihi - 1 : 0, jhi = i + 1 < len ? i + 1 : len - 1;
        uint32_t cnt = 0;
        for (int32_t j = jlo + lane; j <= jhi; j += G) {
          const double ej = i_energy(j);
          const int32_t pj = base + j;
          if (ej > too_hi && ej <= E && pj != cur_p) {
            const bool nz = H[pj].hist != 0;
            H[pj].lnw = nz ? vhi : 0.0;
            cnt += nz ? 1u : 0u;
          }
        }
        cnt = group_sum_u32(cnt);
        if (i >= jlo && i <= jhi) {  // the current bin, whose record every lane holds
          const double ec = i_energy(i);
          if (ec > too_hi && ec <= E) {
            c_lnw = c_hist != 0 ? vhi : 0.0;
            cnt += c_hist != 0 ? 1u : 0u;
          }
        }
        Ns += cnt;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        lam = (E - too_lo) / min_T;
        set_tL();
        double nh = i_energy(i);
        int32_t ihi2 = e_index(nh);
        if (ihi2 > ihi) tmax_scan(ihi + 1, ihi2 < len ? ihi2 : len - 1);
        too_hi = nh;
        ihi = ihi2;
        if (ihi >= len) status = SADMC_WS_INDEX;
      } else if (E < too_lo) {
        grew = true;
        // every bin below too_lo extends from the old ln w(too_lo): the bin
        // of too_lo itself comes last in energy order
        int32_t jlo = i > 0 ? i - 1 : 0, jhi = ilo + 1 < len ? ilo + 1 : len - 1;
        const double vlo = lnw_lo;
        uint32_t cnt = 0;
        for (int32_t j = jlo + lane; j <= jhi; j += G) {
          const double ej = i_energy(j);
          const int32_t pj = base + j;
          if (ej < too_lo && ej >= E && pj != cur_p) {
            const bool nz = H[pj].hist != 0;
            double v = 0.0;
            if (nz) {
              v = vlo + (ej - too_lo) / min_T;
              if (v < 0.0) v = 0.0;
            }
            H[pj].lnw = v;
            cnt += nz ? 1u : 0u;
          }
        }
        cnt = group_sum_u32(cnt);
        if (i >= jlo && i <= jhi) {  // the current bin, whose record every lane holds
          const double ec = i_energy(i);
          if (ec < too_lo && ec >= E) {
            double v = 0.0;
            if (c_hist != 0) {
              v = vlo + (ec - too_lo) / min_T;
              if (v < 0.0) v = 0.0;
            }
            c_lnw = v;
            cnt += c_hist != 0 ? 1u : 0u;
          }
        }
        Ns += cnt;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        lam = (too_hi - E) / min_T;
        set_tL();
        double nl = i_energy(i);
        int32_t ilo2 = e_index(nl);
        if (ilo2 < ilo) tmax_scan(ilo2, ilo - 1);
        too_lo = nl;
        ilo = ilo2;
      }
      if (grew && status == 0) {
        lnw_lo = lnw_at(base + ilo);
        lnw_hi = lnw_at(base + ihi);
      }
    }
    if (tl_now && status == 0 && (ilo >= len || ihi >= len)) status = SADMC_WS_INDEX;
    if (tl_now && status == 0) {
      const uint64_t old_tF = tF;
      tF = tmax;
      if (old_tF != tF && args().move_plan == SADMC_ACCEPTANCE_RATE) {
        double s = acc_rate / args().move_param;
        s = s < 0.8 ? 0.8 : (s > 1.2 ? 1.2 : s);
        tscale *= s;
        if (SYS != SYS_ISING) usc = uniform_scale(-tscale, tscale);
      }
    }
    if (tl_now) gamma_changed();
  }

  // energy.rs:638-756 (WL and 1/t-WL); SAMC after the 1/t switch.
  SADMC_DF void update_wl(int32_t i) {
    if (method == SADMC_SAMC) {
      double t = tm;
      c_lnw += t > t0 ? t0 / t : 1.0;
      return;
    }
    c_lnw += wl_gamma;
    const bool inv_t = method == SADMC_INV_T_WL;
    const bool has_mg = !inv_t && args().has_min_gamma;
    if (has_mg && wl_gamma < args().method_param) {
      if (i >= wl_len) {
        status = SADMC_WS_INDEX;
        return;
      }
      c_wlh += 1;
      WH[cur_p] = c_wlh;
      return;
    }
    if (wl_len != len) {
      if (wl_len == 0 || (wl_gamma != 1.0 && wl_lowest > 0)) {
        wl_gamma = 1.0;
        wl_lowest = 0;
        wl_highest = 0;
        wl_total = 0;
        for (int32_t q = 0; q < len; q++) WH[base + q] = 0;
        c_wlh = 0;
        wl_len = len;
        wl_min_e = bmin;
      } else {
        while (wl_min_e > bmin) {
          wl_min_e -= args().width;
          wl_len += 1;
        }
        while (wl_len < len) wl_len += 1;
        uint64_t mn = ~0ULL;
        for (int32_t q = 0; q < wl_len; q++) {
          uint64_t h = wlh_at(base + q);
          if (h < mn) mn = h;
        }
        wl_lowest = mn;
      }
    }
    if (i >= wl_len) {
      status = SADMC_WS_INDEX;
      return;
    }
    c_wlh += 1;
    WH[cur_p] = c_wlh;
    if (c_wlh > wl_highest) wl_highest = c_wlh;
    wl_total += 1;
    double max_energy = wl_min_e + (double)wl_len * args().width;
    if (c_wlh == wl_lowest + 1 && wl_len > 1 && (!args().has_min_e || args().min_e >= wl_min_e) &&
        (!args().has_max_e || args().max_e <= max_energy)) {
      bool found = false;
      uint64_t mn = ~0ULL;
      for (int32_t q = 0; q < wl_len; q++) {
        if (hist_at(base + q) != 0) {
          found = true;
          uint64_t h = wlh_at(base + q);
          if (h < mn) mn = h;
        }
      }
      if (found && mn == wl_lowest + 1) {
        wl_lowest = c_wlh;
        if ((inv_t && wl_lowest > 0) || (double)wl_lowest >= 0.8 * (double)wl_total / wl_Ns) {
          wl_gamma *= 0.5;
          for (int32_t q = 0; q < wl_len; q++) WH[base + q] = 0;
          c_wlh = 0;
          wl_total = 0;
          wl_lowest = 0;
          wl_highest = 0;
          if (has_mg && wl_gamma < args().method_param) wl_gamma = 0.0;
        }
        if (inv_t && wl_gamma < wl_Ns / tm) {
          method = SADMC_SAMC;
          t0 = wl_Ns;
        }
      }
    }
  }

  // energy.rs:904-974.  One memory round trip per move: both parts of the
  // proposed bin's record are requested as soon as its energy is known, for
  // every lane (a walker whose proposal is void reads its current bin), and
  // what does not need them is computed meanwhile.  What is common is written
  // as selects rather than branches, which the walkers of a wave would
  // otherwise take one after the other; the rare parts stay branches.
  //
  // A move is a proposal and a visit; in between the wave recomputes the
  // energies that the proposals asked for (true) together.
  // `rs`: sqrt(1 / moves), this move counted, where rs_same.
  SADMC_DF bool propose(double rs) {
    bool regrow = false;
    moves += 1;
    tm += 1.0;
    if (METH == M_SAD) tl_now = false;
    if (SYS != SYS_ISING && __builtin_expect(moves == next_check, 0)) {
      const double egood = full_energy();
      if (args().refresh > 0) {
        E = egood;
        next_check += (uint64_t)args().refresh;
        // the refreshed energy may lie in another bin than the tracked one
        // (move_once indexes the bins by the energy itself, energy.rs:904-974),
        // or past the window's edge by the FP32 drift: the window then grows
        // to it as for a proposed energy (energy.rs:400-434), together with
        // the proposal's growth below (the order of the two growths does not
        // change the bins they add)
        if (e_index(E) != cur_i || E < bmin) {
          refresh_indices();
          regrow = cur_p < 0 || E < bmin;
        }
      } else {
        verify_energy(egood);
        next_check += (uint64_t)len * (uint64_t)len * 1000ULL;
      }
    }
    const double e1 = E;
    int32_t i1 = cur_i;
    if (METH == M_SAD) {
      if (g_next >= G) {
        g_lane = sad_gamma(tm + (double)lane);
        g_next = 0;
      }
      g_next += 1;
      gpre = gamma_now();
    }
    if (__builtin_expect(!rs_same, 0)) rs = sqrt(1.0 / tm);
    double e2 = e1;
    bool go = plan_move(tscale, usc, e2);
    acc_rate *= 1.0 - rs;
    // (bitwise on purpose, here and below: && and || become branches)
    go = go & !((e2 > args().ceil_e) & (e2 > e1)) & !((e2 < args().floor_e) & (e2 < e1));
    if (__builtin_expect(regrow | (go & ((e2 < bmin) | (e2 >= btop))), 0)) {
      double lo = go ? e2 : E, hi = lo;
      if (regrow) {
        lo = E < lo ? E : lo;
        hi = E > hi ? E : hi;
      }
      // (also for a walker that the energy check above has stopped)
      const int32_t stopped = status;
      status = 0;
      prepare_for_range(lo, hi);
      status = status ? status : stopped;
    }
    i1 = go ? cur_i : i1;
    const int32_t i2 = e_index(go ? e2 : e1);
    bool bad = (uint32_t)i2 >= (uint32_t)len;
    if (METH == M_SAD) bad = bad | (ilo >= len) | (ihi >= len);
    if (__builtin_expect((status == 0) & ((cur_p < 0) | (go & bad)), 0)) status = SADMC_WS_INDEX;
    from_i = i1;
    bool trip = false;
    if (__builtin_expect(status == 0, 1)) trip = decide(go, e1, e2, i2, rs);
    return trip;
  }
  // The test and the accepted move.
  SADMC_DF bool decide(bool go, double e1, double e2, int32_t i2, double rs) {
    const int32_t p2 = go ? base + i2 : cur_p;
    const HotBin hb = H[p2];
    const ColdBin cb = Cb[p2];
    uint64_t wl2 = 0;
    if (METH == M_WL) wl2 = WH[p2];
    // independent of the record being loaded
    spec_draw();
    double l1 = c_lnw, out2 = 0.0;
    bool ext2 = false;
    if (METH == M_SAD) {
      l1 = sad_lnw_ext(e1, c_lnw);
      out2 = sad_lnw_ext(e2, 0.0);
      ext2 = (e2 < too_lo) | (e2 > too_hi);
    }
    const bool same = p2 == cur_p;
    // The whole record has to be there before the old one's stores are issued:
    // loads and stores complete in order, so any later wait for the loads
    // would be one for the stores too.
    asm volatile("" ::"v"(hb.lnw), "v"(hb.hist), "v"(cb.etot), "v"(cb.esq), "v"(cb.rt), "v"(cb.vep), "v"(wl2));
    const double w2 = same ? c_lnw : hb.lnw, l2 = ext2 ? out2 : w2;
    const uint64_t h2 = same ? c_hist : hb.hist;
    const bool acc = go & !reject_move(go, e1, e2, l1, l2, h2);
    accepted += acc ? 1 : 0;
    acc_rate = acc ? acc_rate + rs : acc_rate;
    const bool trip = take_energy(acc, e2, pdabse);
    if (acc) confirm_system();
    if (acc & !same) set_current(p2, hb, cb, wl2);
    cur_i = acc ? i2 : cur_i;
    return trip;
  }
  // After a recomputed energy, which may lie in another bin.
  SADMC_DF void reindex() {
    const int32_t i = e_index(E);
    if (i != cur_i && idx_ok(i)) {
      load_current(base + i);
      cur_i = i;
    }
  }
  // The update of the bin the walker is in.
  SADMC_DF void visit() {
    const int32_t i1 = from_i;
    const double En = E;
    const int32_t i = cur_i;
    const int32_t p = cur_p;
    if (__builtin_expect(c_hist == 0, 0)) {
      tfound()[p] = moves;
      if (METH == M_SAD && i >= ilo && i <= ihi) tmax = moves;
    }
    c_hist += 1;
    if (SYS == SYS_WCA && args().collect_pressure && __builtin_expect(moves == next_press, 0)) {
      const double pv = pressure();
      PExtra &x = args().extra[(int64_t)wk * args().cap + p];
      rec().has_pressure = 1;
      if (lane == 0) {
        x.count += 1;
        x.total += pv;
      }
      next_press += (uint64_t)n * (uint64_t)n;
    }
    if (METH == M_SAD) {
      update_sad(En, i);
    } else if (METH == M_SAMC) {
      c_lnw += tm > t0 ? t0 / tm : 1.0;
    } else if (METH == M_WL) {
      update_wl(i);
    }
    if (__builtin_expect(status == 0, 1)) after_visit(En, i, i1);
  }
  SADMC_DF void after_visit(double En, int32_t i, int32_t i1) {
    // energy.rs:950-965 and 941-943 (the energy of this move's end is added
    // at the start of the next in the reference; nothing between reads it)
    bool round_trip = true;
    if (__builtin_expect((c_lnw > max_S) | (i == max_S_index), 0)) {
      round_trip = false;
      if (c_lnw > max_S) {
        max_S = c_lnw;
        max_S_index = i;
        epoch += 1;
        bulk = 1;
      } else if (i1 != i) {
        epoch += 1;
        bulk = 0;
      }
    }
    const bool mark = round_trip & !((bulk != 0) | (c_vep == epoch));
    c_vep = mark ? epoch : c_vep;
    c_rt += mark ? 1 : 0;
    c_etot += En;
    c_esq += En * En;
  }

  // rs_wave for the next 64 moves: what every walker needs each move, from one
  // square root per lane.
  SADMC_DF void next_roots() {
    const uint64_t on = __ballot(status == 0);
    const double t = __shfl(tm, (int)__builtin_ctzll(on), 64);
    rs_same = __ballot(1) == ~0ULL && !__any((status == 0) & (tm != t));
    rs_wave = sqrt(1.0 / (t + (double)((threadIdx.x & 63) + 1)));
  }
  // The one of this move, `step` moves on (the same in the whole wave).  Only
  // where the wave's lanes all run: the lane read may belong to a walker that
  // has stopped or to no walker, and what such a lane holds of rs_wave is
  // certain only outside the branches it sits out.
  SADMC_DF double root(int step) const {
    const uint64_t b = __builtin_bit_cast(uint64_t, rs_wave);
    const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, step);
    const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), step);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
  }

  SADMC_DF void run(uint64_t nmoves) {
    // (the loop's exit is the wave's, not a walker's: a divergent exit makes
    // the compiler keep the state of stopped and running walkers apart, which
    // took 80 more registers)
    for (uint64_t k = 0; k < nmoves && __any(status == 0); k++) {
      const int step = (int)(k & 63);
      if (step == 0) next_roots();
      const double rs = root(step);
      bool trip = false;
      if (__builtin_expect(status == 0, 1)) trip = propose(rs);
      if (__builtin_expect(__any(trip), 0)) {
        full_energies(trip);
        if (trip) {
          took_full_energy();
          reindex();
        }
      }
      if (__builtin_expect(status == 0, 1)) visit();
    }
  }

  // energy.rs:830-898 after the system exists (initial energy, greedy
  // descent below max_e, one-bin histogram, method state).
  SADMC_DF void from_params(int walker, double e_lo) {
    const sadmc_walker_state &w = args().ws[walker];
    s0 = w.rng[0];
    s1 = w.rng[1];
    if (SYS != SYS_ISING) {
      if (SYS == SYS_LJ) R2 = w.geom * w.geom;
      L = w.geom;
      halfL = 0.5 * w.geom;
    }
    status = 0;
    E = full_energy();
    err = 0.0;
    if (args().has_max_e) {
      const double sc = SYS == SYS_ISING ? 0.0 : uniform_scale(-0.05, 0.05);
      for (uint64_t k = 0; k < 100000000ULL; k++) {
        double newe;
        if (cube_plan(0.05, sc, newe)) {
          if (newe < E) confirm();
          if (E < args().max_e) break;
        }
      }
    }
    const double width = args().width;
    double emin = (round(E / width) - 0.5) * width;
    bmin = emin;
    len = 1;
    double b = floor((emin - e_lo) / width) + 2.0;
    if (!(b >= 0.0) || b >= (double)(args().cap - 2)) {
      status = SADMC_WS_CAPACITY;
      base = 0;
    } else {
      base = (int32_t)b;
      HotBin hb;
      hb.lnw = 0.0;
      hb.hist = 1;
      H[base] = hb;
      ColdBin cb;
      cb.etot = E;
      cb.esq = E * E;
      cb.rt = 1;
      cb.vep = 0;
      Cb[base] = cb;
    }
    max_S = 0.0;
    max_S_index = 0;
    epoch = 1;
    bulk = 0;
    moves = 0;
    accepted = 0;
    acc_rate = 0.5;
    tscale = args().move_plan == SADMC_TRANSLATION_SCALE ? args().move_param : 0.05;
    method = args().method;
    t0 = 0.0;
    // every method's fields, also those store() leaves to the record
    if (lane == 0) {
      sadmc_walker_state &q = rec();
      q.min_T = args().method == SADMC_SAD ? args().method_param : 0.0;
      q.t0 = args().method == SADMC_SAMC ? args().method_param : 0.0;
      q.too_lo = E;
      q.too_hi = E;
      q.latest_parameter = 0.0;
      q.tL = 0;
      q.tF = 0;
      q.num_states = 1;
      q.highest_hist = 1;
      q.tmax = 0;
      const bool both = args().has_min_e && args().has_max_e;
      q.wl_gamma = 1.0;
      q.wl_lowest_hist = both ? 0 : 1;
      q.wl_highest_hist = 1;
      q.wl_total_hist = 0;
      q.wl_num_states = both ? (args().max_e - args().min_e) / width : 1.0;
      q.wl_len = 0;
      q.wl_min_energy = E;
      q.has_pressure = 0;
    }
    store_common(walker);
  }
};

}  // namespace sadmc
