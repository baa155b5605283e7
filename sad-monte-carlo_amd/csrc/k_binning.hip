// EnergyMC over a histogram Binning (src/mc/energy_binning.rs with
// src/mc/binning/histogram.rs): the walker of the reference's `binning`
// binary, one walker per lane group like the main engine.
//
// The system part (plan_move, confirm, energies, pressure) is the main
// engine's; the bookkeeping is this file's.  Every lane of a group holds the
// walker's scalars (identical values), the bins live in HBM as one 80-byte
// record per bin, the arrays' statistics in LDS.  The O(bins) scans the
// reference makes are either replaced by exact trackers of the extremes
// (BinCounts' min/max recomputations) or split over the group's lanes and
// combined with shuffles (set_lnw, count_states, the trackers' own rescans), so
// that every result is the sequential one.
//
// The histogram walker keeps the record of the bin it is in in registers and
// reads one record a move, the proposed bin's (the linear binning, whose
// visits touch two bins, works on the records in memory).
#define SADMC_KERNEL_TU
#include <type_traits>

#include "sadmc_kernels.h"

namespace sadmc {

namespace {

enum { BC_LNW = 0, BC_EN = 1, BC_TF = 2, BC_HIST = 3, BC_PR = 4 };

// BinCounts' running statistics (histogram.rs:11-33, linear.rs:11-33):
// counts are integers in the histogram, fractions in the linear binning.
// Beside them exact extremes of the array, so that its min_of / max_of /
// min() rescans (histogram.rs:64-80, 226-244) become lookups: the smallest
// total and how many bins hold it, the smallest count and its multiplicity.
// A full rescan is needed only when the last bin holding an extreme leaves
// it, after set_lnw / zero_out, and at the start of a launch.
// One per array and walker, in LDS: in registers the five took 115 of them.
template <typename CT>
struct BC {
  double min_total, max_total, e_max_total, e_max_count;
  CT min_count, max_count;
  uint64_t total_count, exists;
  double tmin;
  uint64_t nmin;
  CT cmin;
  uint64_t ncmin;
};
constexpr int kBinStats = 5;

// Counts live in the 64-bit count fields of the bin records: as integers,
// or as the bits of doubles.
template <typename CT>
__device__ __forceinline__ uint64_t ct_bits(CT v) {
  if constexpr (std::is_floating_point<CT>::value) {
    return __builtin_bit_cast(uint64_t, v);
  } else {
    return (uint64_t)v;
  }
}
template <typename CT>
__device__ __forceinline__ CT ct_from(uint64_t u) {
  if constexpr (std::is_floating_point<CT>::value) {
    return __builtin_bit_cast(double, u);
  } else {
    return (CT)u;
  }
}

__device__ __forceinline__ double shfl_f64(double v, int d) {
  return __builtin_bit_cast(double, (uint64_t)__shfl_xor((long long)__builtin_bit_cast(uint64_t, v), d, 64));
}

}  // namespace

// LIN: the linear interpolation of binning/linear.rs instead of the
// histogram of binning/histogram.rs.
template <int SYS, int KMAX, bool LIN, bool SH>
struct BinWalker {
  using CT = typename std::conditional<LIN, double, uint64_t>::type;
  Engine<SYS, KMAX, 0, M_CAN, 0, 0, SH> e;
  const BinArgs *Bp;
  sadmc_bbin *B;  // this walker's window of bins
  BC<CT> *bc;     // [kBinStats] in LDS
  int lane, G;
  double tm;  // the move count, whole and exact (these walkers start at 0: no state is uploaded)
  SADMC_DF uint64_t moves() const { return (uint64_t)tm; }
  uint64_t accepted;
  double acc_rate, tscale, usc;
  double min, width, inv_width, top, min_e, max_e;  // top = min + width * len
  int32_t len, base, cap;
  int32_t method, status;
  double num_states, tL;
  double min_T, too_lo, too_hi, tF, latest, t0, gamma;
  // 1 / tF, 1 / num_states and whether gamma is 0, after the last change
  double rtF, rNs;
  bool gzero;
  int32_t inv_t, has_min_gamma;
  double min_gamma;
  double lmax;  // the largest ln w total
  double next_verify, next_press;
  // histogram: the record of physical bin cp, and ln w at too_lo / too_hi with
  // the physical bins they are in (-1: none, ln w 0)
  sadmc_bbin C;
  int32_t cp, lo_p, hi_p;
  double lo_l, hi_l;
  // what a proposal leaves for the update
  bool relocate;
  // an extreme lost its last bin: rescan once the move's stores are all in
  // (a rescan between the two bins of a linear update would count the
  // second bin's new value twice); bit k: the totals, bit 8 + k: the counts
  uint32_t stale;
  // the high_resolution side histogram (energy_binning.rs:125, 328-330):
  // counts in HR[hs.base + i], its statistics in *HS (read and written
  // back by each increment, so they hold no registers across the move loop
  // when the histogram is off), and the smallest count's multiplicity
  uint64_t *HR;
  sadmc_hires *HS;
  uint64_t hr_ncmin;

  SADMC_DF const BinArgs &args() const { return *Bp; }

  // ------------------------------------------------------------ state I/O
  SADMC_DF static void bc_load(BC<CT> &c, const sadmc_bcounts &s) {
    c.min_total = s.min_total;
    c.max_total = s.max_total;
    c.e_max_total = s.e_max_total;
    c.e_max_count = s.e_max_count;
    c.min_count = ct_from<CT>(s.min_count);
    c.max_count = ct_from<CT>(s.max_count);
    c.total_count = s.total_count;
    c.exists = s.exists;
  }
  SADMC_DF static void bc_store(const BC<CT> &c, sadmc_bcounts &s) {
    s.min_total = c.min_total;
    s.max_total = c.max_total;
    s.e_max_total = c.e_max_total;
    s.e_max_count = c.e_max_count;
    s.min_count = ct_bits<CT>(c.min_count);
    s.max_count = ct_bits<CT>(c.max_count);
    s.total_count = c.total_count;
    s.exists = (int32_t)c.exists;
    s.reserved = 0;
  }

  SADMC_DF void load_idle(const BinArgs &ba, const SetArgs &sa, int lane_in_group, double *lds_group) {
    Bp = &ba;
    lane = lane_in_group;
    G = sa.G;
    e.load_idle(sa, lane_in_group, lds_group);
    status = e.status;
  }
  SADMC_DF void load(const BinArgs &ba, const SetArgs &sa, int walker, int lane_in_group, double *lds_group,
                     void *stats) {
    Bp = &ba;
    lane = lane_in_group;
    G = sa.G;
    bc = (BC<CT> *)stats;
    e.load_system(sa, walker, lane_in_group, lds_group);
    const sadmc_bwalker_state &w = ba.ws[walker];
    e.s0 = w.rng[0];
    e.s1 = w.rng[1];
    e.E = w.E;
    e.err = w.error;
    if (SYS != SYS_ISING) {
      if (SYS == SYS_LJ) e.R2 = w.geom * w.geom;
      e.L = w.geom;
      e.halfL = 0.5 * w.geom;
    }
    e.status = 0;
    tm = (double)w.moves;
    accepted = w.accepted_moves;
    acc_rate = w.acceptance_rate;
    tscale = w.translation_scale;
    usc = SYS == SYS_ISING ? 0.0 : uniform_scale(-tscale, tscale);
    min = w.min;
    width = w.width;
    min_e = w.min_e;
    max_e = w.max_e;
    inv_width = 1.0 / width;
    len = (int32_t)w.len;
    base = (int32_t)w.base;
    cap = (int32_t)w.cap;
    top = min + width * (double)len;
    method = w.method;
    status = w.status;
    num_states = (double)w.num_states;
    tL = (double)w.tL;
    min_T = w.min_T;
    too_lo = w.too_lo;
    too_hi = w.too_hi;
    tF = w.tF;
    latest = w.latest_parameter;
    t0 = w.t0;
    gamma = w.gamma;
    inv_t = w.inv_t;
    has_min_gamma = w.has_min_gamma;
    min_gamma = w.min_gamma;
    bc_load(bc[BC_LNW], w.lnw);
    bc_load(bc[BC_EN], w.energy);
    bc_load(bc[BC_TF], w.t_found);
    bc_load(bc[BC_HIST], w.hist);
    bc_load(bc[BC_PR], w.pressure);
    B = ba.bins + (int64_t)walker * ba.cap;
    next_verify = (double)((w.moves / 100000000ULL + 1) * 100000000ULL);
    const uint64_t Q = (uint64_t)sa.n * (uint64_t)sa.n;
    next_press = (double)((w.moves / Q + 1) * Q);
    cp = -1;
    stale = 0;
    relocate = false;
    lo_p = hi_p = -1;
    lo_l = hi_l = 0.0;
    gamma_changed();
    rescan_start();
    if (!LIN && !status) edges();
    HR = nullptr;
    HS = nullptr;
    if (ba.hr) {
      HR = ba.hr + (int64_t)walker * ba.hr_cap;
      HS = ba.hrs + walker;
      sadmc_hires hs = *HS;
      hr_rescan(hs);
      *HS = hs;
    }
  }

  SADMC_DF void store(int walker) {
    flush();
    if (SYS != SYS_ISING) {
      // the positions of the group's atoms, from the LDS mirror
      const SetArgs &sa = e.args();
      double *P = sa.pos + (int64_t)walker * 3 * sa.npad;
      for (int j = lane; j < sa.npad; j += G) {
        P[j] = e.lx[j];
        P[sa.npad + j] = e.ly[j];
        P[2 * sa.npad + j] = e.lz[j];
      }
    }
    if (lane != 0) return;
    if (SYS == SYS_ISING) e.args().spins[walker] = e.spins;
    sadmc_bwalker_state &w = args().ws[walker];
    w.rng[0] = e.s0;
    w.rng[1] = e.s1;
    w.E = e.E;
    w.error = e.err;
    w.moves = moves();
    w.accepted_moves = accepted;
    w.acceptance_rate = acc_rate;
    w.translation_scale = tscale;
    w.min = min;
    w.width = width;
    w.min_e = min_e;
    w.max_e = max_e;
    w.len = len;
    w.base = base;
    w.method = method;
    w.status = status;
    w.num_states = (uint64_t)num_states;
    w.tL = (uint64_t)tL;
    w.min_T = min_T;
    w.too_lo = too_lo;
    w.too_hi = too_hi;
    w.tF = tF;
    w.latest_parameter = latest;
    w.t0 = t0;
    w.gamma = gamma;
    bc_store(bc[BC_LNW], w.lnw);
    bc_store(bc[BC_EN], w.energy);
    bc_store(bc[BC_TF], w.t_found);
    bc_store(bc[BC_HIST], w.hist);
    bc_store(bc[BC_PR], w.pressure);
    if (status) *args().flag = 1;
  }

  // ------------------------------------------------------- bin records
  SADMC_DF static double &tot(sadmc_bbin &b, int k) {
    return k == BC_LNW ? b.lnw_total : k == BC_EN ? b.energy_total : k == BC_TF ? b.t_found_total : b.pressure_total;
  }
  SADMC_DF static uint64_t &cnt(sadmc_bbin &b, int k) {
    return k == BC_LNW   ? b.lnw_count
           : k == BC_EN  ? b.energy_count
           : k == BC_TF  ? b.t_found_count
           : k == BC_HIST ? b.hist_count
                          : b.pressure_count;
  }
  SADMC_DF static CT cget(sadmc_bbin &b, int k) { return ct_from<CT>(cnt(b, k)); }
  SADMC_DF static void cset(sadmc_bbin &b, int k, CT v) { cnt(b, k) = ct_bits<CT>(v); }
  // the "hist" extra only ever adds 0.0 to totals that start at 0.0
  SADMC_DF double total_at(int k, int64_t i) const { return k == BC_HIST ? 0.0 : tot(B[base + i], k); }
  SADMC_DF CT count_at(int k, int64_t i) const { return cget(B[base + i], k); }

  // histogram.rs:129-140; -1 or INT32_MAX for the out-of-range cases.  The
  // quotient from the reciprocal, as in the main engine's e_index.
  SADMC_DF int32_t index(double en) const {
    const double v = (en - min) * inv_width;
    if (__builtin_expect(fabs(__builtin_amdgcn_fract(v) - 0.5) < 0.5 - 1e-9 && fabs(v - 5.0e5) < 5.0e5, 1))
      return (int32_t)v;
    if (en < min) return -1;
    const double i = (en - min) / width;
    if (i == (double)len) return len == 0 ? -1 : (int32_t)i - 1;
    if (!(i < 2.0e9)) return INT32_MAX;
    return (int32_t)i;
  }
  SADMC_DF double fidx(double en) const { return (en - min) / width; }  // linear.rs:201-203
  SADMC_DF double energy_of(int32_t i) const { return min + ((double)i + 0.5) * width; }
  // BinCounts::get_total / get_count of linear.rs:139-152 over the
  // interpretation of linear.rs:84-98, in the iterator's order
  SADMC_DF double lin_interp(bool counts, double f) const {
    double t = 0.0;
    if (len == 0 || f < -1.0) return t;
    auto val = [&](int64_t i) -> double {
      return counts ? (double)count_at(BC_LNW, i) : B[base + i].lnw_total;
    };
    if (f < 0.0) {
      t += val(0) * (1.0 - (-f));
    } else if (f < (double)len - 1.0) {
      const int64_t i = (int64_t)f;
      const double o = f - (double)i;
      t += val(i + 1) * o;
      t += val(i) * (1.0 - o);
    } else if (f < (double)len) {
      t += val(len - 1) * (1.0 - (f - ((double)len - 1.0)));
    }
    return t;
  }
  SADMC_DF double get_lnw(double en) const {
    if (LIN) return lin_interp(false, fidx(en));
    const int32_t i = index(en);
    return (i >= 0 && i < len) ? B[base + i].lnw_total : 0.0;
  }
  // get_count as PerEnergy: count / width
  SADMC_DF double get_count(double en) const {
    if (LIN) return lin_interp(true, fidx(en)) / width;
    const int32_t i = index(en);
    return (double)((i >= 0 && i < len) ? (uint64_t)count_at(BC_LNW, i) : 0) / width;
  }

  // ---------------------------------------------------- group reductions
  SADMC_DF uint64_t group_sum_u64(uint64_t v) const {
    for (int d = 1; d < G; d <<= 1) v += (uint64_t)__shfl_xor((long long)v, d, 64);
    return v;
  }
  // Rescans, four bins per lane per step so that their loads overlap.
  // Smallest total of array k and its multiplicity (+inf, 0 when empty).
  SADMC_DF void rescan_total(int k) {
    double m = __builtin_inf();
    uint64_t c = 0;
    if (k != BC_HIST) {
      for (int64_t j0 = lane; j0 < len; j0 += 4 * G) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int64_t j = j0 + u * G;
          v[u] = j < len ? total_at(k, j) : __builtin_inf();
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (j0 + u * G >= len) continue;
          if (v[u] < m) {
            m = v[u];
            c = 1;
          } else if (v[u] == m) {
            c += 1;
          }
        }
      }
    } else if (lane < len) {
      m = 0.0;
      c = (uint64_t)((len - lane + G - 1) / G);
    }
    for (int d = 1; d < G; d <<= 1) {
      const double om = shfl_f64(m, d);
      const uint64_t oc = (uint64_t)__shfl_xor((long long)c, d, 64);
      if (om < m) {
        m = om;
        c = oc;
      } else if (om == m) {
        c += oc;
      }
    }
    bc[k].tmin = m;
    bc[k].nmin = c;
  }
  SADMC_DF void rescan_count(int k) {
    CT big;
    if constexpr (LIN) {
      big = __builtin_inf();
    } else {
      big = ~0ULL;
    }
    CT m = big;
    uint64_t c = 0;
    for (int64_t j0 = lane; j0 < len; j0 += 4 * G) {
      CT v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int64_t j = j0 + u * G;
        v[u] = j < len ? count_at(k, j) : big;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (j0 + u * G >= len) continue;
        if (v[u] < m) {
          m = v[u];
          c = 1;
        } else if (v[u] == m) {
          c += 1;
        }
      }
    }
    for (int d = 1; d < G; d <<= 1) {
      const CT om = ct_from<CT>((uint64_t)__shfl_xor((long long)ct_bits<CT>(m), d, 64));
      const uint64_t oc = (uint64_t)__shfl_xor((long long)c, d, 64);
      if (om < m) {
        m = om;
        c = oc;
      } else if (om == m) {
        c += oc;
      }
    }
    bc[k].cmin = m;
    bc[k].ncmin = c;
  }
  SADMC_DF void rescan_lmax() {
    double m = -__builtin_inf();
    for (int64_t j0 = lane; j0 < len; j0 += 4 * G) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int64_t j = j0 + u * G;
        v[u] = j < len ? B[base + j].lnw_total : -__builtin_inf();
      }
#pragma unroll
      for (int u = 0; u < 4; u++) m = v[u] > m ? v[u] : m;
    }
    for (int d = 1; d < G; d <<= 1) {
      const double om = shfl_f64(m, d);
      m = om > m ? om : m;
    }
    lmax = m;
  }
  // Every array's extremes in one pass over the records: a launch's start
  // would otherwise read the whole window once per statistic (16384 LJ31
  // walkers of 8000 bins: 73 GB and 11.7 ms in seven passes).
  SADMC_DF void rescan_start() {
    const CT big = LIN ? (CT)__builtin_inf() : (CT)~0ULL;
    double m[kBinStats], l = -__builtin_inf();
    CT q[kBinStats];
    uint32_t cm[kBinStats], cq[kBinStats];
#pragma unroll
    for (int k = 0; k < kBinStats; k++) {
      m[k] = __builtin_inf();
      q[k] = big;
      cm[k] = cq[k] = 0;
    }
    for (int32_t j = lane; j < len; j += G) {
      sadmc_bbin r = B[base + j];
      l = r.lnw_total > l ? r.lnw_total : l;
#pragma unroll
      for (int k = 0; k < kBinStats; k++) {
        const double v = k == BC_HIST ? 0.0 : tot(r, k);
        const CT c = cget(r, k);
        cm[k] = v < m[k] ? 1 : cm[k] + (v == m[k] ? 1 : 0);
        m[k] = v < m[k] ? v : m[k];
        cq[k] = c < q[k] ? 1 : cq[k] + (c == q[k] ? 1 : 0);
        q[k] = c < q[k] ? c : q[k];
      }
    }
    for (int d = 1; d < G; d <<= 1) {
      const double ol = shfl_f64(l, d);
      l = ol > l ? ol : l;
#pragma unroll
      for (int k = 0; k < kBinStats; k++) {
        const double om = shfl_f64(m[k], d);
        const uint32_t oc = (uint32_t)__shfl_xor((int)cm[k], d, 64);
        cm[k] = om < m[k] ? oc : cm[k] + (om == m[k] ? oc : 0);
        m[k] = om < m[k] ? om : m[k];
        const CT oq = ct_from<CT>((uint64_t)__shfl_xor((long long)ct_bits<CT>(q[k]), d, 64));
        const uint32_t od = (uint32_t)__shfl_xor((int)cq[k], d, 64);
        cq[k] = oq < q[k] ? od : cq[k] + (oq == q[k] ? od : 0);
        q[k] = oq < q[k] ? oq : q[k];
      }
    }
    if (bc[BC_LNW].exists) lmax = l;
#pragma unroll
    for (int k = 0; k < kBinStats; k++)
      if (bc[k].exists) {
        bc[k].tmin = m[k];
        bc[k].nmin = cm[k];
        bc[k].cmin = q[k];
        bc[k].ncmin = cq[k];
      }
  }
  SADMC_DF void rescan_all(int k) {
    rescan_total(k);
    rescan_count(k);
    if (k == BC_LNW) rescan_lmax();
  }
  // One bin of array k (statistics c) goes from v to w (totals) / from a to b
  // (counts); settle() afterwards, when every bin of the update is stored.
  SADMC_DF void track_total(int k, BC<CT> &c, double v, double w) {
    if (stale & (1u << k)) return;
    const bool below = w < c.tmin, at = w == c.tmin, left = !below & !at & (v == c.tmin);
    c.nmin = below ? 1 : c.nmin + ((at & (v != w)) ? 1 : 0) - (left ? 1 : 0);
    c.tmin = below ? w : c.tmin;
    stale |= (left & (c.nmin == 0)) ? 1u << k : 0u;
  }
  SADMC_DF void track_count(int k, BC<CT> &c, CT a, CT b) {
    if (stale & (256u << k)) return;
    const bool below = b < c.cmin, at = b == c.cmin, left = !below & !at & (a == c.cmin);
    c.ncmin = below ? 1 : c.ncmin + ((at & (a != b)) ? 1 : 0) - (left ? 1 : 0);
    c.cmin = below ? b : c.cmin;
    stale |= (left & (c.ncmin == 0)) ? 256u << k : 0u;
  }
  // `c` is array k's statistics, held by the caller and stored back by it.
  SADMC_DF void settle(int k, BC<CT> &c) {
    if (__builtin_expect(stale != 0, 0)) {
      if (!LIN) flush();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (stale & (1u << k)) {
        rescan_total(k);
        c.tmin = bc[k].tmin;
        c.nmin = bc[k].nmin;
      }
      if (stale & (256u << k)) {
        rescan_count(k);
        c.cmin = bc[k].cmin;
        c.ncmin = bc[k].ncmin;
      }
      stale = 0;
    }
  }
  // a zero bin joins array k
  SADMC_DF void track_new_zero(int k) {
    BC<CT> c = bc[k];
    c.min_total = 0.0;
    c.min_count = 0;
    if (0.0 < c.tmin) {
      c.tmin = 0.0;
      c.nmin = 1;
    } else if (0.0 == c.tmin) {
      c.nmin += 1;
    }
    if ((CT)0 < c.cmin) {
      c.cmin = 0;
      c.ncmin = 1;
    } else if ((CT)0 == c.cmin) {
      c.ncmin += 1;
    }
    bc[k] = c;
    if (k == BC_LNW && !(lmax >= 0.0)) lmax = 0.0;
  }

  // ---------------------------------------- the high_resolution histogram
  // The smallest count and its multiplicity (a count never exceeds the
  // number of moves, so ~0 stands for an empty histogram).
  SADMC_DF void hr_rescan(sadmc_hires &hs) {
    uint64_t m = ~0ULL, c = 0;
    for (int64_t j0 = lane; j0 < hs.len; j0 += 4 * G) {
      uint64_t v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int64_t j = j0 + u * G;
        v[u] = j < hs.len ? HR[hs.base + j] : ~0ULL;
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (j0 + u * G >= hs.len) continue;
        if (v[u] < m) {
          m = v[u];
          c = 1;
        } else if (v[u] == m) {
          c += 1;
        }
      }
    }
    for (int d = 1; d < G; d <<= 1) {
      const uint64_t om = (uint64_t)__shfl_xor((long long)m, d, 64);
      const uint64_t oc = (uint64_t)__shfl_xor((long long)c, d, 64);
      if (om < m) {
        m = om;
        c = oc;
      } else if (om == m) {
        c += oc;
      }
    }
    if (hs.len > 0) hs.min_count = m;
    hr_ncmin = c;
  }
  // insert_zero / push_zero (histogram.rs:47-58) on the side histogram
  SADMC_DF void hr_new_zero(sadmc_hires &hs, int64_t p) {
    HR[p] = 0;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (hs.min_count == 0) {
      hr_ncmin += 1;
    } else {
      hs.min_count = 0;
      hr_ncmin = 1;
    }
    hs.len += 1;
  }
  // Bins::increment_count(e, 0.0) (histogram.rs:182-192, 147-167, 59-81):
  // min_e / max_e, the window grown to hold e, then the bin's count and the
  // count statistics (the totals stay 0)
  SADMC_DF bool hr_increment(double en) {
    sadmc_hires hs = *HS;
    const bool ok = hr_increment(hs, en);
    *HS = hs;
    return ok;
  }
  SADMC_DF bool hr_increment(sadmc_hires &hs, double en) {
    if (en > hs.max_e) hs.max_e = en;
    if (en < hs.min_e) hs.min_e = en;
    if (hs.len == 0) {
      hs.min = floor(en / hs.width) * hs.width;
      const int64_t b0 = (int64_t)floor((hs.min - args().e_lo) / hs.width) + 4;
      hs.base = b0 < 0 ? 0 : (b0 >= args().hr_cap ? args().hr_cap - 1 : b0);
    }
    while (en < hs.min) {
      if (hs.base == 0) {
        status = SADMC_WS_CAPACITY;
        return false;
      }
      hs.base -= 1;
      hr_new_zero(hs, hs.base);
      hs.min -= hs.width;
    }
    while (en >= hs.min + hs.width * (double)hs.len) {
      if (hs.base + hs.len >= args().hr_cap) {
        status = SADMC_WS_CAPACITY;
        return false;
      }
      hr_new_zero(hs, hs.base + hs.len);
    }
    // histogram.rs:129-140
    const double fi = (en - hs.min) / hs.width;
    const int64_t idx = fi == (double)hs.len ? (int64_t)fi - 1 : (int64_t)fi;
    if (!(en >= hs.min) || idx < 0 || idx >= hs.len) {  // an index panic in the reference
      status = SADMC_WS_INDEX;
      return false;
    }
    uint64_t &r = HR[hs.base + idx];
    const uint64_t old_count = r, new_count = old_count + 1;
    r = new_count;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    hs.total_count += 1;
    if (old_count == hs.min_count && --hr_ncmin == 0) hr_rescan(hs);
    if (new_count > hs.max_count) {
      hs.max_count = new_count;
      hs.e_max_count = en;
    }
    return true;
  }

  // ------------------------------------------------------------ growth
  SADMC_DF void zero_bin(int32_t p) {
    {
      sadmc_bbin z;
      z.lnw_total = 0.0;
      z.lnw_count = 0;
      z.energy_total = 0.0;
      z.energy_count = 0;
      z.t_found_total = 0.0;
      z.t_found_count = 0;
      z.hist_count = 0;
      z.pressure_total = 0.0;
      z.pressure_count = 0;
      z.reserved = 0;
      B[p] = z;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  SADMC_DF void grown() {
#pragma unroll 1
    for (int k = 0; k < kBinStats; k++)
      if (bc[k].exists) track_new_zero(k);
    len += 1;
  }
  // histogram.rs:141-158 / linear.rs:204-222 (insert_zero / push_zero on
  // lnw and every extra; the linear binning keeps one more bin above)
  SADMC_DF bool prep(double en) {
    if (len == 0) {
      min = floor(en / width) * width;
      int64_t b0 = (int64_t)floor((min - args().e_lo) / width) + 4;
      base = (int32_t)(b0 < 0 ? 0 : (b0 >= cap ? cap - 1 : b0));
    }
    while (status == 0 && en < min) {
      if (base == 0) {
        status = SADMC_WS_CAPACITY;
      } else {
        base -= 1;
        zero_bin(base);
        grown();
        min -= width;
      }
    }
    while (status == 0 && (LIN ? en >= min + width * ((double)len - 1.0) : en >= min + width * (double)len)) {
      if (base + len >= cap) {
        status = SADMC_WS_CAPACITY;
      } else {
        zero_bin(base + len);
        grown();
      }
    }
    top = min + width * (double)len;
    return status == 0;
  }

  // ------------------------------- the histogram's current record (cp, C)
  SADMC_DF void flush() {
    if (!LIN && cp >= 0 && lane == 0) B[cp] = C;
  }
  SADMC_DF void focus(int32_t p) {
    if (p != cp) {
      flush();
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      C = B[p];
      cp = p;
    }
  }
  SADMC_DF double lnw_of(int32_t p) const { return p < 0 ? 0.0 : p == cp ? C.lnw_total : B[p].lnw_total; }
  // lo_p, hi_p and ln w there: after a change of too_lo, too_hi or the window.
  SADMC_DF void edges() {
    const int32_t i = index(too_lo), j = index(too_hi);
    lo_p = i >= 0 && i < len ? base + i : -1;
    hi_p = j >= 0 && j < len ? base + j : -1;
    lo_l = lnw_of(lo_p);
    hi_l = lnw_of(hi_p);
  }
  // The window grown to hold `en` and its bin's record at hand.
  SADMC_DF bool enter(double en) {
    if (len == 0 || en < min || en >= top) {
      if (!prep(en)) return false;
      edges();
    }
    const int32_t idx = index(en);
    if (idx < 0 || idx >= len) {  // an index panic in the reference
      status = SADMC_WS_INDEX;
      return false;
    }
    focus(base + idx);
    return true;
  }

  // BinCounts::increment_count (histogram.rs:59-81) on lnw, the current bin
  SADMC_DF void lnw_increment(double en, double value) {
    BC<CT> c = bc[BC_LNW];
    c.total_count += 1;
    const CT old_count = cget(C, BC_LNW);
    const CT new_count = old_count + 1;
    const double old_total = C.lnw_total;
    const double new_total = old_total + value;
    cset(C, BC_LNW, new_count);
    C.lnw_total = new_total;
    lo_l = cp == lo_p ? new_total : lo_l;
    hi_l = cp == hi_p ? new_total : hi_l;
    track_total(BC_LNW, c, old_total, new_total);
    track_count(BC_LNW, c, old_count, new_count);
    settle(BC_LNW, c);
    lmax = new_total > lmax ? new_total : lmax;
    // max_of(total) == total[idx], min_of(total) and min(count) after the
    // update are the tracked extremes
    if (new_total > c.max_total && lmax == new_total) {
      c.max_total = new_total;
      c.e_max_total = en;
    }
    if (old_total == c.min_total) c.min_total = c.tmin;
    if (old_count == c.min_count) c.min_count = c.cmin;
    if (new_count > c.max_count) {
      c.max_count = new_count;
      c.e_max_count = en;
    }
    bc[BC_LNW] = c;
  }

  // BinCounts::increment_count of linear.rs:99-137 on lnw: the weight
  // splits over bins idx and idx + 1
  SADMC_DF void lnw_increment_lin(double elo, double ehi, double f, double value) {
    BC<CT> c = bc[BC_LNW];
    const int64_t idx = (int64_t)f;
    const double offset = f - (double)idx;
    sadmc_bbin &r0 = B[base + idx];
    sadmc_bbin &r1 = B[base + idx + 1];
    c.total_count += 1;
    const CT oc = cget(r0, BC_LNW), opc = cget(r1, BC_LNW);
    const CT c0 = oc + (1.0 - offset), c1 = opc + offset;
    const double ot = r0.lnw_total, opt = r1.lnw_total;
    const double t0v = ot + value * (1.0 - offset), t1v = opt + value * offset;
    cset(r0, BC_LNW, c0);
    cset(r1, BC_LNW, c1);
    r0.lnw_total = t0v;
    r1.lnw_total = t1v;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    track_total(BC_LNW, c, ot, t0v);
    track_total(BC_LNW, c, opt, t1v);
    track_count(BC_LNW, c, oc, c0);
    track_count(BC_LNW, c, opc, c1);
    settle(BC_LNW, c);
    if (t0v > lmax) lmax = t0v;
    if (t1v > lmax) lmax = t1v;
    if (t0v > c.max_total && lmax == t0v) {
      c.max_total = t0v;
      c.e_max_total = elo;
    }
    if (t1v > c.max_total && lmax == t1v) {
      c.max_total = t1v;
      c.e_max_total = ehi;
    }
    if (ot == c.min_total || opt == c.min_total) c.min_total = c.tmin;
    if (oc == c.min_count || opc == c.min_count) c.min_count = c.cmin;
    if (c0 > c.max_count) {
      c.max_count = c0;
      c.e_max_count = elo;
    }
    if (c1 > c.max_count) {
      c.max_count = c1;
      c.e_max_count = ehi;
    }
    bc[BC_LNW] = c;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }

  // Bins::accumulate_extra (histogram.rs:219-245, linear.rs:267-310); the
  // histogram's bin is the current one.
  SADMC_DF void new_stat(BC<CT> &c) const {  // BinCounts::new over the current bins
    c.tmin = 0.0;
    c.nmin = (uint64_t)len;
    c.cmin = 0;
    c.ncmin = (uint64_t)len;
    c.exists = 1;
    c.min_total = 0.0;
    c.max_total = 0.0;
    c.e_max_total = -__builtin_inf();
    c.e_max_count = -__builtin_inf();
    c.min_count = 0;
    c.max_count = 0;
    c.total_count = 0;
  }
  SADMC_DF bool accumulate(int k, double en, double value) {
    if constexpr (!LIN) {
      BC<CT> c = bc[k];
      if (__builtin_expect(!c.exists, 0)) new_stat(c);
      c.total_count += 1;
      const CT old_count = cget(C, k);
      const CT new_count = old_count + 1;
      const double old_total = k == BC_HIST ? 0.0 : tot(C, k);
      const double new_total = old_total + value;
      cset(C, k, new_count);
      if (k != BC_HIST) tot(C, k) = new_total;
      track_count(k, c, old_count, new_count);
      if (k != BC_HIST) track_total(k, c, old_total, new_total);
      settle(k, c);
      if (new_count == c.min_count + 1) c.min_count = c.cmin;
      if (new_count > c.max_count) c.max_count = new_count;
      if (new_total > c.max_total) c.max_total = new_total;
      if (old_total == c.min_total) c.min_total = k == BC_HIST ? 0.0 : c.tmin;
      bc[k] = c;
      return true;
    } else {
      if (!prep(en)) return false;
      const double f = fidx(en);
      const int64_t idx = (int64_t)f;
      if (!(f >= 0.0) || idx + 1 >= len) {  // the reference's assert / index panic
        status = SADMC_WS_INDEX;
        return false;
      }
      BC<CT> c = bc[k];
      if (!c.exists) new_stat(c);
      c.total_count += 1;
      const double off = f - (double)idx;
      sadmc_bbin &r0 = B[base + idx];
      sadmc_bbin &r1 = B[base + idx + 1];
      const CT oc = cget(r0, k), opc = cget(r1, k);
      const CT c0 = oc + (1.0 - off), c1 = opc + off;
      const double ot = k == BC_HIST ? 0.0 : tot(r0, k), opt = k == BC_HIST ? 0.0 : tot(r1, k);
      const double t0v = ot + value * (1.0 - off), t1v = opt + value * off;
      cset(r0, k, c0);
      cset(r1, k, c1);
      if (k != BC_HIST) {
        tot(r0, k) = t0v;
        tot(r1, k) = t1v;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      track_count(k, c, oc, c0);
      track_count(k, c, opc, c1);
      if (k != BC_HIST) {
        track_total(k, c, ot, t0v);
        track_total(k, c, opt, t1v);
      }
      settle(k, c);
      if (oc == c.min_count || opc == c.min_count) c.min_count = c.cmin;
      if (c0 > c.max_count) c.max_count = c0;
      if (c1 > c.max_count) c.max_count = c1;
      if (t0v > c.max_total) c.max_total = t0v;
      if (t1v > c.max_total) c.max_total = t1v;
      if (ot == c.min_total || opt == c.min_total) c.min_total = k == BC_HIST ? 0.0 : c.tmin;
      bc[k] = c;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      return true;
    }
  }

  // Bins::zero_out_extra (histogram.rs:246-259) on "hist"
  SADMC_DF void zero_out_hist() {
    BC<CT> c = bc[BC_HIST];
    if (!c.exists) return;
    flush();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int64_t j = lane; j < len; j += G) cset(B[base + j], BC_HIST, (CT)0);
    if (!LIN) cset(C, BC_HIST, (CT)0);
    c.min_total = 0.0;
    c.max_total = -__builtin_inf();
    c.min_count = 0;
    c.max_count = 0;
    c.total_count = 0;
    c.cmin = 0;
    c.ncmin = (uint64_t)len;
    bc[BC_HIST] = c;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }

  // count_states with e >= too_lo && e <= too_hi (histogram.rs:191-200)
  SADMC_DF uint64_t count_states() const {
    uint64_t t = 0;
    for (int32_t j = lane; j < len; j += G) {
      const double en = energy_of(j);
      if (en >= too_lo && en <= too_hi) t += 1;
    }
    return group_sum_u64(t);
  }

  // -------------------------------------------------------------- method
  // energy_binning.rs:503-530; the quotients by tF and the number of states as
  // in the main engine (Engine::quot)
  SADMC_DF double gamma_now() const {
    if (method == SADMC_SAD) {
      const double q = e.quot(tm, tF, rtF);
      const double g = (latest + q) / (latest + e.quot(tm, num_states, rNs) * q);
      return gzero ? 0.0 : g;
    }
    if (method == SADMC_SAMC) return tm > t0 ? t0 / tm : 1.0;
    return gamma;
  }
  SADMC_DF void gamma_changed() {
    rtF = 1.0 / tF;
    rNs = 1.0 / num_states;
    gzero = latest * tF * num_states == 0.0;
  }

  // set_lnw (histogram.rs:182-190, linear.rs:254-262) for SAD's two range
  // extensions (in the linear binning a bin's count is read at its centre,
  // from it and the next bin, before that next bin may be cleared: each
  // step's loads come before its stores); bins
  // above `edge` (up) or below it (down) with a nonzero count take `v` (up)
  // or v + (e - edge)/min_T (down) and lose their count.
  SADMC_DF void set_lnw_sad(bool up, double edge, double v) {
    flush();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int32_t j = lane; j < len; j += G) {
      const double en = energy_of(j);
      const bool side = up ? en > edge : en < edge;
      if (side && get_count(en) > 0.0) {
        sadmc_bbin &r = B[base + j];
        r.lnw_total = up ? v : v + (en - edge) / min_T;
        cset(r, BC_LNW, (CT)0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (!LIN) C = B[cp];
    rescan_all(BC_LNW);
  }

  // energy_binning.rs:276-319: the test, on ln w and the count at the proposed
  // energy's bin; l1 and l2 carry SAD's extension already.
  SADMC_DF bool decide(bool go, double e2, double l1, double l2, bool unseen) {
    const bool rejected = e.mh_test(go & (l2 > l1), l1 - l2);
    if (method == SADMC_SAD && (go & !rejected & unseen) && e2 < too_hi && e2 > too_lo) tL = tm;
    return go & !rejected;
  }

  // energy_binning.rs:566-611 up to the accepted move: the visited energy is
  // added to its bin, then a move is proposed and tested.  True: the
  // system's energy is due for a recomputation.
  SADMC_DF bool propose() {
    tm += 1.0;
    if (SYS != SYS_ISING && __builtin_expect(tm == next_verify, 0)) {
      next_verify += 1.0e8;
      e.verify_energy();
      if (e.status) {
        status = e.status;
        return false;
      }
    }
    const double e1 = e.E;
    if (!LIN && __builtin_expect(cp < 0, 0) && !enter(e1)) return false;
    if (!accumulate(BC_EN, e1, e1)) return false;
    if (SYS == SYS_WCA && args().collect_pressure && __builtin_expect(tm == next_press, 0)) {
      next_press += (double)e.n * (double)e.n;
      const double pv = e.pressure();
      if (!accumulate(BC_PR, e1, pv)) return false;
    }
    const double rs = sqrt(1.0 / tm);
    acc_rate *= 1.0 - rs;
    double e2 = e1;
    bool go = e.cube_plan(tscale, usc, e2);
    if (args().has_max_e) go = go & !((e2 > args().max_e) & (e2 > e1));
    if (args().has_min_e) go = go & !((e2 < args().min_e) & (e2 < e1));
    bool acc, same = true, in = true;
    int32_t p2 = 0;
    sadmc_bbin N;
    if constexpr (!LIN) {
      const int32_t i2 = index(e2);
      in = (i2 >= 0) & (i2 < len);
      p2 = (go & in) ? base + i2 : cp;
      N = B[p2];
      // independent of the record being loaded
      e.spec_draw();
      const bool sad = method == SADMC_SAD, above2 = sad & (e2 > too_hi), below2 = sad & (e2 < too_lo);
      double l1 = (sad & (e1 > too_hi)) ? hi_l : C.lnw_total;
      if (__builtin_expect(sad & (e1 < too_lo), 0)) l1 = lo_l + (e1 - too_lo) / min_T;
      double out2 = hi_l;
      if (__builtin_expect(below2, 0)) out2 = lo_l + (e2 - too_lo) / min_T;
      same = p2 == cp;
      // the record whole before the old one's stores are issued: loads and
      // stores complete in order
      asm volatile("" ::"v"(N.lnw_total), "v"(N.lnw_count), "v"(N.energy_total), "v"(N.energy_count),
                   "v"(N.t_found_total), "v"(N.t_found_count), "v"(N.hist_count), "v"(N.pressure_total),
                   "v"(N.pressure_count), "v"(N.reserved));
      const double w2 = !in ? 0.0 : same ? C.lnw_total : N.lnw_total;
      const uint64_t n2 = !in ? 0 : same ? C.lnw_count : N.lnw_count;
      acc = decide(go, e2, l1, (above2 | below2) ? out2 : w2, n2 == 0);
    } else {
      double l1 = get_lnw(e1), l2 = get_lnw(e2);
      if (method == SADMC_SAD) {
        if (e1 < too_lo)
          l1 = get_lnw(too_lo) + (e1 - too_lo) / min_T;
        else if (e1 > too_hi)
          l1 = get_lnw(too_hi);
        if (e2 < too_lo)
          l2 = get_lnw(too_lo) + (e2 - too_lo) / min_T;
        else if (e2 > too_hi)
          l2 = get_lnw(too_hi);
      }
      e.spec_draw();
      acc = decide(go, e2, l1, l2, get_count(e2) == 0.0);
    }
    accepted += acc ? 1 : 0;
    acc_rate = acc ? acc_rate + rs : acc_rate;
    const bool trip = e.take_energy(acc, e2, e.pdabse);
    if (acc) e.confirm_system();
    if constexpr (!LIN) {
      relocate = trip | (acc & (!in | (e2 < min) | (e2 >= top)));
      if (acc & !relocate & !same) {
        flush();
        C = N;
        cp = p2;
      }
    }
    return trip;
  }

  // energy_binning.rs:320-500 for the energy the walker is at now
  SADMC_DF void update() {
    const double en = e.E;
    const double g = gamma_now();
    const double old_highest = (double)bc[BC_LNW].max_count / width;
    const CT old_max = bc[BC_LNW].max_count;
    max_e = en > max_e ? en : max_e;
    min_e = en < min_e ? en : min_e;
    bool unseen;
    if constexpr (LIN) {
      unseen = get_count(en) == 0.0;
      if (!prep(en)) return;
      const double f = fidx(en);  // linear.rs:237-253
      const int64_t ii = (int64_t)f;
      if (!(f >= 0.0) || ii + 1 >= len) {  // an index panic in the reference
        status = SADMC_WS_INDEX;
        return;
      }
      lnw_increment_lin(energy_of(ii), energy_of(ii + 1), f, g * 1.0 / width);
    } else {
      if (__builtin_expect(relocate, 0)) {
        relocate = false;
        flush();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        unseen = get_count(en) == 0.0;  // before the window grows
        if (!enter(en)) return;
      } else {
        unseen = C.lnw_count == 0;
      }
      lnw_increment(en, g);
    }
    if (HR && !hr_increment(en)) return;
    if (method == SADMC_SAD) {
      if (__builtin_expect(unseen, 0) && !accumulate(BC_TF, en, tm)) return;
      // here > old_highest, both per energy (whole counts compare alike)
      const bool higher = LIN ? get_count(en) > old_highest : ct_bits<CT>(cget(C, BC_LNW)) > ct_bits<CT>(old_max);
      if (__builtin_expect(higher, 0)) {
        const bool up = en > too_hi;
        if (up || en < too_lo) {
          const double v = LIN ? get_lnw(up ? too_hi : too_lo) : up ? hi_l : lo_l;
          set_lnw_sad(up, up ? too_hi : too_lo, v);
          latest = (up ? en - too_lo : too_hi - en) / min_T;
          tL = tm;
          if (up) {
            too_hi = en;
          } else {
            too_lo = en;
          }
          num_states = (double)count_states();
          if (!LIN) edges();
        }
      }
      if (__builtin_expect(tL == tm, 0)) {
        const double old_tF = tF;
        tF = bc[BC_TF].exists ? bc[BC_TF].max_total : 0.0;
        if (old_tF != tF && args().move_plan == SADMC_ACCEPTANCE_RATE) {
          double s = acc_rate / args().move_param;
          s = s < 0.8 ? 0.8 : (s > 1.2 ? 1.2 : s);
          tscale *= s;
          if (SYS != SYS_ISING) usc = uniform_scale(-tscale, tscale);
        }
        gamma_changed();
      }
    } else if (method == SADMC_WL) {
      const double old_lowest = bc[BC_HIST].exists ? (double)bc[BC_HIST].min_count / width : 0.0;
      if (!accumulate(BC_HIST, en, 0.0)) return;
      if (has_min_gamma && gamma < min_gamma) return;
      const double lowest = (double)bc[BC_HIST].min_count / width;
      if (__builtin_expect(lowest > old_lowest, 0)) {
        flush();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const bool ok_lo = !args().has_min_e || get_count(args().min_e) > 0.0;
        const bool ok_hi = !args().has_max_e || get_count(args().max_e) > 0.0;
        if (ok_lo && ok_hi) {
          const double mean = (double)bc[BC_HIST].total_count / (width * (double)len);
          if ((inv_t && lowest > 0.0) || lowest >= 0.8 * mean) {
            gamma *= 0.5;
            zero_out_hist();
            if (has_min_gamma && gamma < min_gamma) gamma = 0.0;
          }
          if (inv_t && gamma < (double)len / tm) {
            method = SADMC_SAMC;
            t0 = (double)len;
          }
        }
      }
    }
  }

  SADMC_DF void run(uint64_t nmoves) {
    for (uint64_t k = 0; k < nmoves && __any(status == 0); k++) {
      bool trip = false;
      if (__builtin_expect(status == 0, 1)) trip = propose();
      if (__builtin_expect(__any(trip), 0)) {
        e.full_energies(trip);
        if (trip) e.took_full_energy();
      }
      if (__builtin_expect(status == 0, 1)) update();
    }
  }

  // energy_binning.rs:533-564: the greedy descent below max_allowed_energy
  // and the initial method state (the histogram stays empty until the
  // first move).
  SADMC_DF void from_params() {
    e.E = e.full_energy();
    e.err = 0.0;
    if (args().has_max_e) {
      const double sc = SYS == SYS_ISING ? 0.0 : uniform_scale(-0.05, 0.05);
      for (uint64_t k = 0; k < 100000000ULL; k++) {
        double newe;
        if (e.cube_plan(0.05, sc, newe)) {
          if (newe < e.E) e.confirm();
          if (e.E < args().max_e) break;
        }
      }
    }
    const double E = e.E;
    too_lo = E;
    too_hi = E;
    num_states = 0.0;
    tL = 0.0;
    tF = 0.0;
    latest = 0.0;
    min = (round(E / width) - 0.5) * width;  // Bins::new (histogram.rs:162-170)
    min_e = E;
    max_e = E;
    len = 0;
    top = min;
    tm = 0.0;
    accepted = 0;
    acc_rate = 0.5;
    tscale = args().move_plan == SADMC_TRANSLATION_SCALE ? args().move_param : 0.05;
    // ln w's BinCounts::new(0); the extras do not exist yet (all zero)
#pragma unroll 1
    for (int k = 0; k < kBinStats; k++) {
      bc[k].exists = 0;
      bc[k].min_total = 0.0;
      bc[k].max_total = 0.0;
      bc[k].e_max_total = 0.0;
      bc[k].e_max_count = 0.0;
      bc[k].min_count = 0;
      bc[k].max_count = 0;
      bc[k].total_count = 0;
    }
    bc[BC_LNW].exists = 1;
    bc[BC_LNW].e_max_total = -__builtin_inf();
    bc[BC_LNW].e_max_count = -__builtin_inf();
    if (HR) {  // Bins::new(system.energy(), de) (energy_binning.rs:568-570)
      sadmc_hires hs;
      hs.width = args().hr_de;
      hs.min = (round(E / hs.width) - 0.5) * hs.width;
      hs.min_e = E;
      hs.max_e = E;
      hs.len = 0;
      hs.base = 0;
      hs.total_count = 0;
      hs.min_count = 0;
      hs.max_count = 0;
      hs.e_max_count = -__builtin_inf();
      *HS = hs;
      hr_ncmin = 0;
    }
    status = e.status;
  }
};

// `per` walkers a wave, as for the main engine's run kernel; registers for two
// waves per SIMD, which 16384 walkers at 8 lanes need.
template <int SYS, int KMAX, bool LIN, bool SH>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void k_bin(BinArgs ba, SetArgs sa, uint64_t nmoves, int init, int per) {
  extern __shared__ double lds[];
  const int G = sa.G, group = threadIdx.x / (SH ? G * KMAX : G);
  const int lane = threadIdx.x & (G - 1);
  const int walker = blockIdx.x * per + group;
  const bool held = group < per && walker < sa.W;
  double *tile = lds + (SYS == SYS_ISING ? 0 : group * 3 * sa.npad);
  char *stats = (char *)(lds + (SYS == SYS_ISING ? 0 : per * 3 * sa.npad)) +
                group * (int)(kBinStats * sizeof(BC<uint64_t>));
  BinWalker<SYS, KMAX, LIN, SH> b;
  if (held) {
    b.load(ba, sa, walker, lane, tile, stats);
  } else {
    b.load_idle(ba, sa, lane, tile);
  }
  if (init) {
    if (held) b.from_params();
  } else {
    b.run(nmoves);
  }
  if (held) b.store(walker);
}

template <int SYS, int KMAX>
static hipError_t launch_bin_t(const BinArgs &ba, const SetArgs &sa, uint64_t moves, int init, hipStream_t s) {
  const int per = walkers_per_wave(sa.W, sa.G);
  const int blocks = (sa.W + per - 1) / per;
  const size_t lds = (SYS == SYS_ISING ? 0 : sizeof(double) * 3 * (size_t)per * sa.npad) +
                     (size_t)per * kBinStats * sizeof(BC<uint64_t>);
  const auto go = [&](auto share) {
    constexpr bool SH = decltype(share)::value;
    if (ba.linear)
      hipLaunchKernelGGL((k_bin<SYS, KMAX, true, SH>), dim3(blocks), dim3(64), lds, s, ba, sa, moves, init, per);
    else
      hipLaunchKernelGGL((k_bin<SYS, KMAX, false, SH>), dim3(blocks), dim3(64), lds, s, ba, sa, moves, init, per);
  };
  if constexpr (SYS != SYS_ISING && KMAX > 1) {
    if (lanes_to_share(per, sa.G, KMAX)) {
      go(std::true_type{});
      return hipGetLastError();
    }
  }
  go(std::false_type{});
  return hipGetLastError();
}

template <int SYS>
static hipError_t launch_bin_s(int kmax, const BinArgs &ba, const SetArgs &sa, uint64_t moves, int init,
                               hipStream_t s) {
  switch (kmax) {
    case 1: return launch_bin_t<SYS, 1>(ba, sa, moves, init, s);
    case 2: return launch_bin_t<SYS, 2>(ba, sa, moves, init, s);
    case 4: return launch_bin_t<SYS, 4>(ba, sa, moves, init, s);
    case 8: return launch_bin_t<SYS, 8>(ba, sa, moves, init, s);
    case 16: return launch_bin_t<SYS, 16>(ba, sa, moves, init, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_binning(int sys, int kmax, const BinArgs &ba, const SetArgs &sa, uint64_t moves, int init,
                          hipStream_t s) {
  if (sys == SYS_ISING) return launch_bin_t<SYS_ISING, 1>(ba, sa, moves, init, s);
  if (sys == SYS_LJ) return launch_bin_s<SYS_LJ>(kmax, ba, sa, moves, init, s);
  if (sys == SYS_WCA) return launch_bin_s<SYS_WCA>(kmax, ba, sa, moves, init, s);
  return hipErrorInvalidValue;
}

}  // namespace sadmc
