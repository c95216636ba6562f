// Plain local search on stencil lattices with the species in LDS, one
// workgroup per lattice.
//
// Same search as hea_mc.hip (accelerate.cpp:601-694; the header there states
// the semantics and the FP64 bookkeeping), for the problems users bring: FCC
// and BCC supercells whose table is the translation stencil (hea_stencil.h).
// Nearly every round of a search accepts (93-99 % on the workloads), so a
// round's cost is the latency of one chain: decide the winner, draw the next
// proposals, walk their neighbours, screen them against the new tables.  The
// kernel is laid out around that chain:
//
//   * worker waves hold one proposal per lane, which computes its sites'
//     neighbours' ids from the sites' coordinates and gathers their species
//     from LDS; no neighbour row is loaded, and whether the two sites are
//     neighbours follows from their distance.  The species bytes hold the
//     histogram shift, so a BCC neighbour costs one three-operand add, one LDS
//     byte and one shift-add; FCC loads a cell's four sites at once (hea_walk.h).
//   * the lane then forms X over all shells from the folded tables
//     (screen_fold) in registers, so a round needs no pass over LDS to
//     combine the shells.
//   * every wave decides the round by itself from the waves' published
//     minima: when the window holds one proposal and its sign is certain
//     (exact_stage's rule), all waves know the winner without another
//     barrier.  The workers go on to draw and walk the next proposals, while
//     the service wave (the last one) forms the winner's exact gamma rows,
//     refreshes the changed table entries and the window: that chain ends
//     before the walk does.
//   * otherwise (first round, several candidates, an undecided sign, fitness
//     near the caller's threshold) the service wave runs exact_stage while
//     the workers wait.
//
// Barriers of a round: B1 minima published; B2 draw counts; B3 proposals
// written; B4 tables and window ready.
//
// What bounds it: LDS (40 to 51 % of a CU's cycles, a third of them bank
// conflicts) and vector issue (61 %), in a chain of dependent steps; of a round of
// 10000 to 13500 cycles the walk is a third, the screen a fifth, drawing and
// listing the proposals a quarter.  Launches on average of a session's searches,
// against k_local_mc: 512 lattices of 8192 sites, 256 proposals, 3.67 ms, 7.47; 256
// of 108000 sites, 512 proposals, 50.7 ms, 155.0; 64 of 256000 sites, two species a
// byte, 2.1 times as fast as the walk through HBM.
#pragma once
#include "hea_exact.h"
#include "hea_internal.h"
#include "hea_screen.h"
#include "hea_walk.h"

namespace {

constexpr int kWaves = 16;               // slots per wave in LDS
constexpr int kMaxSearchThreads = 768;  // 12 waves: at most 168 VGPRs each

// The arguments of the screen templates (hea_screen.h), in LDS: their shell
// varies over the lanes.
struct ShellArgs {
  int N, K, S, stride;
  double delta[HEA_MAX_S], weight[HEA_MAX_S];
  int Z[HEA_MAX_S], off[HEA_MAX_S];
  const int32_t* nbr;
  double thr;
};

struct SearchShared {
  double wm[kWaves];  // smallest X of each worker wave (inf beyond the workers)
  int wj[kWaves];     // its proposal (the first with that X)
  int wc[kWaves];     // proposals of the wave within 2 beta of its smallest X
  int2 wp[kWaves];    // the proposal's sites
  int wab[kWaves];    // and species a | b << 8
  int cnt[kWaves];    // valid draws of each wave
  unsigned long long vb[HEA_MAX_S];  // bits of the largest entry bound of a shell
  double beta;
  ShellArgs args;
  uint32_t next_pos;
  int ncl;
  // the exact stage's state (hea_exact.h)
  double pf, fest;
  unsigned long long res_key;
  int res_j, res_a, res_b, res_kind, pfm;
  unsigned long long bmax[HEA_MAX_S], ubmax[HEA_MAX_S];
  unsigned gmax;
};

// LDS carve-up of one workgroup (byte offsets; every region 16-byte aligned).
// Table rows of UV are padded so that the 16-byte reads of different rows
// start in different banks.
template <int KMAX>
struct SearchLayout {
  static constexpr int TAB = HEA_MAX_S * KMAX * KMAX;
  static constexpr int KP = KMAX == 8 ? 9 : (KMAX + 1) & ~1;
  using PT = typename Pack<KMAX>::T;
  static constexpr size_t up(size_t n) { return (n + 15) & ~(size_t)15; }
  // tables, state and species at fixed offsets, the proposals' arrays behind
  // the species
  static constexpr size_t T8 = up(sizeof(double) * TAB);
  static constexpr size_t UV = 0, G = UV + up(sizeof(double2) * HEA_MAX_S * KMAX * KP), E0 = G + T8,
                          R = E0 + T8, tgt = R + T8, C = tgt + T8, B = C + T8, conc = B + T8,
                          ex = conc + up(sizeof(double) * KMAX), xw = ex + sizeof(double) * 64,
                          sh = xw + sizeof(double) * 64 * (4 + KMAX),
                          sp = sh + up(sizeof(SearchShared));
  size_t WA, WB, WC, prop, xs, cl, total;
  __host__ __device__ SearchLayout(int task, size_t sp_bytes) {
    const size_t t = (size_t)task;
    WA = sp + up(sp_bytes);
    WB = WA + up(sizeof(PT) * HEA_MAX_S * t);
    WC = WB + up(sizeof(PT) * HEA_MAX_S * t);
    prop = WC + up(sizeof(uint32_t) * HEA_MAX_S * t);
    xs = prop + up(sizeof(int2) * t);
    cl = xs + up(sizeof(double) * t);
    total = cl + up(sizeof(int) * t);
  }
};

template <int KMAX, bool NIB>
struct SearchTab {
  using LY = SearchLayout<KMAX>;
  using PT = typename Pack<KMAX>::T;
  using SP = Species<NIB, Pack<KMAX>::W>;
  double *G, *E0, *R, *tgt;  // [S][KMAX][KMAX] as in hea_mc.hip
  double* C;                 // -delta_s / dd_ij
  double* B;                 // fold_bound of the entry
  double2* UV;               // [S][KMAX][KP] folded screen table
  double *conc, *ex, *xw, *xs;
  int2* prop;
  PT *WA, *WB;
  uint32_t* WC;
  int* cl;
  SearchShared* sh;
  SP sp;
  __device__ void carve(unsigned char* base, int task, int n) {
    const LY L(task, SP::bytes(n));
    G = reinterpret_cast<double*>(base + LY::G);
    E0 = reinterpret_cast<double*>(base + LY::E0);
    R = reinterpret_cast<double*>(base + LY::R);
    tgt = reinterpret_cast<double*>(base + LY::tgt);
    C = reinterpret_cast<double*>(base + LY::C);
    B = reinterpret_cast<double*>(base + LY::B);
    UV = reinterpret_cast<double2*>(base + LY::UV);
    conc = reinterpret_cast<double*>(base + LY::conc);
    ex = reinterpret_cast<double*>(base + LY::ex);
    xw = reinterpret_cast<double*>(base + LY::xw);
    xs = reinterpret_cast<double*>(base + L.xs);
    prop = reinterpret_cast<int2*>(base + L.prop);
    WA = reinterpret_cast<PT*>(base + L.WA);
    WB = reinterpret_cast<PT*>(base + L.WB);
    WC = reinterpret_cast<uint32_t*>(base + L.WC);
    cl = reinterpret_cast<int*>(base + L.cl);
    sh = reinterpret_cast<SearchShared*>(base + LY::sh);
    sp.p = base + LY::sp;
  }
  __device__ __forceinline__ int idx(int s, int i, int j) const { return (s * KMAX + i) * KMAX + j; }
  __device__ __forceinline__ int uvx(int s, int i, int j) const { return (s * KMAX + i) * LY::KP + j; }
};

// v, hidden from the compiler: what is computed from it stays where it is
// written instead of occupying registers over the whole search.
__device__ __forceinline__ int opaque(int v) {
  asm("" : "+v"(v));
  return v;
}

// Species histograms of one shell's neighbours of a proposal's two sites.
// All the bytes are in flight before the first is used.
template <int KMAX, int LT, int SHELL, bool NIB>
__device__ __forceinline__ void walk_shell(const SiteTerms* t, typename Pack<KMAX>::T& ma,
                                           typename Pack<KMAX>::T& mb) {
  constexpr int Z = HeaShells<LT>::Z[SHELL];
  uint32_t va[Z], vb[Z];
  load_shell<LT, SHELL>(t[0], va);
  load_shell<LT, SHELL>(t[1], vb);
  __builtin_amdgcn_sched_barrier(0);
  count_shell<KMAX, LT, SHELL, NIB>(t[0], va, ma);
  count_shell<KMAX, LT, SHELL, NIB>(t[1], vb, mb);
}

// The same by cell (both sites' loads are under way before the first count).
template <int KMAX, int LT, int NS, bool NIB>
__device__ __forceinline__ void walk_pair(const HeaCellSite& ca, const HeaCellSite& cb, int L,
                                          uint32_t sp, typename Pack<KMAX>::T* MA,
                                          typename Pack<KMAX>::T* MB) {
  uint32_t va[27], vb[27];
  const CellTerms ta = cell_terms<NIB>(ca, L, sp);
  load_cells<LT, NS, NIB>(ta, va);
  __builtin_amdgcn_sched_barrier(0);
  const CellTerms tb = cell_terms<NIB>(cb, L, sp);
  load_cells<LT, NS, NIB>(tb, vb);
  __builtin_amdgcn_sched_barrier(0);
  count_cells<KMAX, LT, NS, NIB>(ta, va, MA);
  count_cells<KMAX, LT, NS, NIB>(tb, vb, MB);
}

template <int KMAX, int LT, bool NIB>
__device__ __forceinline__ void walk_sites(const HeaCellSite& ca, const HeaCellSite& cb, int L,
                                           uint32_t sp, int S, typename Pack<KMAX>::T* MA,
                                           typename Pack<KMAX>::T* MB) {
#pragma unroll
  for (int s = 0; s < HEA_MAX_S; ++s) MA[s] = MB[s] = 0;
  if constexpr (LT == HEA_LT_FCC || LT == HEA_LT_FCC_REF) {
    if (S == 3)
      walk_pair<KMAX, LT, 3, NIB>(ca, cb, L, sp, MA, MB);
    else if (S == 2)
      walk_pair<KMAX, LT, 2, NIB>(ca, cb, L, sp, MA, MB);
    else
      walk_pair<KMAX, LT, 1, NIB>(ca, cb, L, sp, MA, MB);
  } else {
    const SiteTerms t[2] = {site_terms<LT, NIB>(ca, L, sp), site_terms<LT, NIB>(cb, L, sp)};
    walk_shell<KMAX, LT, 0, NIB>(t, MA[0], MB[0]);
    if (S > 1) walk_shell<KMAX, LT, 1, NIB>(t, MA[1], MB[1]);
    if (S > 2) walk_shell<KMAX, LT, 2, NIB>(t, MA[2], MB[2]);
  }
}

template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_umin_step(uint32_t v) {
  return min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xf, false));
}
// Smallest v over the wave (WAVE) or over each row of 16 lanes; the rows hold
// the same values then.
template <bool WAVE>
__device__ __forceinline__ uint32_t umin_all(uint32_t v) {
  v = dpp_umin_step<0x121, 0xf>(v);
  v = dpp_umin_step<0x122, 0xf>(v);
  v = dpp_umin_step<0x124, 0xf>(v);
  v = dpp_umin_step<0x128, 0xf>(v);
  if constexpr (WAVE) {
    v = dpp_umin_step<0x142, 0xa>(v);
    v = dpp_umin_step<0x143, 0xc>(v);
  }
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Lane of the smallest v (the first of equal ones).  The high words of keys
// that order like the doubles decide alone unless two lanes share the
// smallest: one 32-bit minimum per step instead of a 64-bit one.
template <bool WAVE>
__device__ __forceinline__ int argmin_lane(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const uint32_t flip = (uint32_t)((int32_t)(b >> 32) >> 31);  // all ones below zero
  const uint32_t hi = (uint32_t)(b >> 32) ^ (flip | 0x80000000u);
  const uint32_t m = umin_all<WAVE>(hi);
  unsigned long long at = __ballot(hi == m);
  if (WAVE ? (at & (at - 1)) != 0 : ((uint32_t)at & 0xffffu & ((uint32_t)at - 1u)) != 0) {
    const uint32_t lo = hi == m ? (uint32_t)b ^ flip : ~0u;
    const uint32_t ml = umin_all<WAVE>(lo);
    at = __ballot(hi == m && lo == ml);
  }
  return (int)__builtin_ctzll(at);
}
__device__ __forceinline__ double readlane_f64(double v, int src) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

template <int CTRL>
__device__ __forceinline__ int dpp_add_step(int v) {
  return v + __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false);
}
// Sum of v over each row of 16 lanes, in every lane of the row.
__device__ __forceinline__ int row_sum(int v) {
  v = dpp_add_step<0x121>(v);
  v = dpp_add_step<0x122>(v);
  v = dpp_add_step<0x124>(v);
  return __builtin_amdgcn_readfirstlane(dpp_add_step<0x128>(v));
}

// w mod n for w < 2^31, magic = floor(2^32 / n): the quotient is short by at
// most one (w / 2^32 + 1 < 2).
__device__ __forceinline__ uint32_t stream_mod(uint32_t w, uint32_t n, uint32_t magic) {
  const uint32_t r = w - __umulhi(w, magic) * n;
  return min(r, r - n);
}

// Sum over the shells of twice the largest entry bound (fold_bound), by all
// lanes of one wave.
template <class Tab>
__device__ __forceinline__ double window(const Tab& T, int S, int K, int lane) {
  if (lane < HEA_MAX_S) T.sh->vb[lane] = 0ull;
  wave_sync();
  for (int e = lane; e < S * K * K; e += 64) {
    const int s = e / (K * K), i = (e / K) % K, j = e % K;
    if (i <= j)
      atomicMax(&T.sh->vb[s], (unsigned long long)__double_as_longlong(T.B[T.idx(s, i, j)]));
  }
  wave_sync();
  double b = 0.0;
#pragma unroll
  for (int s = 0; s < HEA_MAX_S; ++s)
    b += __longlong_as_double((long long)T.sh->vb[s]);  // absent shells hold 0
  return 2.0 * 1.01 * b;
}

// What the service wave keeps of a round's winner: the walk record of the
// lane's shell and the two sites.
template <class PT>
struct Winner {
  PT ma, mb;
  int c12, s1, s2;
};

// New gamma entry (a, x) (h = 0) or (b, x) (h = 1) of shell s for the
// winner's swap, as exact_entries gives it; by all lanes of one wave (lanes
// with s >= S idle).  Entries whose step is 0 are replayed addition by
// addition; for the interleaved entry (a, b) the rows' order of additions
// becomes one bit mask per sign and list (a row has at most 64 columns; rows()
// gives lane c column c of the two sites' rows).
template <int KMAX, class Tab, class Rows>
__device__ __forceinline__ double winner_entry(const ShellArgs& A, const Tab& T, int s,
                                               int x, int h, int S, int stride, int a, int b,
                                               const Winner<typename Pack<KMAX>::T>& w, int lane,
                                               const Rows& rows) {
  using PK = Pack<KMAX>;
  double g = 0.0, r = 1.0;
  int up = 0, dn = 0, net = 0;  // additions of +delta and -delta, and their sum
  const bool on = s < S, ab = on && x == (h ? a : b);
  if (on) {
    const int maA = PK::fld(w.ma, a), maB = PK::fld(w.ma, b);
    const int mbA = PK::fld(w.mb, a), mbB = PK::fld(w.mb, b);
    const int e = T.idx(s, h ? b : a, x);
    g = T.G[e];
    r = T.R[e];
    if (ab) {
      up = maA + mbB + 2 * w.c12;
      dn = maB + mbA;
    } else {
      const bool diag = x == (h ? b : a);
      const int max_ = PK::fld(w.ma, x), mbx = PK::fld(w.mb, x);
      dn = h ? mbx : max_;
      up = h ? max_ : mbx;
      if (diag) {
        dn = 2 * (h ? mbB : maA);
        up = 2 * ((h ? maB : mbA) - w.c12);
      }
    }
    net = up - dn;
  }
  double v = fma((double)net, r, g);
  bool slow = on && r == 0.0;
  const double delta = on ? A.delta[s] : 0.0;
  if (__any(slow)) {
    // this swap's own additions reach less far than any swap's
    const double rs = on ? safe_step_within(g, delta, max(up, dn)) : 0.0;
    if (slow && rs != 0.0) {
      v = fma((double)net, rs, g);
      slow = false;
    }
  }
  if (__any(slow)) {
    const bool plain = slow && !ab;
    // (b, x) adds first, the others subtract first
    const double d1 = h ? delta : -delta;
    const int k1 = plain ? (h ? up : dn) : 0;
    const int k2 = plain ? (h ? dn : up) : 0;
    double q = g;
    for (int i = 0; __any(i < k1); i += 4) {
      q = q + (i < k1 ? d1 : 0.0);
      q = q + (i + 1 < k1 ? d1 : 0.0);
      q = q + (i + 2 < k1 ? d1 : 0.0);
      q = q + (i + 3 < k1 ? d1 : 0.0);
    }
    for (int i = 0; __any(i < k2); i += 4) {
      q = q - (i < k2 ? d1 : 0.0);
      q = q - (i + 1 < k2 ? d1 : 0.0);
      q = q - (i + 2 < k2 ? d1 : 0.0);
      q = q - (i + 3 < k2 ? d1 : 0.0);
    }
    if (__any(slow && ab)) {  // replay_ab's additions in row order
      const auto sp = T.sp;
      const int2 col = rows();
      const bool in1 = lane < stride && col.x >= 0, in2 = lane < stride && col.y >= 0;
      const int o1 = in1 ? sp[col.x] : -1, o2 = in2 ? sp[col.y] : -1;
      // species before the swap, whatever sp holds at the two sites
      const int n1 = col.x == w.s2 ? b : o1, n2 = col.y == w.s1 ? a : o2;
      const unsigned long long m1 = __ballot(in1 && n1 == b), m2 = __ballot(in2 && n2 == a);
      const unsigned long long p1 = __ballot(in1 && (col.x == w.s2 || n1 == a));
      const unsigned long long p2 = __ballot(in2 && (col.y == w.s1 || n2 == b));
      const int o = on ? A.off[s] : 0;
      const uint32_t zm = on ? (1u << A.Z[s]) - 1u : 0u;
      double y = g;
#pragma unroll
      for (int list = 0; list < 2; ++list) {
        const uint32_t m = (uint32_t)((list ? m2 : m1) >> o) & zm;
        const uint32_t p = (uint32_t)((list ? p2 : p1) >> o) & zm;
        uint32_t left = (slow && ab) ? m | p : 0u;
        while (__any(left != 0u)) {
          const uint32_t low = left & (0u - left);
          left &= left - 1u;
          y = y - ((m & low) ? delta : 0.0);
          y = y + ((p & low) ? delta : 0.0);
        }
      }
      q = ab ? y : q;
    }
    if (slow) v = q;
  }
  return v;
}

// The exact stage (hea_exact.h) over the candidates T.cl, by the service wave.
// A call of its own: few rounds need it, and inlined its masks and constants
// take scalar registers from every round.
template <int KMAX, bool EXACT, bool NIB>
__device__ __attribute__((noinline)) void undecided(int task, int n, double xmin, double beta) {
  extern __shared__ __align__(16) unsigned char smem[];
  SearchTab<KMAX, NIB> T;
  T.carve(smem, task, n);
  const int lane = threadIdx.x & 63;
  exact_stage<KMAX, EXACT>(T.sh->args, T, T.sp, lane, task,
                           T.sh->ncl, xmin, beta, false);
  if (lane == 0) T.sh->ncl = 0;
}

// A round's decision, the same in every wave (values uniform over the wave).
struct Decision {
  int kind;  // exact_stage's kinds: 0 reject, 1 accept by the exact stage, 2 by the window;
             // -1: undecided
  int j, a, b, s1, s2;  // the winner and its swap
  double xmin;
};

// The rule of exact_stage from the waves' published minima: with prev_fit the
// fitness of the current tables, one candidate of certain sign decides.
__device__ __forceinline__ Decision decide(const SearchShared* sh, int nw, double beta,
                                           double thr, int lane) {
  const int w = lane & (kWaves - 1);
  const double wm = sh->wm[w];
  const int wj = sh->wj[w], wc = sh->wc[w], wab = sh->wab[w];
  const int2 wp = sh->wp[w];
  const double fest = sh->fest;
  const int pfm = sh->pfm;
  const int src = argmin_lane<false>(wm);
  Decision d;
  d.xmin = readlane_f64(wm, src);
  const double mg = 2.0 * beta;
  const uint32_t in = (uint32_t)__ballot(w < nw && !(wm > d.xmin + mg)) & 0xffffu;
  const int n_in = __builtin_amdgcn_readlane(wc, src);
  d.j = __builtin_amdgcn_readlane(wj, src);
  const int ab = __builtin_amdgcn_readlane(wab, src);
  d.a = ab & 255;
  d.b = ab >> 8;
  d.s1 = __builtin_amdgcn_readlane(wp.x, src);
  d.s2 = __builtin_amdgcn_readlane(wp.y, src);
  const bool near = thr > 0.0 && !(fest + d.xmin > thr * thr * 1.01);
  const bool one = __popc(in) == 1 && n_in == 1;
  const int sure = d.xmin - mg > 0.0 ? 0 : (one && d.xmin + mg < 0.0) ? 2 : -1;
  d.kind = __builtin_amdgcn_readfirstlane(pfm != 0 && !near ? sure : -1);
  return d;
}

// The exact stage's decision, for the rounds that decide() leaves open.
__device__ __forceinline__ void read_exact(const SearchShared* sh, const int2* prop, Decision& d) {
  d.kind = __builtin_amdgcn_readfirstlane(sh->res_kind);
  if (d.kind == 0) return;
  d.j = __builtin_amdgcn_readfirstlane(sh->res_j);
  d.a = __builtin_amdgcn_readfirstlane(sh->res_a);
  d.b = __builtin_amdgcn_readfirstlane(sh->res_b);
  const int2 v = prop[d.j];
  d.s1 = __builtin_amdgcn_readfirstlane(v.x);
  d.s2 = __builtin_amdgcn_readfirstlane(v.y);
}

// Rounds of the service wave.  Its barriers pair with worker_rounds'.
template <int KMAX, bool EXACT, bool NIB>
__device__ __forceinline__ void service_rounds(const HeaMcArgs& A, const SearchTab<KMAX, NIB>& T,
                                               int nw, int lane) {
  using PK = Pack<KMAX>;
  SearchShared* sh = T.sh;
  const ShellArgs& SA = sh->args;
  const int K = EXACT ? KMAX : A.K, S = A.S, task = A.task, stride = A.stride;
  const int depth = A.depth, n = A.N;
  const double thr = A.thr;
  const int32_t* nbr = A.nbr;
  // lane (s, h, x) takes entry (a, x) (h = 0) or (b, x) of an accepted swap
  const int sv_s = lane / (2 * K), sv_k = lane - sv_s * 2 * K;
  const int sv_h = sv_k >= K ? 1 : 0, sv_x = sv_k - sv_h * K;
  Winner<typename PK::T> win{};
  int2 col = make_int2(-1, -1);
  Decision d{};
  bool by_window = false;
  double beta = 0.0;
  __builtin_amdgcn_s_setprio(3);
  for (int acc = 0, round = 0; acc < depth; ++round) {
    int found = 0;
    do {
      __syncthreads();  // B2
      found += row_sum(sh->cnt[lane & (kWaves - 1)]);
      if (by_window && lane == 0) {  // every wave has read both (before B2)
        sh->pfm = 2;
        sh->fest = sh->fest + d.xmin;
      }
      by_window = false;
      __syncthreads();  // B3
    } while (found < task);
    if (d.kind != 0) {
      // the winner's exact gamma rows (the exact stage wrote its own), then
      // the tables of the entries that changed
      const int r = sv_h ? d.b : d.a;
      double g = 0.0;
      if (d.kind == 2) {
        g = winner_entry<KMAX>(SA, T, sv_s, sv_x, sv_h, S, stride, d.a, d.b, win, lane,
                               [&]() { return col; });
        wave_sync();  // every lane has read its entries
        if (sv_s < S) {
          T.G[T.idx(sv_s, r, sv_x)] = g;
          T.G[T.idx(sv_s, sv_x, r)] = g;
        }
      } else if (sv_s < S) {
        g = T.G[T.idx(sv_s, r, sv_x)];
      }
      if (sv_s < S) refresh_fold(SA, T, sv_s, r, sv_x, g);
      wave_sync();
    }
    if (d.kind != 0 || round == 0) {
      beta = window(T, S, K, lane);
      if (lane == 0) sh->beta = beta;
    }
    __syncthreads();  // B4
    __syncthreads();  // B1
    d = decide(sh, nw, beta, thr, lane);
    by_window = d.kind == 2;
    if (__builtin_expect(d.kind < 0, 0)) {
      __syncthreads();
      undecided<KMAX, EXACT, NIB>(task, n, d.xmin, beta);
      __syncthreads();
      read_exact(sh, T.prop, d);
      if (d.kind == 2) d.kind = 1;  // the exact stage wrote the rows in any case
    }
    if (d.kind == 0) {
      ++acc;
      continue;
    }
    acc = 0;
    // what the new rows need of the winner, before the next walk replaces its
    // record: the record, and its sites' rows for a replay
    if (sv_s < S) {
      const int w = sv_s * task + d.j;
      win.ma = T.WA[w];
      win.mb = T.WB[w];
      win.c12 = walk_unpack(T.WC[w]).c12;
    }
    win.s1 = d.s1;
    win.s2 = d.s2;
    if (lane < stride)
      col = make_int2(nbr[(size_t)d.s1 * stride + lane], nbr[(size_t)d.s2 * stride + lane]);
  }
}

// What the search reports (uniform).
struct SearchCounts {
  long long rounds, accepts;
  uint32_t pos;
};

// Rounds of a worker wave.
template <int KMAX, bool EXACT, int LT, bool NIB>
__device__ __forceinline__ SearchCounts worker_rounds(const HeaMcArgs& A,
                                                      const SearchTab<KMAX, NIB>& T, int l, int nw,
                                                      int wave, int tid) {
  using PK = Pack<KMAX>;
  using PT = typename PK::T;
  SearchShared* sh = T.sh;
  using SP = Species<NIB, PK::W>;
  const SP sp = T.sp;
  const int lane = tid & 63;
  const uint32_t N = (uint32_t)A.N, nmagic = A.n_magic;
  const int S = A.S, task = A.task, depth = A.depth, edge = A.edge;
  const double thr = A.thr;
  const float inv_edge = A.inv_edge;
  const auto div = [inv_edge](uint32_t n) { return hea_cell_div_small(n, inv_edge); };
  const int dl = A.dl;  // draw lanes, two consecutive draws each
  const bool drawer = __builtin_amdgcn_readfirstlane(wave * 64 < dl ? 1 : 0) != 0;
  // lanes beyond the round's proposals repeat the last one and are masked
  // where results are published
  const bool cand = tid < task;
  const int j_me = min(tid, task - 1);
  const uint32_t iter = *A.iter_ptr, seed_lo = (uint32_t)A.seed,
                 seed_hi = (uint32_t)(A.seed >> 32), phase = A.phase;
  SearchCounts sc{0, 0, 0};
  // this lane's two draws at stream positions 2 (pos >> 1) + 2 tid, + 1, and
  // their species codes a | b << 8
  uint32_t n1[2] = {0, 0}, n2[2] = {0, 0};
  int ab[2] = {0, 0};
  auto draw = [&](uint32_t blk) {  // one Philox block holds two draws
    // (opaque keys: the round keys are scalar sums, not 20 registers kept
    // over the whole search)
    uint32_t k0 = seed_lo, k1 = seed_hi;
    asm("" : "+s"(k0), "+s"(k1));
    const hea_u32x4 o = hea_stream_block(((uint64_t)k1 << 32) | k0, iter, phase, (uint32_t)l, blk);
    n1[0] = stream_mod(o.x, N, nmagic);
    n2[0] = stream_mod(o.y, N, nmagic);
    n1[1] = stream_mod(o.z, N, nmagic);
    n2[1] = stream_mod(o.w, N, nmagic);
  };
  auto look = [&]() {
#pragma unroll
    for (int h = 0; h < 2; ++h) ab[h] = sp.code(n1[h]) | (sp.code(n2[h]) << 8);
  };
  uint32_t pos = 0;
  if (drawer) {
    draw((uint32_t)tid);
    look();
  }

  for (int acc = 0; acc < depth;) {
    // ---- draw `task` valid proposals in stream order (accelerate.cpp:649-655)
    int found = 0;
    for (;;) {
      const uint32_t blk0 = pos >> 1;
      const uint32_t p0 = 2u * (blk0 + (uint32_t)tid);
      const bool v0 = p0 >= pos && (ab[0] & 255) != (ab[0] >> 8);  // ab = 0 beyond the draw lanes
      const bool v1 = (ab[1] & 255) != (ab[1] >> 8);
      const unsigned long long b0 = __ballot(v0), b1 = __ballot(v1);
      if (lane == 0) sh->cnt[wave] = __popcll(b0) + __popcll(b1);
      __syncthreads();  // B2
      // every row of 16 lanes sums the waves' counts (absent waves hold 0)
      const int w = lane & (kWaves - 1), cw = sh->cnt[w];
      const int off = row_sum(w < wave ? cw : 0), tot = row_sum(cw);
      const unsigned long long below = (1ull << lane) - 1ull;
      const int r0 = found + off + __popcll(b0 & below) + __popcll(b1 & below);
      const int r1 = r0 + (v0 ? 1 : 0);
      if (v0 && r0 < task) T.prop[r0] = make_int2((int)n1[0], (int)n2[0]);
      if (v1 && r1 < task) T.prop[r1] = make_int2((int)n1[1], (int)n2[1]);
      if ((v0 && r0 == task - 1) || (v1 && r1 == task - 1))
        sh->next_pos = v0 && r0 == task - 1 ? p0 + 1 : p0 + 2;
      found += tot;
      __syncthreads();  // B3
      if (__builtin_expect(found >= task, 1)) break;
      pos = 2u * (blk0 + (uint32_t)dl);  // rare: the pass held too few valid draws
      if (drawer) {
        draw((pos >> 1) + (uint32_t)tid);
        look();
      }
    }
    pos = __builtin_amdgcn_readfirstlane(sh->next_pos);

    // ---- walk the proposals' neighbours, draw the next round's pairs
    const int2 pr = T.prop[j_me];
    const int sa = sp.code((uint32_t)pr.x), sb = sp.code((uint32_t)pr.y);
    PT MA[HEA_MAX_S], MB[HEA_MAX_S];
    int c12[HEA_MAX_S], d2;
    {
      // (opaque: what follows from L is a few scalar instructions, not
      // registers kept over the search)
      int L = edge;
      asm("" : "+s"(L));
      const uint32_t spa = lds_addr(sp.p);
      const HeaCellSite ca = hea_cell_site<LT>(pr.x, L, div);
      const HeaCellSite cb = hea_cell_site<LT>(pr.y, L, div);
      walk_sites<KMAX, LT, NIB>(ca, cb, L, spa, S, MA, MB);
      d2 = hea_cell_dist2(ca, cb, L);
    }
    const int a = SP::species_of(sa), b = SP::species_of(sb);
#pragma unroll
    for (int s = 0; s < HEA_MAX_S; ++s) {
      c12[s] = d2 == HeaShells<LT>::D2[s] ? 1 : 0;
      if (s < S) {  // (lanes that repeat a proposal write the same values)
        const int w = s * task + j_me;
        T.WA[w] = MA[s];
        T.WB[w] = MB[s];
        T.WC[w] = walk_pack(0, c12[s], c12[s], 0, a, b);
      }
    }
    if (drawer) {
      draw((pos >> 1) + (uint32_t)tid);
      look();
    }
    __syncthreads();  // B4

    // ---- screen: X of every proposal, each wave's minimum
    const double beta = sh->beta;
    const double X = screen_fold<KMAX>(T, S, a, b, MA, MB, c12);
    {
      const double xv = cand ? X : __builtin_inf();
      const int src = argmin_lane<true>(xv);
      const double m = readlane_f64(xv, src);
      const unsigned long long in = __ballot(cand && !(xv > m + 2.0 * beta));
      if (lane == src) {
        sh->wm[wave] = m;
        sh->wj[wave] = j_me;
        sh->wc[wave] = __popcll(in);
        sh->wp[wave] = pr;
        sh->wab[wave] = a | (b << 8);
      }
    }
    __syncthreads();  // B1

    Decision d = decide(sh, nw, beta, thr, lane);
    ++sc.rounds;
    if (__builtin_expect(d.kind < 0, 0)) {
      // the candidates of the window to the exact stage
      const bool f = cand && !(X > d.xmin + 2.0 * beta);
      const unsigned long long bal = __ballot(f);
      if (bal) {
        int base = 0;
        if (lane == 0) base = atomicAdd(&sh->ncl, __popcll(bal));
        base = __builtin_amdgcn_readfirstlane(base);
        if (f) {
          T.cl[base + __popcll(bal & ((1ull << lane) - 1ull))] = j_me;
          T.xs[j_me] = X;
        }
      }
      __syncthreads();
      __syncthreads();
      read_exact(sh, T.prop, d);
      if (d.kind == 1 && tid == 0 && A.first_hit &&
          __longlong_as_double((long long)sh->res_key) <= thr)
        atomicMin(A.first_hit, (unsigned long long)wall_clock64());
    }
    if (d.kind == 0) {
      ++acc;
      continue;
    }
    acc = 0;
    ++sc.accepts;
    const int fa = SP::code_of(d.a), fb = SP::code_of(d.b);
    if (tid == 0) {
      sp.set(d.s1, d.b);
      sp.set(d.s2, d.a);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // the next draws' species after the swap
      const int o1 = ab[h] & 255, o2 = ab[h] >> 8;
      const int t1 = (int)n1[h] == d.s1 ? fb : (int)n1[h] == d.s2 ? fa : o1;
      const int t2 = (int)n2[h] == d.s1 ? fb : (int)n2[h] == d.s2 ? fa : o2;
      ab[h] = t1 | (t2 << 8);
    }
  }
  sc.pos = pos;
  return sc;
}

// Local search of lattice l of the population described by A.
template <int KMAX, bool EXACT, int LT, bool NIB>
__device__ __forceinline__ void search_lattice(const HeaMcArgs& A, int l, unsigned char* smem) {
  using PK = Pack<KMAX>;
  const HeaConst& P = *A.pc;
  const int nthr = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nw = (nthr >> 6) - 1;  // worker waves
  const int N = A.N, K = EXACT ? KMAX : A.K, S = A.S;

  using SP = Species<NIB, PK::W>;
  SearchTab<KMAX, NIB> T;
  T.carve(smem, A.task, N);
  SearchShared* sh = T.sh;
  uint8_t* lat_g = A.lattices + (size_t)l * N;
  uint8_t* sp = T.sp.p;
  if constexpr (NIB) {  // (an even number of sites: two or four a cell)
    for (int i = tid; i < N / 2; i += nthr) sp[i] = (uint8_t)(lat_g[2 * i] | (lat_g[2 * i + 1] << 4));
  } else if ((N & 3) == 0) {  // four bytes at a time: W x species stays below 64
    const uint32_t* g4 = reinterpret_cast<const uint32_t*>(lat_g);
    uint32_t* s4 = reinterpret_cast<uint32_t*>(sp);
    for (int i = tid; i < (N >> 2); i += nthr) s4[i] = g4[i] * (uint32_t)PK::W;
  } else {
    for (int i = tid; i < N; i += nthr) sp[i] = (uint8_t)(lat_g[i] * PK::W);
  }
  // prev_gamma = R_s(pair counts) (accelerate.cpp:636-640) and constants;
  // absent species and padding columns hold zeros
  for (int e = tid; e < HEA_MAX_S * KMAX * SearchLayout<KMAX>::KP; e += nthr)
    T.UV[e] = make_double2(0.0, 0.0);
  if (!EXACT)
    for (int e = tid; e < SearchLayout<KMAX>::TAB; e += nthr) {
      T.G[e] = T.E0[e] = T.R[e] = T.tgt[e] = T.C[e] = T.B[e] = 0.0;
    }
  if (tid < HEA_MAX_S) {
    sh->args.delta[tid] = tid < S ? P.delta[tid] : 0.0;
    sh->args.weight[tid] = tid < S ? P.weight[tid] : 0.0;
    sh->args.Z[tid] = P.Z[tid];
    sh->args.off[tid] = P.off[tid];
  }
  if (tid < K) T.conc[tid] = P.conc[tid];
  if (tid < kWaves) {
    sh->wm[tid] = __builtin_inf();
    sh->cnt[tid] = 0;
  }
  if (tid == 0) {
    const double f0 = A.fitness[l];
    sh->pf = f0;
    sh->pfm = 0;
    sh->fest = f0 * f0;
    sh->ncl = 0;
    sh->args.N = N;
    sh->args.K = K;
    sh->args.S = S;
    sh->args.stride = A.stride;
    sh->args.nbr = A.nbr;
    sh->args.thr = A.thr;
  }
  __syncthreads();
  const ShellArgs& SA = sh->args;
  const int32_t* cnt_g = A.counts + (size_t)l * S * K * K;
  for (int e = tid; e < S * K * K; e += nthr) {
    const int s = e / (K * K), i = (e / K) % K, j = e % K;
    const double c = -SA.delta[s] / (T.conc[i] * T.conc[j]);
    T.G[T.idx(s, i, j)] = hea_r_of_count(P, s, cnt_g[e]);
    T.tgt[T.idx(s, i, j)] = P.target[s][i][j];
    T.C[T.idx(s, i, j)] = c;
    T.UV[T.uvx(s, i, j)].y = 2.0 * SA.weight[s] * c * c;
  }
  __syncthreads();
  for (int e = tid; e < S * K * K; e += nthr) {
    const int s = e / (K * K), i = (e / K) % K, j = e % K;
    if (i <= j) refresh_fold(SA, T, s, i, j, T.G[T.idx(s, i, j)]);
  }

  __syncthreads();

  SearchCounts sc{0, 0, 0};
  if (wave == nw)
    service_rounds<KMAX, EXACT, NIB>(A, T, nw, lane);
  else
    sc = worker_rounds<KMAX, EXACT, LT, NIB>(A, T, l, nw, wave, tid);

  if (tid == 0) {
    double f = sh->pf;
    if (sh->pfm == 2) {  // F of the final gamma (accelerate.cpp:557-569)
      double err = 0.0;
      for (int t = 0; t < S; ++t) {
        double es = 0.0;
        for (int i = 0; i < K * K; ++i) es = es + T.E0[T.idx(t, i / K, i % K)];
        err = err + SA.weight[t] * es;
      }
      f = sqrt(err);
    }
    A.fitness[l] = f;
    int64_t* st = A.stats + (size_t)l * 4;
    st[0] += sc.rounds;
    st[1] += sc.accepts;
    st[2] += sc.rounds * A.task;
    st[3] += (long long)sc.pos;
  }
  if constexpr (NIB) {
    for (int i = tid; i < N / 2; i += nthr) {
      lat_g[2 * i] = sp[i] & 15;
      lat_g[2 * i + 1] = sp[i] >> 4;
    }
  } else if ((N & 3) == 0) {
    const uint32_t* s4 = reinterpret_cast<const uint32_t*>(sp);
    uint32_t* g4 = reinterpret_cast<uint32_t*>(lat_g);
    for (int i = tid; i < (N >> 2); i += nthr) {
      const uint32_t v = s4[i];
      uint32_t o = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        o |= (uint32_t)SP::species_of((int)((v >> (8 * k)) & 255u)) << (8 * k);
      g4[i] = o;
    }
  } else {
    for (int i = tid; i < N; i += nthr) lat_g[i] = (uint8_t)SP::species_of(sp[i]);
  }
}

template <int KMAX, bool EXACT, int LT, bool NIB>
__global__ __launch_bounds__(kMaxSearchThreads, 4) void k_search(HeaMcArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  search_lattice<KMAX, EXACT, LT, NIB>(A, blockIdx.x, smem);
}

}  // namespace

template <int LT, bool NIB>
inline const void* search_fn(int K) {
  switch (K) {
    case 2: return reinterpret_cast<const void*>(k_search<2, true, LT, NIB>);
    case 3: return reinterpret_cast<const void*>(k_search<3, true, LT, NIB>);
    case 4: return reinterpret_cast<const void*>(k_search<4, true, LT, NIB>);
    case 5: return reinterpret_cast<const void*>(k_search<5, true, LT, NIB>);
    case 6: return reinterpret_cast<const void*>(k_search<6, true, LT, NIB>);
    case 7: return reinterpret_cast<const void*>(k_search<8, false, LT, NIB>);
    case 8: return reinterpret_cast<const void*>(k_search<8, true, LT, NIB>);
    default: return nullptr;
  }
}

template <bool NIB>
inline const void* search_fn(int lt, int K) {
  switch (lt) {
    case HEA_LT_FCC: return search_fn<HEA_LT_FCC, NIB>(K);
    case HEA_LT_FCC_REF: return search_fn<HEA_LT_FCC_REF, NIB>(K);
    case HEA_LT_BCC: return search_fn<HEA_LT_BCC, NIB>(K);
    default: return nullptr;
  }
}
