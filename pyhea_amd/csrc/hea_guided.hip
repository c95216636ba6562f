// Guided local search on stencil lattices with the species in LDS, one
// workgroup per lattice.
//
// Same search as the guided mode of hea_mc.hip (the header there and
// hea_session_guide in the public header state the semantics): every slot of
// a round takes the Gumbel-max of the predicted gains of its candidate pairs,
// the round's best proposal is accepted by the exact rule, then up to
// accepts - 1 more come from a shortlist, screened again after every accept.
// Accepted swaps are the same to the bit.
//
// A round spends most of its time in the accepts, one after the other in one
// wave, and the rest in scoring 12 candidates per slot.  So:
//
//   * slot j belongs to lane j of the worker waves.  The lane draws its
//     candidates, scores them, keeps the best in registers and screens it: no
//     exchange of candidates or proposals through LDS.
//   * the service wave makes the accepts with the tables of k_search
//     (winner_entry, refresh_fold, screen_fold): the neighbours whose records
//     change and the adjacency come from coordinates, so no step waits for
//     neighbour rows (only a replay reads them).
//   * a helper wave updates the records and maps of the swap's neighbours (84 on
//     FCC) while the service wave forms the rows and tables: 256 lattices of
//     108000 sites 62.3 -> 56.7 ms, 4000 sites 7.80 -> 7.21 ms.  (That it also
//     screens a shell of the shortlist gained nothing.)
//   * meanwhile the workers draw the next round's candidates (they depend on
//     the stream alone) and fetch their records.  A candidate's records are
//     read one lane at a time, one line per request, and that would bound the
//     scoring.  A block map marks the blocks whose records the accepts change;
//     the lanes that hold such a block read it again.
//   * the gains of a species pair are read from a table of differences built
//     once a round, and record fields sit at compile-time positions.
//
// Records of small lattices stay in LDS (RL), the others' in HBM.
//
// What bounds it: the accepts, half of a round's 65000 cycles at 108000 sites (one
// wave's latency; 5000 each), then the candidates' records (a third).  256 lattices
// of 108000 sites, 512 slots, 12 candidates, up to 8 accepts: 57.9 ms a launch, 148.3
// with k_local_mc; 128 of 4000 sites, 256 slots, a session of two iterations: 12.7
// ms, 36.5.
//
// Barriers of a round: BD difference table ready; B1 minima published; BS
// shortlist ready (accepts only); BA accepts done.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "hea_search.h"

namespace {

constexpr int kPre = 12;           // candidates a lane draws ahead
constexpr int kGroup = 3;          // candidates scored together
constexpr int kCmapWords = 1024;   // conflict map: 32768 hashed bits
__device__ __forceinline__ uint32_t cmap_bit(int i) { return ((uint32_t)i * 0x9e3779b1u) >> 17; }

// Record fields of a shell set (HeaHistLayout of three shells).
template <int LT>
struct RecBits {
  static constexpr int bits(int z) { return z < 8 ? 3 : z < 16 ? 4 : 5; }
  static constexpr int w(int s) { return bits(HeaShells<LT>::Z[s]); }
  static constexpr int o(int s) { return s == 0 ? 0 : s == 1 ? w(0) : w(0) + w(1); }
  static constexpr int W = w(0) + w(1) + w(2);
};
static_assert(RecBits<HEA_LT_FCC>::W == 12 && RecBits<HEA_LT_BCC>::W == 11, "record layout");

template <int P, int W>
__device__ __forceinline__ uint32_t rec_field(uint2 r) {
  if constexpr (P >= 32)
    return __builtin_amdgcn_ubfe(r.y, P - 32, W);
  else if constexpr (P + W <= 32)
    return __builtin_amdgcn_ubfe(r.x, P, W);
  else
    return __builtin_amdgcn_alignbit(r.y, r.x, P) & ((1u << W) - 1u);
}

// Calls f(integral constant) for 0 .. N - 1.
template <int N, class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// Species histogram of shell S in the walk's packing from a record.
template <int KMAX, int LT, int S>
__device__ __forceinline__ uint32_t rec_shell(uint2 r) {
  using RB = RecBits<LT>;
  uint32_t m = 0, sum = 0;
  static_for<KMAX - 1>([&](auto x) {
    const uint32_t f = rec_field<x * RB::W + RB::o(S), RB::w(S)>(r);
    m |= f << (Pack<KMAX>::W * x);
    sum += f;
  });
  return m | ((uint32_t)HeaShells<LT>::Z[S] - sum) << (Pack<KMAX>::W * (KMAX - 1));
}

template <int KMAX>
struct GuidedLayout {
  using B = SearchLayout<KMAX>;
  using PT = uint32_t;
  static constexpr int TAB = B::TAB;
  static constexpr size_t SC = B::sp, H = SC + sizeof(double2) * ((TAB + 1) & ~1),
                          HZ = H + B::up(sizeof(float) * TAB),
                          DH = HZ + B::up(sizeof(float) * TAB),
                          cmap = DH + sizeof(float) * KMAX * KMAX * HEA_MAX_S * 8,
                          vec = cmap + sizeof(uint32_t) * kCmapWords,
                          sl = vec + sizeof(int) * 64, sp = sl + sizeof(int) * 64;
  size_t bmap, rec, WA, WB, WC, prop, xs, cl, total;
  int bwords;
  __host__ __device__ GuidedLayout(int task, int n, int blk, bool rl) {
    const size_t t = (size_t)task;
    bwords = (((n >> blk) + 1 + 31) >> 5);
    bmap = sp + B::up((size_t)n);
    rec = bmap + B::up(sizeof(uint32_t) * (size_t)bwords);
    WA = rec + (rl ? B::up(sizeof(uint64_t) * (size_t)n) : 0);
    WB = WA + B::up(sizeof(PT) * HEA_MAX_S * t);
    WC = WB + B::up(sizeof(PT) * HEA_MAX_S * t);
    prop = WC + B::up(sizeof(uint32_t) * HEA_MAX_S * t);
    xs = prop + B::up(sizeof(int2) * t);
    cl = xs + B::up(sizeof(double) * t);
    total = cl + B::up(sizeof(int) * t);
  }
};

template <int KMAX, bool RL>
struct GuidedTab {
  using LY = GuidedLayout<KMAX>;
  using SL = SearchLayout<KMAX>;
  using PT = uint32_t;
  using SP = Species<false, Pack<KMAX>::W>;
  double *G, *E0, *R, *tgt, *C, *B, *conc, *ex, *xw, *xs;
  double2 *UV, *SC;   // folded screen table; {d_ij + d_ji, -delta/dd_ij} of the first screen
  float *H, *HZ;      // dF2/dn_ij + dF2/dn_ji and Z_s |H| of it
  float* DH;          // [K][K][S][8]: H[b][x] - H[a][x] of species pair (a, b)
  uint32_t *cmap, *bmap;  // hashed sites and blocks touched by the round's accepts
  int *vec, *sl, *cl;     // stencil vectors; shortlist
  unsigned long long* rec;  // neighbour records (RL)
  int2* prop;
  PT *WA, *WB;
  uint32_t* WC;
  SearchShared* sh;
  SP sp;
  int bwords;
  __device__ void carve(unsigned char* base, int task, int n, int blk) {
    const LY L(task, n, blk, RL);
    G = reinterpret_cast<double*>(base + SL::G);
    E0 = reinterpret_cast<double*>(base + SL::E0);
    R = reinterpret_cast<double*>(base + SL::R);
    tgt = reinterpret_cast<double*>(base + SL::tgt);
    C = reinterpret_cast<double*>(base + SL::C);
    B = reinterpret_cast<double*>(base + SL::B);
    UV = reinterpret_cast<double2*>(base + SL::UV);
    conc = reinterpret_cast<double*>(base + SL::conc);
    ex = reinterpret_cast<double*>(base + SL::ex);
    xw = reinterpret_cast<double*>(base + SL::xw);
    sh = reinterpret_cast<SearchShared*>(base + SL::sh);
    SC = reinterpret_cast<double2*>(base + LY::SC);
    H = reinterpret_cast<float*>(base + LY::H);
    HZ = reinterpret_cast<float*>(base + LY::HZ);
    DH = reinterpret_cast<float*>(base + LY::DH);
    cmap = reinterpret_cast<uint32_t*>(base + LY::cmap);
    vec = reinterpret_cast<int*>(base + LY::vec);
    sl = reinterpret_cast<int*>(base + LY::sl);
    sp.p = base + LY::sp;
    bmap = reinterpret_cast<uint32_t*>(base + L.bmap);
    rec = reinterpret_cast<unsigned long long*>(base + L.rec);
    WA = reinterpret_cast<PT*>(base + L.WA);
    WB = reinterpret_cast<PT*>(base + L.WB);
    WC = reinterpret_cast<uint32_t*>(base + L.WC);
    prop = reinterpret_cast<int2*>(base + L.prop);
    xs = reinterpret_cast<double*>(base + L.xs);
    cl = reinterpret_cast<int*>(base + L.cl);
    bwords = L.bwords;
  }
  __device__ __forceinline__ int idx(int s, int i, int j) const { return (s * KMAX + i) * KMAX + j; }
  __device__ __forceinline__ int uvx(int s, int i, int j) const { return (s * KMAX + i) * SL::KP + j; }
};

// refresh_fold_tables and the guided tables of entries (s,i,j) and (s,j,i);
// returns Z_s |H_ij| (refresh_entry_core's formula).
template <int KMAX, class Tab>
__device__ __forceinline__ float refresh_guided(const ShellArgs& A, const Tab& T, int s, int i,
                                                int j, double g) {
  const FoldEntry v = refresh_fold_tables(A, T, s, i, j, g);
  const double D = v.dij + v.dji;
  const int e = T.idx(s, i, j), f = T.idx(s, j, i);
  T.SC[e].x = D;
  T.SC[f].x = D;
  const float h = (float)(2.0 * A.weight[s] * D * T.C[e]);
  T.H[e] = h;
  T.H[f] = h;
  const float hz = fabsf(h) * (float)A.Z[s];
  T.HZ[e] = hz;
  T.HZ[f] = hz;
  return hz;
}

// The window of a round from its entries' bounds (fold_bound_ahead).
__device__ __forceinline__ double round_window(const SearchShared* sh) {
  double b = 0.0;
#pragma unroll
  for (int s = 0; s < HEA_MAX_S; ++s) b += __longlong_as_double((long long)sh->vb[s]);
  return 2.0 * 1.01 * b;
}

// Largest of non-negative floats over the wave.
__device__ __forceinline__ float fmax_all(float v) {
  return __uint_as_float(~umin_all<true>(~__float_as_uint(v)));
}

template <int KMAX, bool RL>
__device__ __attribute__((noinline)) void undecided_guided(int task, int n, int blk, double xmin,
                                                           double beta) {
  extern __shared__ __align__(16) unsigned char smem[];
  GuidedTab<KMAX, RL> T;
  T.carve(smem, task, n, blk);
  const int lane = threadIdx.x & 63;
  exact_stage<KMAX, true>(T.sh->args, T, T.sp, lane, task, T.sh->ncl, xmin, beta, false);
  if (lane == 0) T.sh->ncl = 0;
}

template <bool RL>
__device__ __forceinline__ uint2 load_rec(const unsigned long long* rec, uint32_t i) {
  if constexpr (RL) {
    return *reinterpret_cast<const uint2*>(rec + i);
  } else {
    // every access to a lattice's records comes from its own workgroup:
    // workgroup-scope atomics, loads and barriers order them
    const unsigned long long v =
        __hip_atomic_load(rec + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
  }
}

// What an accepted swap (v.x: species v.z -> v.w, v.y: back) changes besides the
// tables: its sites' neighbours' records, and the round's maps.  By all lanes of
// one wave.
template <int KMAX, int LT, bool RL>
__device__ __forceinline__ void touch(const GuidedTab<KMAX, RL>& T, unsigned long long* rec,
                                      const int4& v, int L, int blk, float inv_edge, int lane) {
  constexpr int K = KMAX;
  constexpr int ZS = HeaShells<LT>::Z[0] + HeaShells<LT>::Z[1] + HeaShells<LT>::Z[2];
  const auto div = [inv_edge](uint32_t x) { return hea_cell_div_small(x, inv_edge); };
  // items lane and lane + 64 of [0, 2 Z): a neighbour of s1, then of s2
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int t = opaque(lane) + 64 * u;
    const bool one = t < ZS, on = t < 2 * ZS;
    const int vec = T.vec[on ? (one ? t : t - ZS) : 0];
    const HeaCellSite c = hea_cell_site<LT>(one ? v.x : v.y, L, div);
    int id = 0;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      int V = 2 * c.c[x] + c.p[x] + ((vec >> (3 * x)) & 7) - 2;
      V = V < 0 ? V + 2 * L : V >= 2 * L ? V - 2 * L : V;
      using ST = HeaShells<LT>;
      const int Bx = ST::BCC ? (x == 2) : x;
      const int Ax = x == 0 ? ST::NB * L * L : x == 1 ? ST::NB * L : ST::NB;
      id += hea_mul24(Ax, V >> 1) + Bx * (V & 1);
    }
    const int s = vec >> 9;
    const int os = s == 0 ? RecBits<LT>::o(0) : s == 1 ? RecBits<LT>::o(1) : RecBits<LT>::o(2);
    // the last species has no field (its count is implied)
    const unsigned long long fa = v.z < K - 1 ? 1ull << (v.z * RecBits<LT>::W + os) : 0ull;
    const unsigned long long fb = v.w < K - 1 ? 1ull << (v.w * RecBits<LT>::W + os) : 0ull;
    const unsigned long long dv = one ? fb - fa : fa - fb;  // modulo 2^64
    if (on) {
      if constexpr (RL)
        atomicAdd(rec + id, dv);
      else
        __hip_atomic_fetch_add(rec + id, dv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      const uint32_t mb = cmap_bit(id);
      atomicOr(&T.cmap[mb >> 5], 1u << (mb & 31u));
      if (!RL) atomicOr(&T.bmap[(uint32_t)id >> (blk + 5)], 1u << (((uint32_t)id >> blk) & 31u));
    }
  }
  if (lane < 2) {
    const uint32_t mb = cmap_bit(lane == 0 ? v.x : v.y);
    atomicOr(&T.cmap[mb >> 5], 1u << (mb & 31u));
  }
}

// The helper wave takes one command at a time from the service wave: the swap
// of touch, or v.x < 0 at the end of a round's accepts.  Both count them; a wait
// ends because the service wave posts the end before it leaves a round and the
// helper answers every swap.  They sit behind the stencil's vectors (at most 42).
constexpr int kCmdSeq = 48, kCmdDone = 49, kCmd = 52;
__device__ __forceinline__ void await(const int* at, int seq) {
  while (__hip_atomic_load(at, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != seq)
    __builtin_amdgcn_s_sleep(1);
}

// Rounds of the helper wave: touch of every accepted swap, while the service
// wave forms its rows and tables.
template <int KMAX, int LT, bool RL>
__device__ __forceinline__ void guided_helper(const HeaMcArgs& A, const GuidedTab<KMAX, RL>& T,
                                              unsigned long long* rec, int nw, int lane) {
  SearchShared* sh = T.sh;
  const int depth = A.depth, multi = A.g_multi, L = A.edge, blk = A.g_blk;
  const double thr = A.thr;
  const float inv_edge = A.inv_edge;
  int seq = 0;
  auto serve = [&]() {
    await(T.vec + kCmdSeq, ++seq);
    const int4 v = *reinterpret_cast<const int4*>(T.vec + kCmd);
    if (__builtin_amdgcn_readfirstlane(v.x) < 0) return false;
    touch<KMAX, LT, RL>(T, rec, v, L, blk, inv_edge, lane);
    if (lane == 0)
      __hip_atomic_store(T.vec + kCmdDone, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    return true;
  };
  __builtin_amdgcn_s_setprio(2);
  for (int acc = 0; acc < depth;) {
    __syncthreads();  // BD
    const double beta = round_window(sh);
    __syncthreads();  // B1
    int kind = decide(sh, nw, beta, thr, lane).kind;
    if (__builtin_expect(kind < 0, 0)) {
      __syncthreads();
      __syncthreads();
      kind = __builtin_amdgcn_readfirstlane(sh->res_kind);
    }
    if (kind == 0) {
      ++acc;
    } else {
      acc = 0;
      serve();
      if (multi > 1) {
        __syncthreads();  // BS
        while (serve()) {
        }
      }
    }
    __syncthreads();  // BA
  }
}

// Rounds of the service wave: the accepts.
template <int KMAX, int LT, bool RL>
__device__ __forceinline__ void guided_service(const HeaMcArgs& A, const GuidedTab<KMAX, RL>& T,
                                               unsigned long long* rec, int l, int nw, bool help,
                                               int lane) {
  using PK = Pack<KMAX>;
  using PT = uint32_t;
  constexpr int K = KMAX, S = 3;
  SearchShared* sh = T.sh;
  const ShellArgs& SA = sh->args;
  const int task = A.task, stride = A.stride, depth = A.depth, n = A.N, L = A.edge, blk = A.g_blk;
  const int multi = A.g_multi;
  const double thr = A.thr;
  const int32_t* nbr = A.nbr;
  const float inv_edge = A.inv_edge;
  int seq = 0;
  auto post = [&](const int4& v) {
    ++seq;
    if (lane == 0) {
      *reinterpret_cast<int4*>(T.vec + kCmd) = v;
      __hip_atomic_store(T.vec + kCmdSeq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  // lane (s, h, x) takes entry (a, x) (h = 0) or (b, x) of an accepted swap
  // (lanes beyond them repeat an entry: they write the same values).  Taken
  // anew where it is used: kept over the rounds, what follows from it spills.
  struct Entry {
    int s, h, x;
  };
  auto entry_of = [](int ln) {
    const int sv = opaque(ln) % (2 * K * S), k = sv % (2 * K);
    return Entry{sv / (2 * K), k >= K ? 1 : 0, k >= K ? k - K : k};
  };
  long long rounds = 0, accepts = 0, screens = 0;
  bool hit = false;
  double beta = 0.0;
  __builtin_amdgcn_s_setprio(3);

  // The fitness after a swap that the window decided (lane 0).  Of a round's
  // first one only behind a barrier: the other waves' decide() reads the old.
  auto estimate = [&](const Decision& d) {
    sh->pfm = 2;
    sh->fest = sh->fest + d.xmin;
  };
  // Accept of swap (s1: a -> b, s2: b -> a): exact rows, tables, species,
  // records and the round's maps.
  auto apply = [&](const Decision& d, const Winner<PT>& win, bool first) {
    if (help)
      post(make_int4(d.s1, d.s2, d.a, d.b));
    else
      touch<KMAX, LT, RL>(T, rec, make_int4(d.s1, d.s2, d.a, d.b), L, blk, inv_edge, lane);
    const Entry en = entry_of(lane);
    const int sv_s = en.s, sv_h = en.h, sv_x = en.x;
    const int r = sv_h ? d.b : d.a;
    double g;
    if (d.kind == 2) {
      g = winner_entry<KMAX>(SA, T, sv_s, sv_x, sv_h, S, stride, d.a, d.b, win, lane, [&]() {
        // (few swaps need the rows: loaded early, they wait behind the
        // workers' record loads)
        int2 col = make_int2(-1, -1);
        if (lane < stride)
          col = make_int2(nbr[(size_t)d.s1 * stride + lane], nbr[(size_t)d.s2 * stride + lane]);
        return col;
      });
      wave_sync();  // every lane has read its entries
      T.G[T.idx(sv_s, r, sv_x)] = g;
      T.G[T.idx(sv_s, sv_x, r)] = g;
    } else {  // the exact stage wrote its rows
      g = T.G[T.idx(sv_s, r, sv_x)];
    }
    const float hz = refresh_guided<KMAX>(SA, T, sv_s, r, sv_x, g);
    float top = fmax_all(hz);
    // the first accept of a round takes the scale of every entry, the others
    // only raise it by the entries they change
    wave_sync();
    if (first) {
      for (int e = lane; e < S * K * K; e += 64) top = fmaxf(top, T.HZ[e]);
      top = fmax_all(top);
    }
    if (lane == 0) {
      T.sp.set(d.s1, d.b);
      T.sp.set(d.s2, d.a);
      if (d.kind == 2 && !first) estimate(d);
      sh->gmax = first ? __float_as_uint(top) : max(sh->gmax, __float_as_uint(top));
    }
    wave_sync();
  };

  for (int acc = 0; acc < depth;) {
    __syncthreads();  // BD
    beta = round_window(sh);
    __syncthreads();  // B1
    Decision d = decide(sh, nw, beta, thr, lane);
    ++rounds;
    screens += task;
    if (__builtin_expect(d.kind < 0, 0)) {
      __syncthreads();
      undecided_guided<KMAX, RL>(task, n, blk, d.xmin, beta);
      __syncthreads();
      read_exact(sh, T.prop, d);
      if (d.kind == 2) d.kind = 1;
      if (d.kind == 1 && __longlong_as_double((long long)sh->res_key) <= thr) hit = true;
    }
    if (d.kind == 0) {
      ++acc;
    } else {
      acc = 0;
      ++accepts;
      for (int e = lane; e < kCmapWords / 4; e += 64)
        reinterpret_cast<uint4*>(T.cmap)[e] = make_uint4(0, 0, 0, 0);
      for (int e = lane; e < T.bwords; e += 64) T.bmap[e] = 0u;
      Winner<PT> win{};
      {
        const int w = entry_of(lane).s * task + d.j;
        win.ma = T.WA[w];
        win.mb = T.WB[w];
        win.c12 = walk_unpack(T.WC[w]).c12;
        win.s1 = d.s1;
        win.s2 = d.s2;
      }
      apply(d, win, true);
      if (multi > 1) {
        __syncthreads();  // BS
        if (d.kind == 2 && lane == 0) estimate(d);
        wave_sync();
        int j, c12[S], a, b;
        int2 pr;
        PT MA[S], MB[S];
        auto load = [&]() {  // the lane's shortlisted proposal
          j = T.sl[opaque(lane)];
          const int jl = max(j, 0);
          pr = T.prop[jl];
          const WalkRec w = walk_unpack(T.WC[jl]);
          a = w.a;
          b = w.b;
#pragma unroll
          for (int s = 0; s < S; ++s) {
            MA[s] = T.WA[s * task + jl];
            MB[s] = T.WB[s * task + jl];
            c12[s] = walk_unpack(T.WC[s * task + jl]).c12;
          }
        };
        load();
        for (int step = 1; step < multi; ++step) {
          if (help) await(T.vec + kCmdDone, seq);
          if (j >= 0) {  // a touched proposal's walk is stale: dropped for good
            const uint32_t b1 = cmap_bit(pr.x), b2 = cmap_bit(pr.y);
            if (((T.cmap[b1 >> 5] >> (b1 & 31u)) | (T.cmap[b2 >> 5] >> (b2 & 31u))) & 1u) j = -1;
          }
          const unsigned long long live = __ballot(j >= 0);
          screens += __popcll(live);
          if (live == 0ull) break;
          double X = __builtin_inf();
          if (j >= 0) X = screen_fold<KMAX>(T, S, a, b, MA, MB, c12);
          int src = argmin_lane<true>(X);
          d.xmin = readlane_f64(X, src);
          const double mg = 2.0 * beta;
          const bool in = j >= 0 && !(X > d.xmin + mg);
          const unsigned long long bal = __ballot(in);
          const double fest = sh->fest;
          const bool near = thr > 0.0 && !(fest + d.xmin > thr * thr * 1.01);
          const bool one = (bal & (bal - 1ull)) == 0ull;
          const int sure = d.xmin - mg > 0.0 ? 0 : (one && d.xmin + mg < 0.0) ? 2 : -1;
          d.kind = __builtin_amdgcn_readfirstlane(sh->pfm != 0 && !near ? sure : -1);
          if (__builtin_expect(d.kind < 0, 0)) {
            if (in) {
              T.cl[__popcll(bal & ((1ull << lane) - 1ull))] = j;
              T.xs[j] = X;
            }
            if (lane == 0) sh->ncl = __popcll(bal);
            T.sl[lane] = j;
            wave_sync();
            undecided_guided<KMAX, RL>(task, n, blk, d.xmin, beta);
            wave_sync();
            load();  // (so that the call keeps none of it)
            read_exact(sh, T.prop, d);
            if (d.kind == 2) d.kind = 1;
            if (d.kind == 1 && __longlong_as_double((long long)sh->res_key) <= thr) hit = true;
            if (d.kind != 0) src = (int)__builtin_ctzll(__ballot(j == d.j));
          }
          if (d.kind == 0) break;
          ++accepts;
          d.a = __builtin_amdgcn_readlane(a, src);
          d.b = __builtin_amdgcn_readlane(b, src);
          d.s1 = __builtin_amdgcn_readlane(pr.x, src);
          d.s2 = __builtin_amdgcn_readlane(pr.y, src);
          win.s1 = d.s1;
          win.s2 = d.s2;
          const int sv_s = entry_of(lane).s;
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const uint32_t ma = (uint32_t)__builtin_amdgcn_readlane((int)MA[s], src);
            const uint32_t mb = (uint32_t)__builtin_amdgcn_readlane((int)MB[s], src);
            const int cc = __builtin_amdgcn_readlane(c12[s], src);
            if (sv_s == s) {
              win.ma = ma;
              win.mb = mb;
              win.c12 = cc;
            }
          }
          apply(d, win, false);
        }
        if (help) {  // (a command is never replaced before it was answered)
          await(T.vec + kCmdDone, seq);
          post(make_int4(-1, 0, 0, 0));
        }
      }
      if (lane < HEA_MAX_S) sh->vb[lane] = 0ull;  // the workers take the new bounds
    }
    __syncthreads();  // BA
    if (multi <= 1 && d.kind == 2 && lane == 0) estimate(d);
    if (hit && lane == 0 && A.first_hit)
      atomicMin(A.first_hit, (unsigned long long)wall_clock64());
    hit = false;
  }
  if (lane == 0) {
    int64_t* st = A.stats + (size_t)l * 4;
    st[0] += rounds;
    st[1] += accepts;
    st[2] += screens;
    st[3] += (long long)((uint32_t)rounds * (uint32_t)(task * A.g_cand));  // the stream position
  }
}

// Rounds of a worker wave.
template <int KMAX, int LT, bool RL>
__device__ __forceinline__ void guided_worker(const HeaMcArgs& A, const GuidedTab<KMAX, RL>& T,
                                              const unsigned long long* rec, int l, int nw,
                                              int wave, int tid, int nthr) {
  using PK = Pack<KMAX>;
  using RB = RecBits<LT>;
  using SP = Species<false, PK::W>;
  constexpr int K = KMAX, S = 3;
  SearchShared* sh = T.sh;
  const SP sp = T.sp;
  const int lane = tid & 63;
  const uint32_t N = (uint32_t)A.N;
  const int task = A.task, depth = A.depth, blk = A.g_blk, g = A.g_cand, edge = A.edge;
  const double thr = A.thr, tau = A.g_tau;
  const float inv_edge = A.inv_edge;
  const auto div = [inv_edge](uint32_t x) { return hea_cell_div_small(x, inv_edge); };
  const bool has = tid < task;
  const int j_me = min(tid, task - 1);
  const uint32_t iter = *A.iter_ptr;
  const uint32_t gk = hea_mix32(hea_mix32(hea_mix32((uint32_t)A.seed ^ 0x6a09e667u) ^
                                          (uint32_t)(A.seed >> 32)) ^
                                (iter * 4u + (A.phase & 3u))) ^
                      hea_mix32((uint32_t)l + 0x3c6ef372u);
  const int nwp = nw, per = (64 + nwp - 1) / nwp;  // shortlist share of a wave
  uint32_t pos = 0;
  // the slot's blocks, and of the candidates drawn ahead: places in the blocks
  // (16 bits each), noise and records
  uint32_t bx = 0, by = 0;
  uint32_t place[kPre] = {};
  float noise[kPre] = {};
  uint2 r1[kPre] = {}, r2[kPre] = {};
  const uint32_t bs = 1u << blk, nb = (N + bs - 1) >> blk;

  auto cand_draw = [&](uint32_t ctr, uint32_t& i1, uint32_t& i2, float& nz) {
    const uint32_t h0 = hea_mix32(gk ^ (ctr * 0x9e3779b9u));
    const uint32_t h1 = hea_mix32(h0 ^ 0x85ebca6bu);
    const uint32_t h2 = hea_mix32(h1 ^ 0xc2b2ae35u);
    i1 = __umulhi(h0, min(N - bx, bs));
    i2 = __umulhi(h1, min(N - by, bs));
    const float U = ((float)(h2 >> 8) + 0.5f) * 0x1p-24f;
    nz = __logf(-__logf(U));
  };
  // the next round's blocks, candidates and their records
  auto ahead = [&]() {
    const uint32_t sctr = pos + (uint32_t)(j_me * g);
    const uint32_t k0 = hea_mix32(gk ^ (sctr * 0x9e3779b9u) ^ 0x27d4eb2fu);
    const uint32_t k1 = hea_mix32(k0 ^ 0x165667b1u);
    bx = __umulhi(k0, nb) << blk;
    by = __umulhi(k1, nb) << blk;
#pragma unroll
    for (int c0 = 0; c0 < kPre; c0 += kGroup) {
      if (c0 < g) {  // (a last, partial group repeats the last candidate)
#pragma unroll
        for (int c = c0; c < c0 + kGroup; ++c) {
          uint32_t i1, i2;
          cand_draw(sctr + (uint32_t)min(c, g - 1), i1, i2, noise[c]);
          place[c] = i1 | (i2 << 16);
          if constexpr (!RL) {
            r1[c] = load_rec<RL>(rec, bx + i1);
            r2[c] = load_rec<RL>(rec, by + i2);
          }
        }
      } else {  // (or the old values stay live over the whole round)
#pragma unroll
        for (int c = c0; c < c0 + kGroup; ++c) {
          noise[c] = 0.0f;
          place[c] = 0u;
          r1[c] = r2[c] = make_uint2(0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  ahead();
  bool changed = false, stale = true;  // the last round accepted swaps; bounds to be taken

  for (int acc = 0; acc < depth;) {
    // ---- differences of the gain rows of every species pair
    for (int e = opaque(tid); e < K * K * S * K; e += nthr) {
      const int p = e / (S * K), q = e - p * S * K, s = q / K, x = q - s * K;
      const int a = p / K, b = p - a * K;
      T.DH[(p * S + s) * 8 + x] = T.H[T.idx(s, b, x)] - T.H[T.idx(s, a, x)];
    }
    // ---- the round's window: bounds that also hold after its accepts
    if (stale) {
      for (int e = opaque(tid); e < S * K * K; e += nthr) {
        const int s = e / (K * K), i = (e / K) % K, j = e % K;
        if (i <= j) {
          const double v = fold_bound_ahead(sh->args, T, s, i, j, T.G[e], A.g_multi);
          atomicMax(&sh->vb[s], (unsigned long long)__double_as_longlong(v));
        }
      }
    }
    const float gs = 2.0f * __uint_as_float(sh->gmax);
    const float inv = (float)(1.0 / (tau * (gs > 0.0f ? (double)gs : 1.0)));
    if (!RL && changed) {  // records that the accepts changed
      const uint32_t q1 = bx >> blk, q2 = by >> blk;
      const bool t1 = (T.bmap[q1 >> 5] >> (q1 & 31u)) & 1u, t2 = (T.bmap[q2 >> 5] >> (q2 & 31u)) & 1u;
      if (t1) {
#pragma unroll
        for (int c = 0; c < kPre; ++c) r1[c] = load_rec<RL>(rec, bx + (place[c] & 0xffffu));
      }
      if (t2) {
#pragma unroll
        for (int c = 0; c < kPre; ++c) r2[c] = load_rec<RL>(rec, by + (place[c] >> 16));
      }
    }
    __syncthreads();  // BD

    // ---- score the candidates, keep the slot's best (ties: the first)
    uint32_t best = 0, s1 = 0, s2 = 0;
    uint2 ra = make_uint2(0, 0), rb = ra;
    int a = 0, b = 0;
    bool found = false;
    auto score = [&](uint32_t i1, uint32_t i2, int ca, int cb, float nz, uint2 q1, uint2 q2) {
      const uint32_t t1 = bx + i1, t2 = by + i2;
      const int xa = SP::species_of(ca), xb = SP::species_of(cb);
      const float* dh = T.DH + (xa * K + xb) * (S * 8);
      float d = 0.0f;
      static_for<S>([&](auto s) {
        const float4 lo = *reinterpret_cast<const float4*>(dh + s * 8);
        float4 hi = make_float4(0, 0, 0, 0);
        if constexpr (K > 4) hi = *reinterpret_cast<const float4*>(dh + s * 8 + 4);
        const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        int rest = 0;
        static_for<K - 1>([&](auto x) {
          const int dc = (int)rec_field<x * RB::W + RB::o(s), RB::w(s)>(q1) -
                         (int)rec_field<x * RB::W + RB::o(s), RB::w(s)>(q2);
          rest -= dc;
          d += v[x] * (float)dc;
        });
        d += v[K - 1] * (float)rest;
      });
      const float sc = -d * inv - nz;
      // order-preserving float bits
      const uint32_t fb = __float_as_uint(sc);
      const uint32_t ob = (fb & 0x80000000u) ? ~fb : (fb | 0x80000000u);
      if (ca != cb && (!found || ob > best)) {
        found = true;
        best = ob;
        s1 = t1;
        s2 = t2;
        ra = q1;
        rb = q2;
        a = xa;
        b = xb;
      }
    };
    // (groups of candidates, or the compiler keeps all of them in flight and
    // spills)
#pragma unroll
    for (int c0 = 0; c0 < kPre; c0 += kGroup) {
      if (c0 < g) {
        int ca[kGroup], cb[kGroup];
#pragma unroll
        for (int k = 0; k < kGroup; ++k) {
          const uint32_t p = place[c0 + k];
          ca[k] = sp.code(bx + (p & 0xffffu));
          cb[k] = sp.code(by + (p >> 16));
          if constexpr (RL) {
            r1[c0 + k] = load_rec<RL>(rec, bx + (p & 0xffffu));
            r2[c0 + k] = load_rec<RL>(rec, by + (p >> 16));
          }
        }
#pragma unroll
        for (int k = 0; k < kGroup; ++k)  // (a repeated candidate never wins)
          score(place[c0 + k] & 0xffffu, place[c0 + k] >> 16, ca[k], cb[k], noise[c0 + k],
                r1[c0 + k], r2[c0 + k]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int c = kPre; c < g; ++c) {
      uint32_t i1, i2;
      float nz;
      cand_draw(pos + (uint32_t)(j_me * g + c), i1, i2, nz);
      score(i1, i2, sp.code(bx + i1), sp.code(by + i2), nz, load_rec<RL>(rec, bx + i1),
            load_rec<RL>(rec, by + i2));
    }
    pos += (uint32_t)(task * g);
    const bool cand = has && found;

    // ---- screen the proposal (screen_shell's order of operations: the
    // shortlist is cut by X)
    __builtin_amdgcn_sched_barrier(0);
    const int jm = opaque(j_me);
    double X = 0.0;
    {
      int L = edge;
      asm("" : "+s"(L));
      const HeaCellSite c1 = hea_cell_site<LT>((int)s1, L, div);
      const HeaCellSite c2 = hea_cell_site<LT>((int)s2, L, div);
      const int d2 = hea_cell_dist2(c1, c2, L);
      static_for<S>([&](auto s) {
        const int c12 = d2 == HeaShells<LT>::D2[s] ? 1 : 0;
        const uint32_t ma = rec_shell<KMAX, LT, s>(ra), mb = rec_shell<KMAX, LT, s>(rb);
        if (has) {
          const int w = s * task + jm;
          T.WA[w] = ma;
          T.WB[w] = mb;
          T.WC[w] = walk_pack(0, c12, c12, 0, a, b);
        }
        X = X + sh->args.weight[s] *
                    screen_shell<KMAX, true>(T, KMAX, s, a, b, ma, mb, 0, c12, c12, 0);
        __builtin_amdgcn_sched_barrier(0);  // one shell's table rows at a time
      });
    }
    const int2 pr = cand ? make_int2((int)s1, (int)s2) : make_int2(-1, -1);
    if (has) T.prop[jm] = pr;
    const double beta = round_window(sh);
    const double xv = cand ? X : __builtin_inf();
    {
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
    if (__builtin_expect(d.kind < 0, 0)) {
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
      d.kind = __builtin_amdgcn_readfirstlane(sh->res_kind);
    }
    changed = stale = d.kind != 0;
    acc = changed ? 0 : acc + 1;
    if (changed && A.g_multi > 1) {
      // the wave's smallest X < 0, for the further accepts
      // (argmin_lane's keys, made once)
      const unsigned long long xb =
          (unsigned long long)__double_as_longlong(cand && X < 0.0 ? X : __builtin_inf());
      const uint32_t flip = (uint32_t)((int32_t)(xb >> 32) >> 31);
      uint32_t hi = (uint32_t)(xb >> 32) ^ (flip | 0x80000000u);
      int mine = -1;
      for (int r = 0; r < per; ++r) {
        const uint32_t m = umin_all<true>(hi);
        if (m >= 0x80000000u) break;  // no X < 0 left
        unsigned long long at = __ballot(hi == m);
        if ((at & (at - 1ull)) != 0ull) {
          const uint32_t lo = hi == m ? (uint32_t)xb ^ flip : ~0u;
          const uint32_t ml = umin_all<true>(lo);
          at = __ballot(hi == m && lo == ml);
        }
        const int src = (int)__builtin_ctzll(at);
        if (lane == src) hi = ~0u;
        if (lane == r) mine = wave * 64 + src;
      }
      if (lane < per && wave * per + lane < 64) T.sl[wave * per + lane] = mine;
      __syncthreads();  // BS
    }
    ahead();
    __syncthreads();  // BA
  }
}

template <int KMAX, int LT, bool RL>
__global__ __launch_bounds__(kMaxSearchThreads, 3) void k_guided(HeaMcArgs A) {
  extern __shared__ __align__(16) unsigned char smem[];
  using PK = Pack<KMAX>;
  constexpr int K = KMAX, S = 3;
  const HeaConst& P = *A.pc;
  const int l = blockIdx.x, nthr = blockDim.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nw = (A.task + 63) >> 6;  // worker waves; then the service wave and the helper
  const int N = A.N;

  GuidedTab<KMAX, RL> T;
  T.carve(smem, A.task, N, A.g_blk);
  SearchShared* sh = T.sh;
  uint8_t* lat_g = A.lattices + (size_t)l * N;
  unsigned long long* rec = RL ? T.rec : A.hist + (size_t)l * N;
  for (int i = tid; i < N; i += nthr) T.sp.p[i] = (uint8_t)(lat_g[i] * PK::W);
  for (int e = tid; e < HEA_MAX_S * KMAX * SearchLayout<KMAX>::KP; e += nthr)
    T.UV[e] = make_double2(0.0, 0.0);
  if (tid < 64) T.sl[tid] = -1;
  if (tid >= kCmdSeq && tid < 64) T.vec[tid] = 0;
  if (tid < HEA_MAX_S) {
    sh->args.delta[tid] = P.delta[tid];
    sh->args.weight[tid] = P.weight[tid];
    sh->args.Z[tid] = P.Z[tid];
    sh->args.off[tid] = P.off[tid];
  }
  if (tid < K) T.conc[tid] = P.conc[tid];
  if (tid < kWaves) sh->wm[tid] = __builtin_inf();
  if (tid < HEA_MAX_S) sh->vb[tid] = 0ull;
  if (tid == 0) {
    const double f0 = A.fitness[l];
    sh->pf = f0;
    sh->pfm = 0;
    sh->fest = f0 * f0;
    sh->ncl = 0;
    sh->gmax = 0u;
    sh->next_pos = 0u;
    sh->args.N = N;
    sh->args.K = K;
    sh->args.S = S;
    sh->args.stride = A.stride;
    sh->args.nbr = A.nbr;
    sh->args.thr = A.thr;
  }
  __syncthreads();
  const ShellArgs& SA = sh->args;
  if (tid < 125) {  // the stencil's vectors, in any order
    const int dx = tid / 25 - 2, dy = tid / 5 % 5 - 2, dz = tid % 5 - 2;
    const int s = HeaShells<LT>::shell(dx, dy, dz);
    if (s >= 0)
      T.vec[atomicAdd(&sh->next_pos, 1u)] = (dx + 2) | ((dy + 2) << 3) | ((dz + 2) << 6) | (s << 9);
  }
  const int32_t* cnt_g = A.counts + (size_t)l * S * K * K;
  for (int e = tid; e < S * K * K; e += nthr) {
    const int s = e / (K * K), i = (e / K) % K, j = e % K;
    const double c = -SA.delta[s] / (T.conc[i] * T.conc[j]);
    T.G[T.idx(s, i, j)] = hea_r_of_count(P, s, cnt_g[e]);
    T.tgt[T.idx(s, i, j)] = P.target[s][i][j];
    T.C[T.idx(s, i, j)] = c;
    T.SC[T.idx(s, i, j)].y = c;
    T.UV[T.uvx(s, i, j)].y = 2.0 * SA.weight[s] * c * c;
  }
  __syncthreads();
  for (int e = tid; e < S * K * K; e += nthr) {
    const int s = e / (K * K), i = (e / K) % K, j = e % K;
    if (i <= j) {
      const float hz = refresh_guided<KMAX>(SA, T, s, i, j, T.G[T.idx(s, i, j)]);
      atomicMax(&sh->gmax, __float_as_uint(hz));
    }
  }
  {  // every site's record
    const float inv_edge = A.inv_edge;
    const auto div = [inv_edge](uint32_t x) { return hea_cell_div_small(x, inv_edge); };
    const uint32_t spa = lds_addr(T.sp.p);
    for (int k = tid; k < N; k += nthr) {
      const HeaCellSite c = hea_cell_site<LT>(k, A.edge, div);
      const SiteTerms t = site_terms<LT, false>(c, A.edge, spa);
      unsigned long long m = 0ull;
      static_for<S>([&](auto s) {
        uint32_t v[HeaShells<LT>::Z[s]], h = 0;
        load_shell<LT, s>(t, v);
        __builtin_amdgcn_sched_barrier(0);
        count_shell<KMAX, LT, s, false>(t, v, h);
        static_for<K - 1>([&](auto x) {
          m |= (unsigned long long)PK::fld(h, x) << (x * RecBits<LT>::W + RecBits<LT>::o(s));
        });
      });
      rec[k] = m;
    }
  }
  __syncthreads();

  if (wave == nw)
    guided_service<KMAX, LT, RL>(A, T, rec, l, nw, nthr > 64 * (nw + 1), lane);
  else if (wave > nw)
    guided_helper<KMAX, LT, RL>(A, T, rec, nw, lane);
  else
    guided_worker<KMAX, LT, RL>(A, T, rec, l, nw, wave, tid, nw * 64);

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
  }
  for (int i = tid; i < N; i += nthr)
    lat_g[i] = (uint8_t)Species<false, PK::W>::species_of(T.sp.p[i]);
}

template <int LT, bool RL>
const void* guided_fn(int K) {
  switch (K) {
    case 2: return reinterpret_cast<const void*>(k_guided<2, LT, RL>);
    case 3: return reinterpret_cast<const void*>(k_guided<3, LT, RL>);
    case 4: return reinterpret_cast<const void*>(k_guided<4, LT, RL>);
    case 5: return reinterpret_cast<const void*>(k_guided<5, LT, RL>);
    case 6: return reinterpret_cast<const void*>(k_guided<6, LT, RL>);
    default: return nullptr;
  }
}
template <bool RL>
const void* guided_fn(int lt, int K) {
  return lt == HEA_LT_FCC       ? guided_fn<HEA_LT_FCC, RL>(K)
         : lt == HEA_LT_FCC_REF ? guided_fn<HEA_LT_FCC_REF, RL>(K)
                                : guided_fn<HEA_LT_BCC, RL>(K);
}

size_t guided_lds(int K, int task, int n, int blk, bool rl) {
  switch (K) {
    case 2: return GuidedLayout<2>(task, n, blk, rl).total;
    case 3: return GuidedLayout<3>(task, n, blk, rl).total;
    case 4: return GuidedLayout<4>(task, n, blk, rl).total;
    case 5: return GuidedLayout<5>(task, n, blk, rl).total;
    default: return GuidedLayout<6>(task, n, blk, rl).total;
  }
}

}  // namespace

// A guided search is this kernel's when the lattice is a stencil with all
// three shells and byte species fit in LDS, candidates come from blocks, and
// a round is one pass of the workers.  `lanes`: workgroup size of the general
// kernel, whose shortlist takes one proposal per lane: beyond it the two
// would cut different shortlists.
HeaSearchPlan hea_guided_plan(const HeaConst& c, int lt, int task, int blk, int lanes,
                              int64_t max_lds) {
  HeaSearchPlan p;
  if (lt == HEA_LT_NONE || c.S != 3 || c.K > 6 || blk < 1 || task > kMaxSearchThreads - 64 ||
      task > lanes)
    return p;
  p.rec_lds = true;  // records in LDS where they fit
  p.lds = guided_lds(c.K, task, c.N, blk, true);
  if ((int64_t)p.lds > max_lds) {
    p.rec_lds = false;
    p.lds = guided_lds(c.K, task, c.N, blk, false);
  }
  if ((int64_t)p.lds > max_lds) return HeaSearchPlan();
  // A helper wave (8 to 10 % of a search, see above) where it costs no resident
  // workgroup, which would cost far more on a full chip: three waves a SIMD fit
  // (registers), and as many workgroups as their LDS.
  const int waves = ((task + 63) >> 6) + 1, by_lds = (int)(160 * 1024 / p.lds);
  const bool help = waves + 1 <= kMaxSearchThreads / 64 &&
                    std::min(12 / (waves + 1), by_lds) == std::min(12 / waves, by_lds);
  p.threads = 64 * (waves + (help ? 1 : 0));
  return p;
}

hipError_t hea_prepare_guided(int lt, int K, bool rec_lds, size_t lds) {
  const void* fn = rec_lds ? guided_fn<true>(lt, K) : guided_fn<false>(lt, K);
  return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

hipError_t hea_launch_guided(const HeaMcArgs& a, const HeaSearchPlan& p, hipStream_t st) {
  const void* fn = p.rec_lds ? guided_fn<true>(a.lt, a.K) : guided_fn<false>(a.lt, a.K);
  if (!fn) return hipErrorInvalidValue;
  void* args[] = {const_cast<HeaMcArgs*>(&a)};
  return hipLaunchKernel(fn, dim3(a.L), dim3(p.threads), args, p.lds, st);
}
