// Wave-level steps that the local-search kernels share: reductions over one
// wave, the walk records, and the exact stage that decides a round.  The
// tables `Tab` are the kernels' LDS tables (hea_screen.h), with the proposals
// prop, their walk records WA, WB, WC and screen values xs, the candidate list
// cl, the work rows xw and ex, and the round's state sh.
#pragma once
#include "hea_internal.h"
#include "hea_screen.h"

namespace {

// Orders LDS traffic between the lanes of one wave (the hardware keeps a
// wave's LDS operations in order; this stops the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Walk record of one (proposal, shell): the adjacency counts c11, c12, c21,
// c22 (each <= HEA_MAX_Z, 5 bits) and the species a, b of the two sites.
struct WalkRec {
  int c11, c12, c21, c22, a, b;
};
__device__ __forceinline__ uint32_t walk_pack(int c11, int c12, int c21, int c22, int a, int b) {
  return (uint32_t)c11 | ((uint32_t)c12 << 5) | ((uint32_t)c21 << 10) | ((uint32_t)c22 << 15) |
         ((uint32_t)a << 20) | ((uint32_t)b << 24);
}
__device__ __forceinline__ WalkRec walk_unpack(uint32_t w) {
  return WalkRec{(int)(w & 31u),         (int)((w >> 5) & 31u), (int)((w >> 10) & 31u),
                 (int)((w >> 15) & 31u), (int)((w >> 20) & 15u), (int)((w >> 24) & 15u)};
}

// One step of a DPP reduction: v = min(v, v of the lane DPP control CTRL
// names), in the rows ROWS enables; lanes of other rows keep v.  Every
// control used here names a lane of the same wave, so no lane reads an
// out-of-range source.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_min_step(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = (int)(uint32_t)b, hi = (int)(uint32_t)(b >> 32);
  const int olo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
  const int ohi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
  const double o = __longlong_as_double(
      (long long)(((unsigned long long)(uint32_t)ohi << 32) | (uint32_t)olo));
  return fmin(v, o);
}

// Smallest v over all 64 lanes (every lane active), returned to every lane.
// row_ror:1,2,4,8 leave each 16-lane row's minimum in all its lanes;
// row_bcast:15 folds rows 0 and 2 into rows 1 and 3, row_bcast:31 folds
// row 1 into rows 2 and 3, so lane 63 holds the wave's minimum.
__device__ __forceinline__ double wave_min(double v) {
  v = dpp_min_step<0x121, 0xf>(v);
  v = dpp_min_step<0x122, 0xf>(v);
  v = dpp_min_step<0x124, 0xf>(v);
  v = dpp_min_step<0x128, 0xf>(v);
  v = dpp_min_step<0x142, 0xa>(v);
  v = dpp_min_step<0x143, 0xc>(v);
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, 63);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 63);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Largest v over all 64 lanes (every lane active), returned to every lane.
__device__ __forceinline__ double wave_max(double v) { return -wave_min(-v); }

// Fitness of the current gamma as the reference computes it
// (accelerate.cpp:557-569): E0 holds the current terms; lane s < S adds its
// shell's K*K terms in row-major order.  Called by all lanes of one wave.
template <int KMAX, bool EXACT, class Args, class Tab>
__device__ __forceinline__ double current_fitness(const Args& A, const Tab& T,
                                                  int lane) {
  const int K = A.K, S = A.S;
  if (lane < S) {
    const double* e0 = T.E0 + T.idx(lane, 0, 0);
    double es = 0.0;
#pragma unroll
    for (int i = 0; i < KMAX; ++i)
#pragma unroll
      for (int y = 0; y < KMAX; ++y)
        if (EXACT || (i < K && y < K)) es = es + e0[i * KMAX + y];
    T.ex[lane] = es;
  }
  wave_sync();
  double err = 0.0;
  for (int t = 0; t < S; ++t) err = err + A.weight[t] * T.ex[t];
  wave_sync();  // ex is reused
  return sqrt(err);
}

__device__ __forceinline__ bool key_less(unsigned long long f1, int j1, unsigned long long f2,
                                         int j2) {
  return (f1 < f2) || (f1 == f2 && j1 < j2);
}

// Exact stage of a round, run by one wave (wave 0): the candidates T.cl[0,
// nsup) (a superset of the proposals whose X lies within 2 beta of xmin),
// first strict minimum of F (accelerate.cpp:663-674) and the accept test
// (:678).  Writes the decision to T.sh (res_kind, res_j, res_a, res_b,
// res_key, pf, pfm, fest) and, for an accept, the winner's new gamma rows;
// with `reset` an accept also clears the bound maxima that the refresh of
// every entry then takes again.
template <int KMAX, bool EXACT, class Args, class Tab, class Sp>
__device__ __forceinline__ void exact_stage(const Args& A, const Tab& T, const Sp sp,
                                            int lane, int task, int nsup, double xmin,
                                            double beta, bool reset) {
  const int K = A.K, S = A.S;
  double prev_fit = T.sh->pf, fest = T.sh->fest;
  int pfm = T.sh->pfm;
  double thr = xmin + 2.0 * beta;
  if (!(thr < __builtin_inf())) thr = __builtin_inf();
  // filter the waves' lists against the workgroup's window, compacting
  // in place (every entry is read before any of its chunk is written)
  int nc = 0, jfirst = -1;  // jfirst = cl[0] after the compaction
  for (int k0 = 0; k0 < nsup; k0 += 64) {
    const int j = (k0 + lane < nsup) ? T.cl[k0 + lane] : -1;
    const bool f = j >= 0 && !(T.xs[j] > thr);
    const unsigned long long bal = __ballot(f);
    if (nc == 0 && bal) jfirst = __builtin_amdgcn_readlane(j, (int)__builtin_ctzll(bal));
    wave_sync();
    if (f) T.cl[nc + __popcll(bal & ((1ull << lane) - 1ull))] = j;
    nc += __popcll(bal);
  }
  wave_sync();
  // lane (c, s, x): candidate c of the chunk, shell s, species x
  const int GS = S * K;      // lanes per candidate
  const int cpc = 64 / GS;   // candidates per chunk
  const int g = lane / K, x = lane - g * K;
  const int c = g / S, s = g - c * S;
  constexpr int XW = 4 + KMAX;
  double* slot = T.xw + lane * XW;
  const double* grp = T.xw + g * K * XW;  // lane (c, s, y) at grp + y * XW
  unsigned long long bk = ~0ull;
  int bj = 0x7fffffff, bc = 0, wc0 = -1;
  int ra = 0, rb = 0;  // window-decided accept: the winner's species (lanes < S*K)
  // When prev_fit = F(gamma), the window decides most rounds: every
  // proposal's err lies within beta of E + X (E common, X = 0 for the
  // current lattice), and 2 beta keeps sqrt's rounding out of the way.
  // One candidate with X < -2 beta is certainly accepted; X > 2 beta for
  // the smallest X is certainly a reject.  Near the threshold, or
  // otherwise, the exact path decides.
  const double mg = 2.0 * beta;
  const bool near = A.thr > 0.0 && !(fest + xmin > A.thr * A.thr * 1.01);
  int kind = -1;
  if (pfm != 0 && !near) {
    if (nc == 1 && xmin + mg < 0.0) kind = 2;
    else if (xmin - mg > 0.0) kind = 0;
  }
  if (kind == -1 && pfm == 2) {  // the exact path compares with prev_fit
    prev_fit = current_fitness<KMAX, EXACT>(A, T, lane);
    pfm = 1;
  }
  if (kind == 0) {
    if (lane == 0) T.sh->res_kind = 0;
    return;
  }
  for (int c0 = 0; c0 < nc; c0 += cpc) {
    int j = -1;
    if (nc == 1)  // the usual case: the candidate came with the filter's ballot
      j = (lane < GS) ? jfirst : -1;
    else if (lane < cpc * GS && c0 + c < nc)
      j = T.cl[c0 + c];
    int a = 0, b = 0;
    double nA = 0.0, nB = 0.0;
    if (j >= 0) {
      const int2 pr = T.prop[j];  // only the rare replay path reads the sites
      const int w = s * task + j;
      const WalkRec r = walk_unpack(T.WC[w]);
      a = r.a;
      b = r.b;
      exact_entries<KMAX>(A, T, sp, s, pr.x, pr.y, a, b, x, T.WA[w], T.WB[w], r.c11, r.c12,
                          r.c21, r.c22, nA, nB);
      slot[0] = nA;
      slot[1] = nB;
      if (kind != 2) {  // alphas feed the terms, which a decided accept skips
        slot[2] = 1.0 - nA / (T.conc[a] * T.conc[x]);
        slot[3] = 1.0 - nB / (T.conc[b] * T.conc[x]);
      }
    }
    wave_sync();
    if (kind == 2) {  // the one candidate is accepted: its new rows only
      if (j >= 0) {
        T.G[T.idx(s, a, x)] = nA;
        T.G[T.idx(s, x, a)] = nA;
        T.G[T.idx(s, b, x)] = nB;
        T.G[T.idx(s, x, b)] = nB;
      }
      bj = jfirst;
      ra = a;
      rb = b;
      break;
    }
    if (j >= 0) {  // terms of row x (accelerate.cpp:560-566)
      const double* tg = T.tgt + T.idx(s, x, 0);
      const double* e0 = T.E0 + T.idx(s, x, 0);
      const double sAx = slot[2], sBx = slot[3];
#pragma unroll
      for (int y = 0; y < KMAX; ++y) {
        if (EXACT || y < K) {
          const bool chg = (x == a) || (x == b) || (y == a) || (y == b);
          const double sro = (x == a)   ? grp[y * XW + 2]
                             : (x == b) ? grp[y * XW + 3]
                             : (y == a) ? sAx
                                        : sBx;
          const double df = sro - tg[y];
          slot[4 + y] = chg ? df * df : e0[y];
        }
      }
    }
    wave_sync();
    if (j >= 0 && x == 0) {  // the shell's K*K terms in row-major order
      double es = 0.0;
#pragma unroll
      for (int i = 0; i < KMAX; ++i)
#pragma unroll
        for (int y = 0; y < KMAX; ++y)
          if (EXACT || (i < K && y < K)) es = es + grp[i * XW + 4 + y];
      T.ex[g] = es;
    }
    wave_sync();
    unsigned long long rk = ~0ull;
    int rj = 0x7fffffff, rc = 0;
    if (j >= 0 && s == 0 && x == 0) {
      double err = 0.0;
      for (int t = 0; t < S; ++t) err = err + A.weight[t] * T.ex[c * S + t];
      rk = (unsigned long long)__double_as_longlong(sqrt(err));
      rj = j;
      rc = c;
    }
    if (nc - c0 == 1) {  // the usual case: one candidate, in lane 0
      rk = ((unsigned long long)(uint32_t)__builtin_amdgcn_readfirstlane((int)(rk >> 32)) << 32) |
           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)rk);
      rj = __builtin_amdgcn_readfirstlane(rj);
      rc = 0;
    } else {
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) {
        const unsigned long long ok =
            ((unsigned long long)(uint32_t)__shfl_xor((int)(rk >> 32), m) << 32) |
            (uint32_t)__shfl_xor((int)(uint32_t)rk, m);
        const int oj = __shfl_xor(rj, m);
        const int oc = __shfl_xor(rc, m);
        if (key_less(ok, oj, rk, rj)) {
          rk = ok;
          rj = oj;
          rc = oc;
        }
      }
    }
    if (key_less(rk, rj, bk, bj)) {
      bk = rk;
      bj = rj;
      bc = rc;
      wc0 = c0;
    }
    if (c0 + cpc < nc) wave_sync();  // the next chunk reuses xw and ex
  }
  if (kind == 2) {
    if (reset && lane < HEA_MAX_S) {  // the refresh below takes new maxima
      T.sh->bmax[lane] = 0ull;
      T.sh->ubmax[lane] = 0ull;
    }
    if (lane == 0) {
      if (reset) T.sh->gmax = 0u;
      T.sh->res_kind = 2;
      T.sh->res_j = bj;
      T.sh->res_a = ra;
      T.sh->res_b = rb;
      T.sh->pfm = 2;
      T.sh->fest = fest + xmin;
    }
    return;
  }
  const double best_fit = __longlong_as_double((long long)bk);
  int a = 0, b = 0;
  if (best_fit < prev_fit) {  // accept: write the winner's rows
    const int2 pr = T.prop[bj];
    {
      const WalkRec r = walk_unpack(T.WC[bj]);  // shell 0's walk holds the species
      a = r.a;
      b = r.b;
    }
    if (wc0 + cpc < nc) {  // a later chunk overwrote the winner's entries
      if (lane < GS) {
        const int w = s * task + bj;
        const WalkRec r = walk_unpack(T.WC[w]);
        double nA, nB;
        exact_entries<KMAX>(A, T, sp, s, pr.x, pr.y, a, b, x, T.WA[w], T.WB[w], r.c11,
                            r.c12, r.c21, r.c22, nA, nB);
        slot[0] = nA;
        slot[1] = nB;
      }
      bc = 0;
    }
    wave_sync();
    // rows a and b of every shell, with their mirrors (columns a and b)
    for (int e = lane; e < S * 2 * K; e += 64) {
      const int t = e / (2 * K), h = (e / K) & 1, y = e % K;
      const double v = T.xw[((bc * S + t) * K + y) * XW + h];
      const int r = h ? b : a;
      T.G[T.idx(t, r, y)] = v;
      T.G[T.idx(t, y, r)] = v;
    }
    if (reset && lane < HEA_MAX_S) {  // the refresh below takes new maxima
      T.sh->bmax[lane] = 0ull;
      T.sh->ubmax[lane] = 0ull;
    }
    if (reset && lane == 0) T.sh->gmax = 0u;
  }
  if (lane == 0) {
    const bool acc1 = best_fit < prev_fit;
    T.sh->res_kind = acc1 ? 1 : 0;
    T.sh->res_key = bk;
    T.sh->res_j = bj;
    T.sh->res_a = a;
    T.sh->res_b = b;
    T.sh->pf = acc1 ? best_fit : prev_fit;
    T.sh->pfm = acc1 ? 1 : pfm;
    if (acc1) T.sh->fest = best_fit * best_fit;
  }
}

}  // namespace
