// Periodic FCC and BCC supercells whose neighbour table is the translation
// stencil of pyhea/lattice/lattice.py (:207-221, 272-287): site ids
// NB ((x L + y) L + z) + loc (lattice.py:105, 142) and shells of all
// lattice vectors of one length.  For such a table a site's neighbours follow
// from its coordinates by a few additions, and whether two sites are
// neighbours from their distance, so the kernels need no table rows.  The
// host compares a problem's whole table with the stencil before it is used
// (hea_stencil_detect); any other table keeps the kernels that read rows.
//
// In half-lattice units a site has coordinates (X, Y, Z) modulo 2L, with
// loc fixed by their parities, and the id is a sum of one term per axis,
//   id = f0(X) + f1(Y) + f2(Z),   f_d(V) = A_d (V >> 1) + B_d (V & 1),
// A = NB (L^2, L, 1); FCC B = (0, 1, 2) (basis order (0,0,0) (1,1,0) (1,0,1)
// (0,1,1), lattice.py:167-190), BCC B = (0, 0, 1).
#pragma once
#include <stdint.h>

#include <vector>

#if defined(__HIPCC__)
#define HEA_ST_HD __host__ __device__ __forceinline__
#else
#define HEA_ST_HD static inline
#endif

// Shell sets (values of HeaMcArgs::lt): FCC 12/6/24 (<110>/2, <100>,
// <211>/2), FCC 12/6/12 (the reference's third shell <110>), BCC 8/6/12.
enum { HEA_LT_NONE = 0, HEA_LT_FCC = 1, HEA_LT_FCC_REF = 2, HEA_LT_BCC = 3 };

// L is at least 3, so that the vectors of up to two half units are distinct
// modulo 2L and two sites have one minimum-image difference, and at most 255
// (hea_cell_div is exact for quotients below L^3 then).
#define HEA_ST_MIN_L 3
#define HEA_ST_MAX_L 255

template <int LT>
struct HeaShells {
  static constexpr bool BCC = LT == HEA_LT_BCC;
  static constexpr int LG = BCC ? 1 : 2, NB = 1 << LG;  // sites per cell
  static constexpr int BIT0 = BCC ? 2 : 1;  // the axis whose parity is bit 0 of the ids
  // squared length of each shell's vectors (half units) and their number
  static constexpr int D2[3] = {BCC ? 3 : 2, 4, LT == HEA_LT_FCC ? 6 : 8};
  static constexpr int Z[3] = {BCC ? 8 : 12, 6, LT == HEA_LT_FCC ? 24 : 12};
  // shell of the vector (dx, dy, dz), or -1
  static constexpr int shell(int dx, int dy, int dz) {
    const int n2 = dx * dx + dy * dy + dz * dz;
    const bool on = BCC ? (((dx ^ dy) | (dy ^ dz)) & 1) == 0 : ((dx + dy + dz) & 1) == 0;
    return !on ? -1 : n2 == D2[0] ? 0 : n2 == D2[1] ? 1 : n2 == D2[2] ? 2 : -1;
  }
};

// n / L for n < L^3, L <= 255: magic = 2^32 / L + 1 is off by e = magic L -
// 2^32 in (0, L], and n e < L^4 < 2^32.
HEA_ST_HD uint32_t hea_cell_magic(int L) { return (uint32_t)((1ull << 32) / (uint64_t)L) + 1u; }
HEA_ST_HD uint32_t hea_cell_div(uint32_t n, uint32_t magic) {
  return (uint32_t)(((uint64_t)n * magic) >> 32);
}

// The same in three full-rate instructions for n < 2^22 - 1, inv = fl(1 / L):
// n + 1/2 is exact, the product is off by less than (n + 1/2) / L 2^-22.9,
// and (n + 1/2) / L lies at least 1 / (2 L) from an integer.
HEA_ST_HD uint32_t hea_cell_div_small(uint32_t n, float inv) {
  return (uint32_t)(((float)n + 0.5f) * inv);
}

// Product of factors below 2^24 (a full-rate instruction on the GPU).
HEA_ST_HD int hea_mul24(int a, int b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (int)__umul24((unsigned)a, (unsigned)b);
#else
  return a * b;
#endif
}

// Cell and parity of a site on each axis.
struct HeaCellSite {
  int c[3], p[3];
};
template <int LT, class Div>
HEA_ST_HD HeaCellSite hea_cell_site(int site, int L, const Div& div) {
  using ST = HeaShells<LT>;
  HeaCellSite s;
  const uint32_t cell = (uint32_t)site >> ST::LG;
  const int loc = site & (ST::NB - 1);
  const uint32_t q = div(cell);
  s.c[0] = (int)div(q);
  s.c[1] = (int)q - hea_mul24(s.c[0], L);
  s.c[2] = (int)cell - hea_mul24((int)q, L);
  s.p[1] = loc & 1;
  s.p[2] = ST::BCC ? loc : loc >> 1;
  s.p[0] = ST::BCC ? loc : s.p[1] ^ s.p[2];
  return s;
}

// f_d(V + d) for d = -2..2 of one axis at cell c and parity p; HALVED: of
// id >> 1 (every term but bit 0 is even).
template <int LT, int AXIS, bool HALVED = false>
HEA_ST_HD void hea_axis_terms(int c, int p, int L, int* f) {
  using ST = HeaShells<LT>;
  constexpr int B = (ST::BCC ? (AXIS == 2) : AXIS) >> (HALVED ? 1 : 0);
  constexpr int NB = ST::NB >> (HALVED ? 1 : 0);
  const int A = AXIS == 0 ? NB * L * L : AXIS == 1 ? NB * L : NB;
  const int at = hea_mul24(A, c), span = A * (L - 1);
  const int up = c == L - 1 ? at - span : at + A;
  const int dn = c == 0 ? at + span : at - A;
  f[0] = dn + B * p;
  f[2] = at + B * p;
  f[4] = up + B * p;
  f[1] = (p ? at : dn) + B * (1 - p);
  f[3] = (p ? up : at) + B * (1 - p);
}

// Squared minimum-image distance (half units) of two sites.
HEA_ST_HD int hea_cell_dist2(const HeaCellSite& s, const HeaCellSite& t, int L) {
  int d2 = 0;
  for (int k = 0; k < 3; ++k) {
    int d = 2 * (s.c[k] - t.c[k]) + s.p[k] - t.p[k];
    d = d < 0 ? -d : d;
    d = d < 2 * L - d ? d : 2 * L - d;
    d2 += d * d;
  }
  return d2;
}

// Whether columns [0, sum Z) of nbr [N][sum Z] are the stencil of shell set
// LT (its first S shells) on an L^3 supercell; host only.
template <int LT>
static bool hea_stencil_matches(const int32_t* nbr, int N, int S, const int32_t* Z, int L) {
  using ST = HeaShells<LT>;
  if (N != ST::NB * L * L * L || L < HEA_ST_MIN_L || L > HEA_ST_MAX_L) return false;
  int sumZ = 0;
  for (int s = 0; s < S; ++s) {
    if (Z[s] != ST::Z[s]) return false;
    sumZ += Z[s];
  }
  // every site's coordinates, 10 bits each
  const uint32_t magic = hea_cell_magic(L);
  const auto div = [magic](uint32_t n) { return hea_cell_div(n, magic); };
  std::vector<uint32_t> at(N);
  for (int i = 0; i < N; ++i) {
    const HeaCellSite c = hea_cell_site<LT>(i, L, div);
    at[i] = (uint32_t)(2 * c.c[0] + c.p[0]) | ((uint32_t)(2 * c.c[1] + c.p[1]) << 10) |
            ((uint32_t)(2 * c.c[2] + c.p[2]) << 20);
  }
  // coordinate difference + 2L -> minimum-image difference + 2, or 125 when
  // it is beyond two units; the three axes' digits in base 5 name a vector
  std::vector<uint8_t> digit(4 * L + 1, 125);
  for (int d = -2 * L + 1; d < 2 * L; ++d) {
    const int m = d > L ? d - 2 * L : d < -L ? d + 2 * L : d;
    if (m >= -2 && m <= 2) digit[d + 2 * L] = (uint8_t)(m + 2);
  }
  int8_t shell[125];
  for (int v = 0; v < 125; ++v) shell[v] = (int8_t)ST::shell(v / 25 - 2, v / 5 % 5 - 2, v % 5 - 2);
  for (int i = 0; i < N; ++i) {
    const int32_t* row = nbr + (size_t)i * sumZ;
    const int x = (int)(at[i] & 1023u) - 2 * L, y = (int)((at[i] >> 10) & 1023u) - 2 * L,
              z = (int)(at[i] >> 20) - 2 * L;
    // a list of Z distinct sites at the shell's vectors holds all of them
    uint64_t seen[2] = {0, 0};
    for (int s = 0, k = 0; s < S; ++s) {
      for (const int end = k + Z[s]; k < end; ++k) {
        const uint32_t t = at[row[k]];
        const unsigned v = 25u * digit[(int)(t & 1023u) - x] +
                           5u * digit[(int)((t >> 10) & 1023u) - y] + digit[(int)(t >> 20) - z];
        if (v >= 125u || shell[v] != s || (seen[v >> 6] >> (v & 63u) & 1u)) return false;
        seen[v >> 6] |= 1ull << (v & 63u);
      }
    }
  }
  return true;
}

// Shell set and edge of a table [N][sum Z] (entries in [0, N)), or
// HEA_LT_NONE.
static inline int hea_stencil_detect(const int32_t* nbr, int N, int S, const int32_t* Z, int* edge) {
  for (int lt = HEA_LT_FCC; lt <= HEA_LT_BCC; ++lt) {
    const int nb = lt == HEA_LT_BCC ? 2 : 4;
    for (int L = HEA_ST_MIN_L; L <= HEA_ST_MAX_L; ++L) {
      if ((int64_t)nb * L * L * L != N) continue;
      const bool ok = lt == HEA_LT_FCC       ? hea_stencil_matches<HEA_LT_FCC>(nbr, N, S, Z, L)
                      : lt == HEA_LT_FCC_REF ? hea_stencil_matches<HEA_LT_FCC_REF>(nbr, N, S, Z, L)
                                             : hea_stencil_matches<HEA_LT_BCC>(nbr, N, S, Z, L);
      if (ok) {
        *edge = L;
        return lt;
      }
    }
  }
  return HEA_LT_NONE;
}
