// Neighbour walks of stencil lattices whose species sit in LDS: a site's
// neighbours' ids from its coordinates (hea_stencil.h), their species gathered
// from LDS, and the shells' species histograms.
#pragma once
#include <type_traits>

#include "hea_exact.h"
#include "hea_screen.h"
#include "hea_stencil.h"

namespace {

// The species in LDS.  Bytes hold the histogram shift W x species, so that a
// gathered byte is a shift amount; lattices beyond that hold species x two a
// byte (site i in nibble i & 1 of byte i >> 1), which costs two more
// instructions per neighbour and reaches twice the sites.
template <bool NIB, int W>
struct Species {
  uint8_t* p;
  static __host__ __device__ __forceinline__ size_t bytes(int n) {
    return NIB ? ((size_t)n + 1) / 2 : (size_t)n;
  }
  // species as stored, equal iff the species are, and back
  __device__ __forceinline__ int code(uint32_t i) const {
    return NIB ? (p[i >> 1] >> (4 * (i & 1u))) & 15 : (int)p[i];
  }
  static __device__ __forceinline__ int code_of(int x) { return NIB ? x : W * x; }
  static __device__ __forceinline__ int species_of(int c) {
    return NIB ? c : W == 8 ? c >> 3 : (c * 205) >> 10;  // c / 5 for codes below 64
  }
  __device__ __forceinline__ int operator[](int i) const { return species_of(code((uint32_t)i)); }
  // one lane at a time: two sites may share a byte
  __device__ __forceinline__ void set(int i, int x) const {
    if (NIB) {
      const int sh = 4 * (i & 1);
      p[i >> 1] = (uint8_t)((p[i >> 1] & (15 << (4 - sh))) | (x << sh));
    } else {
      p[i] = (uint8_t)(W * x);
    }
  }
};

// m += 1 << s: one v_lshl_add_u32 (the compiler does not form it from a shift
// of the constant 1).
__device__ __forceinline__ void count_species(uint32_t& m, uint32_t s) {
  asm("v_lshl_add_u32 %0, 1, %1, %0" : "+v"(m) : "v"(s));
}
__device__ __forceinline__ void count_species(uint64_t& m, uint32_t s) { m += 1ull << s; }
// The same for a shift in the low byte of s: the instruction takes the low five
// (six) bits, and the shifts of species stay below.
__device__ __forceinline__ void count_species_low(uint32_t& m, uint32_t s) { count_species(m, s); }
__device__ __forceinline__ void count_species_low(uint64_t& m, uint32_t s) { m += 1ull << (s & 63u); }

// x + y + z in one instruction (left to itself the compiler shares pair sums
// and needs half as many again).
__device__ __forceinline__ uint32_t add3(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t r;
  asm("v_add3_u32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
  return r;
}

using LdsByte = const __attribute__((address_space(3))) uint8_t;
__device__ __forceinline__ uint32_t lds_addr(const uint8_t* p) {
  return (uint32_t)(uintptr_t)(LdsByte*)p;
}

// LDS addresses' terms of one site's neighbours on each axis; two species a
// byte: half the ids, and the nibble's bit of a neighbour an even or an odd
// step away on the axis that holds bit 0 of the ids.
struct SiteTerms {
  int f[3][5];
  int bit[2];
};
template <int LT, bool NIB>
__device__ __forceinline__ SiteTerms site_terms(const HeaCellSite& c, int L, uint32_t sp) {
  SiteTerms t;
  hea_axis_terms<LT, 0, NIB>(c.c[0], c.p[0], L, t.f[0]);
  hea_axis_terms<LT, 1, NIB>(c.c[1], c.p[1], L, t.f[1]);
  hea_axis_terms<LT, 2, NIB>(c.c[2], c.p[2], L, t.f[2]);
#pragma unroll
  for (int k = 0; k < 5; ++k) t.f[0][k] += (int)sp;
  if constexpr (NIB) {
    t.bit[0] = 4 * c.p[HeaShells<LT>::BIT0];
    t.bit[1] = 4 - t.bit[0];
  }
  return t;
}
template <int LT, int SHELL>
__device__ __forceinline__ void load_shell(const SiteTerms& t, uint32_t* v) {
  int n = 0;
#pragma unroll
  for (int dx = -2; dx <= 2; ++dx)
#pragma unroll
    for (int dy = -2; dy <= 2; ++dy)
#pragma unroll
      for (int dz = -2; dz <= 2; ++dz)
        if (HeaShells<LT>::shell(dx, dy, dz) == SHELL)
          v[n++] = *(LdsByte*)(uintptr_t)add3((uint32_t)t.f[0][dx + 2], (uint32_t)t.f[1][dy + 2],
                                              (uint32_t)t.f[2][dz + 2]);
}
template <int KMAX, int LT, int SHELL, bool NIB>
__device__ __forceinline__ void count_shell(const SiteTerms& t, const uint32_t* v,
                                            typename Pack<KMAX>::T& m) {
  int n = 0;
#pragma unroll
  for (int dx = -2; dx <= 2; ++dx)
#pragma unroll
    for (int dy = -2; dy <= 2; ++dy)
#pragma unroll
      for (int dz = -2; dz <= 2; ++dz)
        if (HeaShells<LT>::shell(dx, dy, dz) == SHELL) {
          uint32_t x = v[n++];
          if constexpr (NIB) {
            const int d = HeaShells<LT>::BIT0 == 1 ? dy : dz;
            x = (uint32_t)Pack<KMAX>::W * __builtin_amdgcn_ubfe(x, (uint32_t)t.bit[d & 1], 4);
          }
          count_species(m, x);
        }
}

// ---- walks by cell: both FCC shell sets ----
//
// The four sites of a cell are the four bytes (or nibbles) of one LDS word, and
// the 42 (30) neighbours of a site lie in 20 (19) cells, those of the first two
// shells, 18, in 10 and the first's 12 in 7: one load per cell
// instead of one per neighbour, and one instruction more per neighbour.  The walk
// is bound by LDS: bytes at random addresses, 6 to 7 cycles a load with their
// bank conflicts, kept it busy 56 % of a search of 108000 sites.  That search
// takes 95.6 ms, 106.5 by neighbour (512 proposals a round); 256000 sites two a
// byte 214.8, 232.0; 4000 sites of 30 neighbours 3.54, 3.65.  BCC's 26
// neighbours lie in 20 cells of two sites, which gains nothing.
// Seen from a site of odd parity on an axis the cells are
// mirrored on it, so with k the mirrored cell of a (mirrored) step d,
//     k = -1, -1, 0, 0, 1 for d = -2 .. 2,
// every lane needs the same cells; the neighbour is site b ^ m of its cell, b the
// site's own number and m the parities of the step.
struct CellTerms {
  uint32_t g[3][3];  // address terms of cells -1, 0, 1 (mirrored) on each axis
  uint32_t sh[4];    // bit of site b ^ m in its cell's word
};
__host__ __device__ constexpr int step_cell(int d) { return d < 0 ? -1 : d > 1 ? 1 : 0; }
// Whether one of LT's first NS shells has a neighbour in cell (x, y, z).
template <int LT, int NS>
__host__ __device__ constexpr bool cell_used(int x, int y, int z) {
  for (int dx = -2; dx <= 2; ++dx)
    for (int dy = -2; dy <= 2; ++dy)
      for (int dz = -2; dz <= 2; ++dz)
        if (HeaShells<LT>::shell(dx, dy, dz) >= 0 && HeaShells<LT>::shell(dx, dy, dz) < NS &&
            step_cell(dx) == x && step_cell(dy) == y && step_cell(dz) == z)
          return true;
  return false;
}
template <bool NIB>
__device__ __forceinline__ CellTerms cell_terms(const HeaCellSite& c, int L, uint32_t sp) {
  constexpr int CB = NIB ? 2 : 4;  // bytes of a cell
  CellTerms t;
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const int A = x == 0 ? CB * L * L : x == 1 ? CB * L : CB;
    const int at = hea_mul24(A, c.c[x]), span = A * (L - 1);
    const int up = c.c[x] == L - 1 ? at - span : at + A;
    const int dn = c.c[x] == 0 ? at + span : at - A;
    t.g[x][0] = (uint32_t)(c.p[x] ? up : dn);
    t.g[x][1] = (uint32_t)at;
    t.g[x][2] = (uint32_t)(c.p[x] ? dn : up);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) t.g[0][k] += sp;
  constexpr uint32_t B = NIB ? 4 : 8;  // bits of a site
  t.sh[0] = B * (uint32_t)(c.p[1] | (c.p[2] << 1));
#pragma unroll
  for (uint32_t m = 1; m < 4; ++m) t.sh[m] = t.sh[0] ^ (B * m);
  return t;
}
template <int LT, int NS, bool NIB>
__device__ __forceinline__ void load_cells(const CellTerms& t, uint32_t* w) {
  using Word = std::conditional_t<NIB, const __attribute__((address_space(3))) uint16_t,
                                  const __attribute__((address_space(3))) uint32_t>;
#pragma unroll
  for (int x = 0; x < 3; ++x)
#pragma unroll
    for (int y = 0; y < 3; ++y)
#pragma unroll
      for (int z = 0; z < 3; ++z)
        if (cell_used<LT, NS>(x - 1, y - 1, z - 1))
          w[(x * 3 + y) * 3 + z] = *(Word*)(uintptr_t)add3(t.g[0][x], t.g[1][y], t.g[2][z]);
}
template <int KMAX, int LT, int NS, bool NIB>
__device__ __forceinline__ void count_cells(const CellTerms& t, const uint32_t* w,
                                            typename Pack<KMAX>::T* m) {
#pragma unroll
  for (int dx = -2; dx <= 2; ++dx)
#pragma unroll
    for (int dy = -2; dy <= 2; ++dy)
#pragma unroll
      for (int dz = -2; dz <= 2; ++dz) {
        const int s = HeaShells<LT>::shell(dx, dy, dz);
        if (s >= 0 && s < NS) {
          const uint32_t c = w[((step_cell(dx) + 1) * 3 + step_cell(dy) + 1) * 3 + step_cell(dz) + 1];
          const uint32_t bit = t.sh[(dy & 1) | ((dz & 1) << 1)];
          if constexpr (NIB)
            count_species(m[s], (uint32_t)Pack<KMAX>::W * __builtin_amdgcn_ubfe(c, bit, 4));
          else
            count_species_low(m[s], c >> bit);
        }
      }
}

// Species histograms m of a site's first NS shells.
template <int KMAX, int LT, int NS, bool NIB>
__device__ __forceinline__ void walk_cells(const HeaCellSite& c, int L, uint32_t sp,
                                           typename Pack<KMAX>::T* m) {
  const CellTerms t = cell_terms<NIB>(c, L, sp);
  uint32_t w[27];
  load_cells<LT, NS, NIB>(t, w);
  __builtin_amdgcn_sched_barrier(0);
  count_cells<KMAX, LT, NS, NIB>(t, w, m);
}

}  // namespace
