// Neighbour walks of stencil lattices whose species sit in LDS: a site's
// neighbours' ids from its coordinates (hea_stencil.h), their species gathered
// from LDS, and the shells' species histograms.
#pragma once
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

}  // namespace
