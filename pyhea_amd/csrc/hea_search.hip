// Launches of the stencil-lattice search (hea_search.h): byte species, and the
// batched launch.  The kernels with two species a byte are instantiated in
// hea_search_nib.hip.
#include "hea_search.h"

const void* hea_search_fn_nib(int lt, int K);

namespace {

// One population each of many problems: workgroup i searches lattice
// items[i].y of problem items[i].x, longest first.  One launch for all of them,
// so that the tail of a phase is made of short searches.  Every species count has
// tables of its own width: padded to 4, 6 and 8 species an odd count paid a fifth
// more screen (uneven problems of 3 to 6 species: 61.3 -> 57.9 ms).
template <int LT>
__device__ __forceinline__ void search_item(const HeaMcArgs& A, int l, unsigned char* smem) {
  switch (A.K) {
    case 2: return search_lattice<2, true, LT, false>(A, l, smem);
    case 3: return search_lattice<3, true, LT, false>(A, l, smem);
    case 4: return search_lattice<4, true, LT, false>(A, l, smem);
    case 5: return search_lattice<5, true, LT, false>(A, l, smem);
    case 6: return search_lattice<6, true, LT, false>(A, l, smem);
    case 8: return search_lattice<8, true, LT, false>(A, l, smem);
    default: return search_lattice<8, false, LT, false>(A, l, smem);
  }
}

__global__ __launch_bounds__(kMaxSearchThreads, 4) void k_search_batch(
    const HeaMcArgs* __restrict__ probs, const int2* __restrict__ items) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int2 it = items[blockIdx.x];
  const HeaMcArgs& A = probs[it.x];
  if (A.lt == HEA_LT_FCC)
    search_item<HEA_LT_FCC>(A, it.y, smem);
  else if (A.lt == HEA_LT_FCC_REF)
    search_item<HEA_LT_FCC_REF>(A, it.y, smem);
  else
    search_item<HEA_LT_BCC>(A, it.y, smem);
}

size_t search_lds(int K, int task, size_t n) {
  switch (K) {
    case 2: return SearchLayout<2>(task, n).total;
    case 3: return SearchLayout<3>(task, n).total;
    case 4: return SearchLayout<4>(task, n).total;
    case 5: return SearchLayout<5>(task, n).total;
    case 6: return SearchLayout<6>(task, n).total;
    default: return SearchLayout<8>(task, n).total;
  }
}

}  // namespace

// Stencil lattices take this search up to 704 proposals (eleven worker waves, the
// most whose registers and the service wave's fit a workgroup), bytes where they
// fit (a nibble costs two instructions more per neighbour), else two species a byte:
// 1.5 to 3 times as fast as k_local_mc at every size measured, 108 to 270000 sites.
HeaSearchPlan hea_search_plan(const HeaConst& c, int lt, int task, int64_t max_lds, bool batch) {
  HeaSearchPlan p;
  if (lt == HEA_LT_NONE || task > kMaxSearchThreads - 64) return p;
  size_t lds = search_lds(c.K, task, Species<false, 5>::bytes(c.N));
  if ((int64_t)lds > max_lds && !batch) {  // two species a byte
    lds = search_lds(c.K, task, Species<true, 5>::bytes(c.N));
    p.nib = true;
  }
  if ((int64_t)lds > max_lds) return HeaSearchPlan();
  p.lds = lds;
  const int workers = (task + 63) & ~63;
  p.threads = workers + 64;
  // draw lanes (two draws each), with the margin of hea_mc_draw_lanes
  p.dl = std::min(workers, (hea_mc_draw_lanes(task, c.conc, c.K, 1 << 20) / 2 + 63) & ~63);
  return p;
}

hipError_t hea_prepare_search(int lt, int K, bool nib, size_t lds) {
  return hipFuncSetAttribute(nib ? hea_search_fn_nib(lt, K) : search_fn<false>(lt, K),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

hipError_t hea_launch_search(const HeaMcArgs& a, const HeaSearchPlan& p, hipStream_t st) {
  const void* fn = p.nib ? hea_search_fn_nib(a.lt, a.K) : search_fn<false>(a.lt, a.K);
  if (!fn) return hipErrorInvalidValue;
  void* args[] = {const_cast<HeaMcArgs*>(&a)};
  return hipLaunchKernel(fn, dim3(a.L), dim3(p.threads), args, p.lds, st);
}

hipError_t hea_prepare_search_batch(size_t lds) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(k_search_batch),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

hipError_t hea_launch_search_batch(const HeaMcArgs* probs, const int2* items, int n_items,
                                   int threads, size_t lds, hipStream_t st) {
  void* args[] = {&probs, &items};
  return hipLaunchKernel(reinterpret_cast<const void*>(k_search_batch), dim3(n_items),
                         dim3(threads), args, lds, st);
}
