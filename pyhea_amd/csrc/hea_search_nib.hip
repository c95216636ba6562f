// The stencil-lattice search with two species a byte in LDS (hea_search.h).
#include "hea_search.h"

const void* hea_search_fn_nib(int lt, int K) { return search_fn<true>(lt, K); }
