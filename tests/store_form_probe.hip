// One instance of every form of vector store in store_form.h, for tests/test_store_form.py to read in assembly.
#include "store_form.h"

using namespace cumo_hip;

extern "C" __global__ void probe_store_cached(store_u4* p, store_u4 v, bool pieces) { store_vector<false>(p + threadIdx.x, v, pieces); }
extern "C" __global__ void probe_store_streamed(store_u4* p, store_u4 v, bool pieces) { store_vector<true>(p + threadIdx.x, v, pieces); }
extern "C" __global__ void probe_tile_cached(store_u4* p, store_u4 v, bool pieces) { store_tile_vector<false>(p + threadIdx.x, v, pieces); }
extern "C" __global__ void probe_tile_streamed(store_u4* p, store_u4 v, bool pieces) { store_tile_vector<true>(p + threadIdx.x, v, pieces); }
