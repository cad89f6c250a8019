// Build-time check (compiled by accy_amd/build.py with hipcc --offload-arch=gfx950): instantiates the
// scatter template with the row shapes the planner emits, so that a host without a GPU still
// verifies that it compiles for CDNA4. Nothing calls these kernels.
#include "common.h"
#include "scatter.h"

template <class IT, int V, int THREADS, int GROUPS, int L, int PL, long N, long ROWS, long WIDTH>
struct CheckTable {
  const float* in;
  const i32_t* ids;
  const float* up;
  float* out;
  typedef IT I;
  typedef float T;
  static constexpr long NI = N, EXT = ROWS, POST = WIDTH, PRE = 2;
  static constexpr int VEC = V, TC = THREADS, KG = GROUPS, LOOP = L, PLOOP = PL;
  static __device__ __forceinline__ T plus(T a, T u) { return a + u; }
  __device__ __forceinline__ I index(I j) const { return (I)ids[j]; }
  __device__ __forceinline__ void init(I p, I k, I c0, T (&v)[VEC]) const {
    for (int u = 0; u < VEC; ++u) v[u] = in[(p * EXT + k) * POST + c0 + u];
  }
  __device__ __forceinline__ void again(I p, I k, I c0, T (&v)[VEC]) const {
    for (int u = 0; u < VEC; ++u) v[u] = out[(p * EXT + k) * POST + c0 + u];
  }
  __device__ __forceinline__ void update(I p, I j, I c0, T (&v)[VEC]) const {
    for (int u = 0; u < VEC; ++u) v[u] = up[(p * NI + j) * POST + c0 + u];
  }
  __device__ __forceinline__ void store(I p, I k, I c0, const T (&v)[VEC]) const {
    for (int u = 0; u < VEC; ++u) out[(p * EXT + k) * POST + c0 + u] = v[u];
  }
};

extern "C" __global__ void __launch_bounds__(256) check_scatter_wide(CheckTable<i32_t, 4, 256, 1, 1, 1, 4096, 32000, 1024> t) {
  accy::scatter::rows(t);
}
extern "C" __global__ void __launch_bounds__(256) check_scatter_narrow(CheckTable<i64_t, 1, 4, 64, 8, 1, 100000, 50000, 3> t) {
  accy::scatter::rows(t);
}
extern "C" __global__ void __launch_bounds__(256) check_scatter_positions(CheckTable<i32_t, 1, 1, 2, 1, 4, 64, 8, 1> t) {
  accy::scatter::rows(t);
}
