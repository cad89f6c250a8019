// Build-time check (compiled by accy_amd/build.py with hipcc --offload-arch=gfx950): instantiates the
// single-query attention template with the shapes the planner emits, so that a host without a GPU
// still verifies that it compiles for CDNA4. Nothing calls these kernels.
#include "common.h"
#include "decode.h"

template <int D, int H, long KEYS, int S, long SHARE>
struct CheckDecode {
  static constexpr int DT = D, HD = H, SPLITS = S;
  static constexpr long SK = KEYS, NB = 128, PER = SHARE, K_S = H, V_S = H;
  static constexpr float SL = 0x1.05p-3f;
  static __device__ __forceinline__ long q_off(long b) { return b * HD; }
  static __device__ __forceinline__ long k_off(long b) { return b * SK * HD; }
  static __device__ __forceinline__ long v_off(long b) { return b * SK * HD; }
};

extern "C" __global__ void __launch_bounds__(256) check_decode_bf16(const u16_t* q, const u16_t* k, const u16_t* v, u16_t* o, float* p) {
  accy::decode::attend<CheckDecode<0, 128, 4096, 8, 512>>(q, k, v, o, p);
}
extern "C" __global__ void __launch_bounds__(256) check_decode_f16(const u16_t* q, const u16_t* k, const u16_t* v, u16_t* o, float* p) {
  accy::decode::attend<CheckDecode<1, 64, 301, 1, 512>>(q, k, v, o, p);
}
extern "C" __global__ void __launch_bounds__(256) check_decode_f32(const float* q, const float* k, const float* v, float* o, float* p) {
  accy::decode::attend<CheckDecode<2, 128, 301, 5, 64>>(q, k, v, o, p);
}
extern "C" __global__ void __launch_bounds__(256) check_decode_join(const float* p, u16_t* o) {
  accy::decode::join<CheckDecode<0, 128, 4096, 8, 512>>(p, o);
}
