// Attention of one query per batch index (a decode step): O[b] = softmax(scale * q[b] K[b]^T) V[b] in one
// pass over K and V, f32 scores, softmax and sums.
//
// Every key and value row is used once, so the rate of reading them bounds it (128 heads x 4096 keys x 128
// bf16 are 268 MB: 41 us at 6.5 TB/s) and the matrix cores, which compute 32 queries at a time, have nothing to
// add. LPK = HD / VEC adjacent lanes read a row 16 bytes each; a wave takes 64 / LPK rows per load and U
// loads of K and of V ahead of their arithmetic, 16 KiB in flight. Each group of LPK lanes keeps its own
// running maximum, sum and output (rescaled per U rows); the groups of a wave meet through shuffles, the
// waves through LDS, the workgroups that share a batch index's keys (SPLITS of them, PER rows each)
// through memory and a second kernel (join). (As two contractions of one row, a softmax kernel and a
// split's sum: 60 us for the above, now 46, 5.8 TB/s.)
//
// C supplies DT (0 bf16, 1 f16, 2 f32), HD, SK, NB, SPLITS, PER (a multiple of STEP), K_S and V_S (row strides in
// elements), SL = scale * log2 e and q_off / k_off / v_off (batch offsets; head dims have stride 1, rows are
// 16-byte aligned). The output is row-major [b][HD]; partial results are [b][split][m, l, HD outputs].
#pragma once

namespace accy {
namespace decode {

typedef u32_t u32x4 __attribute__((ext_vector_type(4)));

template <int DT> struct Elem { typedef u16_t type; static constexpr int VEC = 8; };
template <> struct Elem<2> { typedef float type; static constexpr int VEC = 4; };

template <int DT> __device__ __forceinline__ float elem(u32x4 w, int i) {
  if constexpr (DT == 0) return __builtin_bit_cast(float, i & 1 ? w[i >> 1] & 0xffff0000u : w[i >> 1] << 16);
  else if constexpr (DT == 1) return f16_to_f32((u16_t)(w[i >> 1] >> (16 * (i & 1))));
  else return __builtin_bit_cast(float, (u32_t)w[i]);
}

template <class C> constexpr int lanes_per_key() { return C::HD / Elem<C::DT>::VEC; }
constexpr int WAVES = 4, U = 8;  // rows per lane group and step
template <class C> constexpr int step_keys() { return WAVES * U * (64 / lanes_per_key<C>()); }

template <bool V> struct Flag { static constexpr bool value = V; };

// The exponent's base for a running maximum: nothing is subtracted while every score is -inf.
__device__ __forceinline__ float base_of(float m) { return m == -__builtin_inff() ? 0.0f : m; }

template <class C>
__device__ __forceinline__ void store_out(typename Elem<C::DT>::type* __restrict__ out, long i, float v) {
  if constexpr (C::DT == 0) out[i] = f32_to_bf16(v);
  else if constexpr (C::DT == 1) out[i] = f32_to_f16(v);
  else out[i] = v;
}

template <class C, class T = typename Elem<C::DT>::type>
__device__ __forceinline__ void attend(const T* __restrict__ Q, const T* __restrict__ K, const T* __restrict__ V,
                                       T* __restrict__ out, float* __restrict__ part) {
  constexpr int VEC = Elem<C::DT>::VEC, LPK = lanes_per_key<C>(), KPW = 64 / LPK, STEP = step_keys<C>();
  static_assert(C::PER % STEP == 0 && LPK >= 1 && LPK <= 64 && (LPK & (LPK - 1)) == 0, "whole steps, whole lane groups");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane / LPK, d0 = (lane % LPK) * VEC;
  const long b = blockIdx.x, split = blockIdx.y;
  const u32x4 qw = *(const u32x4*)(Q + C::q_off(b) + d0);
  const T* __restrict__ kp = K + C::k_off(b) + d0;
  const T* __restrict__ vp = V + C::v_off(b) + d0;
  float q[VEC], acc[VEC], m = -__builtin_inff(), l = 0.0f;
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    q[i] = elem<C::DT>(qw, i) * C::SL;
    acc[i] = 0.0f;
  }
  const long first = split * C::PER, end = first + C::PER < C::SK ? first + C::PER : C::SK;
  auto step = [&](long k0, auto tail) {
    u32x4 kw[U], vw[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      long key = k0 + (wave * U + u) * KPW + g;
      if constexpr (decltype(tail)::value) key = key < C::SK ? key : C::SK - 1;
      kw[u] = __builtin_nontemporal_load((const u32x4*)(kp + key * C::K_S));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      long key = k0 + (wave * U + u) * KPW + g;
      if constexpr (decltype(tail)::value) key = key < C::SK ? key : C::SK - 1;
      vw[u] = __builtin_nontemporal_load((const u32x4*)(vp + key * C::V_S));
    }
    float s[U], mx = m;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[u] = 0.0f;
#pragma unroll
      for (int i = 0; i < VEC; ++i) s[u] = __builtin_fmaf(q[i], elem<C::DT>(kw[u], i), s[u]);
#pragma unroll
      for (int o = LPK / 2; o > 0; o >>= 1) s[u] += __shfl_xor(s[u], o, 64);
      if constexpr (decltype(tail)::value) {
        if (k0 + (wave * U + u) * KPW + g >= end) s[u] = -__builtin_inff();
      }
      mx = fmaxf(mx, s[u]);
    }
    const float sub = base_of(mx), alpha = __builtin_amdgcn_exp2f(m - sub);
    m = mx;
    l *= alpha;
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float p = __builtin_amdgcn_exp2f(s[u] - sub);
      l += p;
      bool own = true;  // a row past the end repeats the last one and adds nothing, whatever it holds
      if constexpr (decltype(tail)::value) own = k0 + (wave * U + u) * KPW + g < end;
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[i] = __builtin_fmaf(p, own ? elem<C::DT>(vw[u], i) : 0.0f, acc[i]);
    }
  };
  long k0 = first;
  for (; k0 + STEP <= end; k0 += STEP) step(k0, Flag<false>{});
  if (C::SK % STEP != 0 && k0 < end) step(k0, Flag<true>{});

  // the lane groups of the wave
#pragma unroll
  for (int o = LPK; o < 64; o <<= 1) {
    const float mo = __shfl_xor(m, o, 64), lo = __shfl_xor(l, o, 64), mx = fmaxf(m, mo), sub = base_of(mx);
    const float a = __builtin_amdgcn_exp2f(m - sub), c = __builtin_amdgcn_exp2f(mo - sub);
    m = mx;
    l = l * a + lo * c;
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[i] = acc[i] * a + __shfl_xor(acc[i], o, 64) * c;
  }
  // the waves
  __shared__ float ms[WAVES], ls[WAVES], os[WAVES][C::HD];
  if (lane == 0) {
    ms[wave] = m;
    ls[wave] = l;
  }
  if (lane < LPK)
#pragma unroll
    for (int i = 0; i < VEC; ++i) os[wave][d0 + i] = acc[i];
  __syncthreads();
  m = ms[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) m = fmaxf(m, ms[w]);
  const float sub = base_of(m);
  float scale[WAVES];
  l = 0.0f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) {
    scale[w] = __builtin_amdgcn_exp2f(ms[w] - sub);
    l += ls[w] * scale[w];
  }
  for (int d = threadIdx.x; d < C::HD; d += 64 * WAVES) {
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) o += os[w][d] * scale[w];
    if constexpr (C::SPLITS == 1) {
      store_out<C>(out, b * C::HD + d, o / l);
    } else {
      float* const p = part + (b * C::SPLITS + split) * (C::HD + 2);
      p[2 + d] = o;
      if (d == 0) {
        p[0] = m;
        p[1] = l;
      }
    }
  }
}

// O[b] from its splits' parts, in split order; one thread per output.
template <class C, class T = typename Elem<C::DT>::type>
__device__ __forceinline__ void join(const float* __restrict__ part, T* __restrict__ out) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long)C::NB * C::HD) return;
  const float* const p = part + i / C::HD * (C::SPLITS * (C::HD + 2));
  float m = -__builtin_inff(), l = 0.0f, o = 0.0f;
#pragma unroll 8
  for (int s = 0; s < C::SPLITS; ++s) m = fmaxf(m, p[s * (C::HD + 2)]);
  const float sub = base_of(m);
#pragma unroll 8
  for (int s = 0; s < C::SPLITS; ++s) {
    const float* const q = p + s * (C::HD + 2);
    const float scale = __builtin_amdgcn_exp2f(q[0] - sub);
    l += q[1] * scale;
    o += q[2 + i % C::HD] * scale;
  }
  store_out<C>(out, i, o / l);
}

}  // namespace decode
}  // namespace accy
