// Products of a few activation rows with a packed weight: Gemm with 2 to 32
// rows (a batch of faces, a decode batch), and of one misaligned row.
#include "launch.hpp"

namespace ohip {

// One 16-byte fragment pair on the 16x16 MFMAs: lane l holds row l % 16, and
// of the K range its chunk l / 16.  The result holds, in lane l, rows
// 4 * (l / 16) .. + 3 of column l % 16.
template <Op O> struct Mma16;
template <> struct Mma16<Op::F16> {
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma16<Op::BF16> {
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <> struct Mma16<Op::F32> {   // element e of both chunks is k = 4 * (l / 16) + e
  static __device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(lane_f32(a.x), lane_f32(b.x), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(lane_f32(a.y), lane_f32(b.y), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(lane_f32(a.z), lane_f32(b.z), c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(lane_f32(a.w), lane_f32(b.w), c, 0, 0, 0);
    return c;
  }
};

// Bound: streaming the weight once (HBM), and one CU's share of it.  A block
// takes 16 weight rows; its eight waves split K (four: 12.1 against 8.5 us at
// 2x4096x4096 f16; sixteen: 1.7 us more a launch) and stream both operands
// straight from memory into MFMA fragments, 64 bytes of every row a step, so the 16 weight rows share every
// activation fragment (one row a block re-reads the activations from L2 for
// every weight row: M times the weight's bytes).  The waves' sums meet in LDS
// in wave order.  Activation rows need no alignment and no padding: a row's
// last, partial chunk is read element by element by the last wave.
constexpr int kSkinnyWaves = 8;

template <Op O, class T, int TM>
__global__ void __launch_bounds__(64 * kSkinnyWaves)
skinny_kernel(const T* __restrict__ a, int64_t lda, const T* __restrict__ w, int64_t ldw, int M, int N, int K,
              const u32x4* __restrict__ zeros, const FloatEpi<T> epi) {
  constexpr int E = 16 / (int)sizeof(T), U = TM == 1 ? 8 : 4;
  __shared__ f32x4 red[kSkinnyWaves][TM][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int kf = K / E;           // whole chunks of an activation row
  const int nst = (kf + 3) / 4;   // steps of four chunks a row
  const int per = (nst + kSkinnyWaves - 1) / kSkinnyWaves;
  const int s0 = wave * per, s1 = min(s0 + per, nst);
  const u32x4* wr = reinterpret_cast<const u32x4*>(w + (int64_t)min(n0 + r, N - 1) * ldw);
  const T* ar[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) ar[t] = a + (int64_t)min(t * 16 + r, M - 1) * lda;
  f32x4 acc[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  struct Batch { u32x4 w[U], a[U][TM]; };
  // no branch by lane, so the batch's loads leave together: a lane without a
  // chunk reads the zeros
  auto load = [&](Batch& f, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u < s1) {
        const int c = (s + u) * 4 + q;
        f.w[u] = *(c < kf ? wr + c : zeros);
#pragma unroll
        for (int t = 0; t < TM; ++t) {
          const void* p = c < kf && t * 16 + r < M ? static_cast<const void*>(ar[t] + (int64_t)c * E) : zeros;
          __builtin_memcpy(&f.a[u][t], p, 16);
        }
      } else {
        f.w[u] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int t = 0; t < TM; ++t) f.a[u][t] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  };
  auto sum = [&](const Batch& f) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < TM; ++t) acc[t] = Mma16<O>::mma(f.w[u], f.a[u][t], acc[t]);
  };
  for (int s = s0; s < s1; s += U) {
    Batch f;
    load(f, s);
    sum(f);
  }
  if (K % E != 0 && wave == kSkinnyWaves - 1) {   // the rows' last, partial chunk
    const u32x4 wv = *(q == 0 ? wr + kf : zeros);
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      T e[E];
#pragma unroll
      for (int k = 0; k < E; ++k) e[k] = q == 0 && t * 16 + r < M && kf * E + k < K ? ar[t][(int64_t)kf * E + k] : T(0);
      u32x4 av;
      __builtin_memcpy(&av, e, 16);
      acc[t] = Mma16<O>::mma(wv, av, acc[t]);
    }
  }
#pragma unroll
  for (int t = 0; t < TM; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= TM) return;
  f32x4 v = red[0][wave][lane];
#pragma unroll
  for (int k = 1; k < kSkinnyWaves; ++k) v += red[k][wave][lane];
  const int i = n0 + 4 * q, j = wave * 16 + r;
  if (j >= M) return;
  if (i >= N) return;
  typename FloatEpi<T>::PreI pi;
  typename FloatEpi<T>::PreJ pj;
  epi.load_i(pi, i);
  epi.load_j(pj, j);
  uint32_t bits[4];
  epi.finish(pi, pj, i, j, v, bits);
  const OutAddr out = epi.addr();
  store_group(out, epi.out_bytes(), out.row(i), i, j, bits);
}

template <Op O, class T>
static hipError_t skinny_t(const GemvArgs& g, int K, const void* zero16, const FloatOut& o, hipStream_t st) {
  const T* a = reinterpret_cast<const T*>(g.a);
  const T* w = reinterpret_cast<const T*>(g.w);
  const FloatEpi<T> epi = make_float_epi<T>(o);
  const dim3 grid((unsigned)((g.N + 15) / 16)), block(64 * kSkinnyWaves);
  const u32x4* zeros = static_cast<const u32x4*>(zero16);
  if (g.M <= 16)
    hipLaunchKernelGGL((skinny_kernel<O, T, 1>), grid, block, 0, st, a, g.lda, w, g.ldw, g.M, g.N, K, zeros, epi);
  else if (g.M <= 32)
    hipLaunchKernelGGL((skinny_kernel<O, T, 2>), grid, block, 0, st, a, g.lda, w, g.ldw, g.M, g.N, K, zeros, epi);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t run_skinny(int dtype, const GemvArgs& g, int K, const void* zero16, const FloatOut& o, hipStream_t st) {
  switch (dtype) {
    case DT_F32: return skinny_t<Op::F32, float>(g, K, zero16, o, st);
    case DT_F16: return skinny_t<Op::F16, _Float16>(g, K, zero16, o, st);
    case DT_BF16: return skinny_t<Op::BF16, __bf16>(g, K, zero16, o, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ohip
