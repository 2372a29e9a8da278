// Nearest-codebook search of the VQ autoencoder's four-channel latent (the native search of
// src/lesiondiffusion_mlx/_vq.py:12-82 and VqAutoencoder.quantize, mlx_model.py:742-803).
//
// Distance of latent vector z to code c, with the reference's rounding points in the element
// type T (fp16 or fp32): dot = fma chain of the four products in fp32 (first product plain,
// then three fmas); summed = T(|z|^2 + |c|^2); doubled = T(2 * T(dot)); distance =
// T(summed - doubled). The squared norms are the T-rounded squares summed in fp32 and
// rounded to T once. Selection: the lowest index whose distance is NaN if any is NaN, else
// the lowest index of the smallest distance (argmin's order) -- a function of the distance
// list alone, so any scan order gives the same index.
//
// The dots run on the matrix units: v_mfma_f32_32x32x2_f32 adds its two products in order, each
// as one fp32 fused multiply-add (tests compare every index and value with the fma chain), so
// two of them give the reference's chain for 32 codes x 32 positions (its first product plain
// up to the sign of a zero, which no distance shows). A few codes are scanned on the VALU.
// Integer/index results are bit-exact.

#include "common.h"

#include <cmath>
#include <type_traits>

// Every rounding point above is explicit; no multiply-add may be fused behind the code's back
// (the reference compiles its search with contraction off as well).
#pragma clang fp contract(off)

namespace ldx {

constexpr int VQ_THREADS = 256;
constexpr int VQ_STAGE = 2048;   // codes staged in LDS per round: 2048 x (16 + 4) B = 40 KB
constexpr int VQ_CHUNK = 64;     // codes (two MFMA tiles) per entry of the first pass

// fp32 squared norm of one four-vector as the reference forms it: each square rounded to T,
// the four summed in fp32 in index order, the sum rounded to T once.
template <typename T>
__device__ __forceinline__ T squared_norm4(const T* v) {
  float s = (float)(T)(v[0] * v[0]);
  s += (float)(T)(v[1] * v[1]);
  s += (float)(T)(v[2] * v[2]);
  s += (float)(T)(v[3] * v[3]);
  return (T)s;
}

template <typename T>
__global__ __launch_bounds__(VQ_THREADS) void vq_norms4_kernel(const T* __restrict__ x, int64_t n,
                                                               T* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * VQ_THREADS + threadIdx.x;
  if (i >= n) return;
  T v[4];
#pragma unroll
  for (int c = 0; c < 4; c++) v[c] = x[i * 4 + c];
  out[i] = squared_norm4<T>(v);
}

// Distance of a position to a code from the dot in fp32.
template <typename T>
__device__ __forceinline__ T vq_distance(T zn, T cn, float dot) {
  const T summed = (T)(zn + cn);
  const T doubled = (T)((T)2.f * (T)dot);
  return (T)(summed - doubled);
}

// Distance of code `code` to the position with components zs and squared norm zns.
template <typename T>
__device__ __forceinline__ T code_distance(const float (&zs)[4], T zns, const T* __restrict__ codebook,
                                           const T* __restrict__ cb_norm, int code) {
  const T* e = codebook + (int64_t)code * 4;
  float dot = zs[0] * (float)e[0];
  dot = __builtin_fmaf(zs[1], (float)e[1], dot);
  dot = __builtin_fmaf(zs[2], (float)e[2], dot);
  dot = __builtin_fmaf(zs[3], (float)e[3], dot);
  asm volatile("" : "+v"(dot));   // an fp32 value: not fused with its rounding to fp16 (v_fma_mixlo)
  return vq_distance<T>(zns, cb_norm[code], dot);
}

__device__ __forceinline__ float lane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Bits of the largest absolute component (a NaN is the largest).
__device__ __forceinline__ unsigned max4_bits(float4 v) {
  auto abs_bits = [](float x) { return __float_as_uint(x) & 0x7fffffffu; };
  return max(max(abs_bits(v.x), abs_bits(v.y)), max(abs_bits(v.z), abs_bits(v.w)));
}

// The smallest of three, a NaN if one of them is (v_min3_f32 would drop it).
__device__ __forceinline__ float min3_nan(float a, float b, float c) {
  float r;
  asm("v_minimum3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ f16x2 min3_nan(f16x2 a, f16x2 b, f16x2 c) {
  f16x2 r;
  asm("v_pk_minimum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// (da, ca) chosen over (db, cb): the selection rule for chunks of codes, given by the least
// distance in each (NaN if it holds one).
__device__ __forceinline__ bool vq_chunk_better(float da, int ca, float db, int cb) {
  const bool na = da != da, nb = db != db;
  if (na || nb) return na && (!nb || ca < cb);
  return da < db || (da == db && ca < cb);
}

// The least of 32 MFMA results (none a NaN that matters: such positions are scanned).
__device__ __forceinline__ float minimum16(f32x16 a, f32x16 b) {
  float m[2] = {a[0], b[0]};
#pragma unroll
  for (int i = 1; i < 16; i++) {
    m[0] = __builtin_elementwise_minimum(m[0], a[i]);
    m[1] = __builtin_elementwise_minimum(m[1], b[i]);
  }
  return __builtin_elementwise_minimum(m[0], m[1]);
}

// The least value over the wave's lanes (finite or +inf), in every lane.
__device__ __forceinline__ float wave_min(float v) {
  auto ror = [](float x, auto n) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + decltype(n)::value, 0xf, 0xf, false));
  };
  v = fminf(v, ror(v, std::integral_constant<int, 8>{}));
  v = fminf(v, ror(v, std::integral_constant<int, 4>{}));
  v = fminf(v, ror(v, std::integral_constant<int, 2>{}));
  v = fminf(v, ror(v, std::integral_constant<int, 1>{}));
  return fminf(fminf(lane_f(v, 0), lane_f(v, 16)), fminf(lane_f(v, 32), lane_f(v, 48)));
}

// The largest value over the wave's lanes, in every lane.
__device__ __forceinline__ unsigned wave_max(unsigned v) {
  auto ror = [](unsigned x, auto n) {
    return (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x120 + decltype(n)::value, 0xf, 0xf, false);
  };
  v = max(v, ror(v, std::integral_constant<int, 8>{}));
  v = max(v, ror(v, std::integral_constant<int, 4>{}));
  v = max(v, ror(v, std::integral_constant<int, 2>{}));
  v = max(v, ror(v, std::integral_constant<int, 1>{}));
  auto row = [&](int l) { return (unsigned)__builtin_amdgcn_readlane((int)v, l); };
  return max(max(row(0), row(16)), max(row(32), row(48)));
}

// First pass: the least distance of each position over every chunk of 64 codes and the first
// chunk that has it, from MFMA tiles of 32 codes (rows) x 32 positions (columns; PG column
// groups per wave). Second pass: that chunk alone, in order, for the index. The first pass costs
// 2.5 VALU operations per pair (add, fused multiply-add with 2 * dot in fp32, half a three-way
// minimum) and 128 MFMA cycles per 1,024; a scan that carries the index costs nine. The fused form
// is the reference's unless a finite dot's double overflows (its 2 * dot is then infinite), which
// needs components with |z_c| |e_c| of 2^125: positions that could have such a dot (2^124) are
// scanned with the reference's operations instead (24,000 such positions x 8,192 codes 1,048 us,
// others 44.5; finding the largest component costs 0.7 us of 34 for 500 positions).
// 409,600 positions x 8,192 codes, fp32: 1292 -> 453 us, 7.4e12 pairs per second; bound by the
// sum of the two (about 180 VALU and 128 MFMA cycles per 1,024 pairs: the fp32 MFMAs measured
// without overlap).
//
// Workgroup of four waves. SPLIT = 1: each wave has its own 32 PG positions and scans every
// code. SPLIT = 4: the waves share 32 positions and each scans a quarter of every stage; for
// few positions (launch_vq_nearest4).
template <typename T, int PG, int SPLIT>
__device__ __forceinline__ void exact_search(const T* __restrict__ z, const T* __restrict__ z_norm,
                                             const T* __restrict__ codebook, const T* __restrict__ cb_norm, int64_t P,
                                             int E, int32_t* __restrict__ indices, T* __restrict__ quantized,
                                             float4* cb /* components 0, 2, 1, 3: lane half h reads (h, 2 + h) */,
                                             T* cbn, unsigned* s_em, float* s_best, int* s_chunk) {
  static_assert(SPLIT == 1 || (SPLIT == 4 && PG == 1), "whole scans, or quarters of one column group");
  constexpr bool HALF = sizeof(T) == 2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int64_t p0 = SPLIT == 1 ? ((int64_t)blockIdx.x * 4 + wave) * (32 * PG) : (int64_t)blockIdx.x * 32;
  // B operands (position col of each group: component half, then 2 + half) and |z|^2.
  float zb[PG][2];
  T zn[PG];
#pragma unroll
  for (int g = 0; g < PG; g++) {
    const int64_t pos = p0 + 32 * g + col;
    T v[4] = {};
    zn[g] = (T)0.f;
    if (pos < P) {
#pragma unroll
      for (int c = 0; c < 4; c++) v[c] = z[pos * 4 + c];
      zn[g] = z_norm ? z_norm[pos] : squared_norm4<T>(v);
    }
    zb[g][0] = (float)(half ? v[1] : v[0]);
    zb[g][1] = (float)(half ? v[3] : v[2]);
  }
  float best[PG];
  int chunk[PG];
#pragma unroll
  for (int g = 0; g < PG; g++) { best[g] = INFINITY; chunk[g] = 0x7fffffff; }
  const f32x16 zero = {};
  unsigned em = 0;   // FP32: largest |component| of the staged codes, as bits (a code with a non-finite one has no finite dot)
  for (int base = 0; base < E; base += VQ_STAGE) {
    const int n = min(VQ_STAGE, E - base), nr = (n + VQ_CHUNK - 1) / VQ_CHUNK * VQ_CHUNK;
    __syncthreads();   // the previous stage is no longer read
    // Past the last code: zeros at an infinite norm.
    for (int i = threadIdx.x; i < nr; i += VQ_THREADS) {
      const T* e = codebook + (int64_t)(base + (i < n ? i : 0)) * 4;
      const float4 v = i < n ? make_float4((float)e[0], (float)e[2], (float)e[1], (float)e[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
      cb[i] = v;
      if constexpr (!HALF) {
        const unsigned m = max4_bits(v);
        em = m < 0x7f800000u ? max(em, m) : em;
      }
      cbn[i] = i < n ? cb_norm[base + i] : (T)INFINITY;
    }
    if constexpr (!HALF && SPLIT == 4)
      if (base + VQ_STAGE >= E) {
        em = wave_max(em);
        if (lane == 0) s_em[wave] = em;
      }
    __syncthreads();
    for (int c0 = SPLIT == 1 ? 0 : wave * VQ_CHUNK; c0 < nr; c0 += SPLIT * VQ_CHUNK) {
      float m[PG][2];
      f16x2 mh[PG][2];
#pragma unroll
      for (int g = 0; g < PG; g++)
#pragma unroll
        for (int i = 0; i < 2; i++) { m[g][i] = INFINITY; mh[g][i] = (f16x2)((f16)INFINITY); }
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const int r0 = c0 + 32 * t;
        const float2 a = *(reinterpret_cast<const float2*>(&cb[r0 + col]) + half);
        f32x16 d[PG];
#pragma unroll
        for (int g = 0; g < PG; g++) d[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, zb[g][0], zero, 0, 0, 0);
#pragma unroll
        for (int g = 0; g < PG; g++) d[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, zb[g][1], d[g], 0, 0, 0);
        // Element 4 q + e: code r0 + 8 q + 4 half + e.
#pragma unroll
        for (int q = 0; q < 4; q++) {
          if constexpr (HALF) {
            const f16x4 cn = *reinterpret_cast<const f16x4*>(&cbn[r0 + 8 * q + 4 * half]);
#pragma unroll
            for (int g = 0; g < PG; g++) {
              const f16x2 z2 = {(f16)zn[g], (f16)zn[g]};
              f16x2 dd[2];
#pragma unroll
              for (int e = 0; e < 2; e++) {
                const f16x2 h = {(f16)d[g][4 * q + 2 * e], (f16)d[g][4 * q + 2 * e + 1]};
                dd[e] = (z2 + (f16x2){cn[2 * e], cn[2 * e + 1]}) - (h + h);
              }
              mh[g][q & 1] = min3_nan(mh[g][q & 1], dd[0], dd[1]);
            }
          } else {
            const f32x4 cn = *reinterpret_cast<const f32x4*>(&cbn[r0 + 8 * q + 4 * half]);
#pragma unroll
            for (int g = 0; g < PG; g++) {
              float dd[4];
#pragma unroll
              for (int e = 0; e < 4; e++) dd[e] = __builtin_fmaf(-2.f, d[g][4 * q + e], (float)zn[g] + cn[e]);
              m[g][0] = min3_nan(m[g][0], dd[0], dd[1]);
              m[g][1] = min3_nan(m[g][1], dd[2], dd[3]);
            }
          }
        }
      }
      const int id = (base + c0) / VQ_CHUNK;
#pragma unroll
      for (int g = 0; g < PG; g++) {
        float v;
        if constexpr (HALF) {
          const f16x2 h = min3_nan(mh[g][0], mh[g][1], mh[g][1]);
          v = min3_nan((float)h[0], (float)h[1], (float)h[1]);
        } else {
          v = min3_nan(m[g][0], m[g][1], m[g][1]);
        }
        if (vq_chunk_better(v, id, best[g], chunk[g])) { best[g] = v; chunk[g] = id; }
      }
    }
  }
  if constexpr (!HALF) {   // em over the workgroup
    if constexpr (SPLIT == 1) {
      __syncthreads();   // the last stage, whose memory s_em shares, is no longer read
      em = wave_max(em);
      if (lane == 0) s_em[wave] = em;
      __syncthreads();
    }
    em = max(max(s_em[0], s_em[1]), max(s_em[2], s_em[3]));
  }
  // The two lane halves (codes 0-3 and 4-7 of every eight), then the four waves.
#pragma unroll
  for (int g = 0; g < PG; g++) {
    const float ob = __shfl_xor(best[g], 32, 64);
    const int oc = __shfl_xor(chunk[g], 32, 64);
    if (vq_chunk_better(ob, oc, best[g], chunk[g])) { best[g] = ob; chunk[g] = oc; }
  }
  if constexpr (SPLIT == 4) {
    if (half == 0) { s_best[wave * 32 + col] = best[0]; s_chunk[wave * 32 + col] = chunk[0]; }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 1; w < 4; w++) {
      const float ob = s_best[w * 32 + col];
      const int oc = s_chunk[w * 32 + col];
      if (vq_chunk_better(ob, oc, best[0], chunk[0])) { best[0] = ob; chunk[0] = oc; }
    }
  }
  // Index of that distance in its chunk: a lane per code, one position at a time (64 codes are
  // one contiguous kilobyte; a lane per position gathers: 75 us more at 409,600 positions).
  auto distance = [&](const float (&zs)[4], T zns, int code) {
    return code_distance<T>(zs, zns, codebook, cb_norm, code);
  };
#pragma unroll
  for (int g = 0; g < PG; g++) {
    const float znf = (float)zn[g];
    int found = 0x7fffffff;
#pragma unroll 4
    for (int i = 0; i < 32; i++) {
      const float zs[4] = {lane_f(zb[g][0], i), lane_f(zb[g][0], i + 32), lane_f(zb[g][1], i), lane_f(zb[g][1], i + 32)};
      const float b = lane_f(best[g], i);
      const int code = __builtin_amdgcn_readlane(chunk[g], i) * VQ_CHUNK + lane;
      const float v = (float)distance(zs, (T)lane_f(znf, i), min(code, E - 1));
      const uint64_t hit = __ballot(code < E && (v == b || (v != v && b != b)));
      if (lane == i && hit) found = code - lane + __builtin_ctzll(hit);
    }
    const int64_t pos = p0 + 32 * g + col;
    if (half || pos >= P) continue;
    T zt[4];
#pragma unroll
    for (int c = 0; c < 4; c++) zt[c] = z[pos * 4 + c];
    if constexpr (!HALF) {   // a double may overflow: the plain scan
      const unsigned zm = max4_bits(make_float4(zt[0], zt[1], zt[2], zt[3]));
      if (zm < 0x7f800000u && __uint_as_float(zm) * __uint_as_float(em) >= 0x1p124f) found = 0x7fffffff;
    }
    if (found >= E) {
      // (Also where no real code has the distance: a norm of -inf beside the padding's +inf.)
      const float zs[4] = {(float)zt[0], (float)zt[1], (float)zt[2], (float)zt[3]};
      T d0 = (T)0.f;
      for (int code = 0; code < E; code++) {
        const T d = distance(zs, zn[g], code);
        if (code == 0 || (d != d && d0 == d0) || (d == d && d0 == d0 && d < d0)) { d0 = d; found = code; }
      }
    }
    indices[pos] = found;
    if (quantized) {
      const T* e = codebook + (int64_t)found * 4;
      // The straight-through form z + (selected - z), each operation rounded to T
      // (mlx_model.py:788-789).
#pragma unroll
      for (int c = 0; c < 4; c++) quantized[pos * 4 + c] = (T)(zt[c] + (T)(e[c] - zt[c]));
    }
  }
}

template <typename T, int PG, int SPLIT>
__global__ __launch_bounds__(VQ_THREADS, SPLIT == 1 ? 4 : 3) void vq_nearest4_kernel(
    const T* __restrict__ z, const T* __restrict__ z_norm, const T* __restrict__ codebook,
    const T* __restrict__ cb_norm, int64_t P, int E, int32_t* __restrict__ indices, T* __restrict__ quantized) {
  __shared__ float4 cb[VQ_STAGE];
  __shared__ __attribute__((aligned(16))) T cbn[VQ_STAGE];
  __shared__ float s_best[SPLIT == 4 ? 128 : 1];
  __shared__ int s_chunk[SPLIT == 4 ? 128 : 1];
  __shared__ unsigned s_em[4];
  exact_search<T, PG, SPLIT>(z, z_norm, codebook, cb_norm, P, E, indices, quantized, cb, cbn, s_em, s_best, s_chunk);
}

// 2^e of a nonzero value from its absolute bits; `zero` for 0. Whether it may be scaled.
__device__ __forceinline__ int bits_exponent(unsigned bits, int zero) { return bits ? (int)(bits >> 23) - 127 : zero; }
__device__ __forceinline__ bool bits_scalable(unsigned bits) {
  return bits == 0 || (bits >= (unsigned)(127 - 40) << 23 && bits < (unsigned)(127 + 40) << 23);
}
__device__ __forceinline__ float pow2(int e) { return __int_as_float((127 + e) << 23); }

// FP32 search from bounds. One v_mfma_f32_32x32x16_f16 per 32 codes x 32 positions gives
// |e|^2 - 2 z.e (scaled by powers of two) to within E: z and e as hi + lo fp16 (zh.eh + zh.el +
// zl.eh, twelve of the sixteen products), |e|^2 as three fp16 parts times a power of two. The
// chosen code, whatever the rounding of the exact distances, lies in a 64-code chunk whose least
// value is within 2 E of the least of all. Each lane keeps the two least chunks of its position
// and the third's value: the first chunk, and the second where it is within 2 E, are searched with
// the exact distances; a position whose third is too, or whose values cannot be scaled (zero and
// 2^-40 to 2^40 can), gets an exact scan by its wave; a workgroup with more than VQ_SCANS of those
// (crowded or repeated codes), or a codebook that cannot be scaled, runs the exact search.
//   E, with zm and z1 the largest and the summed |z_c| of the position, em and nm the largest |e_c|
//   and ||e|^2| of the codebook. The largest component is scaled to 2^10 or more, so that a split
//   leaves 2^-12 (half the last bit of lo, and a part below 2^-14 counted as lost): 2^-22 of zm and of
//   em, and lo.lo 2^-22 zm em, over four products and the factor 2; sixteen accumulations at 2^-23 of
//   2.03 z1 em + 1.01 nm; the exact chain's roundings, 2^-24 each: 10 z1 em, 2 nm, 2 |zn|. Together
//   em (3.9e-6 zm + 5e-6 z1) + 2.1e-6 nm + 1.2e-7 |zn|; rounded up below. (How the instruction rounds
//   its sixteen products is not documented: against float64 its error stayed within 2.4 x 2^-23 of
//   their summed sizes over 786,000 sums of search operands and 2.9 over 1.6 million harder mixes.)
// 0.6 VALU operations per pair (half a three-way minimum and the chunk's bookkeeping) beside 32
// MFMA cycles per 1,024, against 2.5 and 128 of the exact pass. us, exact / bounds, normal data:
// 409,600 positions x 8,192 codes 453 / 200, 409,600 x 1,024 92 / 61, 100,000 x 8,192 163 / 75. Bound
// by latency in two rounds of workgroups: 1,600 of them, four per CU, 45 us for one alone. A codebook
// of codes all within 1/8,192 of zero 297, normal codes repeated eightfold 608 (one position
// in a workgroup's 256 to scan is 30 us; the scans of the kernel before the matrix units took 1,292).
constexpr int VQ_BSTAGE = 1024;   // codes per stage: 32 bytes each
constexpr int VQ_SCANS = 16;
__global__ __launch_bounds__(VQ_THREADS, 4) void vq_nearest4_bounds_kernel(
    const float* __restrict__ z, const float* __restrict__ z_norm, const float* __restrict__ codebook,
    const float* __restrict__ cb_norm, int64_t P, int E, int32_t* __restrict__ indices,
    float* __restrict__ quantized) {
  __shared__ __attribute__((aligned(16))) char lds[VQ_STAGE * 20];
  unsigned (*s_max)[2] = reinterpret_cast<unsigned (*)[2]>(lds);   // before the first stage
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int64_t p0 = ((int64_t)blockIdx.x * 4 + wave) * 64;
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
  auto load4 = [](const float* v) { return make_float4(v[0], v[1], v[2], v[3]); };
  auto abs_bits = [](float v) { return (unsigned)__float_as_int(v) & 0x7fffffffu; };
  // Largest component and squared norm of the codebook, as absolute bits (a NaN is the largest).
  unsigned em = 0, nm = 0;
#pragma unroll 8
  for (int i = threadIdx.x; i < E; i += VQ_THREADS) {
    em = max(em, max4_bits(load4(codebook + (int64_t)i * 4)));
    nm = max(nm, abs_bits(cb_norm[i]));
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    em = max(em, (unsigned)__shfl_xor((int)em, o, 64));
    nm = max(nm, (unsigned)__shfl_xor((int)nm, o, 64));
  }
  if (lane == 0) { s_max[wave][0] = em; s_max[wave][1] = nm; }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; w++) { em = max(em, s_max[w][0]); nm = max(nm, s_max[w][1]); }
  bool exact = !bits_scalable(em) || !bits_scalable(nm);
  if (!exact) {
    const int es = 10 - bits_exponent(em, 10), ns = 14 - bits_exponent(nm, 14);
    const float e_scale = -2.f * pow2(es), n_scale = pow2(ns);
    // This lane's position, and the B operands of the wave's two column groups.
    const int64_t pos = p0 + lane;
    const float4 zv = pos < P ? load4(z + pos * 4) : zero4;
    float zn = 0.f;
    if (pos < P) {
      const float v[4] = {zv.x, zv.y, zv.z, zv.w};
      zn = z_norm ? z_norm[pos] : squared_norm4<float>(v);
    }
    const unsigned zm = max4_bits(zv);
    f16x8 zb[2];
#pragma unroll
    for (int g = 0; g < 2; g++) {
      const int64_t q = p0 + 32 * g + col;
      const float4 v4 = q < P ? load4(z + q * 4) : zero4;
      const float v[4] = {v4.x, v4.y, v4.z, v4.w};
      const unsigned m = max4_bits(v4);
      const int zs = bits_scalable(m) ? 10 - bits_exponent(m, 10) : 0;
      const int bs = min(max(zs + es - ns, -14), 15);
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const float x = v[c] * pow2(zs);
        const f16 hi = (f16)x, lo = (f16)(x - (float)hi);
        zb[g][c] = half ? lo : hi;
        zb[g][4 + c] = half ? (c < 3 ? (f16)pow2(bs) : (f16)0.f) : hi;
      }
    }
    float m1 = INFINITY, m2 = INFINITY, m3 = INFINITY;
    int c1 = 0, c2 = 0;
    f16x8* frag = reinterpret_cast<f16x8*>(lds);   // [half][code]
    const f32x16 zero = {};
    for (int base = 0; base < E; base += VQ_BSTAGE) {
      const int n = min(VQ_BSTAGE, E - base), nr = (n + VQ_CHUNK - 1) / VQ_CHUNK * VQ_CHUNK;
      __syncthreads();   // the previous stage is no longer read
      for (int i = threadIdx.x; i < nr; i += VQ_THREADS) {
        f16x8 a = {}, b = {};
        if (i < n) {
          const float4 v4 = load4(codebook + (int64_t)(base + i) * 4);
          const float v[4] = {v4.x, v4.y, v4.z, v4.w};
          const float x = cb_norm[base + i] * n_scale;
          const f16 n0 = (f16)x, n1 = (f16)(x - (float)n0);
          b[4] = n0; b[5] = n1; b[6] = (f16)(x - (float)n0 - (float)n1);
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const float y = v[c] * e_scale;
            a[c] = b[c] = (f16)y;
            a[4 + c] = (f16)(y - (float)a[c]);
          }
        } else {
          b[4] = (f16)INFINITY;   // past the last code
        }
        frag[i] = a;
        frag[VQ_BSTAGE + i] = b;
      }
      __syncthreads();
      for (int c0 = 0; c0 < nr; c0 += VQ_CHUNK) {
        const f16x8 a0 = frag[half * VQ_BSTAGE + c0 + col], a1 = frag[half * VQ_BSTAGE + c0 + 32 + col];
        float m[2];
#pragma unroll
        for (int g = 0; g < 2; g++) {
          const f32x16 d0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, zb[g], zero, 0, 0, 0);
          const f32x16 d1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, zb[g], zero, 0, 0, 0);
          m[g] = minimum16(d0, d1);
        }
        // Lanes 0-31: the chunk's least value of column group 0; lanes 32-63: of group 1.
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(m[0]), __float_as_int(m[1]), false, false);
        const float v = fminf(__int_as_float(sw[0]), __int_as_float(sw[1]));
        const int id = (base + c0) / VQ_CHUNK;
        m3 = __builtin_amdgcn_fmed3f(m2, v, m3);
        c2 = v < m1 ? c1 : (v < m2 ? id : c2);
        m2 = __builtin_amdgcn_fmed3f(m1, v, m2);
        c1 = v < m1 ? id : c1;
        m1 = fminf(m1, v);
      }
    }
    const int zs = bits_scalable(zm) ? 10 - bits_exponent(zm, 10) : 0, bs = zs + es - ns;
    const float zmf = __int_as_float((int)zm), emf = __int_as_float((int)em), nmf = __int_as_float((int)nm);
    const float z1 = __builtin_fabsf(zv.x) + __builtin_fabsf(zv.y) + __builtin_fabsf(zv.z) + __builtin_fabsf(zv.w);
    const float bound = emf * (4e-6f * zmf + 5.1e-6f * z1) + 2.2e-6f * nmf + 2e-7f * __builtin_fabsf(zn);
    const float margin = 2.1f * bound * pow2(zs) * pow2(es);
    const bool scaled = bits_scalable(zm) && bits_scalable(abs_bits(zn)) && bs >= -14 && bs <= 15;
    const bool scan = pos < P && !(scaled && m3 > m1 + margin);
    const bool two = !(m2 > m1 + margin);
    const uint64_t scans = __ballot(scan), twos = __ballot(two);
    int* s_count = reinterpret_cast<int*>(lds);
    __syncthreads();   // the last stage is no longer read
    if (lane == 0) s_count[wave] = __builtin_popcountll(scans);
    __syncthreads();
    exact = s_count[0] + s_count[1] + s_count[2] + s_count[3] > VQ_SCANS;
    if (!exact) {
      const float zl[4] = {zv.x, zv.y, zv.z, zv.w};
      int found = 0;
      // Searches codes k0 and up, a lane per code: the first of the least (d: its distance).
      auto search = [&](int i, int k0, float& d) {
        const float zi[4] = {lane_f(zl[0], i), lane_f(zl[1], i), lane_f(zl[2], i), lane_f(zl[3], i)};
        const float v = code_distance<float>(zi, lane_f(zn, i), codebook, cb_norm, min(k0 + lane, E - 1));
        d = wave_min(v);   // (past the last code: its distance again, at a higher lane)
        return k0 + (int)__builtin_ctzll(__ballot(v == d));
      };
      float best = 0.f;
#pragma unroll 8
      for (int i = 0; i < 64; i++) {
        float d;
        const int code = search(i, __builtin_amdgcn_readlane(c1, i) * VQ_CHUNK, d);
        if (lane == i) { found = code; best = d; }
      }
      for (uint64_t left = __ballot(two && !scan && pos < P); left; left &= left - 1) {
        const int i = __builtin_ctzll(left), k0 = __builtin_amdgcn_readlane(c2, i) * VQ_CHUNK;
        float d;
        const int code = search(i, k0, d);
        if (lane == i && (d < best || (d == best && code < found))) found = code;
      }
      for (uint64_t left = scans; left; left &= left - 1) {
        const int i = __builtin_ctzll(left);
        const float zi[4] = {lane_f(zl[0], i), lane_f(zl[1], i), lane_f(zl[2], i), lane_f(zl[3], i)};
        const float zni = lane_f(zn, i);
        float b = code_distance<float>(zi, zni, codebook, cb_norm, min(lane, E - 1));
        int code = min(lane, E - 1);
#pragma unroll 8
        for (int k = lane + 64; k < E; k += 64) {
          const float d = code_distance<float>(zi, zni, codebook, cb_norm, k);
          const bool better = ((d != d) & (b == b)) | (d < b);   // codes ascend: the first stays
          b = better ? d : b;
          code = better ? k : code;
        }
#pragma unroll
        for (int o = 32; o; o >>= 1) {
          const float ob = __shfl_xor(b, o, 64);
          const int oc = __shfl_xor(code, o, 64);
          if (vq_chunk_better(ob, oc, b, code)) { b = ob; code = oc; }
        }
        if (lane == i) found = code;
      }
      if (pos < P) {
        indices[pos] = found;
        if (quantized) {
          const float* e = codebook + (int64_t)found * 4;
#pragma unroll
          for (int c = 0; c < 4; c++) quantized[pos * 4 + c] = zl[c] + (e[c] - zl[c]);
        }
      }
    }
  }
  if (exact) {
    __syncthreads();
    exact_search<float, 2, 1>(z, z_norm, codebook, cb_norm, P, E, indices, quantized, reinterpret_cast<float4*>(lds),
                              reinterpret_cast<float*>(lds + VQ_STAGE * 16), reinterpret_cast<unsigned*>(lds), nullptr,
                              nullptr);
  }
}

// Few codes: a lane per position scans them all with the reference's operations, from LDS reads that
// all lanes share, eight codes at a time. The searches above cost a stage, a merge and a second pass
// whatever the codes' number (9.6 us for one code, 44 at 409,600 positions); this one thirteen VALU
// operations a pair and nothing else: VALU-bound from 200,000 positions on, one wave's chain (0.04
// us a code) below 100,000.
constexpr int VQ_SCAN_CODES = 256;
static_assert(VQ_SCAN_CODES <= VQ_THREADS && VQ_SCAN_CODES % 8 == 0, "a code per thread, whole eights");
template <typename T>
__global__ __launch_bounds__(VQ_THREADS) void vq_scan4_kernel(
    const T* __restrict__ z, const T* __restrict__ z_norm, const T* __restrict__ codebook,
    const T* __restrict__ cb_norm, int64_t P, int E, int32_t* __restrict__ indices, T* __restrict__ quantized) {
  __shared__ float4 cb[VQ_SCAN_CODES];
  __shared__ T cbn[VQ_SCAN_CODES];
  const int64_t pos = (int64_t)blockIdx.x * VQ_THREADS + threadIdx.x;
  const int nr = (E + 7) / 8 * 8;   // whole eights: the last code again, which never wins twice
  if ((int)threadIdx.x < nr) {
    const int i = min((int)threadIdx.x, E - 1);
    const T* e = codebook + (int64_t)i * 4;
    cb[threadIdx.x] = make_float4((float)e[0], (float)e[1], (float)e[2], (float)e[3]);
    cbn[threadIdx.x] = cb_norm[i];
  }
  __syncthreads();
  if (pos >= P) return;
  T zt[4];
#pragma unroll
  for (int c = 0; c < 4; c++) zt[c] = z[pos * 4 + c];
  const T zn = z_norm ? z_norm[pos] : squared_norm4<T>(zt);
  auto distance = [&](int code) {
    const float4 e = cb[code];
    float dot = (float)zt[0] * e.x;
    dot = __builtin_fmaf((float)zt[1], e.y, dot);
    dot = __builtin_fmaf((float)zt[2], e.z, dot);
    dot = __builtin_fmaf((float)zt[3], e.w, dot);
    if constexpr (sizeof(T) == 2) asm("" : "+v"(dot));   // as in code_distance
    return vq_distance<T>(zn, cbn[code], dot);
  };
  T best = distance(0);
  int found = 0;
  for (int code = 0; code < nr; code += 8) {
    T d[8];
#pragma unroll
    for (int i = 0; i < 8; i++) d[i] = distance(code + i);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const bool better = ((d[i] != d[i]) & (best == best)) | (d[i] < best);
      best = better ? d[i] : best;
      found = better ? code + i : found;
    }
  }
  indices[pos] = found;
  if (quantized) {
#pragma unroll
    for (int c = 0; c < 4; c++) quantized[pos * 4 + c] = (T)(zt[c] + (T)(codebook[found * 4 + c] - zt[c]));
  }
}

// Few codes: the scan. us, scan / the search below: 64 codes 1,000 positions 4.7 / 9.6, 409,600 9.8 /
// 45 (fp16 11 / 45); 128 codes 1,000 7.4 / 9.6 (fp16 8.1 / 9.7), 409,600 17 / 45; 256 codes 50,000
// 13.3 / 13.5 (fp16 14.9 / 20), 100,000 14.3 / 18.2, 409,600 31 / 46 (fp16 34 / 56); 384 codes lose at
// 50,000 (18 estimated / 14).
// Up to 24,576 positions the quarters' workgroups run at once (three per CU), whole scans leave
// waves idle. FP32 above that: bounds. us, quarters / bounds, 8,192 codes: 500 positions 34 / 45,
// 24,000 46 / 76, 28,000 77 / 45, 51,200 111 / 75, 100,000 163 / 75 (whole exact scans); 24,000 x
// 1,024 14 / 17, 32,000 x 300 20 / 14. fp16, whose rounding would make the bounds wide: whole exact
// scans from 81,920 positions (us, whole / quarters, 8,192 codes: 51,200 134 / 112, 100,000 168 /
// 186, 409,600 447 / 667).
template <typename T>
static void launch_vq_nearest4(const T* z, const T* z_norm, const T* codebook, const T* cb_norm, int64_t P, int E,
                               int32_t* indices, T* quantized, hipStream_t st) {
  constexpr bool F32 = sizeof(T) == 4;
  if (E <= 128 || (E <= VQ_SCAN_CODES && P > 32768)) {
    hipLaunchKernelGGL(vq_scan4_kernel<T>, dim3((unsigned)((P + VQ_THREADS - 1) / VQ_THREADS)), dim3(VQ_THREADS), 0, st,
                       z, z_norm, codebook, cb_norm, P, E, indices, quantized);
    return;
  }
  if (P <= (F32 ? 24576 : 81919)) {
    hipLaunchKernelGGL((vq_nearest4_kernel<T, 1, 4>), dim3((unsigned)((P + 31) / 32)), dim3(VQ_THREADS), 0, st, z,
                       z_norm, codebook, cb_norm, P, E, indices, quantized);
    return;
  }
  const dim3 grid((unsigned)((P + 255) / 256));
  if constexpr (F32)
    hipLaunchKernelGGL(vq_nearest4_bounds_kernel, grid, dim3(VQ_THREADS), 0, st, z, z_norm, codebook, cb_norm, P, E,
                       indices, quantized);
  else
    hipLaunchKernelGGL((vq_nearest4_kernel<T, 2, 1>), grid, dim3(VQ_THREADS), 0, st, z, z_norm, codebook, cb_norm, P, E,
                       indices, quantized);
}

}  // namespace ldx

using namespace ldx;

extern "C" int ldx_vq_squared_norms4(const void* x, int64_t n, int32_t dtype, void* out, void* stream) {
  if (!x || !out) return fail("vq_squared_norms4: null pointer");
  if (n < 1) return fail("vq_squared_norms4: n = %lld < 1", (long long)n);
  const unsigned grid = (unsigned)((n + VQ_THREADS - 1) / VQ_THREADS);
  hipStream_t st = as_stream(stream);
  if (dtype == LDX_DTYPE_F16)
    hipLaunchKernelGGL(vq_norms4_kernel<f16>, dim3(grid), dim3(VQ_THREADS), 0, st, (const f16*)x, n, (f16*)out);
  else if (dtype == LDX_DTYPE_F32)
    hipLaunchKernelGGL(vq_norms4_kernel<float>, dim3(grid), dim3(VQ_THREADS), 0, st, (const float*)x, n,
                       (float*)out);
  else
    return fail("vq_squared_norms4: dtype %d is not LDX_DTYPE_F16 or LDX_DTYPE_F32", dtype);
  return check_launch("vq_squared_norms4");
}

extern "C" int ldx_vq_nearest4(const void* z, const void* z_norm, const void* codebook, const void* codebook_norm,
                               int64_t positions, int32_t entries, int32_t dtype, int32_t* indices,
                               void* quantized, void* stream) {
  if (!z || !codebook || !codebook_norm || !indices) return fail("vq_nearest4: null pointer");
  if (positions < 1 || entries < 1)
    return fail("vq_nearest4: empty input (%lld positions, %d codes)", (long long)positions, entries);
  if (positions > ((int64_t)1 << 31)) return fail("vq_nearest4: more than 2^31 positions");
  hipStream_t st = as_stream(stream);
  if (dtype == LDX_DTYPE_F16)
    launch_vq_nearest4<f16>((const f16*)z, (const f16*)z_norm, (const f16*)codebook, (const f16*)codebook_norm,
                            positions, entries, indices, (f16*)quantized, st);
  else if (dtype == LDX_DTYPE_F32)
    launch_vq_nearest4<float>((const float*)z, (const float*)z_norm, (const float*)codebook,
                              (const float*)codebook_norm, positions, entries, indices, (float*)quantized, st);
  else
    return fail("vq_nearest4: dtype %d is not LDX_DTYPE_F16 or LDX_DTYPE_F32", dtype);
  return check_launch("vq_nearest4");
}
