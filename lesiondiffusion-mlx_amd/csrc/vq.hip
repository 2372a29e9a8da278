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
// up to the sign of a zero, which no distance shows). Integer/index results are bit-exact.

#include "common.h"

#include <cmath>

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

// First pass: the least distance of each position over every chunk of 64 codes and the first
// chunk that has it, from MFMA tiles of 32 codes (rows) x 32 positions (columns; PG column
// groups per wave). Second pass: that chunk alone, in order, for the index. The first pass costs
// 2.5 VALU operations per pair (add, fused multiply-add with the exact 2 * dot in fp32, half a
// three-way minimum) and 128 MFMA cycles per 1,024; a scan that carries the index costs nine.
// 409,600 positions x 8,192 codes, fp32: 1292 -> 453 us, 7.4e12 pairs per second; bound by the
// sum of the two (about 180 VALU and 128 MFMA cycles per 1,024 pairs: the fp32 MFMAs measured
// without overlap).
//
// Workgroup of four waves. SPLIT = 1: each wave has its own 32 PG positions and scans every
// code. SPLIT = 4: the waves share 32 positions and each scans a quarter of every stage; for
// few positions (launch_vq_nearest4).
template <typename T, int PG, int SPLIT>
__global__ __launch_bounds__(VQ_THREADS, SPLIT == 1 ? 4 : 3) void vq_nearest4_kernel(
    const T* __restrict__ z, const T* __restrict__ z_norm, const T* __restrict__ codebook,
    const T* __restrict__ cb_norm, int64_t P, int E, int32_t* __restrict__ indices, T* __restrict__ quantized) {
  static_assert(SPLIT == 1 || (SPLIT == 4 && PG == 1), "whole scans, or quarters of one column group");
  constexpr bool HALF = sizeof(T) == 2;
  __shared__ float4 cb[VQ_STAGE];   // components 0, 2, 1, 3: lane half h reads (h, 2 + h)
  __shared__ __attribute__((aligned(16))) T cbn[VQ_STAGE];
  __shared__ float s_best[SPLIT == 4 ? 128 : 1];
  __shared__ int s_chunk[SPLIT == 4 ? 128 : 1];
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
  for (int base = 0; base < E; base += VQ_STAGE) {
    const int n = min(VQ_STAGE, E - base), nr = (n + VQ_CHUNK - 1) / VQ_CHUNK * VQ_CHUNK;
    __syncthreads();   // the previous stage is no longer read
    // Past the last code: zeros at an infinite norm.
    for (int i = threadIdx.x; i < nr; i += VQ_THREADS) {
      const T* e = codebook + (int64_t)(base + (i < n ? i : 0)) * 4;
      cb[i] = i < n ? make_float4((float)e[0], (float)e[2], (float)e[1], (float)e[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
      cbn[i] = i < n ? cb_norm[base + i] : (T)INFINITY;
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
  // A code's distance to the position whose components and |z|^2 are given.
  auto distance = [&](const float (&zs)[4], T zns, int code) {
    const T* e = codebook + (int64_t)code * 4;
    float dot = zs[0] * (float)e[0];
    dot = __builtin_fmaf(zs[1], (float)e[1], dot);
    dot = __builtin_fmaf(zs[2], (float)e[2], dot);
    dot = __builtin_fmaf(zs[3], (float)e[3], dot);
    asm volatile("" : "+v"(dot));   // an fp32 value: not fused with its rounding to fp16 (v_fma_mixlo)
    return vq_distance<T>(zns, cb_norm[code], dot);
  };
#pragma unroll
  for (int g = 0; g < PG; g++) {
    auto lane_f = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
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
    if (found >= E) {
      // No real code has the distance (a norm of -inf beside the padding's +inf): the plain scan.
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

// Fewer than 81,920 positions (320 workgroups of 256) leave waves idle: quarters of the scan
// then. us, whole scans / quarters, 8,192 codes: 500 positions 134 / 33, 51,200 134 / 112,
// 100,000 168 / 186, 409,600 447 / 667.
template <typename T>
static void launch_vq_nearest4(const T* z, const T* z_norm, const T* codebook, const T* cb_norm, int64_t P, int E,
                               int32_t* indices, T* quantized, hipStream_t st) {
  if (P >= 81920)
    hipLaunchKernelGGL((vq_nearest4_kernel<T, 2, 1>), dim3((unsigned)((P + 255) / 256)), dim3(VQ_THREADS), 0, st, z,
                       z_norm, codebook, cb_norm, P, E, indices, quantized);
  else
    hipLaunchKernelGGL((vq_nearest4_kernel<T, 1, 4>), dim3((unsigned)((P + 31) / 32)), dim3(VQ_THREADS), 0, st, z,
                       z_norm, codebook, cb_norm, P, E, indices, quantized);
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
